"""The Q5_0 / Q8_0 layers' fused launches (norm + q, k, v; RoPE + cache append;
partial merge + wo; norm + gate + up + SiLU; the argmax over many workgroups)
at the widths that take each instantiation, through DecodeModel on path 0,
against the CPU reference step.  Bars as tests/test_gpu_q05_model.py: K/V of
layer 0 within one f16 ulp plus 2e-4 of the row RMS (fp32 GEMVs), logits within
2e-3 of their RMS plus four one-step Q8 flips of the head's input, the token the
argmax of the logits that the device holds, exactly.

A value of h that lies on the edge of two Q8 steps may round either way: h is off
by about 1e-6 of its group's largest value (fp32 sums of 64 to 2048 terms), 1e-4 of
a step of 1/127.  A flip moves the hidden row by d8 W_down[:, i], and through the
layer and the Q8 roundings that follow the logits by up to 1e-2 of their RMS (the
model tests' bar past a flip; 5.6e-3 where h[i] of a 32-head layer lay 1.4e-5 of a
step from its edge), four times that at the largest.  Only steps whose h has such a
value in the reference get that bar; their K/V rows carry the flip too, so the
reference goes on with the device's.

The fused launches keep the operations of the separate ones in their order, so
against those the results are equal bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from taraference_amd import synth
from _gpu import P, S, Unaligned, call, dev, empty, host, model_class
from _model_ref import RefModelMixed
from _util import q8_0_dequant
from test_gpu_q05_model import f16, write_model

pytestmark = pytest.mark.gpu


class Ref(RefModelMixed):
    """The reference; `edges` counts the last step's h values that may round either way."""

    def step(self, token, pos):
        self.edges = 0
        return super().step(token, pos)

    def _gemv(self, wm, n_rows, x, bias=None, out=None):
        if n_rows == self.c["n_ff"]:  # down
            d = np.repeat(oracle.quantize_q8(x)[1], 32)
            step = x / np.where(d > 0, d, 1)
            self.edges += int(np.sum(np.abs(step - np.floor(step) - 0.5) < 1e-4))
        return super()._gemv(wm, n_rows, x, bias, out)


@pytest.mark.parametrize("heads,kv,ff,vocab,max_seq", [
    (1, 1, 256, 151, 40),      # two blocks a row; a vocabulary of 3 mod 4
    (4, 2, 512, 257, 40),      # one block a quad
    (17, 17, 768, 1003, 40),   # 34 blocks: the last round of a quad nearly empty
    (32, 4, 256, 130, 1024),   # the widest row, 16 partials
    (8, 8, 256, 64, 1600),     # 24 partials
    (8, 8, 256, 64, 2100),     # 32 partials: merged by their own launch
])
def test_fused_layers(gpu, tmp_path, heads, kv, ff, vocab, max_seq):
    from taraference_amd.model import DecodeModel

    e = 64 * heads
    cfg = dict(n_layer=2, n_embd=e, n_ff=ff, n_head=heads, n_kv=kv, head_dim=64, n_vocab=vocab,
               rope_theta=1e6, rms_eps=1e-6)
    print(f"b32 fused e={e} kv={kv} ff={ff} vocab={vocab} max_seq={max_seq}", flush=True)
    rng = np.random.default_rng(e + ff)
    layers = [synth.qwen05_layer(rng, cfg, li) for li in range(2)]
    emb = synth.qwen05_embedding(rng, cfg)
    path = tmp_path / "m.gguf"
    write_model(path, cfg, layers, emb)
    gm = DecodeModel.from_gguf(path, max_seq)
    rm = Ref(cfg, layers, emb, max_seq)
    nb = e // 32
    wmax = float(np.abs(q8_0_dequant(emb[0][:, : nb * 34].reshape(-1, 34))).max())
    for pos, tok in enumerate(rng.integers(0, vocab, 5).tolist()):
        nxt = gm.forward(tok, pos)
        lg = gm.logits()
        assert nxt == oracle.argmax(lg), pos
        rl, _ = rm.step(tok, pos)
        scale = np.sqrt(np.mean(rl.astype(np.float64) ** 2))
        _, d8 = oracle.quantize_q8(rm.head_x)
        tol = 4e-2 * scale if rm.edges else 2e-3 * scale + 4 * float(d8.max()) * wmax
        assert np.abs(lg.astype(np.float64) - rl).max() <= tol, (pos, rm.edges)
        k, v = gm.kv_cache(0, pos + 1)
        for got, ref in ((k[pos], rm.K[0][pos]), (v[pos], rm.V[0][pos])):
            g, r = f16(got), f16(ref)
            ulp = np.abs(np.spacing(np.asarray(ref, np.uint16).view(np.float16))).astype(np.float64)
            assert np.all(np.abs(g - r) <= ulp + 2e-4 * np.sqrt(np.mean(r ** 2))), pos
        for li in range(2) if rm.edges else ():
            k, v = gm.kv_cache(li, pos + 1)
            rm.K[li][pos], rm.V[li][pos] = k[pos], v[pos]
    gm.close()


def make(cfg, layers, emb, max_seq, shift=()):
    """A DecodeModel; the vectors named in `shift` (attn_norm, ffn_norm or
    output_norm) lie 4 bytes past a 16-byte boundary."""
    rng = np.random.default_rng(9)

    def norm(name, v):
        v = np.asarray(v * rng.uniform(0.8, 1.2, v.size), np.float32)
        return v.view(Unaligned) if name in shift else v

    layers = [dict(L, attn_norm=norm("attn_norm", L["attn_norm"]),
                   ffn_norm=norm("ffn_norm", L["ffn_norm"])) for L in layers]
    onorm = norm("output_norm", np.ones(cfg["n_embd"], np.float32))
    return model_class()(dict(cfg, max_seq=max_seq), layers, emb, output_norm=onorm), layers, onorm


@pytest.mark.parametrize("heads,kv", [(2, 1), (4, 2), (5, 5), (14, 2), (32, 4)])
def test_norm_gate_up_as_separate_launches(gpu, heads, kv):
    """Norms that the fused launches do not take go through tf_rms_norm, the
    GEMVs and silu_mul: the same bits.  (Widths of 4, 8, 10, 28 and 64 blocks.)"""
    cfg = dict(n_layer=2, n_embd=64 * heads, n_ff=512, n_head=heads, n_kv=kv, head_dim=64,
               n_vocab=130, rope_theta=1e6, rms_eps=1e-6)
    rng = np.random.default_rng(heads)
    layers = [synth.qwen05_layer(rng, cfg, li) for li in range(2)]
    emb = synth.qwen05_embedding(rng, cfg)
    print(f"fused norm e={64 * heads}", flush=True)
    a, _, _ = make(cfg, layers, emb, 40)
    b, _, _ = make(cfg, layers, emb, 40, ("attn_norm", "ffn_norm"))
    for pos, tok in enumerate(rng.integers(0, 130, 6).tolist()):
        a.forward(tok, pos)
        b.forward(tok, pos)
        np.testing.assert_array_equal(a.logits(), b.logits())
    a.close()
    b.close()


@pytest.mark.parametrize("heads,kv,max_seq", [(14, 2, 60), (5, 5, 900), (14, 2, 1100), (32, 4, 1535),
                                              (14, 2, 1600), (32, 4, 2047)])
def test_merge_wo_as_separate_launches(gpu, heads, kv, max_seq):
    """One layer whose FFN adds nothing (gate 0): the logits are those of the
    C ABI's own sequence with tf_flash_decode_reduce and tf_gemv_q5_0_f32, at 8,
    16 and 24 partials."""
    e, hd, vocab = 64 * heads, 64, 130
    cfg = dict(n_layer=1, n_embd=e, n_ff=256, n_head=heads, n_kv=kv, head_dim=hd, n_vocab=vocab,
               rope_theta=1e6, rms_eps=1e-6)
    rng = np.random.default_rng(heads + max_seq)
    L0 = synth.qwen05_layer(rng, cfg, 0)
    g, cb, ty = L0["gate"]
    g = g.copy()
    g.reshape(-1, 22)[:, :2] = 0
    L0["gate"] = (g, cb, ty)
    emb = synth.qwen05_embedding(rng, cfg)
    m, (L,), onorm = make(cfg, [L0], emb, max_seq)
    print(f"merge + wo heads={heads} kv={kv} max_seq={max_seq}", flush=True)
    toks = rng.integers(0, vocab, 45).tolist()
    for pos, tok in enumerate(toks):
        m.forward(tok, pos)
    pos, tok = len(toks) - 1, toks[-1]
    ns = m.lib.tf_flash_decode_n_split(kv, max_seq)
    assert ns == max(8, max_seq // 512 * 8) <= 24
    x, xb, q, k, att = empty(e), empty(e), empty(e), empty(kv * hd), empty(e)
    part, lg = empty(heads * ns * (2 + hd)), empty(vocab)
    xq, xd = empty(e, torch.int8), empty(e // 32)
    W = {n: (P(dev(L[n][0])), L[n][1]) for n in ("wq", "wk", "wo")}
    E, ecb = P(dev(emb[0])), emb[1]
    call("tf_embed_row", E, 34, P(x), tok, None, e, ecb, S())
    call("tf_rms_norm", P(x), P(dev(L["attn_norm"])), P(xb), e, cfg["rms_eps"], S())
    call("tf_gemv_q5_0_qk", W["wq"][0], W["wk"][0], P(xb), P(q), P(k), e, e, kv * hd, W["wq"][1], 1,
         P(dev(L["bq"])), P(dev(L["bk"])), S())
    call("tf_rope_neox", P(q), heads, hd, pos, None, cfg["rope_theta"], S())
    call("tf_flash_decode_partial", P(q), m.lib.tf_model_k_cache(m.h, 0),
         m.lib.tf_model_v_cache(m.h, 0), P(part), heads, kv, hd, pos, 1, ns,
         float(np.float32(1) / np.sqrt(np.float32(hd))), S())
    call("tf_flash_decode_reduce", P(part), P(att), heads, hd, ns, 1, S())
    call("tf_gemv_q5_0_f32", W["wo"][0], P(att), P(x), e, e, W["wo"][1], 0, None, 2, None, S())
    call("tf_rms_norm", P(x), P(dev(onorm)), P(xb), e, cfg["rms_eps"], S())
    call("tf_quantize_q8", P(xb), P(xq), P(xd), e, S())
    call("tf_gemv_q8_0_q8", E, P(xq), P(xd), P(lg), e, vocab, ecb, 0, None, 0, None, S())
    np.testing.assert_array_equal(m.logits(), host(lg))
    m.close()


def test_output_norm_4_byte_aligned(gpu):
    """The head's fused norm + Q8 takes 8-byte aligned norms; others go through
    tf_rms_norm and tf_quantize_q8, with the same bits."""
    cfg = dict(n_layer=1, n_embd=896, n_ff=256, n_head=14, n_kv=2, head_dim=64, n_vocab=130,
               rope_theta=1e6, rms_eps=1e-6)
    rng = np.random.default_rng(1)
    layers, emb = [synth.qwen05_layer(rng, cfg, 0)], synth.qwen05_embedding(rng, cfg)
    a, _, _ = make(cfg, layers, emb, 40)
    b, _, _ = make(cfg, layers, emb, 40, ("output_norm",))
    assert a.forward(5, 0) == b.forward(5, 0)
    np.testing.assert_array_equal(a.logits(), b.logits())
    a.close()
    b.close()
