"""The runtime's batched prompt forward (tf_model_prefill: forward.rs:42-71
with the n_tok-row layer of layer.rs) against the CPU reference prefill
(tests/_model_ref.RefModel.prefill: oracle f32 GEMMs, prefill attention,
rope, RMSNorm rows) on tiny random-init Qwen2-shaped Q4_K_M models.

Both sides run fp32 activations through the same operator sequence and
differ only in fp32 summation order.  The K/V rows agree to one f16 ulp plus
2e-4 of the row RMS in layer 0 (the GEMM bound, 1e-5 of sum |terms|, with
sum |terms| about sqrt(K) = 16 row RMS for these rows) and 1e-3 of the row
RMS after it.  The last token's logits (the decode head: RMSNorm, Q8,
lm_head) agree to 5e-3 of their RMS: the hidden row carries the order
differences of every layer (up to 1e-3 of RMS each, as the K/V bound), and
quantizing it to Q8 can flip a value by one step, which moves the logits by
about d8 |w|.  The returned token equals the reference's argmax whenever its
top-two gap exceeds 1e-2 of the RMS.  Prompts end short of, at and past tiles of
32 tokens and chunks of 1024, and a second prefill continues at pos0 > 0.  A prompt
and a width with 192 tiles of 32 x 128 take the gate/up form of whole K, all others
the one that splits K over a workgroup's waves.  The greedy continuation after a prefill
starts with prefill's token and runs on the decode path.
"""
import numpy as np
import pytest
import torch

import oracle
from taraference_amd import synth
from _gpu import Unaligned, model_class
from _model_ref import RefModel, prefill64
from test_gpu_model import TINY, build

pytestmark = pytest.mark.gpu


def f16(a):
    return np.asarray(a, np.uint16).view(np.float16).astype(np.float64)


def check_kv(gm, rm, n_layer, rows):
    for li in range(n_layer):
        gk, gv = gm.kv_cache(li, rows.stop)
        for got, ref in ((gk, rm.K[li]), (gv, rm.V[li])):
            g, r = f16(got[rows]), f16(ref[rows])
            rms = np.sqrt(np.mean(r ** 2, axis=1, keepdims=True))
            ulp = np.abs(r) * 2.0 ** -10 + 2.0 ** -24
            rel = 2e-4 if li == 0 else 1e-3
            assert np.all(np.abs(g - r) <= ulp + rel * rms), (li, np.max(np.abs(g - r) / rms))


def check_logits(gm, ref_logits, ref_tok, tok):
    lg = gm.logits().astype(np.float64)
    rl = ref_logits.astype(np.float64)
    scale = np.sqrt(np.mean(rl ** 2))
    assert np.max(np.abs(lg - rl)) <= 5e-3 * scale
    top = np.sort(rl)[-2:]
    if top[1] - top[0] > 1e-2 * scale:
        assert tok == ref_tok


@pytest.mark.parametrize("ci,n_prompt,n_more", [(0, 300, 21), (1, 40, 7), (2, 37, 0)])
def test_prefill_matches_reference(gpu, ci, n_prompt, n_more):
    cfg = TINY[ci]
    print(f"prefill model cfg {ci} n={n_prompt}+{n_more}", flush=True)
    max_seq = n_prompt + n_more + 8
    gm, rm = build(cfg, 300 + ci, max_seq)
    rng = np.random.default_rng(7 + ci)
    prompt = rng.integers(0, cfg["n_vocab"], n_prompt + n_more).tolist()
    tok = gm.prefill(prompt[:n_prompt], 0)
    rl, rt = rm.prefill(prompt[:n_prompt], 0)
    check_kv(gm, rm, cfg["n_layer"], slice(0, n_prompt))
    check_logits(gm, rl, rt, tok)
    if n_more:
        tok2 = gm.prefill(prompt[n_prompt:], n_prompt)
        rl2, rt2 = rm.prefill(prompt[n_prompt:], n_prompt)
        check_kv(gm, rm, cfg["n_layer"], slice(0, n_prompt + n_more))
        check_logits(gm, rl2, rt2, tok2)
    gm.close()


def calm(layers):
    """Norm weights that bring scores and gates to a few units (the plain synthetic
    rows give hundreds: softmaxes between two close scores, which no two orders of
    summation decide alike)."""
    return [dict(L, attn_norm=L["attn_norm"] * np.float32(0.005),
                 ffn_norm=L["ffn_norm"] * np.float32(0.01)) for L in layers]


def check64(gm, rm, ref, done, tok):
    """K / V rows and the last row's logits against the forward in 64 bits: one f16 ulp
    plus 2e-4 (layer 0) or 1e-3 of the row RMS, and for K what an angle
    pos theta^(-2i/hd) that is off by two roundings of fp32 (2^-22 pos) turns the
    largest pair by (K of a later layer also has the attention before it, whose
    scores turned by the same angles: four times that); the 2-norm over all rows 2.5e-4: f16's rounding is up to 2.1e-4,
    the rest the fp32 sums'."""
    K, V, x = ref
    for li in range(len(K)):
        for got, r, is_k in zip(gm.kv_cache(li, done), (K[li][:done], V[li][:done]), (True, False)):
            g = f16(got)
            rms = np.sqrt(np.mean(r ** 2, axis=1, keepdims=True))
            off = np.abs(r) * 2.0 ** -10 + 2.0 ** -24 + (1e-3 if li else 2e-4) * rms
            if is_k:
                turn = np.arange(done)[:, None] * 2.0 ** -22 * np.abs(r).max(1, keepdims=True)
                off = off + (4 if li else 1) * turn
            assert np.all(np.abs(g - r) <= off), li
            assert np.linalg.norm(g - r) <= 2.5e-4 * np.linalg.norm(r), li
    c = rm.c
    xb = oracle.rms_norm(x[done - 1].astype(np.float32), np.ones(c["n_embd"], np.float32), c["rms_eps"])
    rl = rm._global_q8((rm.E, rm.ecb), c["n_embd"], xb, True)
    check_logits(gm, rl, oracle.argmax(rl), tok)


@pytest.mark.parametrize("n_prompt,n_more,ff", [
    (31, 1, 512), (32, 0, 512), (33, 32, 512), (65, 0, 768),
    (300, 0, 2560),          # gate/up with K whole, a ragged last tile of tokens
    (1024 + 37, 1030, 512),  # a second chunk, and two more from pos0 > 0
    (2048, 0, 512),          # whole chunks
])
def test_prefill_tiles_and_chunks(gpu, n_prompt, n_more, ff):
    from taraference_amd.model import DecodeModel

    cfg = dict(TINY[0], n_ff=ff)
    print(f"prefill n={n_prompt}+{n_more} ff={ff}", flush=True)
    rng = np.random.default_rng(n_prompt)
    layers = calm([synth.qwen_layer(rng, cfg, li) for li in range(cfg["n_layer"])])
    emb = synth.qwen_embedding(rng, cfg)
    gm = DecodeModel(dict(cfg, max_seq=n_prompt + n_more + 8), layers, emb)
    rm = RefModel(cfg, layers, emb, 8)
    prompt = rng.integers(0, cfg["n_vocab"], n_prompt + n_more).tolist()
    ref = prefill64(cfg, layers, emb, prompt)
    done = 0
    for n in (n_prompt, n_more):
        if n:
            tok = gm.prefill(prompt[done:done + n], done)
            done += n
            check64(gm, rm, ref, done, tok)
    gm.close()


@pytest.mark.parametrize("shift", [0, 2])
@pytest.mark.parametrize("e,ff,n,q6", [
    (256, 512, 33, ("wq", "gate")),        # blocks and columns of 210 bytes: every other at 2 mod 4
    (512, 2560, 300, ("wk", "wo", "up")),
    (768, 1024, 70, ("wq", "wk", "gate", "up", "down")),
    (1536, 2048, 40, ("wq", "wo", "gate")),  # rows whose super-blocks are added whole
])
def test_prefill_q6k_matrices(gpu, e, ff, n, q6, shift):
    """Q6_K where the usual mix has Q4_K: q / k / v of mixed types in one launch, gate
    and up apart, raw blocks; `shift` puts all raw Q6_K bytes at 2 mod 4 and takes the
    compact copy of down away."""
    from taraference_amd.model import DecodeModel

    class Shifted(DecodeModel):
        def _q6(self, wm, n_rows, compact):
            m = super()._q6(wm, n_rows, compact)
            raw = torch.from_numpy(np.ascontiguousarray(wm[0])).cuda().reshape(-1)
            t = torch.zeros(raw.numel() + 16, dtype=torch.uint8, device="cuda")
            t[2:2 + raw.numel()] = raw
            self._keep.append(t)
            m.data = t.data_ptr() + 2
            if n_rows == self.cfg["n_ff"]:
                m.compact = None
            return m

    cfg = dict(n_layer=2, n_embd=e, n_ff=ff, n_head=e // 128, n_kv=1, head_dim=128, n_vocab=200,
               rope_theta=1e6, rms_eps=1e-6)
    rng = np.random.default_rng(e + n)
    layers = calm([synth.qwen_layer(rng, cfg, li) for li in range(2)])
    for L in layers:
        for name in q6:
            w, cb = synth.q6k_matrix(rng, ff if name == "down" else e, L[name][0].shape[0])
            if name == "down":
                L["down"], L["down_q6k"] = (w, cb), True
            else:
                L[name] = (w, cb, 14)
    emb = synth.qwen_embedding(rng, cfg)
    gm = (Shifted if shift else DecodeModel)(dict(cfg, max_seq=n + 8), layers, emb)
    print(f"prefill q6k e={e} ff={ff} n={n} {q6} shift={shift}", flush=True)
    toks = rng.integers(0, 200, n).tolist()
    tok = gm.prefill(toks, 0)
    check64(gm, RefModel(cfg, layers, emb, 8), prefill64(cfg, layers, emb, toks), n, tok)
    gm.close()


@pytest.mark.parametrize("name", ["attn_norm", "ffn_norm", "output_norm"])
def test_prefill_norms_4_byte_aligned(gpu, name):
    """A norm vector that starts 4 bytes past a 16-byte boundary: the same bits."""
    cfg = TINY[0]
    rng = np.random.default_rng(77)
    layers = [synth.qwen_layer(rng, cfg, li) for li in range(cfg["n_layer"])]
    emb = synth.qwen_embedding(rng, cfg)
    vec = {n: rng.uniform(0.8, 1.2, cfg["n_embd"]).astype(np.float32)
           for n in ("attn_norm", "ffn_norm", "output_norm")}
    prompt = rng.integers(0, cfg["n_vocab"], 20).tolist()
    out = []
    for u in (False, True):
        v = dict(vec, **({name: vec[name].view(Unaligned)} if u else {}))
        m = model_class()(dict(cfg, max_seq=40),
                          [dict(L, attn_norm=v["attn_norm"], ffn_norm=v["ffn_norm"])
                           for L in layers], emb, output_norm=v["output_norm"])
        print(f"prefill {name} unaligned={u}", flush=True)
        out.append((m.prefill(prompt, 0), m.logits()))
        m.close()
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])


def test_prefill_compact_down_2_byte_aligned(gpu):
    """A compact copy of a Q6_K down that the GEMM cannot load in dwords: the prompt
    reads the raw blocks, with the same bits."""
    from taraference_amd.model import DecodeModel

    class Shifted(DecodeModel):
        def _q6(self, wm, n_rows, compact):
            m = super()._q6(wm, n_rows, compact)
            if n_rows == self.cfg["n_ff"]:
                old = self._keep[-1]
                new = torch.zeros(old.numel() + 16, dtype=torch.uint8, device="cuda")
                new[2:2 + old.numel()] = old
                self._keep.append(new)
                m.compact = new.data_ptr() + 2
            return m

    cfg = TINY[0]
    rng = np.random.default_rng(78)
    layers = [synth.qwen_layer(rng, cfg, li) for li in range(cfg["n_layer"])]
    for L in layers:
        L["down"], L["down_q6k"] = synth.q6k_matrix(rng, cfg["n_ff"], cfg["n_embd"]), True
    emb = synth.qwen_embedding(rng, cfg)
    prompt = rng.integers(0, cfg["n_vocab"], 20).tolist()
    out = []
    for cls in (DecodeModel, Shifted):
        m = cls(dict(cfg, max_seq=40), layers, emb)
        print(f"prefill {cls.__name__}", flush=True)
        out.append((m.prefill(prompt, 0), m.logits()))
        m.close()
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])


def test_generate_after_prefill(gpu):
    cfg = TINY[0]
    gm, _ = build(cfg, 400, 64)
    prompt = np.random.default_rng(3).integers(0, cfg["n_vocab"], 20).tolist()
    out = gm.generate_prefilled(prompt, 6)
    assert len(out) == 6
    # the first token is prefill's; the rest continue on the decode path
    first = gm.prefill(prompt, 0)
    assert out[0] == first
    rest = gm.generate([first], 5, pos0=len(prompt))
    assert list(out[1:]) == list(rest)
    gm.close()
