"""The Q5_0 / Q8_0 layers' fused launches (norm + q, k, v; RoPE + cache append;
partial merge + wo; norm + gate + up + SiLU; the argmax over many workgroups)
at the widths that take each instantiation, through DecodeModel on path 0,
against the CPU reference step.  Bars as tests/test_gpu_q05_model.py: K/V of
layer 0 within one f16 ulp plus 2e-4 of the row RMS (fp32 GEMVs), logits within
2e-3 of their RMS plus four one-step Q8 flips of the head's input, the token the
argmax of the logits that the device holds, exactly."""
import numpy as np
import pytest

import oracle
from taraference_amd import synth
from _model_ref import RefModelMixed
from _util import q8_0_dequant
from test_gpu_q05_model import f16, write_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,ff,vocab,max_seq", [
    (1, 1, 256, 151, 40),      # two blocks a row; a vocabulary of 3 mod 4
    (4, 2, 512, 257, 40),      # one block a quad
    (17, 17, 768, 1003, 40),   # 34 blocks: the last round of a quad nearly empty
    (32, 4, 256, 130, 1024),   # the widest row, 16 partials
    (8, 8, 256, 64, 1600),     # 24 partials: merged by their own launch
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
    rm = RefModelMixed(cfg, layers, emb, max_seq)
    nb = e // 32
    wmax = float(np.abs(q8_0_dequant(emb[0][:, : nb * 34].reshape(-1, 34))).max())
    for pos, tok in enumerate(rng.integers(0, vocab, 5).tolist()):
        nxt = gm.forward(tok, pos)
        lg = gm.logits()
        assert nxt == oracle.argmax(lg), pos
        rl, _ = rm.step(tok, pos)
        scale = np.sqrt(np.mean(rl.astype(np.float64) ** 2))
        _, d8 = oracle.quantize_q8(rm.head_x)
        assert np.abs(lg.astype(np.float64) - rl).max() <= 2e-3 * scale + 4 * float(d8.max()) * wmax
        k, v = gm.kv_cache(0, pos + 1)
        for got, ref in ((k[pos], rm.K[0][pos]), (v[pos], rm.V[0][pos])):
            g, r = f16(got), f16(ref)
            ulp = np.abs(np.spacing(np.asarray(ref, np.uint16).view(np.float16))).astype(np.float64)
            assert np.all(np.abs(g - r) <= ulp + 2e-4 * np.sqrt(np.mean(r ** 2))), pos
    gm.close()
