"""A prompt through a model whose rows do not fit a CU's LDS (n_embd 40960): the
norm of a row reads it back from memory.  The square matrices are 0, so what the
layers compute is small enough for 64 bits: K and V of both layers within one f16
ulp plus 2e-4 of the row RMS (tests/test_gpu_prefill_model.py), the second layer's
input being the first's embedding row plus its FFN."""
import numpy as np
import pytest

from taraference_amd import synth
from _util import q4k_dequant, q6k_dequant, silu64

pytestmark = pytest.mark.gpu

E, F, HD, VOCAB, T = 40960, 256, 128, 64, 5
EPS = 1e-6


def deq(wm, k, q6):
    w = wm[0]
    return (q6k_dequant if q6 else q4k_dequant)(w.reshape(-1, 210 if q6 else 144)).reshape(
        w.shape[0], k).astype(np.float64)


def test_wide_rows(gpu):
    from taraference_amd.model import DecodeModel

    cfg = dict(n_layer=2, n_embd=E, n_ff=F, n_head=E // HD, n_kv=1, head_dim=HD, n_vocab=VOCAB,
               rope_theta=1e6, rms_eps=EPS, max_seq=16)
    rng = np.random.default_rng(40960)
    square = (np.zeros((E, E // 256 * 144), np.uint8), E // 256 * 144)
    layers = []
    for _ in range(2):
        layers.append(dict(
            attn_norm=rng.uniform(0.8, 1.2, E).astype(np.float32),
            ffn_norm=rng.uniform(0.8, 1.2, E).astype(np.float32), wq=square, wo=square,
            wk=synth.q4k_matrix(rng, E, HD), wv=synth.q6k_matrix(rng, E, HD),
            gate=synth.q4k_matrix(rng, E, F), up=synth.q4k_matrix(rng, E, F),
            down=synth.q4k_matrix(rng, F, E), down_q6k=False))
    emb = synth.q6k_matrix(rng, E, VOCAB)
    m = DecodeModel(cfg, layers, emb)
    toks = rng.integers(0, VOCAB, T).tolist()
    print(f"prefill n_embd={E}", flush=True)
    m.prefill(toks, 0)
    assert np.all(np.isfinite(m.logits()))

    def norm(x, w):
        return x / np.sqrt((x * x).mean(1, keepdims=True) + EPS) * w

    x = deq(emb, E, True)[toks]
    i = np.arange(HD // 2)
    ang = np.arange(T)[:, None] * 1e6 ** (-2.0 * i / HD)
    c, s = np.cos(ang), np.sin(ang)
    for li, L in enumerate(layers):
        n = norm(x, L["attn_norm"])
        k, v = n @ deq(L["wk"], E, False).T, n @ deq(L["wv"], E, True).T
        k = np.concatenate([k[:, :64] * c - k[:, 64:] * s, k[:, :64] * s + k[:, 64:] * c], 1)
        for got, ref in zip(m.kv_cache(li, T), (k, v)):
            g = got.view(np.float16).astype(np.float64)
            rms = np.sqrt((ref * ref).mean(1, keepdims=True))
            err = np.abs(g - ref) - np.abs(ref) * 2.0 ** -10 - 2.0 ** -24
            assert np.all(err <= 2e-4 * rms), (li, (err / rms).max())
        n = norm(x, L["ffn_norm"])
        h = silu64(n @ deq(L["gate"], E, False).T) * (n @ deq(L["up"], E, False).T)
        x = x + h @ deq(L["down"], F, False).T
    m.close()
