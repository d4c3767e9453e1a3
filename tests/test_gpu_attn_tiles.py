"""tf_attn_prefill (kernels/attn/fast_v2.cu:12-192) on the matrix cores at the
edges of its tiles: 32 (query, head) rows a workgroup, 32 keys a tile, eight
waves that share the tiles.  Against the fp64 softmax attention of the oracle.

Tolerance: q and 2^14 p are held in two f16 parts (2^-22 of the row's largest q;
2^-22 of each weight p, and of p below 2^-17 2^-39, the largest being 1), K and V
are f16 and the products exact.  A score is off by at most 2^-22 max|q| sum|k| scale
(under 2e-5 here: 2^-22 * 4 * 128 * 0.8 / 8) plus as much again from fp32
summation, and an output is a mean of V rows whose weights are off by that: 4e-5
max|V|, and n 2^-39 max|V| for n keys (6e-8 at 32768).
"""
import numpy as np
import pytest

import oracle
from taraference_amd import synth
from _gpu import P, S, call, dev, empty, host

pytestmark = pytest.mark.gpu


def run(n_head, n_kv, hd, pos0, n_q, shift=0, scale=None):
    rng = np.random.default_rng(n_q * 5 + pos0 + hd)
    L = pos0 + n_q
    K = synth.kv_cache(rng, L + 33, n_kv, hd)
    V = synth.kv_cache(rng, L + 33, n_kv, hd)
    K[L:] = V[L:] = 0x7E00  # f16 NaN past the last query
    q = np.clip(rng.standard_normal((n_q, n_head * hd)), -4, 4).astype(np.float32)
    scale = float(np.float32(hd ** -0.5)) if scale is None else scale
    pad = np.zeros(shift // 2, np.uint16)
    kb = dev(np.concatenate([pad, K.reshape(-1).view(np.uint16)]).view(np.int16))
    vb = dev(np.concatenate([pad, V.reshape(-1).view(np.uint16)]).view(np.int16))
    out = empty(n_q * n_head * hd)
    print(f"attn h={n_head} kv={n_kv} hd={hd} pos0={pos0} n_q={n_q} shift={shift}", flush=True)
    call("tf_attn_prefill", P(dev(q)), P(kb) + shift, P(vb) + shift, P(out), n_head, n_kv, hd, pos0,
         n_q, scale, S())
    y = host(out).reshape(n_q, -1)
    vmax = float(np.abs(V[:L].view(np.float16).astype(np.float32)).max())
    for i in sorted({0, 1, n_q // 2, n_q - 2, n_q - 1} & set(range(n_q))):
        ref = oracle.attn_f64(q[i], K, V, n_head, n_kv, hd, pos0 + i + 1, scale)
        err = np.abs(y[i] - ref).max()
        assert err <= 4e-5 * vmax, (i, err, vmax)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("n_head,n_kv,pos0,n_q", [
    (4, 4, 0, 1),       # one row, one key
    (4, 4, 0, 33),      # one row and one key past a tile
    (14, 2, 31, 5),     # 35 rows of 7 heads: queries cut by a tile of rows
    (16, 2, 0, 32),     # whole tiles
    (28, 4, 255, 9),    # 8 tiles for most rows, 9 for the last
    (40, 1, 511, 3),    # more heads in the group than rows in a tile
    (8, 8, 257, 64),
])
def test_attn_tiles(gpu, hd, n_head, n_kv, pos0, n_q):
    run(n_head, n_kv, hd, pos0, n_q)


@pytest.mark.parametrize("hd", [64, 128])
def test_attn_caches_8_byte_aligned(gpu, hd):
    run(14, 2, hd, 300, 7, shift=8)


@pytest.mark.parametrize("hd", [64, 128])
def test_attn_negative_scale(gpu, hd):
    run(8, 2, hd, 70, 12, scale=-0.1)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("mag", [1e4, 1e9, 1e25])
def test_attn_large_scores(gpu, hd, mag):
    """Scores far beyond 2^24: where the two largest of a row lie further apart than
    they can be off (2^-22 max|q| sum|k| scale for q's parts, as much for fp32
    summation, and 20 for the weights to differ by e^-20), the output is the V row
    of the largest; all others lie within the range of the V rows they see."""
    rng = np.random.default_rng(hd)
    n_head, n_kv, pos0, n_q = 14, 2, 290, 20
    L = pos0 + n_q
    K, V = synth.kv_cache(rng, L, n_kv, hd), synth.kv_cache(rng, L, n_kv, hd)
    q = (rng.standard_normal((n_q, n_head, hd)) * mag).astype(np.float32)
    out = empty(n_q * n_head * hd)
    print(f"attn large scores hd={hd} mag={mag}", flush=True)
    scale = float(np.float32(hd ** -0.5))
    call("tf_attn_prefill", P(dev(q)), P(dev(K)), P(dev(V)), P(out), n_head, n_kv, hd, pos0, n_q,
         scale, S())
    y = host(out).reshape(n_q, n_head, hd)
    k = K.view(np.float16).astype(np.float64).reshape(L, n_kv, hd)
    v = V.view(np.float16).astype(np.float64).reshape(L, n_kv, hd)
    vmax = np.abs(v).max()
    clear = 0
    for i in range(n_q):
        for h in range(n_head):
            kg, vg = (a[:pos0 + i + 1, h // (n_head // n_kv)] for a in (k, v))
            s = kg @ q[i, h].astype(np.float64) * scale
            order = np.argsort(s)
            off = 2.0 ** -21 * np.abs(q[i, h]).max() * np.abs(kg[order[-2:]]).sum(1).max() * scale
            if s[order[-1]] - s[order[-2]] > 2 * off + 20:
                clear += 1
                assert np.abs(y[i, h] - vg[order[-1]]).max() <= 4e-5 * vmax, (i, h)
            assert np.all(y[i, h] <= vg.max(0) + 1e-5) and np.all(y[i, h] >= vg.min(0) - 1e-5)
    assert clear > 0.8 * n_q * n_head


@pytest.mark.parametrize("hd", [64, 128])
def test_attn_sinks(gpu, hd):
    """Eight keys, one in each wave's first tile, 17 above 8000 others and with V = 0:
    the others' weights are e^-17 (below 2^-24), their share of the output 4e-5 max|V|
    of which 4e-5 may be off by the scores, and 1e-7 by the 2^-39 steps (8000 2^-39 =
    1.5e-8) and fp32."""
    rng = np.random.default_rng(hd)
    n_head, n_kv, pos0, n_q = 4, 2, 7990, 18
    L, scale = pos0 + n_q, float(np.float32(hd ** -0.5))
    q = np.zeros((n_q, n_head, hd), np.float32)
    q[..., 0] = np.float32(17 / 16 / scale)
    q[..., 1] = rng.uniform(-1, 1, (n_q, n_head)) / scale
    K = np.zeros((L, n_kv, hd), np.float16)
    V = rng.uniform(0.5, 1, (L, n_kv, hd)).astype(np.float16)
    K[..., 1] = rng.uniform(-0.5, 0.5, (L, n_kv))
    sinks = 32 * np.arange(8)
    K[sinks, :, 0], V[sinks] = 16, 0
    Kb, Vb = K.view(np.uint16).reshape(L, -1), V.view(np.uint16).reshape(L, -1)
    out = empty(n_q * n_head * hd)
    print(f"attn sinks hd={hd}", flush=True)
    call("tf_attn_prefill", P(dev(q)), P(dev(Kb)), P(dev(Vb)), P(out), n_head, n_kv, hd, pos0, n_q,
         scale, S())
    y = host(out).reshape(n_q, -1)
    for i in (0, n_q - 1):
        ref = oracle.attn_f64(q[i].reshape(-1), Kb, Vb, n_head, n_kv, hd, pos0 + i + 1, scale)
        assert 2e-5 < np.abs(ref).min()
        assert np.abs(y[i] - ref).max() <= 4e-5 * np.abs(ref).max() + 1e-7


def rows64(q, K, V, n_head, n_kv, hd, pos0, scale):
    """The outputs in 64 bits where something is infinite or NaN: a NaN or -inf score
    is no key, a +inf one makes the row NaN, and weight 0 times an infinite V is NaN."""
    out = np.empty((len(q), n_head, hd))
    with np.errstate(all="ignore"):
        for i in range(len(q)):
            for h in range(n_head):
                g = h // (n_head // n_kv)
                k, v = K[:pos0 + i + 1, g], V[:pos0 + i + 1, g]
                s = (q[i, h] * k).sum(1) * scale
                e = np.where(s > -1e29, np.exp(s - s[s > -1e29].max(initial=-1e30)), 0)
                out[i, h] = (e[:, None] * v).sum(0) / max(e.sum(), 1e-20)
    return out


def test_attn_hd64_not_finite(gpu):
    """Infinities and NaN at head_dim 64, which takes them as fp32 arithmetic does: in
    a query (alone and beside others of its tile), in a key and in values."""
    rng = np.random.default_rng(64)
    n_head, n_kv, hd, pos0, n_q = 6, 2, 64, 50, 70
    L, scale = pos0 + n_q, 0.125
    q = rng.standard_normal((n_q, n_head, hd)).astype(np.float32)
    K = rng.standard_normal((L, n_kv, hd)).astype(np.float16)
    V = rng.standard_normal((L, n_kv, hd)).astype(np.float16)
    q[2, 0, 5], q[5, 1, 7], q[7, 2, 9] = np.inf, -np.inf, np.nan
    q[30, 4, 1], q[31, 4, 1:3] = np.inf, (np.inf, -np.inf)
    K[95, 0, 3], K[60, 1, 4] = np.inf, -np.inf
    V[100, 0, 9], V[52, 1, 20], V[57, 1, 21] = np.inf, -np.inf, np.nan
    ref = rows64(q.astype(np.float64), K.astype(np.float64), V.astype(np.float64), n_head, n_kv,
                 hd, pos0, scale)
    out = empty(q.size)
    print("attn hd=64 not finite", flush=True)
    call("tf_attn_prefill", P(dev(q)), P(dev(K.view(np.int16))), P(dev(V.view(np.int16))), P(out),
         n_head, n_kv, hd, pos0, n_q, scale, S())
    y = host(out).reshape(ref.shape).astype(np.float64)
    fin = np.isfinite(ref)
    assert 0.3 < fin.mean() < 0.9 and np.isinf(ref).any()
    np.testing.assert_array_equal(np.where(fin, 0, y), np.where(fin, 0, ref))
    assert np.abs(y[fin] - ref[fin]).max() <= 4e-5 * 5


@pytest.mark.parametrize("pos0,n_q,bar", [
    (0, 2, 4.4e-8), (0, 5, 6.7e-8), (0, 12, 9.0e-8), (0, 16, 9.7e-8),  # in fp32
    (20, 5, 1.6e-7), (0, 64, 1.4e-7), (300, 5, 2.6e-7),  # on the matrix cores
])
def test_attn_hd64_error(gpu, pos0, n_q, bar):
    """head_dim 64 is no further from 64 bits than fp32 vector arithmetic: 4.1, 6.3,
    8.5 and 9.1e-8, 1.49, 1.34 and 3.6e-7 of the output's 2-norm for normal q, K and V
    (each bar 7 % above that, the spread over inputs; 2.6e-7 at 300 keys, where two f16
    parts do better)."""
    h, kv, hd = 14, 2, 64
    err = ref = 0.0
    for seed in range(8):
        rng = np.random.default_rng(1000 * n_q + pos0 + seed)
        q = rng.standard_normal((n_q, h, hd)).astype(np.float32)
        q *= np.exp(0.5 * rng.standard_normal((h, hd))).astype(np.float32)
        K, V = (rng.standard_normal((pos0 + n_q, kv, hd)).astype(np.float16) for _ in "kv")
        out = empty(q.size)
        print(f"attn error pos0={pos0} n_q={n_q} seed={seed}", flush=True)
        call("tf_attn_prefill", P(dev(q)), P(dev(K.view(np.int16))), P(dev(V.view(np.int16))),
             P(out), h, kv, hd, pos0, n_q, 0.125, S())
        r = rows64(*(a.astype(np.float64) for a in (q, K, V)), h, kv, hd, pos0, 0.125)
        err += np.sum((host(out).reshape(r.shape) - r) ** 2)
        ref += np.sum(r ** 2)
    assert np.sqrt(err / ref) <= bar
