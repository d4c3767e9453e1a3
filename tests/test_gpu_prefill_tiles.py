"""The prefill GEMMs (tf_gemm_q4k_f32 / tf_gemm_q6k_f32, kernels/gemm.cu:6-121)
at the edges of their tiles and on every branch of their dispatch, against the
fp64 product with numpy-dequantized weights (tests/_util.gemm_ref), within the
fp32 GEMV tolerance (1e-5 relative, floor 0.1 * sum |terms|): the split of x
keeps 22 bits of each value, 2^-23 of a term, and the rest is fp32 summation.

The token tile is 32, a wave's columns 64; the dispatch weighs 256 columns a
workgroup with K whole against fewer columns with K split over its waves, by
the number of output tiles and of super-blocks; the Q6_K loads go by where a
column starts modulo 4 (an odd number of 210-byte blocks makes it alternate).
"""
import numpy as np
import pytest
import torch

from taraference_amd import synth
from _gpu import KEEP, P, S, call, dev, empty, host
from _util import assert_gemv_close, gemm_ref, q6k_dequant

pytestmark = pytest.mark.gpu


def run(fmt, n_rows, n_cols, x, shift=0, seed=0):
    """The GEMM with the weights `shift` bytes into their buffer."""
    rng = np.random.default_rng(n_rows + 3 * n_cols + seed)
    w, cb = (synth.q4k_matrix if fmt == "q4k" else synth.q6k_matrix)(rng, n_rows, n_cols)
    if fmt == "q6k":  # scales over their whole range: products past f16's exact integers
        blk = w.reshape(-1, 210)
        blk[:, 192:208] = rng.integers(-128, 128, (blk.shape[0], 16)).astype(np.int8).view(np.uint8)
    buf = dev(np.concatenate([np.zeros(shift, np.uint8), w.reshape(-1)]))
    n_tok = x.shape[0]
    out = empty(n_tok * n_cols)
    print(f"gemm {fmt} {n_rows}x{n_cols} tok={n_tok} shift={shift}", flush=True)
    call(f"tf_gemm_{fmt}_f32", P(buf) + shift, P(dev(x)), P(out), n_rows, n_cols, cb, n_tok, S())
    y = host(out).reshape(n_tok, n_cols)
    ref, absn = gemm_ref(fmt, w, n_rows, x)
    for t in range(n_tok):
        assert_gemv_close(y[t], ref[t], absn[t], f"{fmt} t={t}")


@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
@pytest.mark.parametrize("n_rows,n_cols,n_tok", [
    (256, 1, 1),        # one value
    (768, 63, 31),      # 3 super-blocks over 4 slices, one short of a tile each way
    (768, 65, 33),      # one past a tile
    (1280, 129, 32),    # 5 super-blocks over 4 slices (Q6_K)
    (512, 4100, 130),   # 128 columns, K over 2 slices (Q6_K)
    (1792, 3200, 200),  # 7 super-blocks over 4 (Q4_K) and 2 (Q6_K) slices
    (256, 8200, 190),   # 256 columns, ragged both ways
    (768, 6145, 260),
])
def test_gemm_tiles(gpu, fmt, n_rows, n_cols, n_tok):
    x = np.random.default_rng(n_tok).standard_normal((n_tok, n_rows)).astype(np.float32)
    run(fmt, n_rows, n_cols, x)


@pytest.mark.parametrize("fmt,shift", [("q4k", 4), ("q4k", 8), ("q6k", 2), ("q6k", 4), ("q6k", 6)])
@pytest.mark.parametrize("n_rows,n_cols,n_tok", [(768, 70, 5), (512, 4100, 130), (768, 6145, 260)])
def test_gemm_unaligned_weights(gpu, fmt, shift, n_rows, n_cols, n_tok):
    x = np.random.default_rng(n_tok).standard_normal((n_tok, n_rows)).astype(np.float32)
    run(fmt, n_rows, n_cols, x, shift)


@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
def test_gemm_scales_of_x(gpu, fmt):
    """Each (token, super-block) has its own power of two: rows and
    super-blocks of very different magnitude, zero rows, the smallest and
    largest scales (the products stay finite)."""
    rng = np.random.default_rng(5)
    x = rng.standard_normal((40, 768)).astype(np.float32)
    x[1] = 0
    x[2, :256] = 0
    x[3] *= np.float32(1e-30)
    x[4] *= np.float32(1e30)
    x[5, 256:512] *= np.float32(1e-12)
    x[6, ::7] *= np.float32(1e4)
    x[7] = np.float32(1e-38)  # subnormal products with the block scales still count
    x[8] = 1
    run(fmt, 768, 200, x)


@pytest.mark.parametrize("k,n,t,bar", [
    (256, 2000, 20, 0.95e-7),   # one super-block
    (512, 900, 64, 1.1e-7),     # 2 of 64 columns and K / 4
    (1280, 4100, 130, 1.1e-7),  # the last width that adds 64 values at a time
    (1536, 1000, 40, 1.85e-7),  # whole super-blocks
])
@pytest.mark.parametrize("shift", [0, 2])
def test_gemm_q6k_error(gpu, k, n, t, bar, shift):
    """Q6_K is no further from 64 bits than sums that were scaled every 16 values: 0.91,
    1.14, 1.70 and 1.85e-7 of the result's 2-norm for normal x and scales over their
    whole range (48 products a value in one sum have 1.7e-7)."""
    rng = np.random.default_rng(k)
    blk = synth.q6k_blocks(rng, n * k // 256)
    blk[:, 192:208] = rng.integers(-128, 128, (len(blk), 16)).astype(np.int8).view(np.uint8)
    w = blk.reshape(n, -1)
    x = rng.standard_normal((t, k)).astype(np.float32)
    buf = dev(np.concatenate([np.zeros(shift, np.uint8), w.reshape(-1)]))
    out = empty(t * n)
    print(f"gemm q6k error {k}x{n} tok={t} shift={shift}", flush=True)
    call("tf_gemm_q6k_f32", P(buf) + shift, P(dev(x)), P(out), k, n, w.shape[1], t, S())
    ref = x.astype(np.float64) @ q6k_dequant(blk).reshape(n, k).astype(np.float64).T
    assert np.linalg.norm(host(out).reshape(t, n) - ref) <= bar * np.linalg.norm(ref)


@pytest.mark.parametrize("fmt,n_rows,n_cols,n_tok", [
    ("q4k", 1 << 27, 64, 1),           # 64 columns of 72 MB: more than 4 GB
    ("q6k", 1 << 27, 64, 1),
    ("q4k", (1 << 25) + 256, 3, 33),   # 32 rows of 128 MB
])
def test_gemm_past_32_bit_offsets(gpu, fmt, n_rows, n_cols, n_tok):
    """Everything 0 but a few super-blocks of the first, the last and the columns and
    rows on either side of 4 GB."""
    rng = np.random.default_rng(n_cols)
    nb, bb = n_rows // 256, 144 if fmt == "q4k" else 210
    make = synth.q4k_blocks if fmt == "q4k" else synth.q6k_blocks
    w = torch.zeros((n_cols, nb, bb), dtype=torch.uint8, device="cuda")
    x = torch.zeros((n_tok, nb, 256), device="cuda")
    KEEP.extend((w, x))
    sbs = [0, 1, nb // 2 + 3, nb - 1]
    cols = sorted({0, n_cols // 2, n_cols - 9, n_cols - 2, n_cols - 1} & set(range(n_cols)))
    cols += [c for c in (36, 37, 55, 56, 57) if c < n_cols and c not in cols]
    wb = np.zeros((n_cols, len(sbs), bb), np.uint8)
    wb[cols] = make(rng, len(cols) * len(sbs)).reshape(len(cols), len(sbs), bb)
    xb = rng.standard_normal((n_tok, len(sbs), 256)).astype(np.float32)
    w[:, sbs] = torch.from_numpy(wb).cuda()
    x[:, sbs] = torch.from_numpy(xb).cuda()
    out = empty(n_tok * n_cols)
    print(f"gemm {fmt} {n_rows}x{n_cols} tok={n_tok}", flush=True)
    call(f"tf_gemm_{fmt}_f32", P(w), P(x), P(out), n_rows, n_cols, nb * bb, n_tok, S())
    y = host(out).reshape(n_tok, n_cols)
    ref, absn = gemm_ref(fmt, wb.reshape(n_cols, -1), 256 * len(sbs), xb.reshape(n_tok, -1))
    for t in range(n_tok):
        assert_gemv_close(y[t], ref[t], absn[t], f"{fmt} t={t}")
    KEEP.clear()
    del w, x
    torch.cuda.empty_cache()
