"""The tiled prefill GEMM kernels at the edges of their tiles.

Each case is a grid, a K range or a remainder at which one of the kernels that
uocr_launch_gemm chooses among could go wrong: partial row and column tiles, K
groups with fewer steps than the others (or none), weight lines that end inside
a group of 64 columns.  The reference is float64 over the operand values that
the kernels define, fp16(q * scale); the bound is one rounding to fp16 (half a
unit, 2^-11 relative, or half the subnormal spacing) plus K fp32 additions of
products no larger than the sum of their magnitudes."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rand_f16, weights_for

pytestmark = pytest.mark.gpu


def operand_values(qtype, w, s) -> np.ndarray:
    """float64 of fp16(q * scale)."""
    if qtype == 1:
        return w.astype(np.float64)
    rows = w.shape[0]
    if qtype == 3:
        q = w.astype(np.float32).reshape(rows, -1, 64)
    else:
        b = w.reshape(rows, -1, 32)
        q = np.concatenate([b & 15, b >> 4], axis=2).astype(np.float32) - 8
    return (q * s.astype(np.float32)[:, :, None]).astype(np.float16).astype(np.float64).reshape(rows, -1)


def check_rows(got, x, wv, add):
    """got fp16 [rows][n] against x . wv^T + add within the bound above."""
    x = x.astype(np.float64)
    ref = x @ wv.T + add
    mag = np.abs(x) @ np.abs(wv).T + np.abs(add)
    bound = np.abs(ref) * 2.0**-11 + 2.0**-25 + mag * wv.shape[1] * 2.0**-24
    err = np.abs(got.astype(np.float64) - ref)
    assert (err <= bound).all(), (float((err / bound).max()), np.argwhere(err > bound)[:4].tolist())


# m x n x k: large tiles (full, ragged rows and columns, the shortest K), 64 x
# 128 tiles with K in two groups (one step: the second group is empty; an odd
# number of steps), K in four groups, 32 x 64 tiles with K in eight groups, and
# K by weight lines (1 row, 1 column piece, a last line with 1, 2 or 3 groups)
SHAPES = [(2561, 2048, 64), (2433, 2056, 320), (1300, 648, 64), (1090, 776, 192), (700, 1000, 4160), (130, 520, 3136),
          (64, 1280, 3072), (1, 8, 64), (33, 72, 192), (95, 200, 448), (32, 64, 832)]


@pytest.mark.parametrize("qtype", [1, 3, 4])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gemm_tile_edges(gpu, qtype, m, n, k):
    uocr = gpu
    rng = np.random.default_rng(m + n + k + qtype)
    w, s = weights_for(qtype, rng, n, k)
    x, res = rand_f16(rng, (m, k)), rand_f16(rng, (m, n))
    of = uocr.DeviceBuffer.of
    dw, ds, dx, dr, dy = of(w), None if s is None else of(s), of(x), of(res), of(np.full((m, n), 7, np.float16))
    rows = np.unique(np.concatenate([np.arange(min(m, 40)), np.arange(max(0, m - 40), m), rng.integers(0, m, 40)]))
    wv = operand_values(qtype, w, s)
    for with_res in (False, True):
        uocr.op_gemm(qtype, dw, ds, m, n, k, dx, dr if with_res else None, dy)
        uocr.sync()
        got = dy.download(np.float16).reshape(m, n)
        check_rows(got[rows], x[rows], wv, res[rows].astype(np.float64) if with_res else np.zeros((rows.size, n)))


@pytest.mark.parametrize("qtype", [1, 3, 4])
def test_gemm_misaligned_rows(gpu, qtype):
    """Widths and pointers whose rows are not whole 16-byte pieces take the
    general kernel and give the same values."""
    uocr = gpu
    rng = np.random.default_rng(qtype)
    m, n, k = 70, 132, 192
    w, s = weights_for(qtype, rng, n, k)
    x = rand_f16(rng, (m, k))
    of = uocr.DeviceBuffer.of
    dw, ds, dx, dy = of(w), None if s is None else of(s), of(x), uocr.DeviceBuffer(m * n * 2 + 16)
    wv = operand_values(qtype, w, s)
    uocr.op_gemm(qtype, dw, ds, m, n, k, dx, None, dy)
    uocr.sync()
    check_rows(dy.download(np.float16, m * n).reshape(m, n), x, wv, np.zeros((m, n)))
    n2 = 128  # whole rows at a pointer 8 bytes off
    uocr.op_gemm(qtype, dw, ds, m, n2, k, dx, None, dy.ptr + 8)
    uocr.sync()
    got = dy.download(np.float16, 4 + m * n2)[4:].reshape(m, n2)
    check_rows(got, x, wv[:n2], np.zeros((m, n2)))
