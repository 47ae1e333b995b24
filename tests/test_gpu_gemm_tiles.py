"""The tiled prefill GEMM kernels at the edges of their tiles.

Each case is a grid, a K range or a remainder at which one of the kernels that
uocr_launch_gemm chooses among could go wrong: partial row and column tiles, K
groups with fewer steps than the others (or none), weight lines that end inside
a group of 64 columns.  The reference is float64 over the operand values that
the kernels define, fp16(q * scale); the bound is one rounding to fp16 (half a
unit, 2^-11 relative, or half the subnormal spacing) plus K fp32 additions of
products no larger than the sum of their magnitudes."""
from __future__ import annotations

import math

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
# K by weight lines (1 row, 1 column piece, a last line with 1, 2 or 3 groups);
# the last two are the first two with a grid on which Q4 takes the large tiles too
SHAPES = [(2561, 2048, 64), (2433, 2056, 320), (1300, 648, 64), (1090, 776, 192), (700, 1000, 4160), (130, 520, 3136),
          (64, 1280, 3072), (1, 8, 64), (33, 72, 192), (95, 200, 448), (32, 64, 832), (3073, 2048, 64), (2945, 2056, 320)]


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


@pytest.mark.parametrize("qtype", [1, 3, 4])
@pytest.mark.parametrize("m,n,k", [(70, 132, 2048), (70, 130, 2048), (257, 132, 192)])
def test_vision_linear_misaligned_rows(gpu, qtype, m, n, k):
    """Widths off 16-byte pieces take the general kernel: split over K with its
    reduce (long K, n % 4 == 0) and unsplit."""
    uocr = gpu
    rng = np.random.default_rng(qtype + n)
    w, s = weights_for(qtype, rng, n, k)
    x, bias = rand_f16(rng, (m, k)), rand_f16(rng, (n,))
    of = uocr.DeviceBuffer.of
    dw, ds, dx, db, dy = of(w), None if s is None else of(s), of(x), of(bias), uocr.DeviceBuffer(m * n * 2)
    uocr.op_vision_linear(qtype, dw, ds, db, m, k, n, 0, 0, dx, dy)
    uocr.sync()
    got = dy.download(np.float16, m * n).reshape(m, n)
    check_rows(got, x, operand_values(qtype, w, s), np.tile(bias.astype(np.float64), (m, 1)))


def activated(x, act):
    """(value, largest slope) of the vision activations in float64."""
    if act == 1:
        return x / (1 + np.exp(-1.702 * x)), 1.1
    if act == 2:
        return 0.5 * x * (1 + np.vectorize(math.erf)(x / math.sqrt(2))), 1.13
    return x, 1.0


# m, n, k, activation, split, kernel: every kernel with an epilogue of its own,
# ragged rows and columns, K groups of 13, 13, 13 and 10 steps (mid_k4), 8 splits
# of 5 steps and fewer in the last (general)
VISION_SHAPES = [(2561, 2568, 128, 2, 0, "large"), (2945, 2064, 64, 1, 688, "large"), (1090, 776, 192, 1, 0, "mid"), (1300, 648, 64, 2, 216, "mid"),
                 (780, 1032, 3136, 1, 0, "mid_k4"), (780, 1032, 3136, 0, 344, "mid_k4"), (330, 1032, 3136, 2, 0, "narrow"), (95, 200, 448, 2, 0, "lines"),
                 (33, 72, 192, 1, 24, "lines"), (100, 256, 2368, 2, 0, "general"), (70, 264, 2368, 1, 88, "general")]


@pytest.mark.parametrize("qtype", [1, 3, 4])
@pytest.mark.parametrize("m,n,k,act,split,kernel", VISION_SHAPES)
def test_vision_tile_edges(gpu, qtype, m, n, k, act, split, kernel):
    """The bound of check_rows through the activation's slope, and 2^-21 of the
    argument for the hardware exp2 and reciprocal and the erf polynomial (1.5e-7
    absolute, times half the argument)."""
    uocr = gpu
    assert uocr.op_gemm_kernel(qtype, m, n, k, True, act) == kernel
    rng = np.random.default_rng(m + n + k + qtype)
    w, s = weights_for(qtype, rng, n, k)
    x, bias = rand_f16(rng, (m, k)), rand_f16(rng, (n,))
    of = uocr.DeviceBuffer.of
    dw, ds, dx, db = of(w), None if s is None else of(s), of(x), of(bias)
    width = split or n
    outs = [of(np.full((m, width), 7, np.float16)) for _ in range(3 if split else 1)]
    uocr.op_vision_linear(qtype, dw, ds, db, m, k, n, act, split, dx, *outs)
    uocr.sync()
    got = np.hstack([o.download(np.float16).reshape(m, width) for o in outs]).astype(np.float64)
    rows = np.unique(np.concatenate([np.arange(min(m, 40)), np.arange(max(0, m - 40), m), rng.integers(0, m, 40)]))
    wv, xd = operand_values(qtype, w, s), x[rows].astype(np.float64)
    pre = xd @ wv.T + bias.astype(np.float64)
    mag = np.abs(xd) @ np.abs(wv).T + np.abs(bias.astype(np.float64))
    ref, slope = activated(pre, act)
    bound = np.abs(ref) * 2.0**-11 + 2.0**-25 + slope * mag * (k + 1) * 2.0**-24 + (np.abs(pre) * 2.0**-21 if act else 0.0)
    err = np.abs(got[rows] - ref)
    assert (err <= bound).all(), (float((err / bound).max()), np.argwhere(err > bound)[:4].tolist())


def test_vision_linear_block_split_in_a_graph(gpu):
    """K split over blocks under capture.  The first capture needs more partials
    than any call of this process has made the library allocate (33 MB), so it
    holds the unsplit kernel; after an eager call, which grows the buffer, it
    holds the split and its reduce and every replay equals the eager result."""
    uocr = gpu
    m, n, k, qtype = 1984, 508, 2048, 3  # 124 tiles, 8 splits; rows off 16-byte pieces
    rng = np.random.default_rng(9)
    w, s = weights_for(qtype, rng, n, k)
    x, bias = rand_f16(rng, (m, k)), rand_f16(rng, (n,))
    of = uocr.DeviceBuffer.of
    dw, ds, dx, db, dy = of(w), of(s), of(x), of(bias), uocr.DeviceBuffer(m * n * 2)
    rows = np.arange(0, m, 37)
    wv, add = operand_values(qtype, w, s), np.tile(bias.astype(np.float64), (rows.size, 1))

    def call():
        uocr.op_vision_linear(qtype, dw, ds, db, m, k, n, 0, 0, dx, dy)

    def result():
        uocr.sync()
        return dy.download(np.uint16).reshape(m, n)

    def captured():
        with uocr.Capture() as g:
            call()
        out = []
        try:
            for _ in range(3):
                dy.zero()
                g.replay(1)
                out.append(result())
        finally:
            g.release()
        assert all(np.array_equal(out[0], o) for o in out)
        return out[0]

    first = captured()
    dy.zero()
    call()
    eager = result()
    second = captured()
    for got in (first, eager):
        check_rows(got.view(np.float16)[rows], x[rows], wv, add)
    assert np.array_equal(second, eager)
    assert not np.array_equal(first, eager)  # another order of the sums: the first was not the split


def routed_rows(rng, counts, P):
    """For each row its 6 experts, so that expert e serves counts[e] rows."""
    left = np.full(P, 6)
    chosen = [[] for _ in range(P)]
    for e in np.argsort(-np.asarray(counts)):
        rows = np.argsort(-left + rng.random(P) * 0.5, kind="stable")[:counts[e]]
        assert (left[rows] > 0).all()
        left[rows] -= 1
        for r in rows:
            chosen[r].append(int(e))
    assert (left == 0).all()
    return chosen


def bucket_counts(P, given):
    """`given` rows for the first experts, the rest of the 6 P spread evenly."""
    rest = 6 * P - sum(given)
    n = 64 - len(given)
    return list(given) + [rest // n + (i < rest % n) for i in range(n)]


@pytest.mark.parametrize("qtype", [1, 3, 4])
@pytest.mark.parametrize("P,given,static", [(1, [], True), (6, [6, 6], True), (7, [7], True), (64, [64, 33, 32, 31, 1], True),
                                            (263, [263, 257, 256, 129, 128, 97, 96, 65, 64, 33, 32, 31, 1], False)])
def test_moe_rows_bucket_edges(gpu, qtype, P, given, static):
    """Expert buckets on both sides of every tile height (and above one tile),
    with few rows (weight lines) and more.  The router is a selector, so the
    bucket sizes are chosen.  Reference: float64 over the kernels' operand
    values with the mids and the shared output rounded to fp16; a mid whose fp32
    sum lies at a rounding boundary may differ by one unit (2^-10), so the bound
    is that share of the magnitudes plus the final rounding."""
    uocr = gpu
    rng = np.random.default_rng(P + qtype)
    counts = [c if c <= P else P for c in bucket_counts(P, given)]
    chosen = routed_rows(rng, counts, P)
    x = rand_f16(rng, (P, 1280), 0.5)
    x[:, :64] = 0
    for t, es in enumerate(chosen):
        x[t, es] = np.float16(1) + np.arange(len(es), dtype=np.float16) / 8
    router = np.zeros((64, 1280), np.float16)
    router[np.arange(64), np.arange(64)] = 8
    res = rand_f16(rng, (P, 1280))
    of = uocr.DeviceBuffer.of
    m, keep, val = uocr.CMoeWeights(), [], {}
    m.expert_qtype = m.shared_qtype = qtype
    for name, rows, k in (("gate", 64 * 896, 1280), ("up", 64 * 896, 1280), ("down", 64 * 1280, 896), ("sgate", 1792, 1280),
                          ("sup", 1792, 1280), ("sdown", 1280, 1792)):
        # a few distinct experts' weights, repeated: the bytes are what the test needs, not their number
        n = rows // 64 if rows > 2000 else rows
        w, s = weights_for(qtype, rng, 4 * n if rows > 2000 else n, k)
        val[name] = operand_values(qtype, w, s)
        if rows > 2000:
            w = np.tile(w, (16, 1))
            s = None if s is None else np.tile(s, (16, 1))
        keep += [of(w), None if s is None else of(s)]
        setattr(m, name + "_w", keep[-2].ptr)
        setattr(m, name + "_s", None if s is None else keep[-1].ptr)
        if name in ("gate", "down"):
            pre = "gu" if name == "gate" else "dn"
            setattr(m, pre + "_w_stride", w.nbytes // 64)
            setattr(m, pre + "_s_stride", 0 if s is None else s.size // 64)
    dr, dx, dres, dout = of(router), of(x), of(res), uocr.DeviceBuffer(P * 2560)
    m.router = dr.ptr
    if static:
        uocr.op_moe_ffn_rows_static(m, dx, None, dres, P, 0, dout)
    else:
        uocr.op_moe_ffn_rows(m, dx, None, dres, P, 0, uocr.moe_rows_workspace(P), dout)
    uocr.sync()
    got = dout.download(np.float16).reshape(P, 1280).astype(np.float64)

    xd = x.astype(np.float64)

    def ffn(xin, g, u, d):
        a = xin @ g.T
        mid = (a / (1 + np.exp(-a)) * (xin @ u.T)).astype(np.float16).astype(np.float64)
        return mid @ d.T, np.abs(mid) @ np.abs(d).T

    y, mag = ffn(xd, val["sgate"], val["sup"], val["sdown"])
    y = y.astype(np.float16).astype(np.float64) + res.astype(np.float64)
    logits = xd[:, :64] * 8
    p = np.exp(logits - logits.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    for e in range(64):
        rows = [t for t in range(P) if e in chosen[t]]
        if rows:
            part = lambda name, n: val[name][(e % 4) * n:(e % 4 + 1) * n]  # noqa: E731
            o, a = ffn(xd[rows], part("gate", 896), part("up", 896), part("down", 1280))
            y[rows] += p[rows, e, None] * o
            mag[rows] += p[rows, e, None] * a
    bound = np.abs(y) * 2.0**-11 + mag * 2.0**-10 + 2.0**-24
    err = np.abs(got - y)
    assert (err <= bound).all(), float((err / bound).max())


@pytest.mark.parametrize("P", [1, 170, 171, 1365, 1366, 4096, 4097])
def test_moe_rows_routing_edges(gpu, P):
    """Row counts at which the bucket build changes its pairs per thread (8 up to
    1,365 rows, 24 up to 4,096, two passes above) and the edges of its batches:
    every row equals its own single-row MoE of the decode operators up to the
    rounding of fp16 (the single-row path rounds the same values)."""
    uocr = gpu
    rng = np.random.default_rng(P)
    of = uocr.DeviceBuffer.of
    m, keep = uocr.CMoeWeights(), []
    m.expert_qtype = m.shared_qtype = 4
    for name, rows, k in (("gate", 64 * 896, 1280), ("up", 64 * 896, 1280), ("down", 64 * 1280, 896), ("sgate", 1792, 1280),
                          ("sup", 1792, 1280), ("sdown", 1280, 1792)):
        w, s = weights_for(4, rng, rows, k)
        keep += [of(w), of(s)]
        setattr(m, name + "_w", keep[-2].ptr)
        setattr(m, name + "_s", keep[-1].ptr)
        if name in ("gate", "down"):
            pre = "gu" if name == "gate" else "dn"
            setattr(m, pre + "_w_stride", w.nbytes // 64)
            setattr(m, pre + "_s_stride", s.size // 64)
    router = of(rand_f16(rng, (64, 1280), 0.03))
    m.router = router.ptr
    x, res = rand_f16(rng, (P, 1280)), rand_f16(rng, (P, 1280))
    dx, dres, dout = of(x), of(res), uocr.DeviceBuffer(P * 2560)
    uocr.op_moe_ffn_rows(m, dx, None, dres, P, 1, uocr.moe_rows_workspace(P), dout)
    uocr.sync()
    got = dout.download(np.float16).reshape(P, 1280).astype(np.float64)
    ws, one, ids, wts = uocr.workspace(), uocr.DeviceBuffer(2560), uocr.DeviceBuffer(64), uocr.DeviceBuffer(64)
    for t in np.unique(np.concatenate([np.arange(min(P, 20)), np.arange(max(0, P - 20), P)])):
        uocr.op_moe_ffn(m, dx.ptr + 2560 * int(t), None, dres.ptr + 2560 * int(t), 1, ws, one, ids, wts)
        uocr.sync()
        ref = one.download(np.float16).astype(np.float64)
        # weights rounded to fp16(q * scale) here and exact there: 2^-11 of each
        # product, which add up like a random walk; 2^-7 of the row's size is
        # over ten times that, a wrong expert or weight is 0.1 and more of it
        size = np.sqrt(np.mean((ref - res[t].astype(np.float64)) ** 2))
        assert np.abs(got[t] - ref).max() <= 2.0**-7 * size + 2.0**-10 * np.abs(ref).max(), int(t)
