"""Causal prefill attention at the edges of its query and key tiles.

The prompt lengths sit on both sides of every size at which the kernel's tiling
or its choice of tiles changes: one query, a full and a started 32-key tile, the
last length of each query tile shape and the first of the next.  The reference
is float64; the bound is the rounding of each probability to fp16 (2^-11
relative, each weighing |v|), of the output (2^-11), and 2^-13 of that sum for
the fp32 scores and sums (scores below 32 in magnitude, exp2 to 2 ulp)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rand_f16

pytestmark = pytest.mark.gpu


def reference(q, kc, vc, rows):
    """(context, sum of p |v|) of the query rows, float64 [rows][1280]."""
    out, mag = [], []
    for i in rows:
        o, a = [], []
        for h in range(10):
            k, v = kc[h, :i + 1].astype(np.float64), vc[h, :i + 1].astype(np.float64)
            s = k @ q[i, 128 * h:128 * h + 128].astype(np.float64) / np.sqrt(128.0)
            p = np.exp(s - s.max())
            p /= p.sum()
            o.append(p @ v)
            a.append(p @ np.abs(v))
        out.append(np.concatenate(o))
        mag.append(np.concatenate(a))
    return np.array(out), np.array(mag)


@pytest.mark.parametrize("P,offset", [(P, 0) for P in (1, 31, 32, 33, 64, 65, 127, 129, 255, 256, 257, 319, 700, 3300, 3301)] +
                         [(P, 4) for P in (1, 33, 256, 257, 3301)])
def test_prefill_attention_tile_edges(gpu, P, offset):
    """offset 4: cache pointers 8 bytes off a 16-byte boundary."""
    uocr = gpu
    rng = np.random.default_rng(P)
    cap = P + 5
    kc, vc, q = rand_f16(rng, (10, cap, 128)), rand_f16(rng, (10, cap, 128)), rand_f16(rng, (P, 1280), 1.5)
    # growing keys: the running maximum keeps moving; slots past the prompt hold NaN
    kc *= np.linspace(0.2, 1.5, cap, dtype=np.float16)[None, :, None]
    kc[:, P:], vc[:, P:] = np.nan, np.nan
    dk, dv = (uocr.DeviceBuffer(x.nbytes + 16) for x in (kc, vc))
    pad = np.zeros(offset, np.float16)
    dk.upload(np.concatenate([pad, kc.ravel()]))
    dv.upload(np.concatenate([pad, vc.ravel()]))
    dq, dctx = uocr.DeviceBuffer.of(q), uocr.DeviceBuffer.of(np.full((P, 1280), 9, np.float16))
    uocr.op_prefill_attention(dq, dk.ptr + 2 * offset, dv.ptr + 2 * offset, cap, P, dctx)
    uocr.sync()
    got = dctx.download(np.float16).reshape(P, 1280).astype(np.float64)
    rows = np.unique(np.concatenate([np.arange(min(P, 34)), np.arange(max(0, P - 34), P), rng.integers(0, P, 8)]))
    ref, mag = reference(q, kc, vc, rows)
    bound = (mag * (1 + 2.0**-2) + np.abs(ref)) * 2.0**-11 + 2.0**-24
    err = np.abs(got[rows] - ref)
    assert (err <= bound).all(), float((err / bound).max())
