"""The prompt's expert choice: router logits, top-6 ids and the pair lists of
the bucketed MoE, read from the operator's workspace for every row."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rand_f16, weights_for

pytestmark = pytest.mark.gpu


def workspace_views(buf, P):
    """(logits [P][64], ids [P][6], list_tok, list_pair) of a workspace after a
    call: pieces of 256 bytes in the order of the operator's layout."""
    raw = buf.download(np.uint8)
    tiles = (6 * P + 63) // 64 + 64
    at, off = {}, 0
    for name, nbytes in (("xn", 2560 * P), ("logits", 256 * P), ("ids", 24 * P), ("wts", 24 * P), ("offsets", 256), ("te", 4 * tiles),
                         ("ts0", 4 * tiles), ("ts1", 4 * tiles), ("nt", 4), ("tok", 24 * P), ("pair", 24 * P)):
        at[name] = raw[off:off + nbytes]
        off += (nbytes + 255) // 256 * 256
    return at["logits"].view(np.float32).reshape(P, 64), at["ids"].view(np.int32).reshape(P, 6), at["tok"].view(np.int32), at["pair"].view(np.int32)


class Layer:
    """A MoE layer of 64 identical experts; the choice is what is looked at."""

    def __init__(self, uocr, rng, router, shared_offset=0):
        """shared_offset: bytes by which the shared experts' payloads miss a 16-byte boundary."""
        self.uocr, self.m, self.keep = uocr, uocr.CMoeWeights(), []
        self.m.expert_qtype = self.m.shared_qtype = 4
        for name, rows, k in (("gate", 896, 1280), ("up", 896, 1280), ("down", 1280, 896), ("sgate", 1792, 1280), ("sup", 1792, 1280),
                              ("sdown", 1280, 1792)):
            w, s = weights_for(4, rng, rows, k)
            pad = np.zeros(shared_offset if name[0] == "s" else 0, np.uint8)
            self.keep += [uocr.DeviceBuffer.of(np.concatenate([pad, w.view(np.uint8).ravel()])), uocr.DeviceBuffer.of(s)]
            setattr(self.m, name + "_w", self.keep[-2].ptr + pad.size)
            setattr(self.m, name + "_s", self.keep[-1].ptr)
        # strides of 0: every expert reads the same weights
        self.keep.append(uocr.DeviceBuffer.of(router))
        self.m.router = self.keep[-1].ptr

    def choose(self, x):
        uocr, P = self.uocr, x.shape[0]
        of, ws, out = uocr.DeviceBuffer.of, uocr.moe_rows_workspace(P), uocr.DeviceBuffer(2560 * P)
        dx, dres = of(x), of(np.zeros((P, 1280), np.float16))
        uocr.op_moe_ffn_rows(self.m, dx, None, dres, P, 0, ws, out)
        uocr.sync()
        return workspace_views(ws, P)


@pytest.mark.parametrize("shared_offset", [0, 8])
@pytest.mark.parametrize("P", [1, 31, 33, 65, 200])
def test_router_logits_are_one_ordered_sum(gpu, P, shared_offset):
    """2^24 first, fifteen products of 1 spread over K, -2^24 last: an fp32 sum
    in ascending K loses every 1 and ends at 0 (2^24 + 1 rounds to 2^24), a sum
    in parts keeps some of them.  Six experts have that logit, six the plain
    logit 3, the others -48 and less.  Off a 16-byte boundary the router is a
    launch of its own."""
    rng = np.random.default_rng(P)
    x, router = np.zeros((P, 1280), np.float16), np.zeros((64, 1280), np.float16)
    parts, plain = rng.permutation(64)[:12].reshape(2, 6)
    steps = 64 * np.arange(3, 18)
    x[:, 0], x[:, 1279], x[:, steps], x[:, 1] = 4096, 4096, 1, 3
    router[:, 1] = -16
    router[plain, 1] = 1
    router[parts, 1] = 0
    router[parts, 0], router[parts, 1279] = 4096, -4096
    router[np.ix_(parts, steps)] = 1
    logits, ids, _, _ = Layer(gpu, rng, router, shared_offset).choose(x)
    assert (logits[:, parts] == 0).all() and (logits[:, plain] == 3).all()
    assert (np.sort(ids, 1) == np.sort(plain)).all()


@pytest.mark.parametrize("P", [1, 6, 7, 64, 932, 1366, 4001, 4097])
def test_every_pair_is_routed_once(gpu, P):
    """The slot lists hold each (token, rank) pair once, grouped by expert, and
    the ids are the six largest float64 logits wherever the 6th and 7th lie
    further apart than the fp32 sums can err: 1,280 additions of 2^-24 of the
    magnitudes, on both sides."""
    rng = np.random.default_rng(P)
    router, x = rand_f16(rng, (64, 1280), 0.03), rand_f16(rng, (P, 1280))
    logits, ids, tok, pair = Layer(gpu, rng, router).choose(x)
    assert (np.sort(pair) == np.arange(6 * P)).all() and (tok == pair // 6).all()
    assert (np.diff(ids.ravel()[pair]) >= 0).all()
    ref = x.astype(np.float64) @ router.astype(np.float64).T
    err = (np.abs(x.astype(np.float64)) @ np.abs(router.astype(np.float64)).T) * 1280 * 2.0**-24
    assert (np.abs(logits - ref) <= err).all()
    order = np.argsort(-ref, 1)
    gap = np.take_along_axis(ref, order, 1)
    sure = gap[:, 5] - gap[:, 6] > 2 * err.max(1)
    assert sure.mean() > 0.9 or P < 64
    assert (np.sort(ids, 1)[sure] == np.sort(order[:, :6], 1)[sure]).all()
