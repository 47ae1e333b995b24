"""Which kernel a plain GEMM takes: both sides of every line of the rule, with
the sizes that were measured for it."""
from __future__ import annotations

import pytest

F16, Q8, Q4 = 1, 3, 4
NONE, QUICK, ERF = 0, 1, 2

# qtype, m, n, k, kernel
PLAIN = [
    (Q8, 4001, 6848, 1280, "large"), (Q4, 2000, 1280, 6848, "mid"), (F16, 2400, 1280, 6848, "mid"), (Q8, 3300, 1280, 6848, "large"),
    (Q8, 3264, 1280, 6848, "mid"), (Q8, 1664, 1280, 6848, "mid"), (Q8, 1600, 1280, 6848, "mid_k4"), (Q4, 932, 1280, 6848, "mid_k4"),
    (F16, 500, 1280, 6848, "mid_k4"), (Q4, 500, 1280, 6848, "mid_k4"), (Q4, 384, 1280, 6848, "narrow"), (F16, 2, 1280, 6848, "narrow"),
    (Q4, 932, 1280, 1280, "mid"), (Q8, 500, 1280, 1280, "mid"), (F16, 400, 1280, 1280, "mid"), (Q4, 500, 1280, 1280, "lines"),
    (Q4, 640, 1280, 1280, "mid"), (Q8, 384, 1280, 1280, "lines"), (F16, 384, 1280, 1280, "narrow"), (F16, 257, 1280, 1024, "lines"),
    (Q4, 3264, 1280, 1280, "mid"), (Q4, 3265, 1280, 1280, "general"), (Q4, 4864, 1280, 6848, "general"), (Q4, 4865, 1280, 1280, "large"),
    (Q8, 3265, 1280, 1280, "large"), (F16, 3265, 1280, 1280, "large"), (Q4, 33, 1280, 1792, "lines"), (Q4, 70, 132, 192, "general"),
]
# qtype, m, n, k, act, kernel
VISION = [
    (Q8, 4096, 3072, 768, ERF, "large"), (Q4, 4096, 3072, 768, ERF, "large"), (Q4, 1600, 3072, 768, ERF, "general"), (Q4, 1176, 3072, 768, ERF, "general"),
    (Q8, 1600, 3072, 768, ERF, "large"), (Q8, 1176, 3072, 768, ERF, "mid"), (Q4, 1600, 3072, 768, NONE, "large"), (Q4, 588, 3072, 768, ERF, "mid"),
    (Q4, 1028, 4096, 1024, QUICK, "general"), (Q4, 1960, 2304, 768, NONE, "large"), (Q4, 1960, 768, 768, NONE, "mid"), (Q8, 392, 3072, 768, ERF, "mid"),
    (Q4, 784, 768, 768, NONE, "lines"), (Q8, 784, 768, 768, NONE, "mid"),
    (Q4, 101, 1024, 4096, NONE, "general"), (F16, 101, 1024, 4096, NONE, "general"), (Q4, 200, 1024, 4096, NONE, "general"),
    (Q8, 200, 1024, 4096, NONE, "narrow"), (Q4, 257, 1024, 4096, NONE, "narrow"), (F16, 257, 1024, 4096, NONE, "narrow"),
    (Q4, 514, 1024, 4096, NONE, "general"), (Q8, 514, 1024, 4096, NONE, "general"), (F16, 514, 1024, 4096, NONE, "mid_k4"),
    (Q4, 771, 1024, 4096, NONE, "mid_k4"), (F16, 2313, 1024, 4096, NONE, "mid"), (F16, 200, 1280, 2048, NONE, "narrow"),
]


@pytest.fixture(scope="module")
def kernel_of():
    import uocr
    return uocr.op_gemm_kernel


@pytest.mark.parametrize("qtype,m,n,k,kernel", PLAIN)
def test_plain(kernel_of, qtype, m, n, k, kernel):
    assert kernel_of(qtype, m, n, k) == kernel


@pytest.mark.parametrize("qtype,m,n,k,act,kernel", VISION)
def test_vision(kernel_of, qtype, m, n, k, act, kernel):
    assert kernel_of(qtype, m, n, k, True, act) == kernel


def test_bad_arguments(kernel_of):
    for args in ((2, 4, 128, 128), (Q4, 0, 128, 128), (Q4, 4, 128, 100), (Q4, 4, 128, 128, True, 3)):
        with pytest.raises(ValueError):
            kernel_of(*args)


def test_value_tests_reach_every_kernel(kernel_of):
    """The shapes of the value tests are on the kernels that their comments name."""
    import test_gpu_gemm_tiles as t
    rest = ["mid", "mid", "mid_k4", "narrow", "narrow", "lines", "lines", "lines", "lines", "large", "large"]
    for q in (F16, Q8, Q4):
        assert [kernel_of(q, *s) for s in t.SHAPES] == (["general"] * 2 if q == Q4 else ["large"] * 2) + rest
        for m, n, k, act, _, kernel in t.VISION_SHAPES:
            assert kernel_of(q, m, n, k, True, act) == kernel
