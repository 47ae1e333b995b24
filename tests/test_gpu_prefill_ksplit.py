"""The prompt's O projection and dense down with K split over blocks (and the
residual and next norm in its reduce) against the unsplit kernels."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_engine import model, prompt

pytestmark = pytest.mark.gpu

# prompts on both sides of the sizes where the split begins and ends
ROWS = {1: (40, 600, 1600, 1601), 2: (384, 385, 1216), 3: (385, 932, 1217)}


@pytest.mark.parametrize("qprofile", [3, 2, 1])
def test_split_k_agrees_with_unsplit(gpu, monkeypatch, qprofile):
    """Only fp32 summation order differs; the hidden state of the last row after
    12 layers that round to fp16 then moves by its rounding noise (up to 7e-3 of
    its norm between the library's own forms of one prompt, 3.1e-2 with an expert
    changed at a near-tie), a wrong plane or row by its whole size."""
    uocr = gpu
    m = model(uocr, qprofile)
    got = {}
    for unsplit in (False, True):
        if unsplit:
            monkeypatch.setenv("UOCR_HIP_NO_PREFILL_KSPLIT", "1")
        eng = uocr.Engine.from_memory(m, backend="hip", max_prompt_tokens=1664, max_gen_tokens=8)
        for P in ROWS[qprofile]:
            ids, mask, rows = prompt(np.random.default_rng(P), 20, P - 20)
            _, score, _, _ = eng.generate_embeddings(ids, mask, rows, 1, flags=uocr.GEN_IGNORE_EOS)
            hidden = eng.trace_read()[1].astype(np.float64)
            if not unsplit:
                got[P] = float(score[0]), hidden
                continue
            a, b = got[P]
            assert np.linalg.norm(hidden - b) <= 5e-2 * np.linalg.norm(b), P
            assert abs(a - float(score[0])) <= 2e-2 + 1e-2 * abs(a), P
        eng.close()
