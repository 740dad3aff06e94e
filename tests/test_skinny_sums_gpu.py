"""Rounding of the streaming kernel for small m, n (no counterpart in SPLA).

The shape with one accumulator per output (real, m > 32, n > 16) plans twice the partial
results for a long reduction, so its sums are as long as those of a narrower product of the
same data.
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle
import spla_amd as spla
from helpers import OPS, make_buffer, to_device

pytestmark = pytest.mark.gpu


def test_error_does_not_grow_with_the_outputs(ctx, device):
    """Columns that both products have, against the double-double oracle: the two root mean
    squares over 1024 elements differ by chance by 3 % (one standard deviation); sums twice
    as long would be off by a third more."""
    m, n, narrow, k = 64, 32, 16, 600000
    A = make_buffer(91, 1, k, m, k, np.float64)
    B = make_buffer(91, 2, k, n, k, np.float64)
    ref = np.zeros(m * narrow)
    oracle.gemm(OPS["T"], 0, m, narrow, k, 1.0, A, k, B, k, 0.0, ref, m, accurate=True)
    dA, dB = to_device(A, device), to_device(B, device)
    rms = []
    for cols in (n, narrow):
        dC = to_device(np.zeros(m * cols), device)
        spla.gemm(OPS["T"], 0, m, cols, k, 1.0, dA, k, dB, k, 0.0, dC, m, ctx)
        rms.append(float(np.sqrt(np.mean((dC.cpu().numpy()[:m * narrow] - ref) ** 2))))
    print("rms error:", rms)
    assert rms[0] <= 1.15 * rms[1]
