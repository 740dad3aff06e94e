"""Products whose splits add up sums of a bounded length (no counterpart in SPLA): the tiles'
accumulators are added to totals every few k-blocks, so that a plan with fewer splits rounds
no worse than one with more (tests/test_plan_sums_host.py holds the shapes to that kernel).
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle
import spla_amd as spla
from helpers import OPS, make_buffer, op_shape, to_device, to_matrix

pytestmark = pytest.mark.gpu

SHAPES = {np.complex128: [(354, 550, 165), (330, 300, 2100)],
          np.float64: [(385, 553, 301), (400, 300, 4000)]}


def apply(op, x):
    return x if op == "N" else (x.T if op == "T" else x.conj().T)


@pytest.mark.parametrize("dtype", list(SHAPES), ids=["z", "d"])
@pytest.mark.parametrize("opA", "NTC")
@pytest.mark.parametrize("opB", "NTC")
def test_exact(ctx, device, dtype, opA, opB):
    """Integers: bit for bit, in one split and in several, a partial stretch at the end."""
    for m, n, k in SHAPES[dtype]:
        (ra, ca), (rb, cb) = op_shape(OPS[opA], m, k), op_shape(OPS[opB], k, n)
        lda, ldb, ldc = ra + 1, rb + 3, m + 2
        A = make_buffer(81, 1, ra, ca, lda, dtype, "int")
        B = make_buffer(81, 2, rb, cb, ldb, dtype, "int")
        C0 = make_buffer(81, 3, m, n, ldc, dtype, "int")
        dC = to_device(C0, device)
        spla.gemm(OPS[opA], OPS[opB], m, n, k, 2.0, to_device(A, device), lda,
                  to_device(B, device), ldb, 3.0, dC, ldc, ctx)
        ref = 3 * to_matrix(C0, m, n, ldc) + 2 * (apply(opA, to_matrix(A, ra, ca, lda)) @
                                                  apply(opB, to_matrix(B, rb, cb, ldb)))
        assert np.array_equal(to_matrix(dC.cpu().numpy(), m, n, ldc), ref), (m, n, k)


@pytest.mark.parametrize("m,n,k,dtype,splits", [(534, 597, 1523, np.complex128, 11),
                                                (801, 590, 3905, np.float64, 14)],
                         ids=["z", "d"])
def test_error_of_many_splits(device, m, n, k, dtype, splits, monkeypatch):
    """Against the double-double oracle, the planned product is no further off than the same
    product forced into as many splits of that length (root mean square over 3e5 elements: the
    two differ by chance by under 1 %, one long sum is off by more than half as much again)."""
    op = "C" if dtype == np.complex128 else "T"
    A = make_buffer(82, 1, k, m, k, dtype)
    B = make_buffer(82, 2, k, n, k, dtype)
    ref = np.zeros(m * n, dtype=dtype)
    oracle.gemm(OPS[op], 0, m, n, k, 1.0, A, k, B, k, 0.0, ref, m, accurate=True)
    dA, dB = to_device(A, device), to_device(B, device)
    rms = []
    for forced in (None, str(splits)):
        if forced:
            monkeypatch.setenv("SPLA_AMD_SPLITS", forced)
        ctx = spla.Context(spla.ProcessingUnit.GPU)
        ctx.set_gemm_mode(spla.GemmMode.FP64)
        dC = to_device(np.zeros(m * n, dtype=dtype), device)
        spla.gemm(OPS[op], 0, m, n, k, 1.0, dA, k, dB, k, 0.0, dC, m, ctx)
        rms.append(float(np.sqrt(np.mean(np.abs(dC.cpu().numpy() - ref) ** 2))))
    print("rms error planned, forced:", rms)
    assert rms[0] <= 1.05 * rms[1]
