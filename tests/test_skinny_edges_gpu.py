"""Edges of the streaming kernel for small m, n (no counterpart in SPLA).

The kernel reads the reduction in chunks of 128 bytes of a row, times the number
of stretches that small outputs put side by side, and leaves the partial chunk at
the end to one wave. Integer inputs small enough for every product and partial sum
to be exact, so the results must equal the oracle bit for bit.
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle
import spla_amd as spla
from helpers import OPS, make_buffer, to_device

pytestmark = pytest.mark.gpu

# (m, n): the smallest and largest of every number of stretches and of fragments
SHAPES = {np.complex128: [(1, 1), (2, 1), (2, 2), (3, 4), (1, 5), (8, 8), (9, 2), (16, 16), (1, 17),
                          (16, 32), (17, 1), (32, 16), (32, 32)],
          np.float64: [(1, 1), (2, 2), (4, 3), (8, 5), (16, 16), (3, 32), (17, 16), (32, 32),
                       (33, 1), (64, 17)]}


@pytest.mark.parametrize("dtype", [np.complex128, np.float64], ids=["z", "d"])
@pytest.mark.parametrize("op", ["T", "C"])
def test_chunk_edges(ctx, device, dtype, op):
    """From the shortest reduction that takes the kernel: whole chunks, one element more or
    less, and odd leading dimensions (16-byte loads at 8-byte addresses)."""
    comps = 2 if dtype == np.complex128 else 1
    shortest = 8192 // comps
    for i, (m, n) in enumerate(SHAPES[dtype]):
        for k in (shortest, shortest + 1, shortest + 129 * (i + 1), 3 * shortest - 1):
            lda, ldb, ldc = k + 1 + i % 2, k + 3, m + 1
            A = make_buffer(31, 1, k, m, lda, dtype, "int")
            B = make_buffer(31, 2, k, n, ldb, dtype, "int")
            C0 = make_buffer(31, 3, m, n, ldc, dtype, "int")
            dC = to_device(C0, device)
            spla.gemm(OPS[op], OPS["N"], m, n, k, 2.0, to_device(A, device), lda,
                      to_device(B, device), ldb, 3.0, dC, ldc, ctx)
            oracle.gemm(OPS[op], OPS["N"], m, n, k, 2.0, A, lda, B, ldb, 3.0, C0, ldc,
                        accurate=True)
            assert np.array_equal(dC.cpu().numpy(), C0), (m, n, k)


@pytest.mark.parametrize("k", [8192, 300000])
def test_values_past_the_reduction_are_not_used(ctx, device, k):
    """NaN behind the last reduction index of every row of A and B."""
    m, n, k = 5, 7, k + 3
    A = make_buffer(32, 1, k, m, k + 13, np.complex128, "int").reshape(m, k + 13)
    B = make_buffer(32, 2, k, n, k + 13, np.complex128, "int").reshape(n, k + 13)
    A[:, k:] = np.nan
    B[:, k:] = np.nan
    dC = to_device(np.zeros(m * n, dtype=np.complex128), device)
    spla.gemm(OPS["C"], OPS["N"], m, n, k, 1.0, to_device(A.reshape(-1), device), k + 13,
              to_device(B.reshape(-1), device), k + 13, 0.0, dC, m, ctx)
    ref = A[:, :k].conj() @ B[:, :k].T
    assert np.array_equal(dC.cpu().numpy().reshape(n, m).T, ref)
