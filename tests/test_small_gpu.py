"""Products of the small-product kernel (no counterpart in SPLA, which calls a vendor BLAS).

Sizes around its 16 x 16 tiles, its MFMA steps (4, 8 or 16 reduction indices), the 32
indices that a wave loads together, its 16 waves and the largest products that take it.
Integer inputs small enough for every product and partial sum to be exact in the type,
so the results must equal the oracle bit for bit.
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle
import spla_amd as spla
from helpers import OPS, make_buffer, op_shape, to_device

pytestmark = pytest.mark.gpu

WIDE = {np.float32: np.float64, np.complex64: np.complex128, np.float64: np.float64,
        np.complex128: np.complex128}
DTYPES = list(WIDE)
IDS = ["s", "c", "d", "z"]
# (m, n, k); the last of every row is the largest its type takes for the kernel, or just past it
SIZES = [(1, 1, 1), (1, 17, 3), (16, 16, 4), (17, 1, 5), (15, 33, 16), (31, 2, 31), (16, 48, 32),
         (3, 16, 33), (33, 17, 63), (13, 32, 263), (5, 5, 511), (17, 16, 512), (4, 4, 513),
         (2, 3, 1024), (1, 1, 1025), (3, 1, 2048), (2, 2, 2049)]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("opA", "NTC")
@pytest.mark.parametrize("opB", "NTC")
def test_small_products_exact(ctx, device, dtype, opA, opB):
    oa, ob = OPS[opA], OPS[opB]
    for m, n, k in SIZES:
        ra, ca = op_shape(oa, m, k)
        rb, cb = op_shape(ob, k, n)
        lda, ldb, ldc = ra + 1, rb + 3, m + 2
        A = make_buffer(51, 1, ra, ca, lda, dtype, "int")
        B = make_buffer(51, 2, rb, cb, ldb, dtype, "int")
        C0 = make_buffer(51, 3, m, n, ldc, dtype, "int")
        for beta in (3.0, 0.0):
            dC = to_device(C0 if beta else np.full_like(C0, np.nan), device)
            spla.gemm(oa, ob, m, n, k, 2.0, to_device(A, device), lda, to_device(B, device), ldb,
                      beta, dC, ldc, ctx)
            wide = WIDE[dtype]
            ref = C0.astype(wide)
            oracle.gemm(oa, ob, m, n, k, 2.0, A.astype(wide), lda, B.astype(wide), ldb, beta, ref,
                        ldc, accurate=True)
            got = dC.cpu().numpy().reshape(n, ldc)[:, :m]
            assert np.array_equal(got, ref.astype(dtype).reshape(n, ldc)[:, :m]), (m, n, k, beta)


@pytest.mark.parametrize("opA,opB", [("T", "N"), ("N", "C")])
def test_reduction_padding_is_not_used(ctx, device, opA, opB):
    """NaN behind the reduction's last index (K-major rows, MN-major columns)."""
    m, n, k = 7, 19, 37
    ra, ca = op_shape(OPS[opA], m, k + 9)
    rb, cb = op_shape(OPS[opB], k + 9, n)
    A = make_buffer(52, 1, ra, ca, ra, np.complex128, "int").reshape(ca, ra)
    B = make_buffer(52, 2, rb, cb, rb, np.complex128, "int").reshape(cb, rb)
    (A[k:] if opA == "N" else A[:, k:])[...] = np.nan
    (B[k:] if opB != "N" else B[:, k:])[...] = np.nan
    dC = to_device(np.zeros(m * n, dtype=np.complex128), device)
    spla.gemm(OPS[opA], OPS[opB], m, n, k, 1.0, to_device(A.reshape(-1), device), ra,
              to_device(B.reshape(-1), device), rb, 0.0, dC, m, ctx)
    a = A[:k].T if opA == "N" else A[:, :k]
    b = B[:k].conj() if opB == "C" else B[:, :k].T
    assert np.array_equal(dC.cpu().numpy().reshape(n, m).T, a @ b)
    assert np.isfinite(dC.cpu().numpy()).all()


@pytest.mark.parametrize("dtype", [np.float64, np.complex128], ids=["d", "z"])
@pytest.mark.parametrize("fill", [spla.FillMode.UPPER, spla.FillMode.LOWER])
def test_small_triangle(ctx, device, dtype, fill):
    """One triangle of a small C inside a larger matrix: that triangle equals the oracle's."""
    m, k, row, col = 45, 40, 3, 1
    ldc = m + row + 4
    dist = spla.MatrixDistribution.create_blacs_block_cyclic(spla.MPI_COMM_SELF, "R", 1, 1, 16, 16)
    A = make_buffer(53, 1, k, m, k, dtype, "int")
    B = make_buffer(53, 2, k, m, k, dtype, "int")
    C0 = make_buffer(53, 3, ldc, m + col, ldc, dtype, "int")
    dC = to_device(C0, device)
    spla.pgemm_ssbtr(m, m, k, OPS["C"], 1.0, to_device(A, device), k, to_device(B, device), k, 2.0,
                     dC, ldc, row, col, fill, dist, ctx)
    full = 2.0 * C0.reshape(m + col, ldc)[col:, row:row + m].T + \
        A.reshape(m, k).conj() @ B.reshape(m, k).T
    got = dC.cpu().numpy().reshape(m + col, ldc)[col:, row:row + m].T
    i, j = np.meshgrid(np.arange(m) + row, np.arange(m) + col, indexing="ij")
    keep = (i <= j) if fill == spla.FillMode.UPPER else (i >= j)
    assert np.array_equal(got[keep], full[keep])
