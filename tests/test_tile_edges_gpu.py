"""Edges of the MFMA tile kernels (no counterpart in SPLA, which calls a vendor BLAS).

The k loop of the tile kernels loads whole 128-byte k-blocks with 32-bit lane
offsets and clamps the rows of ragged tiles; a partial last k-block and leading
dimensions whose rows lie too far apart for 32-bit offsets take code of their
own. Integer inputs small enough for every product and partial sum to be exact
in the type, so the results must equal the oracle bit for bit.
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
LAYOUTS = [("C", "N"), ("T", "C"), ("N", "N"), ("N", "C"), ("C", "C"), ("C", "T")]


def reference(oa, ob, m, n, k, A, lda, B, ldb, C0, ldc, dtype):
    wide = WIDE[dtype]
    ref = C0.astype(wide)
    oracle.gemm(oa, ob, m, n, k, 2.0, A.astype(wide), lda, B.astype(wide), ldb, 3.0, ref, ldc,
                accurate=True)
    return ref.astype(dtype)


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("tile", ["M", "L"])
@pytest.mark.parametrize("opA,opB", LAYOUTS)
def test_ragged_tiles_and_partial_kblocks(ctx, device, dtype, tile, opA, opB, monkeypatch):
    """One row or column more or less than a wave's, a tile's and two tiles' share; k one
    less, equal to and one more than one to five k-blocks of each type (8, 16, 32)."""
    monkeypatch.setenv("SPLA_AMD_TILE", tile)
    oa, ob = OPS[opA], OPS[opB]
    for i, (m, n) in enumerate([(1, 65), (31, 129), (33, 63), (65, 1), (130, 127)]):
        for k in ((1, 9, 33, 64), (7, 16, 31, 97), (8, 17, 40, 65))[i % 3]:
            ra, ca = op_shape(oa, m, k)
            rb, cb = op_shape(ob, k, n)
            lda, ldb, ldc = ra + 1, rb + 3, m + 2
            A = make_buffer(5, 1, ra, ca, lda, dtype, "int")
            B = make_buffer(5, 2, rb, cb, ldb, dtype, "int")
            C0 = make_buffer(5, 3, m, n, ldc, dtype, "int")
            dC = to_device(C0, device)
            spla.gemm(oa, ob, m, n, k, 2.0, to_device(A, device), lda, to_device(B, device), ldb,
                      3.0, dC, ldc, ctx)
            ref = reference(oa, ob, m, n, k, A, lda, B, ldb, C0, ldc, dtype)
            assert np.array_equal(dC.cpu().numpy(), ref), (m, n, k)


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("tile", ["M", "L", "XL"])
@pytest.mark.parametrize("opA,opB", [("C", "N"), ("N", "C")])
def test_rows_further_apart_than_32_bit_offsets(ctx, device, dtype, tile, opA, opB, monkeypatch):
    """Leading dimensions just past 4 GiB / 33 elements of the type, where the kernels switch to
    64-bit lane addresses; only the operand's own entries are ever initialised."""
    import torch

    monkeypatch.setenv("SPLA_AMD_TILE", tile)
    oa, ob = OPS[opA], OPS[opB]
    m, n, k = (35, 33, 41) if opA == "C" else (139, 131, 21)
    ld = (1 << 32) // (33 * np.dtype(dtype).itemsize) + 1
    ra, ca = op_shape(oa, m, k)
    rb, cb = op_shape(ob, k, n)
    A = make_buffer(6, 1, ra, ca, ra, dtype, "int")
    B = make_buffer(6, 2, rb, cb, rb, dtype, "int")
    C0 = make_buffer(6, 3, m, n, m, dtype, "int")
    spread = []
    for X, rows, cols in ((A, ra, ca), (B, rb, cb)):
        x = torch.empty(ld * (cols - 1) + rows, dtype=to_device(X[:1], device).dtype,
                        device=device)
        x.as_strided((cols, rows), (ld, 1)).copy_(to_device(X, device).view(cols, rows))
        spread.append(x)
    dC = to_device(C0, device)
    spla.gemm(oa, ob, m, n, k, 2.0, spread[0], ld, spread[1], ld, 3.0, dC, m, ctx)
    ref = reference(oa, ob, m, n, k, A, ra, B, rb, C0, m, dtype)
    assert np.array_equal(dC.cpu().numpy(), ref)
    del spread
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dtype", [np.float64, np.complex128], ids=["d", "z"])
@pytest.mark.parametrize("opA", [2, 0], ids=["ssb", "sbs"])
def test_batch_rows_further_apart_than_32_bit_offsets(ctx, device, dtype, opA):
    """The same switch in the batched launch, beside a block with ordinary rows."""
    import torch

    cplx = dtype == np.complex128
    opA = 1 if opA == 2 and not cplx else opA
    ld = (1 << 32) // (33 * np.dtype(dtype).itemsize) + 1
    blocks, keep, refs = [], [], []
    for i, (m, n, k, lda) in enumerate([(67, 130, 19, ld), (40, 70, 300, None)]):
        ra, ca = op_shape(opA, m, k)
        A = make_buffer(8, 1 + i, ra, ca, ra, dtype, "int")
        B = make_buffer(8, 3 + i, k, n, k, dtype, "int")
        C0 = make_buffer(8, 5 + i, m, n, m, dtype, "int")
        lda = lda or ra
        dA = torch.empty(lda * (ca - 1) + ra, dtype=to_device(A[:1], device).dtype, device=device)
        dA.as_strided((ca, ra), (lda, 1)).copy_(to_device(A, device).view(ca, ra))
        dB, dC = to_device(B, device), to_device(C0, device)
        keep += [dA, dB]
        refs.append((dC, reference(opA, 0, m, n, k, A, ra, B, k, C0, m, dtype)))
        blocks.append(dict(m=m, n=n, k=k, A=dA, lda=lda, B=dB, ldb=k, C=dC, ldc=m))
    batch = spla.Batch(ctx, blocks, 2.0, 3.0, complex_=cplx, opA=opA)
    batch.execute()
    for dC, ref in refs:
        assert np.array_equal(dC.cpu().numpy(), ref)
    batch.close()
    del keep
    torch.cuda.empty_cache()
