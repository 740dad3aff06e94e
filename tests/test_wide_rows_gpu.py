"""Operands whose rows lie too far apart for 32-bit lane offsets (no counterpart in SPLA), over
reductions long enough for the pipelined k loop, for several tiles in each direction and for
sums in stretches. Integer inputs, so the results must equal the product bit for bit.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import spla_amd as spla
from helpers import OPS, make_buffer, op_shape, to_device, to_matrix

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.complex64, np.float64, np.complex128]


def apply(op, x):
    return x if op == "N" else (x.T if op == "T" else x.conj().T)


def wide_ld(dtype):
    """Just past the leading dimension where 33 rows span 4 GiB."""
    return (1 << 32) // (33 * np.dtype(dtype).itemsize) + 1


def spread(x, rows, cols, ld, device):
    """Packed columns of x, ld apart; nothing else is initialised."""
    out = torch.empty(ld * (cols - 1) + rows, dtype=to_device(x[:1], device).dtype, device=device)
    out.as_strided((cols, rows), (ld, 1)).copy_(to_device(x, device).view(cols, rows))
    return out


def product(ctx, device, dtype, opA, opB, m, n, k, wideA, wideB):
    (ra, ca), (rb, cb) = op_shape(OPS[opA], m, k), op_shape(OPS[opB], k, n)
    A = make_buffer(85, 1, ra, ca, ra, dtype, "int")
    B = make_buffer(85, 2, rb, cb, rb, dtype, "int")
    C0 = make_buffer(85, 3, m, n, m, dtype, "int")
    lda, ldb = (wide_ld(dtype) if wideA else ra), (wide_ld(dtype) if wideB else rb)
    dA, dB = spread(A, ra, ca, lda, device), spread(B, rb, cb, ldb, device)
    dC = to_device(C0, device)
    spla.gemm(OPS[opA], OPS[opB], m, n, k, 2.0, dA, lda, dB, ldb, 3.0, dC, m, ctx)
    wide = np.complex128 if np.iscomplexobj(C0) else np.float64
    ref = 3 * to_matrix(C0, m, n, m).astype(wide) + \
        2 * (apply(opA, to_matrix(A, ra, ca, ra).astype(wide)) @
             apply(opB, to_matrix(B, rb, cb, rb).astype(wide)))
    assert np.array_equal(to_matrix(dC.cpu().numpy(), m, n, m), ref.astype(dtype)), (m, n, k)


@pytest.mark.parametrize("dtype", DTYPES, ids=["s", "c", "d", "z"])
@pytest.mark.parametrize("tile", ["M", "L", "XL"])
@pytest.mark.parametrize("opA,opB,m,n,k", [("C", "N", 140, 131, 301), ("N", "N", 139, 131, 130),
                                           ("T", "C", 67, 161, 97), ("N", "T", 130, 65, 128)])
def test_pipelined_loop(ctx, device, dtype, tile, opA, opB, m, n, k, monkeypatch):
    monkeypatch.setenv("SPLA_AMD_TILE", tile)
    for wideA, wideB in ((True, False), (False, True)):
        product(ctx, device, dtype, opA, opB, m, n, k, wideA, wideB)
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dtype,m,n,k", [(np.complex128, 354, 550, 165), (np.float64, 385, 553, 301)],
                         ids=["z", "d"])
def test_stretches(ctx, device, dtype, m, n, k):
    product(ctx, device, dtype, "C", "N", m, n, k, True, False)
    product(ctx, device, dtype, "N", "N", m, n, k, True, False)
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dtype", [np.float64, np.complex128], ids=["d", "z"])
@pytest.mark.parametrize("opA", "CN")
@pytest.mark.parametrize("persistent", [False, True], ids=["grouped", "persistent"])
def test_batches(ctx, device, dtype, opA, persistent):
    """Blocks of one to several tiles and k-blocks beside one with wide rows, more than enough of
    them for large tiles as well."""
    opA = "T" if opA == "C" and dtype == np.float64 else opA
    specs, keep, want = [], [], []
    sizes = [(130, 161, 100)] + [(150 + 9 * i, 270 - 3 * i, 700 + 11 * i) for i in range(60)]
    for i, (m, n, k) in enumerate(sizes):
        ra, ca = op_shape(OPS[opA], m, k)
        A = make_buffer(86 + i, 1, ra, ca, ra, dtype, "int")
        B = make_buffer(86 + i, 2, k, n, k, dtype, "int")
        lda = wide_ld(dtype) if i == 0 else ra
        dA, dB = spread(A, ra, ca, lda, device), to_device(B, device)
        dC = to_device(np.zeros(m * n, dtype=dtype), device)
        keep.append((dA, dB, dC))
        specs.append(dict(m=m, n=n, k=k, A=dA, lda=lda, B=dB, ldb=k, C=dC, ldc=m))
        want.append(apply(opA, to_matrix(A, ra, ca, ra)) @ to_matrix(B, k, n, k))
    batch = spla.Batch(ctx, specs, 1.0, 0.0, complex_=dtype == np.complex128, opA=OPS[opA],
                       persistent=persistent)
    assert batch.info()["persistent"] == persistent
    batch.execute()
    for (m, n, k), (_, _, dC), ref in zip(sizes, keep, want):
        assert np.array_equal(to_matrix(dC.cpu().numpy(), m, n, m), ref), (m, n, k)
    batch.close()
    del keep, specs
    torch.cuda.empty_cache()


def test_measuring_leaves_the_context_alone(device):
    """A batch with wide rows that measures its candidates does not decide how the context runs
    ordinary batches: their plans are the same as without it."""
    def ordinary(ctx):
        x = torch.zeros(500 * 300, dtype=torch.float64, device=device)
        c = torch.zeros(300 * 300, dtype=torch.float64, device=device)
        specs = [dict(m=300, n=290 - i, k=500, A=x, lda=500, B=x, ldb=500, C=c, ldc=300)
                 for i in range(40)]
        batch = spla.Batch(ctx, specs, 1.0, 0.0, complex_=False, opA=OPS["T"])
        info = batch.info()
        batch.close()
        return info

    contexts = [spla.Context(spla.ProcessingUnit.GPU) for _ in range(2)]
    ld = wide_ld(np.float64)
    x = torch.zeros(ld * 15 + 400, dtype=torch.float64, device=device)
    c = torch.zeros(256, dtype=torch.float64, device=device)
    specs = [dict(m=16, n=16, k=400, A=x, lda=ld, B=x, ldb=400, C=c, ldc=16)]
    measured = spla.Batch(contexts[1], specs, 1.0, 0.0, complex_=False, opA=OPS["T"],
                          measure=True)
    measured.close()
    assert ordinary(contexts[0]) == ordinary(contexts[1])
