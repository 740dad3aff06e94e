"""Half tiles and fill modes of the tile kernels (no counterpart in SPLA).

Tiles of which at most half the columns exist or are needed run as half tiles, and only
the tiles that a fill mode needs are launched. Integer inputs, so the triangle must equal
the oracle bit for bit; the rest of C must hold either its old or its computed value.
"""

from __future__ import annotations

import numpy as np
import pytest

import spla_amd as spla
from helpers import OPS, make_buffer, to_device

pytestmark = pytest.mark.gpu

TYPES = [np.float64, np.complex128, np.float32, np.complex64]
IDS = ["d", "z", "s", "c"]


@pytest.mark.parametrize("dtype", TYPES, ids=IDS)
@pytest.mark.parametrize("tile", ["M", "L", "XL"])
@pytest.mark.parametrize("splits", ["1", "3"])
@pytest.mark.parametrize("fill", [spla.FillMode.UPPER, spla.FillMode.LOWER, spla.FillMode.FULL])
def test_triangles_at_offsets(ctx, device, dtype, tile, splits, fill, monkeypatch):
    monkeypatch.setenv("SPLA_AMD_TILE", tile)
    monkeypatch.setenv("SPLA_AMD_SPLITS", splits)
    dist = spla.MatrixDistribution.create_blacs_block_cyclic(spla.MPI_COMM_SELF, "R", 1, 1, 64, 64)
    # (m, n, row, col): half and whole last tiles, the diagonal through halves, beside C
    for m, n, row, col in [(130, 130, 0, 0), (97, 161, 2, 2), (200, 33, 40, 0), (65, 190, 0, 37),
                           (60, 96, 300, 0), (60, 96, 0, 300), (64, 129, 64, 0)]:
        k, ldc = 800, m + row + 1
        A = make_buffer(61, 1, k, m, k, dtype, "int")
        B = make_buffer(61, 2, k, n, k, dtype, "int")
        C0 = make_buffer(61, 3, ldc, n + col, ldc, dtype, "int")
        dC = to_device(C0, device)
        args = (m, n, k, OPS["C"], 1.0, to_device(A, device), k, to_device(B, device), k, 2.0, dC,
                ldc, row, col)
        if fill == spla.FillMode.FULL:
            spla.pgemm_ssb(*args, dist, ctx)
        else:
            spla.pgemm_ssbtr(*args, fill, dist, ctx)
        old = C0.reshape(n + col, ldc)[col:, row:row + m].T
        a, b = A.reshape(m, k), B.reshape(n, k)
        new = (2 * old.astype(np.complex128) +
               a.astype(np.complex128).conj() @ b.astype(np.complex128).T)
        new = (new if np.iscomplexobj(C0) else new.real).astype(dtype)
        got = dC.cpu().numpy().reshape(n + col, ldc)[col:, row:row + m].T
        i, j = np.meshgrid(np.arange(m) + row, np.arange(n) + col, indexing="ij")
        need = {spla.FillMode.UPPER: i <= j, spla.FillMode.LOWER: i >= j}.get(fill, i >= 0)
        assert np.array_equal(got[need], new[need]), (m, n, row, col)
        assert np.all((got == new) | (got == old)), (m, n, row, col)


@pytest.mark.parametrize("type_", ["d", "z"])
@pytest.mark.parametrize("opA", ["C", "N"])
def test_batched_half_tiles(ctx, device, type_, opA):
    """Blocks whose last tile has one column, half of its columns and one more."""
    dtype = np.complex128 if type_ == "z" else np.float64
    keep, specs, want = [], [], []
    for i, n in enumerate([1, 31, 32, 33, 63, 64, 65, 96, 97, 160, 161]):
        m, k = 20 + 7 * i, 600 + i
        rows = m if opA == "N" else k
        A = make_buffer(62 + i, 1, rows, m + k - rows, rows, dtype, "int")
        B = make_buffer(62 + i, 2, k, n, k, dtype, "int")
        dA, dB = to_device(A, device), to_device(B, device)
        dC = to_device(np.zeros(m * n, dtype=dtype), device)
        keep.append((dA, dB, dC))
        specs.append(dict(m=m, n=n, k=k, A=dA.data_ptr(), lda=rows, B=dB.data_ptr(), ldb=k,
                          C=dC.data_ptr(), ldc=m))
        a = A.reshape(m + k - rows, rows)
        want.append((a.T if opA == "N" else a.conj()) @ B.reshape(n, k).T)
    batch = spla.Batch(ctx, specs, 1.0, 0.0, complex_=type_ == "z", opA=OPS[opA])
    batch.execute()
    for (_, _, dC), w in zip(keep, want):
        assert np.array_equal(dC.cpu().numpy().reshape(w.shape[1], w.shape[0]).T, w), w.shape
