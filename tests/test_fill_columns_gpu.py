"""Fill modes over hundreds of tile columns (no counterpart in SPLA): wide and square
triangles whose workgroups look their tile up among all columns. Integer inputs, so the
triangle must equal the product bit for bit; the rest of C holds its old or its computed value.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import spla_amd as spla
from helpers import OPS, make_buffer, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.complex64], ids=["d", "c"])
@pytest.mark.parametrize("fill", [spla.FillMode.UPPER, spla.FillMode.LOWER])
def test_many_tile_columns(ctx, device, dtype, fill):
    dist = spla.MatrixDistribution.create_blacs_block_cyclic(spla.MPI_COMM_SELF, "R", 1, 1, 64, 64)
    for m, n, k, row, col in [(70, 40001, 33, 0, 0), (70, 40001, 33, 30000, 3),
                              (3001, 2987, 600, 5, 0)]:
        ldc = m + row
        A = make_buffer(71, 1, k, m, k, dtype, "int")
        B = make_buffer(71, 2, k, n, k, dtype, "int")
        C0 = make_buffer(71, 3, m, n, m, dtype, "int").reshape(n, m)
        # only the product's own part of the larger C is initialised
        dC = torch.empty((n + col) * ldc, dtype=to_device(C0[:1], device).dtype, device=device)
        view = dC.view(n + col, ldc)[col:, row:row + m]
        view.copy_(to_device(C0, device))
        spla.pgemm_ssbtr(m, n, k, OPS["C"], 1.0, to_device(A, device), k, to_device(B, device), k,
                         2.0, dC, ldc, row, col, fill, dist, ctx)
        got = view.cpu().numpy().T
        a, b = (x.astype(np.complex128) for x in (A.reshape(m, k), B.reshape(n, k)))
        new = 2 * C0.T.astype(np.complex128) + a.conj() @ b.T
        new = (new if np.iscomplexobj(C0) else new.real).astype(dtype)
        i, j = np.arange(m)[:, None] + row, np.arange(n)[None, :] + col
        need = i <= j if fill == spla.FillMode.UPPER else i >= j
        assert np.array_equal(got[need], new[need]), (m, n, row, col)
        assert np.all((got == new) | (got == C0.T)), (m, n, row, col)
