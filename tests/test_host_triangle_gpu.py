"""Triangles of products whose operands are streamed from host memory in several chunks of the
reduction (no counterpart in SPLA). Integer inputs: the triangle equals the product bit for
bit, and every other element of C holds either its old value or the whole product, whatever
kernel the short last chunk would take by itself.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import spla_amd as spla
from helpers import OPS, make_buffer, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.complex128], ids=["d", "z"])
@pytest.mark.parametrize("fill", [spla.FillMode.UPPER, spla.FillMode.LOWER])
@pytest.mark.parametrize("pinned", [True, False], ids=["pinned", "pageable"])
def test_chunks_share_their_tiles(device, dtype, fill, pinned):
    dist = spla.MatrixDistribution.create_blacs_block_cyclic(spla.MPI_COMM_SELF, "R", 1, 1, 64, 64)
    ctx = spla.Context(spla.ProcessingUnit.GPU)
    # tiles in front of 16 x 16 ones; the streaming kernel in front of tiles; small ones only
    for m, n, chunk, tail, row, col in [(200, 200, 2048, 500, 0, 0), (190, 170, 4096, 100, 3, 40),
                                        (30, 31, 8192, 300, 0, 0), (100, 90, 448, 65, 0, 5)]:
        k = 2 * chunk + tail
        ctx.set_stream_chunk_bytes(chunk * (m + n) * np.dtype(dtype).itemsize)
        A = make_buffer(97, 1, k, m, k, dtype, "int")
        B = make_buffer(97, 2, k, n, k, dtype, "int")
        ldc = m + row
        C0 = make_buffer(97, 3, ldc, n + col, ldc, dtype, "int")
        hA, hB = torch.from_numpy(A), torch.from_numpy(B)
        if pinned:
            hA, hB = (torch.empty(x.shape, dtype=x.dtype, pin_memory=True).copy_(x)
                      for x in (hA, hB))
        dC = to_device(C0, device)
        spla.pgemm_ssbtr(m, n, k, OPS["C"], 1.0, hA, k, hB, k, 2.0, dC, ldc, row, col, fill, dist,
                         ctx)
        a, b = A.reshape(m, k), B.reshape(n, k)
        old = C0.reshape(n + col, ldc)[col:, row:].T
        new = 2 * old + a.conj() @ b.T
        got = dC.cpu().numpy().reshape(n + col, ldc)[col:, row:].T
        i, j = np.arange(m)[:, None] + row, np.arange(n)[None, :] + col
        need = i <= j if fill == spla.FillMode.UPPER else i >= j
        assert np.array_equal(got[need], new[need]), (m, n, k)
        assert np.all((got == new) | (got == old)), (m, n, k)
