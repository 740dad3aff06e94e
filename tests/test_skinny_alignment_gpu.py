"""The streaming kernel for small m, n on operands that start and step on cache lines and on
operands that do not (no counterpart in SPLA).

How the operands lie in memory decides how they are loaded, not which sums an element goes
to: a product of the same numbers has the same bits. Every number of fragments and of
stretches side by side, reductions on and off the edges of a turn.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
import spla_amd as spla
from helpers import OPS, make_buffer, to_device

pytestmark = pytest.mark.gpu

# (m, n): stretches 16, 8, 4, 2, 1 and every pair of fragment counts
SHAPES = {np.complex128: [(1, 1), (2, 2), (4, 3), (8, 5), (16, 16), (9, 12), (16, 17), (17, 16),
                          (32, 32)],
          np.float64: [(1, 1), (2, 1), (3, 4), (7, 8), (16, 16), (11, 9), (16, 32), (32, 3),
                       (30, 31), (64, 16), (64, 32)]}


def place(x, device, ld, offset):
    """Rows of x at `offset` elements into a buffer, ld apart, NaN in between and behind."""
    rows, k = x.shape
    buf = torch.full((offset + ld * rows + 64,), float("nan"),
                     dtype=to_device(x[:1, :1], device).dtype, device=device)
    assert buf.data_ptr() % 128 == 0
    view = buf[offset:].as_strided((rows, k), (ld, 1))
    view.copy_(to_device(x, device))
    return buf[offset:]


@pytest.mark.parametrize("dtype", list(SHAPES), ids=["z", "d"])
@pytest.mark.parametrize("op", ["T", "C"])
def test_bits_do_not_depend_on_the_alignment(ctx, device, dtype, op):
    line = 128 // np.dtype(dtype).itemsize
    shortest = 8192 // (2 if dtype == np.complex128 else 1)
    for m, n in SHAPES[dtype]:
        for k in (shortest, shortest + 1, 5 * shortest + line, 3 * shortest - 1,
                  4 * shortest + line + 3):
            ld = -(-k // line) * line
            for kind in ("int", "uniform"):
                A = make_buffer(95, m, k, m, k, dtype, kind).reshape(m, k)
                B = make_buffer(95, 70 + n, k, n, k, dtype, kind).reshape(n, k)
                got = []
                # on lines; every row off them; a view one element in; only B off
                for lda, ldb, offset in [(ld, ld, 0), (k | 1, (k + 2) | 1, 0),
                                         (ld, ld, 1), (ld, ld + 1, 0)]:
                    dC = torch.zeros(m * n, dtype=to_device(A[:1, :1], device).dtype, device=device)
                    spla.gemm(OPS[op], OPS["N"], m, n, k, 1.0, place(A, device, lda, offset), lda,
                              place(B, device, ldb, offset), ldb, 0.0, dC, m, ctx)
                    got.append(dC.cpu().numpy())
                if kind == "int":
                    ref = np.zeros(m * n, dtype=dtype)
                    oracle.gemm(OPS[op], OPS["N"], m, n, k, 1.0, A.reshape(-1), k, B.reshape(-1),
                                k, 0.0, ref, m, accurate=True)
                    got.append(ref)
                for other in got[1:]:
                    assert np.array_equal(got[0], other), (m, n, k, kind)
