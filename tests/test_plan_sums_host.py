"""Host tests of the partial sums that whole-device plans keep and of how long their sums
are (spla_amd/csrc/runtime/tuner.cpp), against the coarse plan of the same product.
"""

import ctypes
import random
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
ll = ctypes.c_longlong


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    out = tmp_path_factory.mktemp("sums") / "libsums.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC",
                    "-I", str(ROOT / "spla_amd" / "csrc"), "-I", str(ROOT / "include"),
                    str(ROOT / "spla_amd" / "csrc" / "runtime" / "tuner.cpp"),
                    str(ROOT / "tests" / "cpp" / "plan_sums_capi.cpp"), "-o", str(out)],
                   check=True)
    lib = ctypes.CDLL(str(out))
    lib.plan_sums_c.argtypes = [ctypes.c_int, ll, ll, ll, ctypes.c_int, ctypes.c_int,
                                ctypes.POINTER(ll)]

    def call(cplx, m, n, k, scalar, mode):
        out = (ll * 5)()
        lib.plan_sums_c(cplx, m, n, k, scalar, mode, out)
        return list(out)

    return call


def test_allocation_free_products_stay_accepted(plan):
    """The allocation-free entry point takes what the coarse plan fits into 64 MiB, one split
    of a large C (no partial sums) included."""
    rng = random.Random(7)
    shapes = [(2335, 3446, 41573), (6274, 1169, 12259), (8478, 812, 1808)]
    shapes += [(rng.randint(64, 9000), rng.randint(64, 9000), round(16 * 2 ** rng.uniform(0, 15)))
               for _ in range(3000)]
    for m, n, k in shapes:
        splits, _, coarse, _, _ = plan(1, m, n, k, 8, 0)
        if coarse == 1 or coarse * m * n * 16 <= 64 << 20:
            assert splits == 1 or splits * m * n * 16 <= 64 << 20, (m, n, k)
