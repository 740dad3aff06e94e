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
        out = (ll * 6)()
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
        splits, _, coarse, *_ = plan(1, m, n, k, 8, 0)
        if coarse == 1 or coarse * m * n * 16 <= 64 << 20:
            assert splits == 1 or splits * m * n * 16 <= 64 << 20, (m, n, k)


@pytest.mark.parametrize("scalar", [8, 4])
def test_sums_are_no_longer_than_the_coarse_plan(plan, scalar):
    """The rounding error of a sum grows with its length. Small products (their own kernel) share
    the reduction among up to 16 waves."""
    rng = random.Random(11)
    block = 128 // scalar
    shapes = [(1, 1238, 1207, 4119), (1, 534, 1797, 9523), (0, 1601, 1190, 20905),
              (1, 1560, 1626, 252100), (1, 256, 256, 4096)]
    shapes += [(rng.randint(0, 1), *(round(2 ** rng.uniform(0, e)) for e in (12, 12, 19)))
               for _ in range(4000)]
    for cplx, m, n, k in shapes:
        kp = k * (1 + cplx)
        for mode in (0, 1, 2):
            splits, per, coarse, longest, small, ksum = plan(cplx, m, n, k, scalar, mode)
            if small:
                waves = min(16, -(-k // 32))
                step = 64 // (scalar * (1 + cplx))  # of one MFMA and 16-byte piece
                length = -(-(-(-k // step)) // waves) * step * (1 + cplx)
                assert length <= longest or waves == 1, (cplx, m, n, k, mode)
                continue
            assert ksum == 0 or (scalar == 8 and ksum % 32 == 0 and 0 < ksum < per)
            unit = block if scalar == 4 else 1  # whole k-blocks
            assert min(ksum or per, kp) < longest + unit, (cplx, m, n, k, mode)


def test_shapes_that_add_up_stretches(plan):
    """The shapes of tests/test_stretch_gpu.py take the kernel that it means to test."""
    for cplx, m, n, k, one in [(1, 354, 550, 165, True), (1, 330, 300, 2100, False),
                               (0, 385, 553, 301, True), (0, 400, 300, 4000, False),
                               (1, 534, 597, 1523, False), (0, 801, 590, 3905, False)]:
        splits, _, coarse, _, _, ksum = plan(cplx, m, n, k, 8, 0)
        assert ksum > 0 and (splits == 1) == one and coarse > splits, (m, n, k)
