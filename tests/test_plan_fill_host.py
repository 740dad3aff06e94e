"""Host tests of the whole-device planner's fill modes and single-precision plans
(spla_amd/csrc/runtime/tuner.cpp).

* the closed form of the active tiles equals SPLA's block_is_active
  (src/block_generation/block.hpp:58-66) counted tile by tile;
* plans of every fill mode and scalar size cover the reduction in whole 128-byte
  k-blocks with no empty split; double partial sums stay within 256 MiB (single
  precision may take more, to keep its sums short).
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
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("plan") / "libplan.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC",
                    "-I", str(ROOT / "spla_amd" / "csrc"), "-I", str(ROOT / "include"),
                    str(ROOT / "spla_amd" / "csrc" / "runtime" / "tuner.cpp"),
                    str(ROOT / "tests" / "cpp" / "plan_fill_capi.cpp"), "-o", str(out)],
                   check=True)
    lib = ctypes.CDLL(str(out))
    lib.plan_active_tiles_c.argtypes = [ll, ll, ctypes.c_int, ctypes.c_int, ctypes.c_int, ll, ll]
    lib.plan_active_tiles_c.restype = ll
    lib.plan_fill_c.argtypes = [ctypes.c_int, ll, ll, ll, ctypes.c_int, ctypes.c_int, ll, ll,
                                ctypes.POINTER(ll)]
    return lib


def active(mode, ro, co, r, c, nr, nc):
    if mode == 1:
        return c + nc + co > r + ro
    if mode == 2:
        return r + nr + ro > c + co
    return True


def test_active_tiles_equal_the_predicate(lib):
    rng = random.Random(3)
    for _ in range(3000):
        m, n = rng.randint(1, 700), rng.randint(1, 700)
        rows, cols = rng.choice([(32, 64), (64, 64), (64, 128), (128, 128)])
        ro, co = rng.choice([(0, 0), (2, 3), (rng.randint(0, 900), rng.randint(0, 900))])
        for mode in (0, 1, 2):
            want = sum(active(mode, ro, co, r, c, min(rows, m - r), min(cols, n - c))
                       for r in range(0, m, rows) for c in range(0, n, cols))
            got = lib.plan_active_tiles_c(m, n, rows, cols, mode, ro, co)
            assert got == want, (m, n, rows, cols, mode, ro, co)


@pytest.mark.parametrize("scalar", [8, 4])
@pytest.mark.parametrize("cplx", [0, 1])
def test_plans_cover_the_reduction(lib, cplx, scalar):
    unit = 128 // scalar
    for m in (1, 33, 263, 700, 2048):
        for n in (1, 64, 263, 2048):
            for k in (1, 263, 4096, 30011, 200000):
                for mode in (0, 1, 2):
                    out = (ll * 5)()
                    lib.plan_fill_c(cplx, m, n, k, scalar, mode, 2, 2, out)
                    _, splits, per, tm, tn = list(out)
                    kp = k * (1 + cplx)
                    assert per > 0 and per % unit == 0 and tm > 0 and tn > 0
                    assert splits * per >= kp and (splits - 1) * per < kp
                    if splits > 1 and scalar == 8:
                        assert splits * n * m * (1 + cplx) * scalar <= 256 << 20
