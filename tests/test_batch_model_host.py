"""Host tests of the batched launch's cost model (spla_amd/csrc/runtime/batch_schedule.cpp)."""

import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
ll = ctypes.c_longlong


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    out = tmp_path_factory.mktemp("model") / "libmodel.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC",
                    "-I", str(ROOT / "spla_amd" / "csrc"), "-I", str(ROOT / "include"),
                    str(ROOT / "spla_amd" / "csrc" / "runtime" / "batch_schedule.cpp"),
                    str(ROOT / "tests" / "cpp" / "batch_schedule_capi.cpp"), "-o", str(out)],
                   check=True)
    lib = ctypes.CDLL(str(out))
    lib.bs_plan.restype = ctypes.c_void_p
    lib.bs_plan.argtypes = [ctypes.POINTER(ll), ctypes.c_int, ctypes.c_int, ctypes.c_int,
                            ctypes.c_int, ctypes.c_double, ctypes.c_int, ctypes.c_double]
    lib.bs_counts.argtypes = [ctypes.c_void_p, ctypes.POINTER(ll)]
    lib.bs_model_seconds.restype = ctypes.c_double
    lib.bs_model_seconds.argtypes = [ctypes.c_void_p]
    lib.bs_free.argtypes = [ctypes.c_void_p]

    def call(shapes, cplx, cfg, scale, eff):
        """(workgroups of the products, seconds by the model)"""
        flat = (ll * (6 * len(shapes)))(*[x for s in shapes for x in (*s, 0, 0, 0)])
        h = lib.bs_plan(flat, len(shapes), cplx, 0, cfg, scale, 256, eff)
        counts = (ll * 4)()
        lib.bs_counts(h, counts)
        seconds = lib.bs_model_seconds(h)
        lib.bs_free(h)
        return counts[0], seconds

    return call


def test_equal_blocks_fill_whole_rounds(plan):
    """16 complex blocks of 256 x 256 make 128 large tiles, whose splits fill the 512 resident
    workgroups three times whatever the rate (a rounding error once made a 13th split)."""
    for percent in range(50, 96):
        items, _ = plan([(256, 256, 16384)] * 16, 1, 0, 1.0, percent / 100)
        assert items == 1536, percent


def test_many_partial_sums_take_their_time(plan):
    """The reduction of one 64 x 64 tile over 256 splits was measured at about 0.3 ms: 16 elements
    a thread, 256 loads each, eight in flight."""
    items, seconds = plan([(64, 64, 65536)], 0, 1, 2.0, 0.83)
    assert items == 256
    assert 0.2e-3 < seconds < 0.5e-3
