"""Host tests of the enumeration of a fill mode's tiles (spla_amd/csrc/kernels/fill_tiles.hpp).

The closed form must count the tiles of SPLA's block_is_active
(src/block_generation/block.hpp:58-66) and give each of them once, column by column, for
every ratio of tile rows to columns that the kernels have and for diagonals beside the
matrix; finding one tile among a million tile columns must not walk them.
"""

import ctypes
import random
import shutil
import subprocess
import time
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
ll = ctypes.c_longlong
SHAPES = [(16, 16), (32, 64), (32, 32), (64, 64), (64, 128), (128, 128), (128, 64), (256, 128),
          (256, 64)]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("fill") / "libfill.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC",
                    "-I", str(ROOT / "spla_amd" / "csrc"), "-I", str(ROOT / "include"),
                    str(ROOT / "tests" / "cpp" / "fill_tiles_capi.cpp"), "-o", str(out)],
                   check=True)
    lib = ctypes.CDLL(str(out))
    lib.fill_total.argtypes = [ctypes.POINTER(ll)]
    lib.fill_total.restype = ll
    lib.fill_locate.argtypes = [ctypes.POINTER(ll), ll, ctypes.POINTER(ctypes.c_int)]
    return lib


def active(mode, off, r, c, nr, nc):
    return c + nc + off > r if mode == 1 else r + nr > c + off


@pytest.mark.parametrize("rows,cols", SHAPES)
@pytest.mark.parametrize("mode", [1, 2], ids=["upper", "lower"])
def test_every_tile_once(lib, rows, cols, mode):
    rng = random.Random(rows * 7 + cols)
    for i in range(150):
        m, n = rng.randint(1, 900), rng.randint(1, 900)
        off = rng.choice((0, 1, -1, 37, rng.randint(-1000, 1000), -m, n, -m + 1, n - 1))
        want = [(r // rows, c // cols) for c in range(0, n, cols) for r in range(0, m, rows)
                if active(mode, off, r, c, min(rows, m - r), min(cols, n - c))]
        p = (ll * 6)(m, n, rows, cols, mode, off)
        assert lib.fill_total(p) == len(want), (m, n, off)
        out = (ctypes.c_int * 2)()
        for t, tile in enumerate(want):
            lib.fill_locate(p, t, out)
            assert tuple(out) == tile, (m, n, off, t)


@pytest.mark.parametrize("mode", [1, 2], ids=["upper", "lower"])
def test_many_columns_are_not_walked(lib, mode):
    """One tile row, 16 million tile columns: 2000 tiles in well under a second (walking them
    takes several seconds each)."""
    n = 1 << 30
    p = (ll * 6)(64, n, 64, 64, mode, -n if mode == 2 else 0)
    total = lib.fill_total(p)
    assert total == n // 64
    out = (ctypes.c_int * 2)()
    begin = time.perf_counter()
    for i in range(2000):
        t = i * 8191 % total
        lib.fill_locate(p, t, out)
        assert tuple(out) == (0, t)
    assert time.perf_counter() - begin < 1.0
