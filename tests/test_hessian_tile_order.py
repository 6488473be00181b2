"""The Hessian kernel numbers the tiles of the upper triangle whole super-tiles first (`tile_coords` in
csrc/hessian_tiles.h, compiled for the host here): a restatement of that order, which the function has to follow, has to reach
every tile once, and to keep the 32 tiles that one L2 serves together."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm-compressor_amd", "csrc")
WRAPPER = """
#define __host__
#define __device__
#define __forceinline__ inline
#include "hessian_tiles.h"
extern "C" void tiles(int n, int nb, int SH, int SW, int* ij) {
  for (int c = 0; c < n; ++c) tile_coords(c, nb, SH, SW, ij[2 * c], ij[2 * c + 1]);
}
"""


def _tiles(nb, SH, SW):
    rows, cols, rest = nb // SH, nb // SW, nb % SW
    right = lambda si: (si * SH + SH - 1 + SW - 1) // SW  # noqa: E731
    for si in range(rows):
        for sj in range(right(si), cols):
            for i in range(SH):
                for j in range(SW):
                    yield si * SH + i, sj * SW + j
    for si in range(rows):
        if rest and right(si) <= cols:
            for i in range(SH):
                for j in range(rest):
                    yield si * SH + i, cols * SW + j
    for si in range((nb + SH - 1) // SH):
        f = right(si)
        end = f * SW if si < rows and (f < cols or (f == cols and rest)) else nb
        for i in range(si * SH, min(nb, (si + 1) * SH)):
            for j in range(i, end):
                yield i, j


@pytest.mark.parametrize("SH,SW", [(4, 8), (8, 8)])
def test_every_tile_of_the_upper_triangle_once(SH, SW):
    for nb in range(1, 90):
        tiles = list(_tiles(nb, SH, SW))
        assert len(tiles) == nb * (nb + 1) // 2 == len(set(tiles))
        assert all(i <= j < nb for i, j in tiles)


@pytest.mark.parametrize("nb", [56, 32, 28])
def test_groups_of_32_share_their_panels(nb):
    tiles = list(_tiles(nb, 4, 8))
    whole = len(tiles) // 256 * 256
    per = whole // 8
    groups = [tiles[x * per + g:x * per + g + 32] for x in range(8) for g in range(0, per, 32)]
    panels = [len({p for t in group for p in t}) for group in groups]
    assert sum(panels) / len(panels) <= 12.5


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("tiles") / "tiles.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", "-x", "c++", "-", "-o", lib],
                   input=WRAPPER.encode(), check=True)
    return ctypes.CDLL(lib).tiles


@pytest.mark.parametrize("SH,SW", [(4, 8), (8, 8)])
def test_the_kernel_takes_the_tiles_in_this_order(compiled, SH, SW):
    for nb in range(1, 90):
        want = list(_tiles(nb, SH, SW))
        got = ((ctypes.c_int * 2) * (len(want) + 1))()
        compiled(len(want) + 1, nb, SH, SW, ctypes.byref(got))
        assert [tuple(t) for t in got] == want + [(-1, -1)]
