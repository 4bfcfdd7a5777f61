"""The merge table of the PME tiles (csrc/tiles.h) on the CPU, against whole-number arithmetic without a limit.

For every grid coordinate the two offsets per axis are rebuilt from the numbering itself: tile u of the axis lies in cube
u // 2 and octant u % 2, the fine key is cube * 8 + octant, and point l of the tile's block is l strides in.  Past 2^31
block values (768^3 points at order 6, 864^3 at order 4) the offsets need all 32 bits; past 2^32 there are no tiles.
"""

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pgm-jax_amd", "csrc")

SHIM = r"""
#include "tiles.h"
extern "C" int tiles(const int *K, int P, int cap, int *out, unsigned *tab) {
    pgm::PMETiles t{};
    if (!pgm::pme_tiles(K, P, cap, t)) return 0;
    const int v[12] = {t.T[0], t.T[1], t.T[2], t.nt[0], t.nt[1], t.nt[2], t.nc[0], t.nc[1], t.nc[2], t.ntiles, t.bsize, t.ncubes};
    for (int k = 0; k < 12; ++k) out[k] = v[k];
    const std::vector<unsigned> m = pgm::pme_merge_table(K, P, t);
    for (size_t k = 0; k < m.size(); ++k) tab[k] = m[k];
    return 1;
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC, str(d / "shim.cpp"), "-o", str(d / "shim.so")],
                   check=True)
    return C.CDLL(str(d / "shim.so"))


def _tiles(host, K, P, cap=8):
    k, out, tab = np.array(K, np.int32), np.zeros(12, np.int32), np.zeros(2 * sum(K), np.uint32)
    ok = host.tiles(k.ctypes.data_as(C.c_void_p), P, cap, out.ctypes.data_as(C.c_void_p), tab.ctypes.data_as(C.c_void_p))
    return (out, tab) if ok else None


@pytest.mark.parametrize("K, P, cap", [((32, 32, 32), 6, 8), ((24, 36, 27), 4, 8), ((56, 48, 63), 8, 8), ((126, 66, 95), 6, 6),
                                       ((768, 768, 768), 6, 8), ((864, 864, 864), 4, 8), ((24, 4096, 4096), 6, 8)])
def test_merge_table_offsets(host, K, P, cap):
    out, tab = _tiles(host, K, P, cap)
    T, nt, nc = [int(v) for v in out[:3]], [int(v) for v in out[3:6]], [int(v) for v in out[6:9]]
    B = [t + P - 1 for t in T]
    bsize = B[0] * B[1] * 16
    assert (int(out[9]), int(out[10])) == (8 * nc[0] * nc[1] * nc[2], bsize)
    cube, octant, stride = (nc[1] * nc[2], nc[2], 1), (4, 2, 1), (B[1] * 16, 16, 1)
    at = 0
    for a in range(3):
        for g in range(K[a]):
            u = min(g // T[a], nt[a] - 1)
            left = g - u * T[a]
            key = 8 * (u // 2) * cube[a] + (u % 2) * octant[a]
            assert int(tab[at]) == key * bsize + left * stride[a], (a, g)
            if left <= P - 2:
                v = (u - 1) % nt[a]
                width = K[a] - (nt[a] - 1) * T[a] if v == nt[a] - 1 else T[a]
                key = 8 * (v // 2) * cube[a] + (v % 2) * octant[a]
                assert int(tab[at + 1]) == key * bsize + (left + width) * stride[a], (a, g)
            else:
                assert int(tab[at + 1]) == 2**32 - 1
            at += 2


@pytest.mark.parametrize("K, P", [((1024, 1024, 1024), 6), ((8, 32, 32), 6), ((32, 16384, 16), 6)])
def test_no_tiles(host, K, P):
    """Too many block values, too few points for three tiles, too many cubes along an axis."""
    assert _tiles(host, K, P) is None
