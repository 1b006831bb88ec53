"""The x-axis auxiliary layout, compiled for the host: every absorbing cell has
an element of its own inside the field, and what one 64-column tile touches of a
row, or of neighbouring rows, lies together."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = '''
#include <hip/hip_runtime.h>
#include "cgfd_device.h"
extern "C" unsigned aux_x(int n0, int n1, int ni, int nj, int nk, int x, int y, int z)
{
    return cgfd::aux_x_index(cgfd::aux_x_layout(n0, n1, ni, nj, nk), n0, nj, x, y, z);
}
'''


@pytest.fixture(scope="module")
def aux_x(tmp_path_factory):
    d = tmp_path_factory.mktemp("aux")
    (d / "aux.cpp").write_text(SRC)
    so = d / "aux.so"
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "copara-cgfd3d_amd", "csrc"),
                    str(d / "aux.cpp"), "-o", str(so)], check=True)
    f = ctypes.CDLL(str(so)).aux_x
    f.restype = ctypes.c_uint
    return f


# one tile, one column short of and past it, several tiles; layers on both
# sides, of different depth, on one side
@pytest.mark.parametrize("ni", [33, 63, 64, 65, 200])
@pytest.mark.parametrize("n0,n1", [(5, 5), (3, 9), (0, 7), (4, 0)])
def test_every_absorbing_cell_has_its_own_element(aux_x, ni, n0, n1):
    nj, nk = 7, 4
    cells = [(x, y, z) for z in range(nk) for y in range(nj) for x in range(ni) if x < n0 or x >= ni - n1]
    at = [aux_x(n0, n1, ni, nj, nk, *c) for c in cells]
    assert sorted(at) == list(range(len(cells)))


# where each side lies in one tile, a tile's cells of 4 rows of a plane are one run of
# elements
@pytest.mark.parametrize("ni", [40, 64, 75, 200])
def test_a_tiles_cells_of_neighbouring_rows_are_one_run(aux_x, ni):
    n0, n1, nj, nk = 5, 6, 12, 3
    for x0 in range(0, ni, 64):
        cells = [(x, y, 1) for y in range(4, 8) for x in range(x0, min(ni, x0 + 64)) if x < n0 or x >= ni - n1]
        at = sorted(aux_x(n0, n1, ni, nj, nk, *c) for c in cells)
        assert at == list(range(at[0], at[0] + len(at))) if at else True
