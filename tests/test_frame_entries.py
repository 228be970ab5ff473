"""The absorbing frame's entries that the update kernels fetch, over every
cell that they ask for: shapes of 2 and 4 cells per thread also ask for the
cells past the last column.  Every fetch lies in its array, and there is none
where the arrays are absent (no frame, or no CPML)."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include "sofi_frame.h"
struct G { int nx, ny, fw, abs_type, gx2, gx3, gy2, gy3, wx, wy; };
template <bool PAST> int bad(const G &g, int vw)
{
    const int nxp = (g.ny + 1) * g.wx, nyp = g.wx * g.wy;
    const bool any = g.abs_type == 1 && g.fw > 0;
    for (int j = 1; j <= g.ny; ++j)
        for (int i0 = 1; i0 <= g.nx; i0 += vw)
            for (int i = i0; i < i0 + vw; ++i) {
                const bool xf = frame_x<PAST>(g, i), yf = frame_y<PAST>(g, i, j), get = cpml_fetch<PAST>(g);
                bool ok = any || !(get && (xf || yf));
                if (get && xf) {
                    const int h = hx(g, i), q = x_entry(g, h, j);
                    ok = ok && h >= 0 && h < g.wx && q >= 0 && q < nxp;
                }
                if (get && yf) {
                    const int q = y_entry(g, i, j);
                    ok = ok && q >= 0 && q < nyp;
                }
                // and a cell of the grid has what its update reads
                if (i <= g.nx) ok = ok && xf == in_xframe(g, i) && yf == in_yframe(g, j) && (get || !any);
                if (!ok) return i + 100000 * j;
            }
    return 0;
}
// the first cell whose fetch lies outside (i + 100000 * j), or 0
extern "C" int bad_cell(int nx, int ny, int fw, int abs_type, int surf, int vw)
{
    const G g = { nx, ny, fw, abs_type, fw, nx - fw, surf ? 0 : fw, ny - fw, 2 * fw + 1, nx + 1 };
    return vw > 1 ? bad<true>(g, vw) : bad<false>(g, vw);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("frame")
    (d / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "gpi_project_amd", "csrc", "device"), str(d / "t.cpp"), "-o", str(d / "t.so")],
                   check=True)
    return C.CDLL(str(d / "t.so"))


@pytest.mark.parametrize("vw", [1, 2, 4])
@pytest.mark.parametrize("nx,ny,fw", [(64, 48, 20), (65, 49, 20), (126, 47, 1), (63, 9, 4), (67, 33, 0), (64, 5, 0),
                                      (5, 5, 0), (2, 2, 1)])
@pytest.mark.parametrize("abs_type,surf", [(1, 0), (1, 1), (2, 0), (0, 0)])
def test_fetches_lie_in_their_arrays(lib, nx, ny, fw, abs_type, surf, vw):
    bad = lib.bad_cell(nx, ny, fw, abs_type, surf, vw)
    assert bad == 0, (bad % 100000, bad // 100000)
