"""The columns that a chunk of the ray-driven FP stages (csrc/fp_span.hpp, the
kernel's own header compiled for the host) hold every tap that its rays read:
the fixed-point positions, row chunks, view groups and column bounds of
fp_stream_kernel restated on the host, on the library's own tables.  A tap
outside them is whatever LDS held before."""
import ctypes as C
import math
import os
import subprocess

import pytest

from ct_recon_extensions_amd import _lib

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))

SOURCE = r"""
#include "ct_recon_extensions_amd/csrc/fp_span.hpp"
using namespace ctr;

// taps read outside the staged columns (and how many were read); -1: no shape applies
extern "C" long long outside(const ctr_geom* g, const double* bo, const int* usex, int rows,
                             long long* taps, int* widest)
{
    int shape = 0;
    while (shape < 4 && !fp_stream_applies(*g, shape < 2 ? 4 : 1, 4, shape & 1 ? 256 : 128)) ++shape;
    if (shape == 4) return -1;
    const int views = shape < 2 ? 4 : 1, most = shape & 1 ? 256 : 128;
    const int na = g->na, ns = g->ns;
    long long bad = 0;
    *taps = 0;
    *widest = 0;
    for (int xb = 0; xb < 2; ++xb)
        for (int a0 = 0; a0 < na; a0 += views)
            for (int s0 = 0; s0 < ns; s0 += 64) {
                const int nsteps = xb ? g->ny : g->nx, rowlen = xb ? g->nx : g->ny;
                for (int k0 = 0; k0 < nsteps; k0 += rows) {
                    float xmin = 1e30f, xmax = -1e30f;
                    for (int a = a0; a < a0 + views && a < na; ++a) {
                        if ((usex[a] != 0) != (xb != 0)) continue;
                        const double* p = bo + 2 * (size_t)a * ns;
                        const float xa = (float)p[2 * s0], sl = (float)p[2 * s0 + 1];
                        const float xz = (float)p[2 * std::min(s0 + 63, ns - 1)];
                        const float drift = (rows - 1) * sl;
                        const float lo = fminf(xa, xz) + fminf(0.0f, drift);
                        const float hi = fmaxf(xa, xz) + fmaxf(0.0f, drift);
                        xmin = fminf(xmin, fmaf((float)k0, sl, lo));
                        xmax = fmaxf(xmax, fmaf((float)k0, sl, hi));
                    }
                    if (xmin > xmax) continue;
                    const FpSpan c = fp_span(xmin, xmax, rowlen, most);
                    *widest = std::max(*widest, c.cols);
                    for (int a = a0; a < a0 + views && a < na; ++a) {
                        if ((usex[a] != 0) != (xb != 0)) continue;
                        for (int s = s0; s < s0 + 64 && s < ns; ++s) {
                            const double *r = bo + 2 * ((size_t)a * ns + s);
                            const long long off = (long long)rint(r[1] * 0x1p32);
                            for (int k = k0; k < k0 + rows && k < nsteps; ++k) {
                                const double x = r[0] + k * r[1];
                                if (!(x >= 0 && x <= rowlen - 1)) continue;
                                const long long f = (long long)rint(r[0] * 0x1p32) + k * off;
                                const int i = f < 0 ? 0 : (int)(f >> 32);
                                *taps += 2;
                                bad += i < c.first || i >= c.first + c.cols;
                                bad += i + 1 < c.first || i + 1 >= c.first + c.cols;
                            }
                        }
                    }
                }
            }
    return bad;
}
"""


@pytest.fixture(scope="module")
def outside(tmp_path_factory):
    d = tmp_path_factory.mktemp("spans")
    src, so = d / "spans.cpp", d / "spans.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", f"-I{ROOT}", str(src), "-o",
                    str(so)], check=True)
    f = C.CDLL(str(so)).outside
    f.restype = C.c_longlong
    return f


# (nx, ny, channels, views, ds, offset, start): rays on the last column with 63, 64,
# 65 and 128 columns to it, and off it; narrow images; coarse and fine channels
CASES = [
    (64, 64, 64, 90, 1.0, 0.0, 0.0), (63, 63, 63, 90, 1.0, 0.0, 0.0), (65, 65, 65, 90, 1.0, 0.0, 0.0),
    (128, 128, 250, 90, 1.0, 0.0, 0.0), (256, 256, 378, 90, 1.0, 0.0, 0.0),
    (256, 256, 382, 90, 1.0, 0.0, 0.0), (129, 129, 253, 60, 1.0, 0.0, 0.0),
    (195, 195, 307, 60, 1.0, 0.0, 0.0), (195, 195, 311, 60, 1.0, 0.0, 0.0),
    (128, 128, 65, 40, 2.0, 0.0, 0.0), (130, 130, 70, 40, 2.0, 0.0, 0.0),
    (64, 48, 80, 37, 1.0, 0.3, 0.1), (48, 64, 80, 37, 1.0, -0.3, -0.7), (5, 3, 12, 9, 1.0, 0.0, 0.0),
    (3, 70, 90, 22, 0.8, 0.0, 0.3), (130, 130, 150, 6, 1.0, 0.0, 0.05), (90, 90, 70, 45, 2.5, 0.2, 0.2),
    (200, 200, 41, 50, 1.0, 0.0, 0.0), (257, 255, 257, 16, 1.0, 0.0, math.pi / 4),
]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("rows", [2, 4])
def test_every_tap_is_staged(outside, case, rows):
    nx, ny, ns, na, ds, offset, start = CASES[case]
    g = _lib.CtrGeom()
    g.nx, g.ny, g.ns, g.na, g.ds, g.dx, g.dy = nx, ny, ns, na, ds, 1.0, 1.0
    g.offset_x, g.offset_y, g.offset_s = offset, -offset, offset
    g.orbit, g.orbit_start = math.pi / na, start
    sc, bo, usex = (C.c_double * (2 * na))(), (C.c_double * (2 * na * ns))(), (C.c_int * na)()
    _lib.call("ctr_fp_tables", C.byref(g), sc, bo, usex)
    taps, widest = C.c_longlong(), C.c_int()
    bad = outside(C.byref(g), bo, usex, rows, C.byref(taps), C.byref(widest))
    assert taps.value > 0 and widest.value > 0
    assert bad == 0, f"{bad} of {taps.value} taps"
