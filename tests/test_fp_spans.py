"""The ray-driven FP's host and device arithmetic (csrc/fp_span.hpp, the kernel's own
header compiled for the host): the rows of a ray are those that the reference's
accumulation admits, and the columns that a chunk stages hold every tap its rays read:
the fixed-point positions, row chunks, view groups and column bounds of
fp_stream_kernel restated on the host, on the library's own tables.  A tap
outside them is whatever LDS held before."""
import ctypes as C
import math
import os
import subprocess

import numpy as np
import pytest

from ct_recon_extensions_amd import _lib

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))

SOURCE = r"""
#include "ct_recon_extensions_amd/csrc/fp_span.hpp"
using namespace ctr;

// rays of `count` whose rows differ from the accumulation's, or whose rows without a
// test (fin to fout) are not all inside
extern "C" long long wrong_rows(const double* x0, const double* off, const int* hi, const int* n,
                                long long count)
{
    long long bad = 0;
    for (long long i = 0; i < count; ++i) {
        int kin, kout, fin, fout, a = 0, b = 0;
        fp_ray_rows(x0[i], off[i], hi[i], n[i], kin, kout, fin, fout);
        bool seen = false, free = true;
        double x = x0[i];
        for (int k = 0; k < n[i]; ++k, x += off[i]) {
            const bool inside = x >= 0 && x <= hi[i];
            if (inside && !seen) a = k;
            if (inside) b = k + 1;
            seen = seen || inside;
            free = free && (inside || k < fin || k >= fout);
        }
        bad += a != kin || b != kout || !free;
    }
    return bad;
}

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
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("spans")
    src, so = d / "spans.cpp", d / "spans.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-shared", "-fPIC", f"-I{ROOT}", str(src), "-o",
                    str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.outside.restype = lib.wrong_rows.restype = C.c_longlong
    return lib


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
def test_every_tap_is_staged(lib, case, rows):
    nx, ny, ns, na, ds, offset, start = CASES[case]
    g = _lib.CtrGeom()
    g.nx, g.ny, g.ns, g.na, g.ds, g.dx, g.dy = nx, ny, ns, na, ds, 1.0, 1.0
    g.offset_x, g.offset_y, g.offset_s = offset, -offset, offset
    g.orbit, g.orbit_start = math.pi / na, start
    sc, bo, usex = (C.c_double * (2 * na))(), (C.c_double * (2 * na * ns))(), (C.c_int * na)()
    _lib.call("ctr_fp_tables", C.byref(g), sc, bo, usex)
    taps, widest = C.c_longlong(), C.c_int()
    bad = lib.outside(C.byref(g), bo, usex, rows, C.byref(taps), C.byref(widest))
    assert taps.value > 0 and widest.value > 0
    assert bad == 0, f"{bad} of {taps.value} taps"


@pytest.mark.parametrize("decade", range(0, 15))
@pytest.mark.parametrize("size", [300, 6000])
def test_rows_are_those_of_the_accumulation(lib, decade, size):
    """Steps from 2 columns a row down to 1e-14, of rays anywhere, on an end of the
    image, crossing it exactly at a row, and near that."""
    count = 40000 if size == 300 else 2500
    rng = np.random.default_rng(2000 + decade)
    n, hi = rng.integers(1, size, count), rng.integers(1, size, count)
    off = np.minimum(10.0 ** (rng.uniform(0, 1, count) - decade), 2.0) * rng.choice([-1, 1], count)
    off[rng.random(count) < 0.02] = 0.0
    end, row = np.where(rng.random(count) < 0.5, 0, hi), rng.integers(0, n + 1)
    kind = rng.integers(0, 5, count)
    x0 = np.select(
        [kind == 0, kind == 1, kind == 2, kind == 3],
        [rng.uniform(-0.2, 1.2, count) * hi, end, end - off * row,
         end - off * row + rng.uniform(-2e-13, 2e-13, count)],
        end - off * rng.uniform(0, 1, count) * n + rng.uniform(-2e-8, 2e-8, count))
    x0, off = np.ascontiguousarray(x0, np.float64), np.ascontiguousarray(off, np.float64)
    hi, n = hi.astype(np.int32), n.astype(np.int32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    assert lib.wrong_rows(p(x0), p(off), p(hi), p(n), C.c_longlong(count)) == 0
