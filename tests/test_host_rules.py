"""Rules that size launches and place boundaries, from the headers the kernels include and the
library's host code, compiled for the CPU."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "dplus-dev_amd")
LIB = os.path.join(PKG, "dplus_mi355x")
SOURCE = r"""
#include "device.hpp"
using namespace dplus;
extern "C" void patch_sets(long long nchunks, int *D, int *nset) { mc_patch_sets(nchunks, *D, *nset); }
extern "C" void rebin(const double *w, const double *b, double *out) {  // vegas_rebin's sums, one axis
    double cum[kVB], c = 0.0;
    for (int i = 0; i < kVB; i++) cum[i] = c += w[i];
    out[0] = b[0];
    for (int i = 0; i < kVB; i++)
        out[i + 1] = i == kVB - 1 ? b[i + 1] : vegas_boundary(w, cum, b + 1, b[0], i + 1, b[i + 1]);
}
// the mesh builder's plan of one class of n sources in [lo, hi]: 0 refused, else the mesh's sizes
static bool plan(const double *lo, const double *hi, int N, double step, int fp64, long long n, MeshPlan &P, MeshSizes &Z) {
    MeshSources S;
    S.ok = true;
    S.nfield = 1;
    S.natoms = n;
    for (int a = 0; a < 3; a++) {
        S.lo[a] = S.cell0[a] = lo[a];
        S.hi[a] = hi[a];
        S.cell_inv[a] = 1.0 / std::max(kMeshCell, (hi[a] - lo[a]) / kMeshCells);
    }
    return mesh_plan(S, N, step, fp64 != 0, 1, kMeshRoom, P, Z);
}
extern "C" int mesh_sizes(const double *lo, const double *hi, int N, double step, int fp64, int *m, int *k, long long *bytes) {
    MeshPlan P;
    MeshSizes Z;
    if (!plan(lo, hi, N, step, fp64, 1000, P, Z)) return 0;
    for (int a = 0; a < 3; a++) {
        m[a] = P.ax[a].m;
        k[a] = P.ax[a].k;
    }
    *bytes = (long long)Z.bytes;
    return 1;
}
// the most that a patch's planes and z windows need, over every patch of the grid, against what
// the launch gives them; 0: refused
extern "C" int mesh_patches(const double *lo, const double *hi, int N, double step, int fp64, long long *need, long long *have, int *zmost) {
    MeshPlan P;
    MeshSizes Z;
    if (!plan(lo, hi, N, step, fp64, 1000, P, Z)) return 0;
    std::vector<MeshBand> bands;
    int ntiles;
    mesh_bands(P, Z, N, fp64 != 0, bands, ntiles);
    const int W = fp64 ? 16 : 8;
    *need = 0;
    *zmost = 0;
    *have = (long long)mesh_lds(Z, fp64 != 0);
    for (const MeshBand &B : bands) {
        const int n6 = 6 * B.shell, half = 3 * B.shell;
        const double q = B.shell * step;
        auto place = [](double r, double inv) { return (int)ceil(r * inv); };
        for (int k0 = 0; k0 < n6; k0 += B.cols) {
            int x0 = 1 << 30, x1 = -x0, y0 = x0, y1 = x1, z0 = x0, z1 = x1;
            for (int r = 0; r < B.rows; r++) {
                const double t = kPi * (B.j0 + r) / half;
                const int iz = place(q * cos(t), P.ax[2].dkinv);
                z0 = std::min(z0, iz);
                z1 = std::max(z1, iz);
                for (int k = k0; k < std::min(k0 + B.cols, n6); k++) {
                    const int ix = place(q * sin(t) * cos(k2Pi * k / n6), P.ax[0].dkinv);
                    const int iy = place(q * sin(t) * sin(k2Pi * k / n6), P.ax[1].dkinv);
                    x0 = std::min(x0, ix);
                    x1 = std::max(x1, ix);
                    y0 = std::min(y0, iy);
                    y1 = std::max(y1, iy);
                }
            }
            *need = std::max(*need, (long long)B.rows * (y1 - y0 + W) * ((x1 - x0 + W) | 1) * (fp64 ? 16 : 8));
            *zmost = std::max(*zmost, z1 - z0 + W);
        }
    }
    return 1;
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, out = str(d / "rules.cpp"), str(d / "librules.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(PKG, "csrc"), "-I" + os.path.join(ROOT, "include"), src, "-L" + LIB,
                    "-ldplus_mi355x", "-Wl,-rpath," + LIB, "-o", out], check=True)
    return ctypes.CDLL(out)


def test_mc_patch_sets_fit_the_partial_sums(rules):
    """Every count of chunks: the sets cover the chunks, no set is empty, and the workgroups write
    no more blocks than the partial sums' buffer holds (chunk / 256 a chunk)."""
    D, nset = ctypes.c_int(), ctypes.c_int()
    for n in list(range(4, 5000)) + [10 ** 6, 10 ** 6 + 1]:
        rules.patch_sets(ctypes.c_longlong(n), ctypes.byref(D), ctypes.byref(nset))
        per = 4 * D.value
        assert D.value in (1, 2, 4) and (nset.value - 1) * per < n <= nset.value * per
        for chunk in (256, 512, 768, 8192):
            assert chunk // 64 * nset.value <= n * chunk // 256, (n, chunk)


def _rebin(rules, w, b):
    out = np.empty(33)
    p = ctypes.POINTER(ctypes.c_double)
    w, b = np.ascontiguousarray(w, float), np.ascontiguousarray(b, float)
    rules.rebin(w.ctypes.data_as(p), b.ctypes.data_as(p), out.ctypes.data_as(p))
    return out


def _sweep(w, b):
    """The serial sweep over the bins: a boundary wherever the running weight passes a share."""
    new, j, dw, x, pts = b.copy(), 0, 0.0, b[0], w.sum() / 32
    for i in range(32):
        dw += w[i]
        old, x = x, b[i + 1]
        while dw > pts:
            dw -= pts
            if j < 31:
                new[j + 1] = x - dw * (x - old) / w[i]
            j += 1
    return new


def test_vegas_boundaries_of_general_weights_are_the_sweeps(rules):
    rng = np.random.default_rng(3)
    for _ in range(1000):
        b = np.concatenate([[0.0], np.sort(rng.random(31)), [1.0]])
        w = rng.random(32) ** rng.uniform(0.2, 4.0)
        # a sum's rounding (32 terms: 2^-48 of the total) moves a boundary by that over the weight's density
        tol = 2.0 ** -48 * w.sum() / w.min() + 1e-15
        assert np.max(np.abs(_rebin(rules, w, b) - _sweep(w, b))) < tol


def test_vegas_boundaries_with_zero_and_equal_weights(rules):
    """Zero weights beside equal ones, where shares meet running sums exactly up to rounding: every
    boundary is finite, in order, and lies in a bin of nonzero weight that holds its share."""
    rng = np.random.default_rng(4)
    cases = [np.zeros(32), np.eye(32)[0], np.eye(32)[31], np.eye(32)[17] * 1e-300, np.ones(32) * 0.1]
    cases += [np.where(rng.random(32) < rng.random(), rng.random(), 0.0) for _ in range(4000)]
    cases += [np.where(rng.random(32) < rng.random(), rng.random(32), 0.0) for _ in range(1000)]
    for w in cases:
        b = np.concatenate([[0.0], np.sort(rng.random(31)), [1.0]])
        out = _rebin(rules, w, b)
        assert np.isfinite(out).all() and out[0] == 0.0 and out[32] == 1.0
        if not w.any():
            assert np.array_equal(out, b)
            continue
        c = np.concatenate([[0.0], np.cumsum(w)])
        eps = 2.0 ** -48 * c[32]
        # the shares that a sum exceeds come first; boundaries past the last keep their value
        taken = [i for i in range(1, 32) if c[32] > (c[32] / 32) * i]
        assert (np.diff(out[[0] + taken]) >= 0).all()
        for i in taken:
            share = (c[32] / 32) * i
            assert any(w[n] > 0 and b[n] <= out[i] <= b[n + 1] and c[n] - eps <= share <= c[n + 1] + eps
                       for n in range(32))


@pytest.mark.parametrize("fp64", [0, 1])
def test_mesh_plan_refuses_extents_it_has_no_sizes_for(rules, fp64):
    """One long axis or three, from a protein to beyond any structure, and steps that are no
    numbers: a plan has positive sizes within the workspace, or is refused."""
    arr = lambda v: (ctypes.c_double * 3)(*v)
    m, k, nb = (ctypes.c_int * 3)(), (ctypes.c_int * 3)(), ctypes.c_longlong()
    for X in (0.0, 1.0, 50.0, 1e3, 1e6, 1e8, 1e9, 1e12, 1e200):
        for axes in ((0,), (1,), (2,), (0, 1, 2)):
            for step in (0.05, 1.0, 1e9, float("inf"), float("nan")):
                half = [X if a in axes else 1.0 for a in range(3)]
                ok = rules.mesh_sizes(arr([-x for x in half]), arr(half), 53, ctypes.c_double(step), fp64, m, k,
                                      ctypes.byref(nb))
                if not ok:
                    assert X > 5.0 or step > 1.0 or step != step
                    continue
                assert all(0 < v < 4096 + 32 for v in m) and all(0 < v < 2 * 65536 + 2 for v in k)
                assert 0 < nb.value <= 512 << 20


@pytest.mark.parametrize("fp64", [0, 1])
def test_mesh_patches_fit_their_planes(rules, fp64):
    """Every patch of the interpolation at node spacings from far below a frequency step to far
    above, equal and unequal axes: its (x, y) planes fit the launch's LDS (64 KB a workgroup mixed,
    128 KB FP64) and its z points the rows' windows."""
    arr = lambda v: (ctypes.c_double * 3)(*v)
    need, have, z = ctypes.c_longlong(), ctypes.c_longlong(), ctypes.c_int()
    tried = 0
    for N in (4, 13, 28, 53):
        for half in ((0.3, 0.3, 0.3), (1.0, 0.8, 0.6), (2.0, 2.0, 2.0), (4.0, 1.0, 7.0), (9.0, 6.0, 5.0), (3.0, 30.0, 2.0)):
            for step in (0.02, 0.05, 0.11, 0.23, 0.6):
                if not rules.mesh_patches(arr([-h for h in half]), arr(half), N, ctypes.c_double(step), fp64,
                                          ctypes.byref(need), ctypes.byref(have), ctypes.byref(z)):
                    continue
                tried += 1
                assert 0 < need.value <= have.value <= (128 if fp64 else 64) << 10, (N, half, step)
                assert (z.value + 7) // 8 * 8 <= 40
    assert tried > 80
