"""The benchmark workloads at their stated sizes on the GPU, against the FP64
oracle on the same seeded inputs.

* 50,000 atoms + hydration layer, grid 250, 1,000 q: sampled grid nodes against
  the oracle's direct atom and box sums, VEGAS 10 x 100,352 and Gauss-Kronrod
  (tolerance 1e-4) mixed against FP64, and the oracle's VEGAS on the FP64 grid.
* 5,000-atom subunit on a grid of 200 docked as a 1,000-copy helix, 800 q, MC
  over 2 x 10^6 directions: mixed against FP64 and the closed form at q = 0;
  the oracle's docked MC on the same grids.
* 512-request serving stream, every request its own structure (500..200,000
  atoms): alone against in the mix (bit-identical), mixed against FP64, and
  eight requests (largest atom count, largest grid) against the oracle.
* 16 fit sessions (2,000..20,000-atom subunits on grids of 150..250, 60..1,980
  helix or icosahedral copies, 600 q): one evaluation each against the oracle's
  docked MC on the downloaded grids, chi^2 against the host's.

Directions are keyed by (seed, direction, shell layer), so the oracle can check
the q values of a few shell layers of a full-size average exactly.
Tolerances: FP64 mode 1e-6 relative on I(q) (grid nodes 1e-9 of the shell's RMS
amplitude); mixed 1e-4 on I(q) (grid nodes 2e-5 of the shell's RMS amplitude).
"""
import os
import sys
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FP64_TOL = 1e-6
MIXED_TOL = 1e-4


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def rel(a, b):
    return float(np.max(np.abs(np.asarray(a) - np.asarray(b)) / np.abs(np.asarray(b))))


def sample_nodes(O, gs, qmax, per_shell=48, nshells=40, seed=0):
    """Node indices: the origin, and per_shell nodes in each of ~nshells shells
    (always the first three and the last two), among them both poles, the
    equator row (when 3i is even) and random (theta row, phi) pairs."""
    N = gs // 2 + 3
    rng = np.random.default_rng(seed)
    shells = sorted(set([1, 2, 3, N - 1, N] + [int(x) for x in np.linspace(1, N, nshells)]))
    idx, shell_of = [0], [0]
    for i in shells:
        picks = [(0, 0), (0, 3 * i), (3 * i, 0), (3 * i, 5)]
        if (3 * i) % 2 == 0:
            picks += [(3 * i // 2, 0), (3 * i // 2, 3 * i), (3 * i // 2, 1)]
        while len(picks) < per_shell:
            picks.append((int(rng.integers(0, 3 * i + 1)), int(rng.integers(0, 6 * i))))
        for t, p in picks:
            idx.append(O.index_from_indices(i, t, p % (6 * i)))
            shell_of.append(i)
    idx = np.array(idx, dtype=np.int64)
    qv = np.array([O.qvector_from_index(gs, qmax, int(k)) for k in idx])
    return idx, np.array(shell_of), qv


def node_errors(vals, ref, shell_of):
    """Per shell: max |vals - ref| over the sampled nodes / the RMS of |ref| there."""
    worst = 0.0
    for i in np.unique(shell_of):
        m = shell_of == i
        scale = np.sqrt(np.mean(np.abs(ref[m]) ** 2))
        worst = max(worst, float(np.max(np.abs(vals[m] - ref[m])) / scale))
    return worst


def grid_values(g, idx):
    d = g.data
    return d[2 * idx] + 1j * d[2 * idx + 1]


def layer_subset(q, step, layers):
    """Indices of the q values that fall in the given shell layers (q in
    (l step, (l+1) step], q = 0 in layer 0)."""
    lay = np.maximum(np.ceil(q / step) - 1, 0).astype(int)
    return np.nonzero(np.isin(lay, layers))[0]


def oracle_ions(O, coef9, rad, ion, sol=333.0):
    return O.Ions(coef9, rad, np.bincount(ion, minlength=len(coef9)), sol, 1.0,
                  O.CALC_ATOMIC_FORMFACTORS | O.CALC_DUMMY_SOLVENT)


# ---------------------------------------------------------------- mesh builder
def _mesh_case(kind, seed=3):
    """(atoms xyz, elements, layer (dims, com), excluded (dims, com), voxel, grid size, qmax) of shapes
    that the frequency-mesh builder has to place right."""
    rng = np.random.default_rng(seed)
    el4 = np.array(["C", "N", "O", "S"])
    none = (np.zeros((0, 3), np.int32), np.zeros((0, 3)))

    def atoms(n, half, shift=(0, 0, 0), el=el4):
        return rng.uniform(-1, 1, (n, 3)) * half + shift, el[rng.integers(0, len(el), n)]

    def boxes(n, most, half, shift=(0, 0, 0)):
        return rng.integers(1, most + 1, (n, 3)).astype(np.int32), rng.uniform(-1, 1, (n, 3)) * half + shift

    if kind == "slab":  # one axis without extent
        return (*atoms(9001, (5.0, 0.0, 3.0)), none, none, 0.05, 60, 5.0)
    if kind == "apart":  # two clusters far from the origin and from each other
        a, b = atoms(4000, (1.0, 1.0, 1.0), (14.0, 3.0, -2.0)), atoms(3001, (1.0, 1.0, 1.0), (5.0, -6.0, 9.0))
        return (np.concatenate([a[0], b[0]]), np.concatenate([a[1], b[1]]), none, none, 0.05, 90, 4.0)
    if kind == "boxes":  # both box sets, edges up to 2.4 nm, and as many atoms
        return (*atoms(1500, (3.0, 3.0, 3.0), (1.0, 0.0, 0.0)), boxes(1500, 24, (3.0, 3.0, 3.0), (1.0, 0.0, 0.0)),
                boxes(700, 7, (2.0, 3.0, 1.0)), 0.1, 70, 4.0)
    if kind == "boxes alone":
        return (np.zeros((1, 3)), np.array(["C"]), boxes(9000, 3, (4.0, 2.0, 3.0)), none, 0.05, 60, 6.0)
    if kind == "coarse grid":  # nodes further apart than the frequency mesh's points
        return (*atoms(30011, (6.0, 6.0, 6.0)), none, none, 0.05, 44, 6.5)
    if kind == "fine grid":
        return (*atoms(2000, (1.2, 1.2, 1.2)), none, none, 0.05, 150, 5.0)
    el12 = np.array(["H", "C", "N", "O", "P", "S", "Na", "Mg", "Cl", "K", "Ca", "Zn"])
    return (*atoms(8000, (3.0, 3.5, 4.0), (0, 0, 0), el12), none, none, 0.05, 70, 7.0)


@pytest.mark.parametrize("kind", ["slab", "apart", "boxes", "boxes alone", "coarse grid", "fine grid", "12 ions"])
def test_mesh_builder_vs_oracle(dplus, oracle, kind, monkeypatch):
    """Grids built through the frequency mesh (also those that the direct builder takes at this size,
    with few nodes or many box pieces) against the oracle's direct sums at sampled nodes.
    Tolerances of the shell's RMS: the mixed windows' 6e-8 per axis and side, FP32 sums of 72
    terms (1e-7) and the largest of ~2,000 nodes make 2e-6, times 5; FP64 6e-14 times 16."""
    import dplus_mi355x.synth as S
    O = oracle
    xyz, el, layer, excl, vox, gs, qmax = _mesh_case(kind)
    coef9, rad, ion, _ = S.structure_tables(el)
    flags = 0 if kind == "boxes alone" else 3
    idx, shell_of, qv = sample_nodes(O, gs, qmax)
    ref = np.zeros(len(idx), complex)
    if flags:
        ref += O.amp_atoms(xyz, ion, oracle_ions(O, coef9, rad, ion), qv)
    for (dims, com), contrast in ((layer, 33.3), (excl, -333.0)):
        if len(dims):
            ref += O.amp_boxes(dims, com, vox, contrast, qv)
    st = dplus.Structure(xyz, ion, coef9, rad, sol_ed=333.0, flags=flags, scale=0.5, box_dims=layer[0],
                         box_com=layer[1], vox_step=vox, box_contrast=33.3, excl_dims=excl[0], excl_com=excl[1],
                         excl_contrast=-333.0)
    for prec, tol in ((0, 1e-12), (1, 1e-5)):
        g = dplus.Grid(gs, qmax, prec)
        monkeypatch.setenv("DPLUS_BUILD_ROUTE", "mesh")
        assert st.build_route(g) == "mesh"
        st.build(g, host_copy=True)
        vals = grid_values(g, idx)
        e = node_errors(vals, 0.5 * ref, shell_of)
        say(f"  [mesh] {kind}, precision {prec}: nodes max err / shell RMS {e:.3e}")
        assert e < tol
        first = g.data.copy()
        st.build(g, host_copy=True)
        assert np.array_equal(first, g.data)


@pytest.mark.parametrize("n,gs,qmax,half,shift", [(2000, 100, 5.0, (3.0, 3.0, 3.0), 0.0), (5000, 120, 6.1, (3.5, 2.7, 2.2), 0.0),
                                                  (2000, 40, 3.0, (1.5, 1.5, 1.5), 0.0),
                                                  (4000, 90, 4.0, (1.0, 1.0, 1.0), (14.0, 3.0, -2.0))])
def test_fp64_mesh_is_as_precise_as_direct_sums(dplus, n, gs, qmax, half, shift, monkeypatch):
    """FP64 grids through the mesh and by direct sums against 80-bit sums at 24 nodes of 17 shells:
    the median over the shells of |dA| / |A| of the mesh is no larger than the direct builder's (a
    quarter allowed for the sampled nodes; a table of six digits less would be twice or more)."""
    import dplus_mi355x.synth as S
    LD = np.longdouble
    pi = LD("3.14159265358979323846264338327950288")
    rng = np.random.default_rng(n + gs)
    xyz = rng.normal(size=(n, 3))
    xyz *= np.array(half) * rng.uniform(0, 1, (n, 1)) ** (1 / 3) / np.linalg.norm(xyz, axis=1)[:, None]
    xyz = xyz + shift
    coef9, rad, ion, _ = S.structure_tables(np.array(["C"] * n))
    N = gs // 2 + 3
    idx, shell, qv = [], [], []
    for i in sorted(set(range(1, 6)) | set(np.linspace(1, N, 14).astype(int).tolist())):
        for _ in range(24):
            j, k = int(rng.integers(0, 3 * i + 1)), int(rng.integers(0, 6 * i))
            idx.append(1 + 6 * (i - 1) * i * i + j * 6 * i + k)
            shell.append(i)
            q, th, ph = LD(i) * LD(qmax) / LD(gs // 2), pi * j / (3 * i), pi * k / (3 * i)
            qv.append([q * np.sin(th) * np.cos(ph), q * np.sin(th) * np.sin(ph), q * np.cos(th)])
    shell, qv = np.array(shell), np.array(qv, dtype=LD)
    ref = np.zeros((len(idx), 2), LD)
    for c in range(0, n, 500):
        p = qv @ xyz[c:c + 500].astype(LD).T
        ref += np.stack([np.cos(p).sum(1), np.sin(p).sum(1)], axis=1)
    st = dplus.Structure(xyz, ion, coef9, rad, sol_ed=0.0, flags=dplus.CALC_ATOMIC_FORMFACTORS)
    med = {}
    for route in ("mesh", "direct"):
        monkeypatch.setenv("DPLUS_BUILD_ROUTE", route)
        g = dplus.Grid(gs, qmax, 0)
        assert st.build_route(g) == route
        st.build(g, host_copy=True)
        a = np.stack([g.data[0::2][idx], g.data[1::2][idx]], axis=1).astype(LD)
        e = []
        for i in np.unique(shell):
            m = shell == i
            f = (a[m] * ref[m]).sum() / (ref[m] ** 2).sum()  # the shell's form factor
            e.append(float(np.sqrt(((a[m] - f * ref[m]) ** 2).sum() / ((f * ref[m]) ** 2).sum())))
        med[route] = np.median(e)
    say(f"  [80-bit] {n} atoms, grid {gs}: mesh {med['mesh']:.2e}, direct {med['direct']:.2e}")
    assert med["mesh"] <= 1.25 * med["direct"]


def test_one_large_box_stays_whole(dplus, oracle, monkeypatch):
    """A box that would make a million pieces beside 500 atoms: the structure keeps it whole and its
    grids are direct sums whatever the route asked for; a box of a tenth of its edge goes through the
    mesh.  FP64 nodes against the oracle, and the mesh's mixed ones (the direct builder's mixed sinc
    of 45 rad has FP32's error of that angle, which the mesh's bound does not cover)."""
    import dplus_mi355x.synth as S
    rng = np.random.default_rng(5)
    xyz, el = rng.uniform(-1, 1, (500, 3)), np.array(["C", "N", "O", "S"])[rng.integers(0, 4, 500)]
    coef9, rad, ion, _ = S.structure_tables(el)
    monkeypatch.setenv("DPLUS_BUILD_ROUTE", "mesh")
    gs, qmax = 24, 3.0
    idx, shell_of, qv = sample_nodes(oracle, gs, qmax)
    atoms = oracle.amp_atoms(xyz, ion, oracle_ions(oracle, coef9, rad, ion), qv)
    for edge, route in ((300, "direct"), (30, "mesh")):
        dims, com = np.array([[edge] * 3], np.int32), np.array([[0.1, -0.2, 0.3]])
        st = dplus.Structure(xyz, ion, coef9, rad, sol_ed=333.0, flags=3, box_dims=dims, box_com=com, vox_step=0.1,
                             box_contrast=33.3)
        ref = atoms + oracle.amp_boxes(dims, com, 0.1, 33.3, qv)
        for prec, tol in ((0, 1e-12), (1, 1e-5)):
            g = dplus.Grid(gs, qmax, prec)
            assert st.build_route(g) == route
            st.build(g, host_copy=True)
            if prec == 0 or route == "mesh":
                assert node_errors(grid_values(g, idx), ref, shell_of) < tol


ARENA_BUILD = r"""
#include "device.hpp"
using namespace dplus;
// a build whose buffers come from `size` bytes of one allocation: 0, or an error's code
extern "C" int build_in_arena(void *st, void *gh, size_t size, int *mesh, size_t *mesh_bytes, size_t *used) {
    const Structure &S = *(const Structure *)st;
    Grid &g = *(Grid *)gh;
    hipStream_t s = Device::get().stream;
    MeshPlan mp;
    MeshSizes mz;
    *mesh_bytes = S.mesh_route(g, mp, mz) ? mz.bytes : 0;
    Arena a;
    if (hipMalloc((void **)&a.base, size) != hipSuccess) return -1;
    a.size = size;
    set_arena(&a);
    int rc = 0;
    try {
        Structure::Pending P;
        const BuildShape sh = S.shape_for(g);
        BuildJob J = S.prepare(g, sh.slices, P, s);
        S.launch(g, J, sh.wg, P, s);
        S.enqueue_finish(g, P, s, false);
        check_hip(hipStreamSynchronize(s), "build");
        *mesh = P.mesh ? 1 : 0;
        *used = a.used;
    } catch (const Error &e) {
        (void)hipStreamSynchronize(s);
        rc = e.code;
    }
    set_arena(nullptr);
    (void)hipFree(a.base);
    return rc;
}
"""


@pytest.mark.parametrize("prec", [0, 1])
def test_build_without_room_for_the_mesh_is_direct(dplus, prec, tmp_path, monkeypatch):
    """A build that the mesh would take, where its workspace cannot be had but the direct builder's
    can: the bits of a direct build.  With room for the workspace, the mesh's."""
    import ctypes
    import subprocess
    import dplus_mi355x.synth as S
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    pkg, lib = os.path.join(root, "dplus-dev_amd"), os.path.join(root, "dplus-dev_amd", "dplus_mi355x")
    src, out = tmp_path / "arena.cpp", tmp_path / "libarena.so"
    src.write_text(ARENA_BUILD)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(pkg, "csrc"), "-I" + os.path.join(root, "include"), str(src), "-L" + lib,
                    "-ldplus_mi355x", "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + lib, "-o", str(out)], check=True)
    fn = ctypes.CDLL(str(out)).build_in_arena
    xyz, el, _, _, _, gs, qmax = _mesh_case("coarse grid")
    coef9, rad, ion, _ = S.structure_tables(el)
    st = dplus.Structure(xyz, ion, coef9, rad, sol_ed=333.0, flags=3)
    want = {}
    for route in ("mesh", "direct"):
        monkeypatch.setenv("DPLUS_BUILD_ROUTE", route)
        g = dplus.Grid(gs, qmax, prec)
        st.build(g, host_copy=True)
        want[route] = g.data.copy()
    assert not np.array_equal(want["mesh"], want["direct"])
    monkeypatch.setenv("DPLUS_BUILD_ROUTE", "mesh")
    mesh, nb, used = ctypes.c_int(), ctypes.c_size_t(), ctypes.c_size_t()
    for size, route in ((256 << 20, "mesh"), (10 << 20, "direct")):
        g = dplus.Grid(gs, qmax, prec)
        rc = fn(st._h, g.handle, ctypes.c_size_t(size), ctypes.byref(mesh),
                ctypes.byref(nb), ctypes.byref(used))
        say(f"  [arena] precision {prec}, {size >> 20} MB, workspace {nb.value}: rc {rc}, mesh {mesh.value}, used {used.value}")
        assert rc == 0 and 10 << 20 < nb.value and used.value <= size
        assert mesh.value == (route == "mesh")
        g.download()
        assert np.array_equal(g.data, want[route])
    # no room for either: refused as before
    g = dplus.Grid(gs, qmax, prec)
    assert fn(st._h, g.handle, ctypes.c_size_t(1 << 20), ctypes.byref(mesh),
              ctypes.byref(nb), ctypes.byref(used)) == 21



# ---------------------------------------------------------------- 50,000 atoms + hydration, grid 250
def test_50k_atoms_hydration_grid250_vs_oracle(dplus, oracle):
    import dplus_mi355x.synth as S
    O = oracle
    say("[case] 50k atoms + 0.3 nm hydration layer, grid 250, qmax 7.5, 1000 q")
    t0 = time.time()
    xyz, el = S.walk_structure(2024, 50000, (8.0, 6.0, 5.0))
    coef9, rad, ion, _ = S.structure_tables(el)
    dims, com = dplus.hydration_boxes(xyz, rad[ion], probe=0.14, thickness=0.3, vox=0.05)
    vox, contrast, gs, qmax = 0.05, 366.3 - 333.0, 250, 7.5
    say(f"  {len(xyz)} atoms, {len(dims)} boxes, host prep {time.time() - t0:.1f} s")
    st = dplus.Structure(xyz, ion, coef9, rad, sol_ed=333.0, c1=1.0, flags=3, box_dims=dims, box_com=com,
                         vox_step=vox, box_contrast=contrast)
    grids = {}
    for prec in (0, 1):
        say(f"  [step] build precision {prec}")
        g = dplus.Grid(gs, qmax, prec)
        st.build(g, host_copy=True)
        grids[prec] = g
    # sampled nodes against the oracle's direct sums
    idx, shell_of, qv = sample_nodes(O, gs, qmax)
    assert len(idx) >= 2000
    say(f"  [step] oracle direct sums at {len(idx)} nodes")
    ref = O.amp_atoms(xyz, ion, oracle_ions(O, coef9, rad, ion), qv) + O.amp_boxes(dims, com, vox, contrast, qv)
    for prec, tol in ((0, 1e-9), (1, 2e-5)):
        vals = grid_values(grids[prec], idx)
        e = node_errors(vals, ref, shell_of)
        e0 = abs(vals[0] - ref[0]) / abs(ref[0])
        say(f"  precision {prec}: nodes max err / shell RMS {e:.3e}, origin {e0:.3e}")
        assert e < tol and e0 < tol
    # VEGAS 10 x 100,352 and Gauss-Kronrod, mixed against FP64
    q = np.linspace(0.0, qmax, 1000)
    curves, gks = {}, {}
    for prec in (0, 1):
        say(f"  [step] VEGAS and GK precision {prec}")
        curves[prec], _ = dplus.orientation_average(dplus.Docking.single(grids[prec]), q, method=dplus.OA_VEGAS,
                                                    seed=7, vegas_iterations=10, vegas_points_per_bin=98)
        gks[prec], _ = dplus.orientation_average(dplus.Docking.single(grids[prec]), q, method=dplus.OA_GK,
                                                 eps=1e-4, gk_max_depth=8)
    ev, eg = rel(curves[1], curves[0]), rel(gks[1], gks[0])
    say(f"  mixed vs FP64: VEGAS {ev:.3e}, GK {eg:.3e}")
    assert ev < MIXED_TOL and eg < MIXED_TOL
    # the oracle's VEGAS on the downloaded FP64 grid, on the q of five shell layers
    step = grids[0].step_size
    sub = layer_subset(q, step, [0, 1, 40, 90, 124])
    say(f"  [step] oracle VEGAS on {len(sub)} q")
    d64 = O.Docked.single(gs, qmax, grids[0].data, grids[0].interp)
    orc, _ = O.vegas_oa(d64, q[sub], 7, 10, 98)
    e64, e32 = rel(curves[0][sub], orc), rel(curves[1][sub], orc)
    say(f"  VEGAS vs oracle: FP64 {e64:.3e}, mixed {e32:.3e}")
    assert e64 < FP64_TOL and e32 < MIXED_TOL


# ---------------------------------------------------------------- 1,000-copy helix, 2 x 10^6 directions
def test_helix_of_1000_copies_2e6_directions(dplus, oracle):
    """A 5,000-atom subunit (2.5 nm sphere) on a grid of 200 (qmax 6) docked as a
    1,000-copy helix (radius 12 nm, rise 0.9 nm, twist 27.7 deg; translations to
    ~450 nm), 800 q on [0, 6], MC over 2 x 10^6 directions in both precisions:
    mixed within 1e-4 of FP64 and I(0) = (1000 A(0))^2; the oracle's docked MC on
    the downloaded grids (8 shell layers, 4,096 directions)."""
    import dplus_mi355x.synth as S
    O = oracle
    say("[case] 5000-atom subunit gs 200, helix of 1000 copies, 800 q, MC 2e6 directions")
    xyz, el = S.walk_structure(3, 5000, (2.5, 2.5, 2.5))
    coef9, rad, ion, _ = S.structure_tables(el)
    rot, nt, tr = S.rows_to_docking(S.helix_rows(1000, 12.0, 0.9, 27.7))
    q = np.linspace(0.0, 6.0, 800)
    st = dplus.Structure(xyz, ion, coef9, rad, sol_ed=333.0, flags=3)
    out, grids = {}, {}
    for prec in (0, 1):
        g = dplus.Grid(200, 6.0, prec)
        st.build(g, host_copy=True)
        grids[prec] = g
        say(f"  [step] MC 2e6 directions precision {prec}")
        t0 = time.time()
        I, stt = dplus.orientation_average(dplus.Docking([(g, rot, nt, tr)]), q, seed=5, max_dirs=2_000_000,
                                           chunk=8192)
        say(f"    {stt.dirs_used} directions in {time.time() - t0:.1f} s")
        assert stt.dirs_used >= 2_000_000
        out[prec] = I
        closed = (1000.0 * float(g.data[0])) ** 2
        assert I[0] == pytest.approx(closed, rel=1e-12 if prec == 0 else 1e-4)
    err = rel(out[1], out[0])
    say(f"  mixed vs FP64 {err:.3e}")
    assert err < MIXED_TOL
    step = grids[0].step_size
    sub = layer_subset(q, step, [0, 1, 5, 20, 45, 70, 95, 99])
    say(f"  [step] oracle docked MC on {len(sub)} q, 4096 directions")
    for prec, tol in ((0, FP64_TOL), (1, MIXED_TOL)):
        g = grids[prec]
        mine, _ = dplus.orientation_average(dplus.Docking([(g, rot, nt, tr)]), q[sub], seed=9, max_dirs=4096,
                                            chunk=4096)
        ref, _ = O.mc_oa(O.Docked([(200, 6.0, g.data, g.interp, rot, nt, tr)]), q[sub], 9, 4096, 4096)
        e = rel(mine, ref)
        say(f"    precision {prec} vs oracle {e:.3e}")
        assert e < tol


# ---------------------------------------------------------------- 512-request serving stream
def test_serving_stream_512_distinct_structures(dplus, oracle):
    from dplus_mi355x.serving import Engine
    import dplus_mi355x.synth as S
    O = oracle
    t0 = time.time()
    _, reqs, _ = S.serving_workload(512)
    say(f"[case] serving: 512 requests, {sum(n for *_, n in reqs)} atoms in 512 distinct structures "
        f"(prepared in {time.time() - t0:.1f} s)")
    say("  [step] mixed, one request at a time on one stream, eager launches")
    e1 = Engine(hbm_budget_bytes=200 * 10 ** 9, streams=1, graphs=False)
    alone = [e1.wait(e1.submit(q, precision=dplus.PRECISION_MIXED, **kw))[0] for q, kw, _ in reqs]
    e1.close()
    say("  [step] mixed, all submitted at once on 16 streams, one captured graph per request")
    e16 = Engine(hbm_budget_bytes=200 * 10 ** 9, streams=16, graphs=True)
    tickets = [e16.submit(q, precision=dplus.PRECISION_MIXED, **kw) for q, kw, _ in reqs]
    mix = [e16.wait(t)[0] for t in tickets]
    st = e16.stats()
    e16.close()
    say(f"    max concurrent {st['max_concurrent']}, cache hits {st['cache_hits']}, graph launches "
        f"{st['graph_launches']} (updated {st['graph_updates']})")
    assert st["max_concurrent"] > 1 and st["graph_launches"] == len(reqs)
    for i, (a, m) in enumerate(zip(alone, mix)):
        assert np.array_equal(a, m), i
    say("  [step] FP64, 16 streams")
    e64 = Engine(hbm_budget_bytes=200 * 10 ** 9, streams=16)
    tickets = [e64.submit(q, precision=dplus.PRECISION_FP64, **kw) for q, kw, _ in reqs]
    fp64 = [e64.wait(t)[0] for t in tickets]
    e64.close()
    errs = [rel(m, f) for m, f in zip(mix, fp64)]
    say(f"  mixed vs FP64: max {max(errs):.3e}")
    assert max(errs) < MIXED_TOL
    # eight requests against the oracle: the largest atom count, the largest grid,
    # and six more of both averaging methods
    n_at = np.array([n for *_, n in reqs])
    gsz = np.array([kw["grid_size"] for _, kw, _ in reqs])
    chosen = [int(np.argmax(n_at)), int(np.argmax(gsz))]
    for k in np.argsort(n_at)[::64]:
        if int(k) not in chosen and len(chosen) < 8:
            chosen.append(int(k))
    for k in chosen:
        q, kw, n = reqs[k]
        p = kw["pdb"]
        gs, qmax = kw["grid_size"], kw["qmax"]
        say(f"  [step] oracle: request {k}, {n} atoms, grid {gs}, qmax {qmax:.2f}, {len(q)} q, "
            f"{'MC' if kw['method'] == dplus.OA_MC else 'VEGAS'}")
        g = dplus.Grid(gs, qmax, dplus.PRECISION_FP64)
        dplus.Structure(p["xyz"], p["ion"], p["coef9"], p["rad"], sol_ed=p["sol_ed"], flags=p["flags"]).build(
            g, host_copy=True)
        idx, shell_of, qv = sample_nodes(O, gs, qmax, per_shell=12, nshells=12, seed=k)
        ref = O.amp_atoms(p["xyz"], p["ion"], oracle_ions(O, p["coef9"], p["rad"], p["ion"], p["sol_ed"]), qv)
        assert node_errors(grid_values(g, idx), ref, shell_of) < 1e-9
        step = g.step_size
        nl = int(np.ceil(q[-1] / step))
        sub = layer_subset(q, step, sorted({0, 1, nl // 3, (2 * nl) // 3, nl - 1}))
        dock = O.Docked.single(gs, qmax, g.data, g.interp)
        if kw["method"] == dplus.OA_MC:
            orc, _ = O.mc_oa(dock, q[sub], kw["seed"], kw["max_dirs"], kw["chunk"])
        else:
            orc, _ = O.vegas_oa(dock, q[sub], kw["seed"], kw["vegas_iterations"], kw["vegas_points_per_bin"])
        e64, e32 = rel(fp64[k][sub], orc), rel(mix[k][sub], orc)
        say(f"    vs oracle on {len(sub)} q: FP64 {e64:.3e}, mixed {e32:.3e}")
        assert e64 < FP64_TOL and e32 < MIXED_TOL


# ---------------------------------------------------------------- 16 fit sessions
def test_16_fit_sessions_vs_oracle(dplus, oracle):
    from dplus_mi355x.serving import FitSession
    import dplus_mi355x.synth as S
    O = oracle
    t0 = time.time()
    plans = S.session_plans(16, 5)
    say(f"[case] 16 fit sessions (prepared in {time.time() - t0:.1f} s): grids "
        f"{[p['gs'] for p in plans]}, copies {[p['copies'] for p in plans]}")
    qmax, nq, dirs = 5.0, 600, 2048
    q = np.linspace(0.01, qmax, nq)
    rng = np.random.default_rng(3)
    for si, p in enumerate(plans):
        say(f"  [step] session {si}: {p['kind']}, {len(p['leaves'])} subunits "
            f"({[len(l[0]) for l in p['leaves']]} atoms), grid {p['gs']}, {p['copies']} copies")
        grids = []
        for xyz, ion, coef9, rad in p["leaves"]:
            g = dplus.Grid(p["gs"], qmax, dplus.PRECISION_MIXED)
            dplus.Structure(xyz, ion, coef9, rad, sol_ed=333.0, flags=3).build(g, host_copy=True)
            grids.append(g)
        y = rng.uniform(0.5, 2.0, nq)
        sig = rng.uniform(0.05, 0.2, nq)
        sess = FitSession(grids, q, y, sig, seed=p["seed"], directions=dirs)
        pl = S.session_placements(p, 1.03, 1.5)
        I, c2 = sess.evaluate(pl, fit_scale=2e-7, fit_constant=0.3)
        sess.close()
        host = float(np.sum(((2e-7 * I + 0.3 - y) / sig) ** 2))
        assert c2 == pytest.approx(host, rel=1e-12)
        step = grids[0].step_size
        nl = int(np.ceil(q[-1] / step))
        sub = layer_subset(q, step, [1, nl // 2, nl - 1])
        dock = O.Docked([(p["gs"], qmax, g.data, g.interp, rot, nt, tr) for g, (rot, nt, tr) in zip(grids, pl)])
        ref, _ = O.mc_oa(dock, q[sub], p["seed"], dirs, dirs)
        e = rel(I[sub], ref)
        say(f"    vs oracle on {len(sub)} q: {e:.3e}")
        assert e < MIXED_TOL
        del grids, dock
