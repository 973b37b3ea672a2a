"""The work that programs have this library do on one GPU, as cases that can be timed
and whose results can be compared.

A case is one of six kinds of call:
  curve    a resident PDB structure -> amplitude grid -> orientation average -> I(q)
  helix    a resident subunit grid docked as a helix -> Monte Carlo average -> I(q)
  session  one evaluation of a fit session (re-docked subunits, chi^2 on the device)
  ring     grid-level manual symmetry into a new grid -> VEGAS average -> I(q)
  matrix   the 2-D (q_z, q_perp) generate path over a resident grid
  stream   a burst of curve requests through the request engine
Mixed precision computes in FP32 and its curves are kept as float32; FP64 curves are
kept as float64.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "dplus-dev_amd"))

import dplus_mi355x as D  # noqa: E402
from dplus_mi355x import synth  # noqa: E402
from dplus_mi355x.grid import (Docking, Grid, Structure, azimuthal_average, dock_grid, hydration_boxes,  # noqa: E402
                               orientation_average)
from dplus_mi355x.serving import Engine, FitSession  # noqa: E402

SOLVENT, LAYER_CONTRAST, VOXEL = 333.0, 33.3, 0.05


# ------------------------------------------------------------------ the cases
def curve(name, atoms, gs, qmax, nq, method, precision="mixed", layer=False, points=0, iters=0, ppb=0, tol=0.0):
    """points: MC directions; iters, ppb: VEGAS iterations and points per bin; tol: Gauss-Kronrod."""
    return {"name": name, "kind": "curve", "atoms": atoms, "layer": layer, "gs": gs, "qmax": qmax, "nq": nq,
            "precision": precision, "method": method, "points": points, "iters": iters, "ppb": ppb, "tol": tol}


def listed():
    return [
        # the smallest request of a serving stream: latency and launches count
        curve("small_curve", 500, 30, 4.0, 200, "vegas", iters=5, ppb=4),
        # an ordinary protein at the default accuracy: 2,000 atoms, 10^6 MC directions
        curve("protein_mc", 2000, 100, 5.0, 500, "mc", points=1_000_000),
        # the same protein where a user asks for double precision
        curve("protein_mc_fp64", 2000, 100, 5.0, 500, "mc", precision="fp64", points=262_144),
        # a complex with its hydration layer, the benchmark's headline curve
        curve("complex_layer_vegas", 50_000, 250, 7.5, 1000, "vegas", layer=True, iters=10, ppb=98),
        # a hydrated protein in double precision, odd sizes
        curve("hydrated_fp64", 4999, 120, 6.1, 701, "vegas", precision="fp64", layer=True, iters=10, ppb=24),
        # the largest structure a serving stream carries
        curve("largest_mc", 199_999, 110, 8.0, 997, "mc", points=65_536),
        # the adaptive quadrature users take for publication curves
        curve("protein_gk", 5000, 150, 6.0, 501, "gk", tol=1e-3),
        # a microtubule-like helix: 1,000 copies of a subunit
        {"name": "helix_mc", "kind": "helix", "atoms": 5000, "gs": 200, "qmax": 6.0, "nq": 800, "copies": 1000,
         "radius": 12.0, "rise": 0.9, "twist": 27.7, "points": 65_536, "precision": "mixed"},
        # one evaluation of a fitting loop: a capsid-like shell of two subunits
        {"name": "capsid_session", "kind": "session", "atoms": 6000, "leaves": 2, "gs": 150, "qmax": 5.0, "nq": 600,
         "copies": 900, "radius": 14.0, "points": 8192},
        # a 13-unit ring assembled on a grid of its own
        {"name": "ring_grid", "kind": "ring", "atoms": 3000, "gs": 150, "qmax": 5.0, "nq": 500, "copies": 13,
         "radius": 9.0, "iters": 5, "ppb": 16, "precision": "mixed"},
        # a 2-D detector pattern of an oriented sample
        {"name": "matrix_2d", "kind": "matrix", "atoms": 3000, "gs": 100, "qmax": 5.0, "side": 64, "nphi": 1024,
         "precision": "mixed"},
        # a burst of requests on the engine, sizes as a serving stream mixes them
        {"name": "request_stream", "kind": "stream", "requests": 64, "least": 500, "most": 60_000},
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["curve"] * 6 + ["helix", "session", "ring", "matrix", "stream"])
    if kind == "curve":
        precision = rng.choice(["mixed", "mixed", "mixed", "fp64"])
        method = rng.choice(["mc", "vegas", "vegas", "gk"])
        layer = rng.random() < 0.3
        atoms = _log(rng, 500, (60_000 if layer else 200_000) if precision == "mixed" else 6000)
        qmax = round(rng.uniform(2.0, 8.0), 2)
        # the grid size that fits the structure's diameter, up to three times finer
        diameter = 2.5 * (3.0 * atoms / (4.0 * math.pi * 50.0)) ** (1.0 / 3.0)
        need = 2.0 * qmax * diameter / math.pi + 3.0
        gs = 2 * int(min(250 if precision == "mixed" else 120, max(20, need * rng.uniform(1.0, 2.5))) / 2)
        return {"kind": "curve", "atoms": atoms, "layer": layer, "gs": gs, "qmax": qmax, "nq": _log(rng, 100, 1000),
                "precision": precision, "method": method, "points": _log(rng, 8192, 1_000_000) if method == "mc" else 0,
                "iters": rng.randint(3, 10) if method == "vegas" else 0,
                "ppb": _log(rng, 4, 98) if method == "vegas" else 0,
                "tol": 10.0 ** rng.uniform(-4, -2) if method == "gk" else 0.0}
    qmax = round(rng.uniform(3.0, 6.0), 2)
    if kind == "helix":
        return {"kind": kind, "atoms": _log(rng, 1000, 10_000), "gs": 2 * rng.randint(40, 100), "qmax": qmax,
                "nq": rng.randint(200, 800), "copies": rng.randint(40, 1000), "radius": rng.uniform(6.0, 12.0),
                "rise": rng.uniform(0.2, 0.9), "twist": rng.uniform(20.0, 40.0), "points": _log(rng, 8192, 65_536),
                "precision": rng.choice(["mixed", "mixed", "fp64"])}
    if kind == "session":
        return {"kind": kind, "atoms": _log(rng, 2000, 8000), "leaves": rng.randint(1, 3), "gs": 2 * rng.randint(60, 100),
                "qmax": qmax, "nq": rng.randint(200, 600), "copies": 60 * rng.randint(1, 15),
                "radius": rng.uniform(10.0, 20.0), "points": 8192}
    if kind == "ring":
        return {"kind": kind, "atoms": _log(rng, 1000, 5000), "gs": 2 * rng.randint(40, 75), "qmax": qmax,
                "nq": rng.randint(100, 500), "copies": rng.randint(5, 24), "radius": rng.uniform(5.0, 10.0),
                "iters": rng.randint(3, 6), "ppb": rng.randint(4, 32), "precision": rng.choice(["mixed", "mixed", "fp64"])}
    if kind == "matrix":
        return {"kind": kind, "atoms": _log(rng, 1000, 5000), "gs": 2 * rng.randint(30, 75), "qmax": qmax,
                "side": rng.randint(20, 90), "nphi": _log(rng, 64, 2048), "precision": rng.choice(["mixed", "mixed", "fp64"])}
    return {"kind": kind, "requests": rng.randint(8, 64), "least": 500, "most": _log(rng, 5000, 60_000)}


# ------------------------------------------------------------------ inputs
def _structure(seed, atoms, layer=False):
    """A random-walk chain in an ellipsoid of 50 atoms / nm^3, C/N/O/S, with the dummy-atom solvent."""
    k = (3.0 * atoms / (4.0 * math.pi * 50.0)) ** (1.0 / 3.0)
    axes = (1.29 * k, 0.97 * k, 0.80 * k) if layer else (k, k, k)
    xyz, el = synth.walk_structure(seed, atoms, axes)
    coef9, rad, ion, _ = synth.structure_tables(el)
    pdb = dict(xyz=xyz, ion=ion, coef9=coef9, rad=rad, sol_ed=SOLVENT, c1=1.0, flags=3, scale=1.0)
    if layer:
        dims, com = hydration_boxes(xyz, rad[ion], probe=0.14, thickness=0.3, vox=VOXEL)
        pdb.update(box_dims=dims, box_com=com, vox_step=VOXEL, box_contrast=LAYER_CONTRAST)
    return pdb


def _precision(case):
    return D.PRECISION_FP64 if case.get("precision") == "fp64" else D.PRECISION_MIXED


def _ring_rows(case, rng):
    n = case["copies"]
    ang = 2.0 * np.pi * np.arange(n) / n
    z = rng.normal(scale=0.3, size=n)
    return np.stack([case["radius"] * np.cos(ang), case["radius"] * np.sin(ang), z, rng.uniform(0, 30, n),
                     rng.uniform(0, 30, n), np.rad2deg(ang)], axis=1)


def _helix_rows(case, rng):
    return synth.helix_rows(case["copies"], case["radius"] * (1.0 + 0.01 * rng.random()), case["rise"],
                            case["twist"] + 0.01 * rng.random())


def _requests(case, seed):
    """(q, submit arguments) of a burst: sizes log-uniform, grid size from qmax and the diameter."""
    rng = np.random.default_rng(seed)
    sizes = np.random.default_rng(17).uniform(math.log(case["least"]), math.log(case["most"]), case["requests"])
    out = []
    for i, s in enumerate(np.exp(sizes)):
        pdb = _structure(int(rng.integers(1 << 30)), int(round(s)))
        shape = np.random.default_rng(1000 + i)
        qmax = float(shape.uniform(2.0, 8.0))
        size = 2.0 * (3.0 * s / (4.0 * math.pi * 50.0)) ** (1.0 / 3.0)
        kw = dict(pdb=pdb, grid_size=int(math.ceil((2.0 * qmax * size / math.pi + 3.0) / 10.0) * 10), qmax=qmax,
                  seed=int(rng.integers(1 << 30)))
        if shape.random() < 0.5:
            kw.update(method=D.OA_MC, max_dirs=65_536)
        else:
            kw.update(method=D.OA_VEGAS, vegas_iterations=5, vegas_points_per_bin=4)
        out.append((np.linspace(0.0, qmax, int(shape.integers(200, 1001))), kw))
    return out


def _inputs(case, seed):
    """The host data of a case, as `prepare` and `exact` take it."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    I = {"seed": int(rng.integers(1 << 30))}
    if kind == "stream":
        I["requests"] = _requests(case, seed)
        return I
    I["pdbs"] = [_structure(int(rng.integers(1 << 30)), case["atoms"], case.get("layer", False))
                 for _ in range(case.get("leaves", 1))]
    I["q"] = np.linspace(0.0, case["qmax"], case["nq"]) if kind != "matrix" else None
    if kind == "helix":
        I["placements"] = [synth.rows_to_docking(_helix_rows(case, rng))]
    elif kind == "ring":
        I["placements"] = [synth.rows_to_docking(_ring_rows(case, rng))]
    elif kind == "session":
        n, per = case["leaves"], case["copies"]
        I["placements"] = [synth.rows_to_docking(synth.icosahedral_rows(case["radius"] * (1.0 + 0.05 * l), per,
                                                                        seed=int(rng.integers(1 << 30))))
                           for l in range(n)]
        I["data"] = 1e9 * np.exp(-I["q"]) * (1.0 + 0.02 * rng.normal(size=case["nq"]))
        I["sigma"] = 0.02 * np.abs(I["data"]) + 1.0
    elif kind == "matrix":
        x = np.linspace(0.0, case["qmax"] / math.sqrt(2.0), case["side"])
        qz, qp = (a.ravel() for a in np.meshgrid(x, x, indexing="ij"))
        I["q"], I["theta"] = np.hypot(qz, qp), np.arctan2(qp, qz)
    return I


def prepare(case, seed):
    I = _inputs(case, seed)
    s = {"case": case, "in": I}
    kind = case["kind"]
    if kind == "stream":
        s["engine"] = Engine(hbm_budget_bytes=64 << 30, streams=16)
        return s
    s["structures"] = [Structure(**p) for p in I["pdbs"]]
    s["grids"] = [Grid(case["gs"], case["qmax"], _precision(case)) for _ in I["pdbs"]]
    if kind == "curve":
        s["dock"] = Docking.single(s["grids"][0])
        return s
    for st, g in zip(s["structures"], s["grids"]):
        st.build(g)
    if kind in ("helix", "ring"):
        s["dock"] = Docking([(s["grids"][0], *I["placements"][0])])
    if kind == "ring":
        s["out"] = Grid(case["gs"], case["qmax"], _precision(case))
        s["out_dock"] = Docking.single(s["out"])
    if kind == "session":
        s["session"] = FitSession(s["grids"], I["q"], I["data"], I["sigma"], seed=I["seed"], directions=case["points"])
    if kind == "matrix":
        s["dock"] = Docking.single(s["grids"][0])
    return s


_METHOD = {"mc": D.OA_MC, "vegas": D.OA_VEGAS, "gk": D.OA_GK}


def _average(dock, I, case, method):
    if method == "mc":
        return orientation_average(dock, I["q"], method=D.OA_MC, seed=I["seed"], max_dirs=case["points"])[0]
    if method == "vegas":
        return orientation_average(dock, I["q"], method=D.OA_VEGAS, seed=I["seed"], vegas_iterations=case["iters"],
                                   vegas_points_per_bin=case["ppb"])[0]
    return orientation_average(dock, I["q"], method=D.OA_GK, eps=case["tol"], gk_max_depth=8)[0]


def _keep(case, curve):
    return curve if case.get("precision") == "fp64" else curve.astype(np.float32)


def run(state):
    case, I, kind = state["case"], state["in"], state["case"]["kind"]
    if kind == "curve":
        state["structures"][0].build(state["grids"][0])
        return _keep(case, _average(state["dock"], I, case, case["method"]))
    if kind == "helix":
        return _keep(case, _average(state["dock"], I, case, "mc"))
    if kind == "session":
        curve, chi2 = state["session"].evaluate(I["placements"])
        return {"I": curve.astype(np.float32), "chi2": np.float32(chi2)}
    if kind == "ring":
        dock_grid(state["out"], state["dock"])
        return _keep(case, _average(state["out_dock"], I, case, "vegas"))
    if kind == "matrix":
        return _keep(case, azimuthal_average(state["dock"], I["q"], I["theta"], nphi=case["nphi"], seed=I["seed"]))
    tickets = [state["engine"].submit(q, **kw) for q, kw in I["requests"]]
    # the curves one after the other
    return np.concatenate([state["engine"].wait(t)[0] for t in tickets]).astype(np.float32)


# ------------------------------------------------------------------ the work a pass cannot do without
def _points(gs):
    n = gs // 2 + 3
    return 1 + 6 * n * (n + 1) ** 2


def _layers(qmax, gs, nq):
    return min(nq, gs // 2)


def work(case):
    """Sources read, grids written (values and slopes) and read once, curves written; per grid node
    its spline (20 flops), per lookup 4 planes of 8 nodes (300 flops), per copy and q its phase (10)."""
    kind = case["kind"]
    if kind == "stream":
        sizes = np.exp(np.random.default_rng(17).uniform(math.log(case["least"]), math.log(case["most"]), case["requests"]))
        b = f = 0.0
        for i, s in enumerate(sizes):
            qmax = float(np.random.default_rng(1000 + i).uniform(2.0, 8.0))
            gs = 2.0 * qmax * 2.0 * (3.0 * s / (4.0 * math.pi * 50.0)) ** (1.0 / 3.0) / math.pi + 8.0
            P = 6.0 * (gs / 2 + 3) ** 3
            b += 16.0 * s + 32.0 * P
            f += 20.0 * P + 300.0 * gs / 2 * 20_480
        return {"bytes": b, "flops": f}
    node = 32 if case.get("precision") == "fp64" else 16
    P = _points(case["gs"])
    ng = _layers(case["qmax"], case["gs"], case.get("nq", 1))
    if kind == "curve":
        lookups = {"mc": case["points"], "vegas": case["iters"] * case["ppb"] * 1024, "gk": 225 * case["nq"] / max(1, ng)}
        return {"bytes": 16.0 * case["atoms"] + 2.0 * node * P + 8.0 * case["nq"],
                "flops": 20.0 * P + 300.0 * ng * lookups[case["method"]]}
    copies = case.get("copies", 1) * case.get("leaves", 1)
    if kind in ("helix", "session"):
        lookups = ng * case["points"] * (copies if kind == "helix" else 60 * case["leaves"])
        return {"bytes": node * P * case.get("leaves", 1), "flops": 300.0 * lookups + 10.0 * case["points"] * case["nq"] * copies}
    if kind == "ring":
        return {"bytes": 3.0 * node * P, "flops": (310.0 * copies + 20.0) * P + 300.0 * ng * case["iters"] * case["ppb"] * 1024}
    return {"bytes": 1.0 * node * P, "flops": 300.0 * case["side"] ** 2 * case["nphi"]}


# ------------------------------------------------------------------ the same results in 64 bits
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(x, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=dtype, device=_dev())


def _form_factors(pdb, q):
    """Four Gaussians and a constant less the dummy atom's Gaussian, per ion, at radius q."""
    c, rad = pdb["coef9"].reshape(-1, 9), pdb["rad"]
    s2 = (q / (40.0 * math.pi)) ** 2
    f = c[:, 8] + sum(c[:, 2 * k] * np.exp(-s2 * c[:, 2 * k + 1]) for k in range(4))
    counts = np.bincount(pdb["ion"], minlength=len(c))
    rm = np.cbrt((rad ** 3 * counts).sum() / counts.sum())
    return f - 4.0 / 3.0 * math.pi * rad ** 3 * np.exp(-(rm * q) ** 2 * 0.2067834969664667) * pdb["sol_ed"]


def _amplitudes(pdb, gs, qmax):
    """A at every grid node by direct summation, and its periodic-spline slope along phi."""
    N, step, dev = gs // 2 + 3, qmax / (gs // 2), _dev()
    xyz, ion = _t(pdb["xyz"]).T.contiguous(), torch.as_tensor(pdb["ion"], dtype=torch.int64, device=dev)
    boxes = pdb.get("box_dims") is not None and len(pdb["box_dims"]) > 0
    if boxes:
        com = _t(pdb["box_com"]).T.contiguous()
        edge = [np.unique(pdb["box_dims"][:, a], return_inverse=True) for a in range(3)]
        length = [_t(e[0] * VOXEL) for e in edge]
        which = [torch.as_tensor(e[1].ravel(), dtype=torch.int64, device=dev) for e in edge]
    A = torch.zeros(_points(gs), dtype=torch.complex128, device=dev)
    S = torch.zeros_like(A)
    A[0] = float(_form_factors(pdb, 0.0)[pdb["ion"]].sum())
    if boxes:
        A[0] += float(np.prod(pdb["box_dims"].astype(float) * VOXEL, axis=1).sum() * LAYER_CONTRAST)
    base = 1
    for i in range(1, N + 1):
        n, m = 6 * i, 3 * i
        f = _t(_form_factors(pdb, i * step))[ion]
        rows = m // 2 + 1
        th = (torch.arange(rows, dtype=torch.float64, device=dev) * (math.pi / m)).repeat_interleave(n)
        ph = (torch.arange(n, dtype=torch.float64, device=dev) * (2.0 * math.pi / n)).repeat(rows)
        qv = i * step * torch.stack([th.sin() * ph.cos(), th.sin() * ph.sin(), th.cos()], dim=1)
        half = torch.empty(rows * n, dtype=torch.complex128, device=dev)
        per = max(1, int(6e7 // max(xyz.shape[1], com.shape[1] if boxes else 1)))
        for k in range(0, rows * n, per):
            p = qv[k:k + per] @ xyz
            re, im = p.cos() @ f, p.sin() @ f
            if boxes:
                p = qv[k:k + per] @ com
                w = torch.full_like(p, LAYER_CONTRAST)
                for a in range(3):
                    x = 0.5 * qv[k:k + per, a:a + 1] * length[a]
                    w *= (torch.sinc(x / math.pi) * length[a])[:, which[a]]
                re, im = re + (p.cos() * w).sum(1), im + (p.sin() * w).sum(1)
            half[k:k + per] = torch.complex(re, im)
        half = half.view(rows, n)
        V = torch.empty(m + 1, n, dtype=torch.complex128, device=dev)
        V[:rows] = half
        V[m + 1 - rows:] = torch.where(torch.arange(m + 1 - rows, m + 1, device=dev)[:, None] >= rows,
                                       half.flip(0).roll(m, 1).conj(), V[m + 1 - rows:])
        A[base:base + n * (m + 1)] = V.reshape(-1)
        S[base:base + n * (m + 1)] = _slopes(V).reshape(-1)
        base += n * (m + 1)
    return A, S


def _slopes(V):
    """Periodic cubic spline: D[k-1] + 4 D[k] + D[k+1] = 3 (V[k+1] - V[k-1])."""
    n = V.shape[1]
    w = 2.0 * math.pi * torch.arange(n, dtype=torch.float64, device=V.device) / n
    return torch.fft.ifft(torch.fft.fft(V, dim=1) * (6j * w.sin() / (4.0 + 2.0 * w.cos())), dim=1)


def _cubic(a, b, da, db, t):
    return a + t * (da + t * (3.0 * (b - a) - 2.0 * da - db + t * (2.0 * (a - b) + da + db)))


def _four(y, t):
    """The cubic through the middle interval of four points, slopes of the natural-like spline."""
    d0, d1, d2, d3 = y[1] - y[0], y[2] - y[0], y[3] - y[1], y[3] - y[2]
    return _cubic(y[1], y[2], (-7.0 * d0 + 14.0 * d1 - 4.0 * d2 + 2.0 * d3) / 15.0,
                  (2.0 * d0 - 4.0 * d1 + 14.0 * d2 - 7.0 * d3) / 15.0, t)


def _plane(G, i, ut, up):
    """Shell i at theta = pi ut, phi = 2 pi up: cubic in phi on four rows, then in theta."""
    A, S = G
    n, m = 6 * i, 3 * i
    base = 1 + 6 * (i - 1) * i * i
    xt, xp = ut * m, up * n
    ti, pi = xt.to(torch.int64), xp.to(torch.int64)
    tt, tp = xt - ti, xp - pi
    y = []
    for r in range(-1, 3):
        v = ti + r
        past = (v < 0) | (v > m)
        row = base + torch.remainder(v, m + 1) * n
        k0 = torch.remainder(pi + torch.where(past, m, 0), n)
        k1 = torch.remainder(k0 + 1, n)
        y.append(_cubic(A[row + k0], A[row + k1], S[row + k0], S[row + k1], tp))
    return _four(y, tt)


def _planes(G, layer, th, ph):
    out = []
    for i in range(layer - 1, layer + 3):
        if i == -1:
            b = ph + math.pi
            out.append(_plane(G, 1, ((math.pi - th) / math.pi).clamp(0.0, 1.0),
                              torch.where(b >= 2.0 * math.pi, b - 2.0 * math.pi, b) / (2.0 * math.pi)))
        elif i == 0:
            out.append(G[0][0].expand(th.shape))
        else:
            out.append(_plane(G, i, th / math.pi, ph / (2.0 * math.pi)))
    return out


def _groups(q, step):
    """(layer, indices) of the q that share a shell interval (layer step, (layer + 1) step]."""
    layer = np.maximum(np.ceil(q / step) - 1, 0).astype(int)
    layer = np.where(q > (layer + 1) * step, layer + 1, np.where((q <= layer * step) & (layer > 0), layer - 1, layer))
    return [(int(l), np.flatnonzero(layer == l)) for l in np.unique(layer)]


def _uniform(seed, c0, c1, c2, c3):
    """Two 53-bit uniforms from Philox4x32-10 with the counter (c0, c1, c2, c3)."""
    M, k0, k1 = 0xFFFFFFFF, seed & 0xFFFFFFFF, seed >> 32
    full = torch.zeros_like(c0)
    c = [c0 & M, full + c1, full + c2, full + c3]

    def mul(a, x):  # the high and low 32 bits of a x
        lo, hi = a * (x & 0xFFFF), a * (x >> 16)
        t = hi + (lo >> 16)
        return t >> 16, ((t & 0xFFFF) << 16) | (lo & 0xFFFF)

    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c[0])
        h1, l1 = mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
    return [(((a >> 6) << 27 | b >> 5).to(torch.float64) + 0.5) / 2.0 ** 53 for a, b in ((c[0], c[1]), (c[2], c[3]))]


def _directions(seed, count, layer, chunk=8192):
    """Stratified directions: every run of 64 fills one of the chunk's equal-area patches."""
    d = torch.arange(count, dtype=torch.int64, device=_dev())
    u, v = _uniform(seed, d, 0, layer, 0x4D43)
    W = chunk // 64
    nu = max(a for a in range(1, W + 1) if 2 * a * a <= W and W % a == 0 or a == 1)
    nv = W // nu
    w = (d % chunk) // 64
    return torch.acos(2.0 * ((w // nv + u) / nu) - 1.0), 2.0 * math.pi * ((w % nv + v) / nv)


def _unit(th, ph):
    return torch.stack([th.sin() * ph.cos(), th.sin() * ph.sin(), th.cos()])


def _rotation(a, b, c):
    sa, ca, sb, cb, sc, cc = math.sin(a), math.cos(a), math.sin(b), math.cos(b), math.sin(c), math.cos(c)
    X = np.array([[1, 0, 0], [0, ca, -sa], [0, sa, ca]])
    Y = np.array([[cb, 0, sb], [0, 1, 0], [-sb, 0, cb]])
    Z = np.array([[cc, -sc, 0], [sc, cc, 0], [0, 0, 1]])
    return X @ Y @ Z


def _copies(placements):
    """(leaf, R^T, scale, translations) of every placed rotation."""
    out = []
    for leaf, (rot, nt, tr) in enumerate(placements):
        t0 = 0
        for r, n in zip(rot, nt):
            out.append((leaf, _t(_rotation(*r[:3]).T), float(r[3]), _t(tr[t0:t0 + n])))
            t0 += n
    return out


def _intensities(Gs, copies, layer, q, step, th, ph):
    """|A(q_j)|^2 of the docked leaves along every direction, for the q of one shell interval."""
    t = [float(x / step - layer) for x in q]
    if copies is None:
        p = _planes(Gs[0], layer, th, ph)
        return [_four(p, x).abs() ** 2 for x in t]
    qv = _unit(th, ph)
    acc = [torch.zeros(th.shape, dtype=torch.complex128, device=_dev()) for _ in t]
    for leaf, rt, scale, tr in copies:
        v = rt @ qv
        nph = torch.atan2(v[1], v[0])
        p = _planes(Gs[leaf], layer, torch.acos(v[2].clamp(-1.0, 1.0)), torch.where(nph < 0, nph + 2.0 * math.pi, nph))
        along = tr @ qv
        for j, x in enumerate(t):
            d = float(q[j]) * along
            acc[j] += scale * _four(p, x) * torch.complex(d.cos().sum(0), d.sin().sum(0))
    return [a.abs() ** 2 for a in acc]


def _mc(Gs, copies, q, step, seed, count):
    out, total = np.zeros(len(q)), -(-count // 8192) * 8192
    for layer, idx in _groups(q, step):
        th, ph = _directions(seed, total, layer)
        for j, I in zip(idx, _intensities(Gs, copies, layer, q[idx], step, th, ph)):
            out[j] = float(I.mean())
    return out


def _rebin(var, b):
    """New boundaries of one axis from its 32 variances: damped equal shares."""
    total = var.sum()
    if total == 0.0:
        return b
    local = np.array([var[max(0, i - 1):i + 2].mean() for i in range(32)])
    with np.errstate(all="ignore"):
        x = total / local
        w = ((x - 1.0) / (x * np.log(x))) ** 1.5
    w = np.where(np.isnan(w), 0.0, w)
    share, new, dw, j, xnew = w.sum() / 32, b.copy(), 0.0, 0, 0.0
    for i in range(32):
        dw += w[i]
        xold, xnew = xnew, b[i + 1]
        while dw > share:
            dw -= share
            if j < 31:
                new[j + 1] = xnew - dw * (xnew - xold) / w[i]
            j += 1
    return new


def _vegas(Gs, q, step, seed, iters, ppb):
    out = np.zeros(len(q))
    index = torch.arange(1024 * ppb, dtype=torch.int64, device=_dev())
    ti, pj = (index // ppb) // 32, (index // ppb) % 32
    for layer, idx in _groups(q, step):
        bt, bp = np.linspace(0.0, 1.0, 33), np.linspace(0.0, 1.0, 33)
        mean = np.zeros(len(idx))
        for k in range(iters):
            u, v = _uniform(seed, index, k, layer, 0x5645)
            T, P = _t(bt), _t(bp)
            th = torch.acos(1.0 - 2.0 * (u * (T[ti + 1] - T[ti]) + T[ti]))
            ph = 2.0 * math.pi * (v * (P[pj + 1] - P[pj]) + P[pj])
            vol = ((T[1:] - T[:-1])[:, None] * (P[1:] - P[:-1])[None, :]).reshape(-1)
            I = torch.stack(_intensities(Gs, None, layer, q[idx], step, th, ph)).view(len(idx), 1024, ppb)
            mean = (mean * k + (I.mean(2) @ vol).cpu().numpy()) / (k + 1)
            S = vol[:, None] * I.sum(0)
            var = (((S - S.mean(1, keepdim=True)) ** 2).sum(1) * ppb).view(32, 32).cpu().numpy()
            bt, bp = _rebin(var.sum(1), bt), _rebin(var.sum(0), bp)
        out[idx] = mean
    return out


def _sphr(G, N, step, q, th, ph):
    """The amplitude at (q, theta, phi) points, shell by shell."""
    out = torch.empty(q.shape, dtype=torch.complex128, device=_dev())
    ratio = q / step
    cell = (ratio * (1.0 + 1e-15)).to(torch.int64)
    for i in torch.unique(cell).tolist():
        at = torch.nonzero(cell == i, as_tuple=True)
        t = (ratio[at] - i).clamp(min=0.0)
        p = _planes(G, i, th[at], ph[at]) if i + 2 < N else None
        if p is None:
            p = [_plane(G, k, th[at] / math.pi, ph[at] / (2.0 * math.pi)) for k in range(i - 1, min(i + 2, N + 1))]
            p += [p[-1]] * (4 - len(p))
        out[at] = torch.where(t < 1e-9, p[1], _four(p, t))
    return out


def _docked_nodes(G, N, gs, step, copies):
    """The docked amplitude at every node of a grid."""
    A = torch.empty(_points(gs), dtype=torch.complex128, device=_dev())
    S = torch.zeros_like(A)
    A[0] = sum(scale * tr.shape[0] for _, _, scale, tr in copies) * G[0][0]
    base = 1
    for i in range(1, N + 1):
        n, m = 6 * i, 3 * i
        th = (torch.arange(m + 1, dtype=torch.float64, device=_dev()) * (math.pi / m)).repeat_interleave(n)
        ph = (torch.arange(n, dtype=torch.float64, device=_dev()) * (2.0 * math.pi / n)).repeat(m + 1)
        qv = _unit(th, ph)
        acc = torch.zeros(th.shape, dtype=torch.complex128, device=_dev())
        for _, rt, scale, tr in copies:
            v = rt @ qv
            nph = torch.atan2(v[1], v[0])
            nph = torch.where(nph < 0, nph + 2.0 * math.pi, nph)
            d = i * step * (tr @ qv)
            acc += scale * _plane(G, i, torch.acos(v[2].clamp(-1.0, 1.0)) / math.pi, nph / (2.0 * math.pi)) * \
                torch.complex(d.cos().sum(0), d.sin().sum(0))
        A[base:base + n * (m + 1)] = acc
        S[base:base + n * (m + 1)] = _slopes(acc.view(m + 1, n)).reshape(-1)
        base += n * (m + 1)
    return A, S


def exact(case, seed):
    kind = case["kind"]
    # the adaptive quadrature's value depends on its accept decisions; bursts, helices
    # and the largest sums take too long
    if kind in ("stream", "helix") or case.get("method") == "gk":
        return None
    sources = case["atoms"] * (4.0 if case.get("layer") else 1.0) * case.get("leaves", 1)
    if _points(case["gs"]) / 2 * sources > 6e10:
        return None
    I = _inputs(case, seed)
    step, N = case["qmax"] / (case["gs"] // 2), case["gs"] // 2 + 3
    Gs = [_amplitudes(p, case["gs"], case["qmax"]) for p in I["pdbs"]]
    if kind == "curve" and case["method"] == "mc":
        return _mc(Gs, None, I["q"], step, I["seed"], case["points"])
    if kind == "curve":
        return _vegas(Gs, I["q"], step, I["seed"], case["iters"], case["ppb"])
    if kind == "session":
        curve = _mc(Gs, _copies(I["placements"]), I["q"], step, I["seed"], case["points"])
        return {"I": curve, "chi2": float((((curve - I["data"]) / I["sigma"]) ** 2).sum())}
    if kind == "ring":
        G = _docked_nodes(Gs[0], N, case["gs"], step, _copies(I["placements"]))
        return _vegas([G], I["q"], step, I["seed"], case["iters"], case["ppb"])
    q, th = _t(I["q"]), _t(I["theta"])
    k = torch.arange(case["nphi"], dtype=torch.int64, device=_dev())
    out = np.empty(len(q))
    per = max(1, (1 << 20) // case["nphi"])
    for a in range(0, len(q), per):
        point = torch.arange(a, min(a + per, len(q)), dtype=torch.int64, device=_dev())
        kk, pp = k.repeat(len(point)), point.repeat_interleave(case["nphi"])
        u, _ = _uniform(I["seed"], kk, pp, 0, 0x415A)
        ph = 2.0 * math.pi * (kk + u) / case["nphi"]
        amp = _sphr(Gs[0], N, step, q[pp], th[pp], ph)
        out[a:a + len(point)] = (amp.abs() ** 2).view(len(point), -1).mean(1).cpu().numpy()
    return out
