"""Timed cases of the COORDINATION and METAD paths.

``listed()`` gives the cases, ``draw(rng)`` one more of the same ranges,
``prepare(case, seed)`` what a program holds before the call (positions on the
GPU, or on the host where the caller is an MD engine on the host; the action;
a bias grid that already has hills), ``run(state)`` one pass through the
package's entry points, ``work(case)`` the bytes and operations that a pass
cannot do without, and ``exact(case, seed)`` the same outputs in FP64 from
plain torch and numpy.

Positions are uniform in the cell at the densities of the repository's
benchmark (33.4 atoms/nm^3: atoms of a liquid; 100 /nm^3: with hydrogens), and
frames of one run are steps of a random walk of 0.005 nm, as in an MD run.
"""
import math

import numpy as np
import torch

import plumed2_amd as P
from plumed2_amd.autograd import coordination
from plumed2_amd.synthetic import batch_systems

SIGMA = 0.005  # nm a frame
KB = 0.0083144621  # kJ/mol/K
DISTS = "RATIONAL R_0=0.3 NN=6 MM=12 D_MAX=1.2"


def listed():
    return [
        # what most inputs are: a few hundred atoms, default keywords (no
        # D_MAX), positions handed over by an MD engine on the host, each step
        {"name": "host_contacts_300", "kind": "host", "na": 100, "nb": 200, "side": 3.0},
        # a cluster or nanoparticle without a cell: every pair of the group
        {"name": "open_cluster_5k", "kind": "open", "na": 5001, "nb": 0, "rho": 60.0},
        # a solute and its solvent in a small cell with NLIST: one list
        # build and nine steps on the kept list
        {"name": "nlist_small_cell", "kind": "nlist", "na": 700, "nb": 5300, "side": 4.2, "mode": "NLIST"},
        # two groups of 1,000 atoms in a 5 nm cell, no list keyword
        {"name": "two_groups_2k", "kind": "two", "na": 1000, "nb": 1000, "side": 5.0},
        # the repository's headline workload: NLISTCELLS, NL_STRIDE=10; a pass
        # is one list build and the ten steps that use it
        {"name": "liquid_50k_cells", "kind": "cells", "n": 50000},
        # a triclinic cell and a switch other than RATIONAL n, 2n; the list is
        # built at every call
        {"name": "triclinic_20k_exp", "kind": "tric", "n": 20011, "switch": "EXP R_0=0.15 D_MAX=1.0"},
        # per-atom coordination numbers and the forces a function of them sends
        # back, no list keyword
        {"name": "numbers_30k", "kind": "rows", "n": 30000},
        # METAD on a coordination and a distance between two centres, forces on
        # the atoms; ten steps
        {"name": "metad_step_100k", "kind": "chain", "n": 100000},
        # training with the CV: forward and backward in float32 on five frames,
        # the list kept within a 0.1 nm skin
        {"name": "autograd_500k", "kind": "grad", "na": 10000, "nb": 490000},
        # frames and walkers of many systems in one step, list built each time
        {"name": "batch_48_systems", "kind": "batch", "nsys": 48, "lo": 6000, "hi": 64000},
        # replaying the hills of a run on two open CVs, 512 x 512 bins
        {"name": "hills_open_4000", "kind": "hills", "periodic": False, "ncv": 2, "bins": 512, "hills": 4000},
        # the same on two torsions (periodic, 100 x 100 bins)
        {"name": "hills_torsions_500", "kind": "hills", "periodic": True, "ncv": 2, "bins": 100, "hills": 500},
    ]


SWITCHES = ["EXP R_0=0.15 D_MAX=1.0", "GAUSSIAN R_0=0.25 D_MAX=1.0", "RATIONAL R_0=0.3 NN=8 MM=20 D_MAX=1.1",
            "RATIONAL R_0=0.25 NN=6 MM=10 D_0=0.05 D_MAX=1.0", "RATIONAL R_0=0.35 NN=8 MM=16 D_MAX=1.0"]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["host", "open", "nlist", "two", "cells", "tric", "rows", "chain", "grad", "batch", "hills"])
    if kind == "host":
        return {"kind": kind, "na": size(10, 400), "nb": rng.choice([0, size(10, 400)]),
                "side": round(rng.uniform(2.2, 4.0), 3)}
    if kind == "open":
        two = rng.random() < 0.5
        return {"kind": kind, "na": size(150, 2500 if two else 5000), "nb": size(150, 2500) if two else 0,
                "rho": round(rng.uniform(20.0, 100.0), 2)}
    if kind == "nlist":
        return {"kind": kind, "na": size(50, 700), "nb": size(300, 5300), "side": round(rng.uniform(3.3, 4.3), 3),
                "mode": rng.choice(["NLIST", "NLISTCELLS"])}
    if kind == "two":
        return {"kind": kind, "na": size(100, 4000), "nb": size(100, 4000), "side": round(rng.uniform(3.0, 6.0), 3)}
    if kind == "cells":
        return {"kind": kind, "n": size(2000, 50000)}
    if kind == "tric":
        return {"kind": kind, "n": size(2000, 20000), "switch": rng.choice(SWITCHES)}
    if kind == "rows":
        return {"kind": kind, "n": size(2000, 30000)}
    if kind == "chain":
        return {"kind": kind, "n": size(8000, 100000)}
    if kind == "grad":
        return {"kind": kind, "na": size(500, 10000), "nb": size(10000, 490000)}
    if kind == "batch":
        return {"kind": kind, "nsys": rng.randint(2, 48), "lo": 6000, "hi": size(8000, 64000)}
    per = rng.random() < 0.5
    if per:
        return {"kind": kind, "periodic": True, "ncv": rng.randint(1, 2), "bins": rng.randint(60, 150),
                "hills": size(50, 500)}
    return {"kind": kind, "periodic": False, "ncv": rng.randint(1, 2), "bins": rng.randint(200, 512),
            "hills": size(200, 1000)}


# ---- inputs ---------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _frames(n, box, seed, steps):
    """[steps][n, 3] float64 positions: uniform in the cell, then a random walk."""
    g = _gen(seed)
    b = torch.tensor(np.asarray(box), dtype=torch.float64, device="cuda")
    x = torch.rand((n, 3), generator=g, device="cuda", dtype=torch.float64) @ b
    out = [x]
    for _ in range(steps - 1):
        x = x + SIGMA * torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float64)
        out.append(x)
    return out


def _cube(n, rho):
    return np.diag([(n / rho) ** (1.0 / 3.0)] * 3)


def _tric(n, rho):
    b = np.array([[1.0, 0.0, 0.0], [0.08, 1.1, 0.0], [-0.06, 0.09, 0.95]])
    return b * (n / rho / abs(np.linalg.det(b))) ** (1.0 / 3.0)


def _groups(na, nb):
    return f"GROUPA=1-{na}" + (f" GROUPB={na + 1}-{na + nb}" if nb else "")


def _outs(n):
    f64 = dict(dtype=torch.float64, device="cuda")
    return (torch.empty(1, **f64), torch.empty((n, 3), **f64), torch.empty((3, 3), **f64))


def _line(c):
    """The COORDINATION line of a case (without the batch, row and hill kinds)."""
    k = c["kind"]
    if k == "host":
        return f"c: COORDINATION {_groups(c['na'], c['nb'])} R_0=0.3"
    if k == "open":
        return f"c: COORDINATION {_groups(c['na'], c['nb'])} SWITCH={{RATIONAL R_0=0.3}} NOPBC"
    if k == "nlist":
        return (f"c: COORDINATION {_groups(c['na'], c['nb'])} SWITCH={{RATIONAL R_0=0.3 D_MAX=1.6}} {c['mode']} "
                "NL_CUTOFF=2.2 NL_STRIDE=10")
    if k == "two":
        return f"c: COORDINATION {_groups(c['na'], c['nb'])} SWITCH={{RATIONAL R_0=0.3 NN=6 MM=12 D_MAX=1.0}}"
    if k in ("cells", "chain"):
        return f"c: COORDINATION {_groups(c['n'], 0)} SWITCH={{{DISTS}}} NLISTCELLS NL_CUTOFF=1.5 NL_STRIDE=10"
    if k == "tric":
        return f"c: COORDINATION {_groups(c['n'], 0)} SWITCH={{{c['switch']}}}"
    return f"c: COORDINATION {_groups(c['na'], c['nb'])} SWITCH={{RATIONAL R_0=0.35 NN=8 MM=16 D_MAX=1.0}}"


def _setup(c, seed):
    """(box, frames) of a case."""
    k = c["kind"]
    if k in ("host", "nlist", "two"):
        s = c["side"]
        box = np.diag([s, 1.05 * s, 0.97 * s] if k == "nlist" else [s] * 3)
        return box, _frames(c["na"] + c["nb"], box, seed, 10 if k == "nlist" else 1)
    if k == "open":
        box = _cube(c["na"] + c["nb"], c["rho"])
        return box, _frames(c["na"] + c["nb"], box, seed, 1)
    if k in ("cells", "chain"):
        return _cube(c["n"], 33.4), _frames(c["n"], _cube(c["n"], 33.4), seed, 10)
    if k == "tric":
        return _tric(c["n"], 100.0), _frames(c["n"], _tric(c["n"], 100.0), seed, 1)
    if k == "rows":
        return _cube(c["n"], 33.4), _frames(c["n"], _cube(c["n"], 33.4), seed, 1)
    n = c["na"] + c["nb"]  # grad
    return _cube(n, 100.0), _frames(n, _cube(n, 100.0), seed, 5)


def _chain_inputs(c, x0, box, seed):
    """Two compact groups, the METAD line and the hills already on its grid."""
    n, L = c["n"], float(box[0, 0])
    x = x0.cpu().numpy()
    size = max(50, n // 200)

    def nearest(point, skip):
        r = ((x - point) ** 2).sum(1)
        r[skip] = np.inf
        return np.argpartition(r, size)[:size]

    g1 = np.sort(nearest(np.array([0.3, 0.35, 0.3]) * L, []))
    g2 = np.sort(nearest(np.array([0.55, 0.5, 0.45]) * L, g1))
    mid, half = 2.9107 * n, 3000.0 * math.sqrt(n / 1e5)
    sig, dist = 20.0 * math.sqrt(n / 1e5), 0.33 * L
    line = (f"m: METAD ARG=c,d SIGMA={sig:.4f},0.05 HEIGHT=1.2 PACE=500 BIASFACTOR=10 TEMP=300 "
            f"GRID_MIN={mid - half:.3f},0 GRID_MAX={mid + half:.3f},6 GRID_BIN=512,512")
    rng = np.random.default_rng(seed + 7)
    hills = np.column_stack([rng.uniform(mid - half / 2, mid + half / 2, 4000),
                             np.clip(rng.uniform(dist - 0.35, dist + 0.25, 4000), 0.01, 5.99)])
    return g1, g2, line, hills, rng.uniform(0.3, 1.2, 4000)


def _hills_inputs(c, seed):
    """METAD line, periodic domains and the walk of the CVs."""
    rng = np.random.default_rng(seed)
    d, m = c["ncv"], c["hills"]
    if c["periodic"]:
        names = ["phi", "psi"][:d]
        lo, hi, sig = [-math.pi] * d, [math.pi] * d, [0.35] * d
        steps = rng.normal(0.0, 0.5, (m, d))
        walk = (np.cumsum(steps, axis=0) - 1.0 + math.pi) % (2 * math.pi) - math.pi
        line = (f"m: METAD ARG={','.join(names)} SIGMA={','.join(['0.35'] * d)} HEIGHT=1.2 PACE=500 BIASFACTOR=8 "
                f"TEMP=300 GRID_MIN={','.join(['-pi'] * d)} GRID_MAX={','.join(['pi'] * d)} "
                f"GRID_BIN={','.join([str(c['bins'])] * d)}")
        return line, {a: ("-pi", "pi") for a in names}, walk, lo, hi, sig
    lo, hi, sig = [0.0, 0.0][:d], [5000.0, 6.0][:d], [20.0 * 512 / c["bins"], 0.05 * 512 / c["bins"]][:d]
    walk, p = np.empty((m, d)), np.array([2500.0, 3.0])[:d]
    for k in range(m):
        p = np.clip(p + rng.normal(0.0, np.array([20.0, 0.05])[:d]), lo, np.array(hi) * 0.9999)
        walk[k] = p
    line = (f"m: METAD ARG={','.join(['c', 'd'][:d])} SIGMA={','.join(repr(s) for s in sig)} HEIGHT=1.2 PACE=500 "
            f"BIASFACTOR=10 TEMP=300 GRID_MIN={','.join(['0'] * d)} GRID_MAX={','.join(['5000', '6'][:d])} "
            f"GRID_BIN={','.join([str(c['bins'])] * d)}")
    return line, {}, walk, lo, hi, sig


def _systems(c, seed):
    """Atom counts and cells of the batch (the case's own), positions of the seed."""
    natoms, boxes, _ = batch_systems(c["nsys"], c["lo"], c["hi"])
    g = _gen(seed)
    b = torch.tensor(boxes, device="cuda").repeat_interleave(torch.tensor(natoms, device="cuda"), dim=0)
    x = torch.rand((len(b), 1, 3), generator=g, device="cuda", dtype=torch.float64)
    return natoms, boxes, (x.transpose(1, 2) * b).sum(1).contiguous()


def prepare(case, seed):
    c, k = case, case["kind"]
    if k == "hills":
        line, periodic, walk = _hills_inputs(c, seed)[:3]
        return {"case": c, "metad": P.MetaD(line, periodic=periodic), "walk": walk}
    if k == "batch":
        natoms, boxes, pos = _systems(c, seed)
        b = P.CoordinationBatch(natoms, DISTS, 1.2)
        b.set_boxes(boxes)
        b.set_graph(True)
        out = (torch.empty(c["nsys"], dtype=torch.float64, device="cuda"), torch.empty_like(pos),
               torch.empty((c["nsys"], 3, 3), dtype=torch.float64, device="cuda"))
        return {"case": c, "batch": b, "pos": pos, "out": out}
    box, frames = _setup(c, seed)
    st = {"case": c, "box": box, "frames": frames}
    if k == "rows":
        st["cn"] = P.CoordinationNumbers(DISTS, species=range(c["n"]))
        st["w"] = torch.rand(c["n"], generator=_gen(seed + 1), device="cuda", dtype=torch.float64)
        return st
    st["act"] = act = P.Coordination(_line(c))
    if k == "host":
        st["frames"] = [f.cpu().numpy() for f in frames]
    elif k == "grad":
        act.set_skin(0.1)
        st["frames"] = [f.to(torch.float32).requires_grad_(True) for f in frames]
    elif k == "chain":
        g1, g2, line, hills, heights = _chain_inputs(c, frames[0], box, seed)
        m = P.MetaD(line)
        m.add_hills(hills, heights)
        st["chain"] = P.MetadStep(act, m, P.CenterDistance(c["n"], g1, g2))
        st["step"] = 0
    else:
        st["out"] = [_outs(len(f)) for f in frames]
    return st


# ---- one pass ---------------------------------------------------------------------
def run(state):
    c, k = state["case"], state["case"]["kind"]
    if k == "host":
        return state["act"].calculate(state["frames"][0], state["box"])
    if k == "hills":
        m = state["metad"]
        heights = m.deposit(state["walk"])
        return (heights, *m.grid())
    if k == "batch":
        return state["batch"].calculate_torch(state["pos"], state["out"])
    if k == "rows":
        return state["cn"](state["frames"][0], state["box"], weights=state["w"])
    if k == "grad":
        got = []
        for s, x in enumerate(state["frames"]):
            x.grad = None
            v = coordination(x, state["act"], state["box"], s)
            v.backward()
            got.append((v.detach(), x.grad))
        return got
    if k == "chain":
        s0 = state["step"]
        for s, x in enumerate(state["frames"]):
            out = state["chain"].step(s0 + s, x, state["box"])
        state["step"] = s0 + len(state["frames"])
        return out
    act, box = state["act"], state["box"]
    return [act.calculate_torch(x, box, s, o) for s, (x, o) in enumerate(zip(state["frames"], state["out"]))]


# ---- what a pass cannot do without -----------------------------------------------
def _pairs(c):
    """Pairs within D_MAX of one frame, from the mean density (or every pair)."""
    k = c["kind"]
    if k in ("host", "open"):
        n, m = c["na"], c["nb"]
        return n * m if m else n * (n - 1) / 2
    if k in ("cells", "rows", "chain"):
        return c["n"] / 2 * 33.4 * 4.18879 * 1.2 ** 3
    if k == "tric":
        return c["n"] / 2 * 100.0 * 4.18879 * float(c["switch"].split("D_MAX=")[1]) ** 3
    if k == "grad":
        return c["na"] * 100.0 * c["nb"] / (c["na"] + c["nb"]) * 4.18879
    v = c["side"] ** 3 * (1.0185 if k == "nlist" else 1.0)
    return c["na"] * c["nb"] / v * 4.18879 * (1.6 if k == "nlist" else 1.0) ** 3


def work(case):
    c, k = case, case["kind"]
    if k == "hills":
        d, m = c["ncv"], c["hills"]
        support = (41.0 * c["bins"] / 100 if c["periodic"] else 17.0 if d == 1 else 23.7) ** d
        nodes = (c["bins"] + (0 if c["periodic"] else 1)) ** d
        return {"bytes": 8.0 * (m * (d + 1) + 2 * nodes * (1 + d)), "flops": m * support * (12.0 * d + 10)}
    if k == "batch":
        hi, lo = float(c["hi"]), float(c["lo"])
        n = c["nsys"] * (hi - lo) / math.log(hi / lo)
        return {"bytes": 48.0 * n, "flops": 49.0 * n / 2 * 33.4 * 4.18879 * 1.2 ** 3}
    n = c["n"] if "n" in c else c["na"] + c["nb"]
    steps = {"nlist": 10, "cells": 10, "chain": 10, "grad": 5}.get(k, 1)
    per = 24.0 if k == "grad" else 64.0 if k == "rows" else 72.0 if k == "chain" else 48.0
    return {"bytes": steps * per * n, "flops": steps * 49.0 * _pairs(c)}


# ---- the same in FP64, without the package ---------------------------------------
def _switch(text):
    """(D_MAX, f) with f(r2) -> (s, (1/r) ds/dr) for r <= D_MAX, stretched."""
    w = text.split()
    kv = dict(t.split("=") for t in w[1:])
    r0, d0, dmax = float(kv["R_0"]), float(kv.get("D_0", 0.0)), float(kv.get("D_MAX", "inf"))
    n = int(kv.get("NN", 6))
    m = int(kv.get("MM", 2 * n))

    def base(x):
        if w[0] == "EXP":
            e = torch.exp(-x)
            return e, -e
        if w[0] == "GAUSSIAN":
            e = torch.exp(-0.5 * x * x)
            return e, -x * e
        if m == 2 * n:
            xn = x ** (n - 1)
            s = 1.0 / (1.0 + xn * x)
            return s, -n * xn * s * s
        near = (x - 1.0).abs() < 1.1e-5
        y = torch.where(near, torch.full_like(x, 0.5), x)
        s = (1.0 - y ** n) / (1.0 - y ** m)
        ds = (m * y ** (m - 1) * s - n * y ** (n - 1)) / (1.0 - y ** m)
        d1, t = 0.5 * n * (n - m) / m, x - 1.0
        d2 = n * (m * m - 3.0 * m * (n - 1) + n * (2 * n - 3)) / (6.0 * m)
        return torch.where(near, n / m + t * (d1 + 0.5 * t * d2), s), torch.where(near, d1 + t * d2, ds)

    stretch, shift = 1.0, 0.0
    if math.isfinite(dmax):
        end = base(torch.tensor([0.0, (dmax - d0) / r0], dtype=torch.float64))[0].tolist()
        stretch = 1.0 / (end[0] - end[1])
        shift = -end[1] * stretch

    def f(r2):
        r = torch.sqrt(r2)
        x = (r - d0) / r0
        s, ds = base(torch.clamp(x, min=0.0))
        flat = x <= 0.0
        s = torch.where(flat, torch.ones_like(s), s) * stretch + shift
        return s, torch.where(flat, torch.zeros_like(s), ds * stretch / (r0 * torch.clamp(r, min=1e-300)))

    return dmax, f


def _sums(xa, xb, box, switch, weights=None):
    """Sums over the ordered pairs (a, b) of s, its gradients and -(dfunc d x d):
    (rows of a, gradient of a, gradient of b or None, virial over ordered pairs).
    xb None: one group with itself.  box None: no cell.  weights: each pair is
    weighted with w_a + w_b (one group)."""
    dmax, f = _switch(switch)
    same = xb is None
    xb = xa if same else xb
    dev, nb = xa.device, len(xb)
    rows = torch.zeros(len(xa), dtype=torch.float64, device=dev)
    ga, gb = torch.zeros_like(xa), None if same else torch.zeros_like(xb)
    vir = torch.zeros((3, 3), dtype=torch.float64, device=dev)
    oa = torch.arange(len(xa), device=dev)
    ob = torch.arange(nb, device=dev)
    slabs = box is not None and math.isfinite(dmax)
    if box is not None:
        B = torch.tensor(np.asarray(box), dtype=torch.float64, device=dev)
        inv = torch.linalg.inv(B)
    if slabs:  # sorted by fractional c; a partner within D_MAX is within `reach` of it
        reach = dmax * float(torch.linalg.norm(inv[:, 2])) + 1e-9
        slabs = 2 * reach < 0.9
    if slabs:
        fa, fb = ((x @ inv)[:, 2] for x in (xa, xb))
        fa, fb = fa - fa.floor(), fb - fb.floor()
        oa = torch.argsort(fa)
        fa = fa[oa]
        fb = torch.cat([fb - 1.0, fb, fb + 1.0])
        ob = torch.arange(nb, device=dev).repeat(3)
        keep = (fb > -reach - 1e-6) & (fb < 1.0 + reach + 1e-6)
        fb, ob = fb[keep], ob[keep]
        order = torch.argsort(fb)
        fb, ob = fb[order], ob[order]
        edges = fa.cpu().numpy()
        fbh = fb.cpu().numpy()
    step = 512 if slabs else max(1, min(512, int(2e7) // max(nb, 1)))
    for i0 in range(0, len(xa), step):
        ia = oa[i0:i0 + step]
        jb = ob
        if slabs:
            e0, e1 = edges[i0], edges[min(i0 + step, len(xa)) - 1]
            if e1 - e0 + 2 * reach < 1.0:
                jb = ob[int(np.searchsorted(fbh, e0 - reach)):int(np.searchsorted(fbh, e1 + reach))]
            else:  # the window goes round the cell: every partner once
                jb = torch.arange(nb, device=dev)
        d = xb[jb][None, :, :] - xa[ia][:, None, :]
        if box is not None:
            t = d @ inv
            d = d - torch.round(t) @ B
        r2 = (d * d).sum(2)
        ok = r2 <= dmax * dmax
        if same:
            ok &= ia[:, None] != jb[None, :]
        p, q = torch.nonzero(ok, as_tuple=True)
        d, r2 = d[p, q], r2[p, q]
        s, df = f(r2)
        pa, pb = ia[p], jb[q]
        rows.index_add_(0, pa, s)
        if weights is not None:
            df = df * (weights[pa] + weights[pb])
        g = df[:, None] * d
        ga.index_add_(0, pa, -g)
        if not same:
            gb.index_add_(0, pb, g)
        vir -= g.T @ d
    return rows, ga, gb, vir


def _coordination(x, na, nb, box, switch):
    """(value, derivatives, virial) of one frame."""
    if nb:
        rows, ga, gb, vir = _sums(x[:na], x[na:], box, switch)
        return rows.sum().reshape(1), torch.cat([ga, gb]), vir
    rows, ga, _, vir = _sums(x, None, box, switch)
    return (0.5 * rows.sum()).reshape(1), ga, 0.5 * vir


class _Bias:
    """A METAD grid (first CV fastest) with hills, in numpy."""

    def __init__(self, lo, hi, bins, sig, periodic):
        self.lo, self.sig, self.per = np.array(lo), np.array(sig), periodic
        self.dx = (np.array(hi) - self.lo) / np.array(bins)
        self.n = [b + (0 if periodic else 1) for b in bins]
        self.half = np.ceil(math.sqrt(12.5) * self.sig / self.dx).astype(int)
        self.d = len(bins)
        self.v = np.zeros(self.n[::-1])
        self.g = np.zeros(self.n[::-1] + [self.d])

    def cell(self, x):
        return np.floor((x - self.lo) / self.dx).astype(int)

    def add(self, x, h):
        at, dp, e2 = [], [], 0.0
        for i, c in enumerate(self.cell(x)):
            k = np.arange(c - self.half[i], c + self.half[i] + 1)
            k = k % self.n[i] if self.per else k[(k >= 0) & (k < self.n[i])]
            u = self.lo[i] + k * self.dx[i] - x[i]
            if self.per:
                L = self.n[i] * self.dx[i]
                u = u - L * np.round(u / L)
            shape = [1] * self.d
            shape[self.d - 1 - i] = len(k)
            at.append(k)
            dp.append((u / self.sig[i]).reshape(shape))
            e2 = e2 + 0.5 * dp[-1] ** 2
        a, b = 1.00193418799744762399, -0.00193418799744762399
        inside = e2 < 6.25
        e = np.where(inside, np.exp(-e2), 0.0)
        ix = np.ix_(*at[::-1])
        self.v[ix] += np.where(inside, h * (a * e + b), 0.0)
        for i in range(self.d):
            self.g[ix + (i,)] += -h * a * e * dp[i] / self.sig[i]

    def spline(self, x):
        """Bias and its gradient."""
        c = self.cell(x)
        v, dv = 0.0, np.zeros(self.d)
        for corner in range(1 << self.d):
            up = np.array([(corner >> i) & 1 for i in range(self.d)])
            k = c + up
            if not self.per and any(k[i] >= self.n[i] for i in range(self.d)):
                continue
            node = tuple(int(k[i]) % self.n[i] for i in range(self.d))[::-1]
            val = self.v[node]
            C, D = np.empty(self.d), np.empty(self.d)
            for i in range(self.d):
                h, sg = self.dx[i], 1.0 - 2.0 * up[i]
                X = abs((x[i] - self.lo[i] - c[i] * h) / h - up[i])
                yy = 0.0 if abs(val) < 1e-7 else -self.g[node][i] / val
                C[i] = 1 - 3 * X ** 2 + 2 * X ** 3 - sg * yy * (X - 2 * X ** 2 + X ** 3) * h
                D[i] = (-6 * X + 6 * X ** 2 - sg * yy * (1 - 4 * X + 3 * X ** 2) * h) * sg / h
            v += val * np.prod(C)
            for i in range(self.d):
                dv[i] += val * D[i] * np.prod(np.delete(C, i))
        return v, dv


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "hills":
        _, _, walk, lo, hi, sig = _hills_inputs(c, seed)
        b = _Bias(lo, hi, [c["bins"]] * c["ncv"], sig, c["periodic"])
        kt = KB * 300.0 * ((8.0 if c["periodic"] else 10.0) - 1.0)
        heights = []
        for x in walk:
            heights.append(1.2 * math.exp(-b.spline(x)[0] / kt))
            b.add(x, heights[-1])
        return np.array(heights), b.v.reshape(-1), b.g.reshape(-1, c["ncv"])
    if k == "batch":
        natoms, boxes, x = _systems(c, seed)
        got, at = [], 0
        for n, box in zip(natoms, boxes):
            got.append(_coordination(x[at:at + n], int(n), 0, box, DISTS))
            at += n
        return torch.cat([g[0] for g in got]), torch.cat([g[1] for g in got]), torch.stack([g[2] for g in got])
    box, frames = _setup(c, seed)
    if k == "rows":
        w = torch.rand(c["n"], generator=_gen(seed + 1), device="cuda", dtype=torch.float64)
        rows, g, _, vir = _sums(frames[0], None, box, DISTS, w)
        return rows, g, 0.5 * vir
    na, nb = c.get("n") or c["na"], c.get("nb", 0)
    if k == "host":  # R_0 alone: D_MAX where the switch has fallen to 1e-5, and the stretch of that
        sw = f"RATIONAL R_0=0.3 D_MAX={0.3 * 0.00001 ** (-1.0 / 6.0)!r}"
        v, d, w = _coordination(frames[0], na, nb, box, sw)
        return float(v), d.cpu().numpy(), w.cpu().numpy()
    sw = _line(c).split("{")[1].split("}")[0]
    if k == "chain":
        g1, g2, line, hills, heights = _chain_inputs(c, frames[0], box, seed)
        kv = dict(t.split("=") for t in line.split()[2:])
        b = _Bias(*([float(t) for t in kv[w].split(",")] for w in ("GRID_MIN", "GRID_MAX")), [512, 512],
                  [float(t) for t in kv["SIGMA"].split(",")], False)
        for x, h in zip(hills, heights):
            b.add(x, h)
        x = frames[-1]
        v, d, w = _coordination(x, na, 0, box, sw)
        r = x[torch.as_tensor(g2)].mean(0) - x[torch.as_tensor(g1)].mean(0)
        u = r / r.norm()
        cv = np.array([float(v), float(r.norm())])
        bias, dv = b.spline(cv)
        f = d * -dv[0]
        f[torch.as_tensor(g1, device=f.device)] += dv[1] * u / len(g1)
        f[torch.as_tensor(g2, device=f.device)] -= dv[1] * u / len(g2)
        return {"cv": cv, "bias": np.array([bias]), "cv_force": -dv, "forces": f,
                "virial": -dv[0] * w + dv[1] * torch.outer(r, u), "height": np.zeros(1)}
    if k == "grad":
        frames = [x.to(torch.float32).to(torch.float64) for x in frames]
        got = [_coordination(x, na, nb, box, sw) for x in frames]
        return [(v.reshape(()), g) for v, g, _ in got]
    return [_coordination(x, na, nb, None if k == "open" else box, sw) for x in frames]
