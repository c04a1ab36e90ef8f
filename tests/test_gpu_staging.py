"""Pairs exactly at D_MAX where the cut decision needs the requested index of a
staged atom: weighted COORDINATIONNUMBER rows (whose staged atoms carry their
weight in the index's place) and groups that share atoms, on the lattice
geometry (spacing D_MAX/2, six partners exactly at D_MAX) with every other atom
off its site, against the oracle.  The group sizes leave ragged clusters and
items of few entries; NL_CUTOFF sets how many listed entries D_MAX leaves.

A pair at D_MAX adds nothing to a value (stretched switch) but has a derivative
of about 1e-3 of the largest.  Tolerances: FP32 pair arithmetic with FP64 sums,
values 1e-6, derivatives and box derivatives 1e-5 of their largest entry, as
for the same entry points off the lattice."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

TOL, F_TOL = 1e-6, 1e-5
A, M = 0.2, 14


def lattice(seed):
    g = np.arange(M) * A
    x = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3) + 0.013
    x[::2] += np.random.default_rng(seed).normal(0.0, 0.005, x[::2].shape)
    return x, np.diag([M * A] * 3)


def close(got, want, tol):
    assert np.max(np.abs(got - want)) <= tol * np.max(np.abs(want))


SWITCHES = [f"RATIONAL R_0=0.15 NN=6 MM=12 D_MAX={2 * A}", f"RATIONAL R_0=0.18 NN=8 MM=16 D_MAX={2 * A}"]


@pytest.mark.parametrize("defn", SWITCHES)
@pytest.mark.parametrize("groups", ["one", "apart", "shared", "few"])
def test_weighted_rows_with_pairs_at_dmax(defn, groups):
    import torch
    import plumed2_amd as P
    x, box = lattice(11)
    n = len(x)
    order = np.random.default_rng(12).permutation(n)
    kw = {"one": dict(species=order[:2501]), "apart": dict(species_a=order[:701], species_b=order[701:]),
          "shared": dict(species_a=order[:1203], species_b=order[601:2603]),
          "few": dict(species_a=order[:9], species_b=order[4:])}[groups]
    rows = kw.get("species", kw.get("species_a"))
    w = np.random.default_rng(13).normal(size=len(rows))
    cn = P.CoordinationNumbers(defn, **kw)
    got, vjp, vir = cn(torch.tensor(x, dtype=torch.float64, device="cuda:0"), box, weights=w)
    assert cn.action.stats()["path"] == 0
    want, owant, ovir = O.coordination_numbers(O.Switch(defn), box, x, weights=w, **kw)
    close(got.cpu().numpy(), want, TOL)
    close(vjp.cpu().numpy(), owant, F_TOL)
    close(vir.cpu().numpy(), ovir, F_TOL)


@pytest.mark.parametrize("margin", [0.0, 0.12])
@pytest.mark.parametrize("na,lo", [(1203, 601), (2744, 0), (9, 4)])
@pytest.mark.parametrize("defn", SWITCHES)
def test_shared_groups_with_pairs_at_dmax(defn, na, lo, margin):
    import plumed2_amd as P
    x, box = lattice(14)
    x = x[np.random.default_rng(15).permutation(len(x))]
    n = len(x)
    req = np.concatenate([np.arange(na), np.arange(lo, n)])
    nl = f" NLIST NL_CUTOFF={2 * A + margin} NL_STRIDE=1" if margin else ""
    act = P.Coordination(f"c: COORDINATION GROUPA=1-{na} GROUPB={lo + 1}-{n}{nl} SWITCH={{{defn}}}")
    v, d, w = act.calculate(x[req], box, 0)
    assert act.stats()["path"] == 0
    ov, od, ow, npair = O.coordination(O.Switch(defn), box, x[req], na, n - lo, absidx=req)
    assert act.stats()["contributing_pairs"] == npair
    assert abs(v - ov) <= TOL * abs(ov)
    close(d, od, F_TOL)
    close(w, ow, F_TOL)


@pytest.mark.parametrize("layout", ["plain", "offset", "strided", "grad"])
def test_all_atoms_in_order_are_not_gathered(layout):
    """Rows over all atoms in order take the positions as they are, whatever
    their layout: the same bits as through the gather (the same atoms listed as
    rows of a longer array whose last atom is left out)."""
    import torch
    import plumed2_amd as P
    x, box = lattice(16)
    n = len(x)
    w = np.random.default_rng(17).normal(size=n)
    y = torch.tensor(np.vstack([x, [[0.5, 0.5, 0.5]]]), dtype=torch.float64, device="cuda:0")
    t = {"plain": y[:n].clone(), "grad": y[:n].clone().requires_grad_(),
         "offset": torch.cat([y[:1, 0], y[:n].reshape(-1)])[1:].view(n, 3),
         "strided": torch.cat([y[:n], y[:n]], 1)[:, 3:]}[layout]
    cn = P.CoordinationNumbers(SWITCHES[0], species=range(n))
    a = cn(t, box, weights=w)
    b = cn(y, box, weights=w)
    assert a[1].shape == (n, 3) and b[1].shape == (n + 1, 3)
    assert not any(q.requires_grad for q in a) and torch.all(b[1][n] == 0.0)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1][:n]) and torch.equal(a[2], b[2])
