"""Atoms whose coordinates are not numbers (a run that blew up) on the cluster
path: the call ends, the value and the pair count are those of the other atoms
(a pair that is not within D_MAX adds nothing), and the context's next call at
finite positions gives the bits of a fresh one.  NaN atoms fall into column 0:
one, most of a cluster, whole clusters."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

N = 3000
BOX = np.diag([(N / 33.4) ** (1 / 3)] * 3)
SWITCHES = ["RATIONAL R_0=0.3 NN=6 MM=12 D_MAX=1.2", "EXP R_0=0.2 D_MAX=1.0", "RATIONAL R_0=0.3 NN=5 MM=11 D_MAX=0.6"]


def _positions(bad, seed=31):
    x = np.random.default_rng(seed).uniform(0, BOX[0, 0], (N, 3))
    y = x.copy()
    at = np.random.default_rng(seed + bad).permutation(N)[:bad]
    y[at[::2]] = np.nan
    y[at[1::2], 2] = np.nan
    return x, y, np.setdiff1d(np.arange(N), at)


@pytest.mark.parametrize("chunk", [64, 32])
@pytest.mark.parametrize("sw", SWITCHES)
@pytest.mark.parametrize("bad", [1, 7, 8, 30])
def test_one_group(bad, sw, chunk):
    import plumed2_amd as P

    x, y, ok = _positions(bad)
    line = f"c: COORDINATION GROUPA=1-{N} SWITCH={{{sw}}}"
    act, fresh = P.Coordination(line), P.Coordination(line)
    for a in (act, fresh):
        a.set_tuning(chunk, 4)
    ov, _, _, npair = O.coordination(O.Switch(sw), BOX, y[ok], len(ok), 0)
    for _ in range(2):  # the second build takes the atoms in the first one's order
        v, _, _ = act.calculate(y, BOX)
        st = act.stats()
        assert st["path"] == 0 and st["contributing_pairs"] == npair
        assert abs(v - ov) <= 1e-6 * abs(ov)
    got, want = act.calculate(x, BOX), fresh.calculate(x, BOX)
    assert all(np.array_equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("groups", ["one", "apart", "shared"])
@pytest.mark.parametrize("bad", [1, 7, 30])
def test_weighted_rows(bad, groups):
    import torch
    import plumed2_amd as P

    x, y, ok = _positions(bad)
    rows, env = {"one": (N, None), "apart": (900, range(900, N)), "shared": (900, range(N))}[groups]
    kw = dict(species=range(N)) if env is None else dict(species_a=range(rows), species_b=env)
    w = np.random.default_rng(33).normal(size=rows)
    cn, fresh = P.CoordinationNumbers(SWITCHES[0], **kw), P.CoordinationNumbers(SWITCHES[0], **kw)
    got = cn(torch.tensor(y, dtype=torch.float64, device="cuda:0"), BOX, weights=w)[0].cpu().numpy()
    assert cn.action.stats()["path"] == 0
    finite = np.intersect1d(ok, np.arange(rows))
    # rows that are numbers, over the environment atoms that are
    e = np.intersect1d(ok, np.arange(N) if env is None else np.array(env))
    want = O.coordination_numbers(O.Switch(SWITCHES[0]), BOX, y, species_a=finite, species_b=e)
    assert np.max(np.abs(got[finite] - want)) <= 1e-6 * np.max(np.abs(want))
    t = torch.tensor(x, dtype=torch.float64, device="cuda:0")
    assert all(torch.equal(a, b) for a, b in zip(cn(t, BOX, weights=w), fresh(t, BOX, weights=w)))


@pytest.mark.parametrize("bad", [1, 7, 30])
def test_batch(bad):
    import torch
    import plumed2_amd as P

    x, y, ok = _positions(bad)
    b = P.CoordinationBatch([N, N], SWITCHES[0], 1.3)
    b.set_boxes(np.array([BOX, BOX]))
    v, d, _ = b.calculate_torch(torch.tensor(np.vstack([y, x]), dtype=torch.float64, device="cuda:0"))
    for k, q in enumerate((y[ok], x)):
        ov, od, _, npair = O.coordination(O.Switch(SWITCHES[0]), BOX, q, len(q), 0)
        assert b.pair_counts()[k] == npair and abs(float(v[k]) - ov) <= 1e-6 * abs(ov)
    # the system whose atoms are all numbers
    assert np.max(np.abs(d[N:].cpu().numpy() - od)) <= 1e-5 * np.max(np.abs(od))
