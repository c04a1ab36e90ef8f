"""Hills deposited in one call against one call per hill (bit for bit: every
node and corner receives the same FP64 additions in the same order) and
against the FP64 oracle (1e-10 relative, as the other METAD tests), at the
edges of the runs and epochs (2^CVs corners on a 64-lane wave, 1,024 corners an
epoch), with open, periodic and mixed CVs."""
import math

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
KB = 0.0083144621


def _line(ncv, periodic, bins, wt=True):
    names = "abcd"[:ncv]
    lo = ["-pi" if p else "-2" for p in periodic]
    hi = ["pi" if p else "2" for p in periodic]
    return (f"m: METAD ARG={','.join(names)} SIGMA={','.join(['0.3'] * ncv)} HEIGHT=1.1 PACE=5 "
            + ("BIASFACTOR=6 TEMP=300 " if wt else "")
            + f"GRID_MIN={','.join(lo)} GRID_MAX={','.join(hi)} GRID_BIN={','.join([str(b) for b in bins])}",
            {names[i]: ("-pi", "pi") for i in range(ncv) if periodic[i]})


def _walk(n, periodic, seed):
    rng = np.random.default_rng(seed)
    x, out = np.zeros(len(periodic)), []
    for _ in range(n):
        x = x + rng.normal(0, 0.25, len(x))
        x = np.where(periodic, (x + math.pi) % (2 * math.pi) - math.pi, np.clip(x, -2.0, 1.9999))
        out.append(x)
    return np.array(out)


CASES = [(1, (False,), (60,)), (1, (True,), (70,)), (2, (False, False), (40, 33)), (2, (True, True), (50, 64)),
         (2, (False, True), (45, 40)), (3, (True, False, True), (40, 17, 31)), (4, (False, True, False, True), (9, 40, 11, 35))]


@pytest.mark.parametrize("ncv,periodic,bins", CASES)
@pytest.mark.parametrize("count", [1, 4, 5, 17, "epoch-1", "epoch", "epoch+1", "2epoch+3"])
def test_one_call_equals_hill_by_hill(ncv, periodic, bins, count):
    import plumed2_amd as P

    e = 1024 >> ncv
    n = {"epoch-1": e - 1, "epoch": e, "epoch+1": e + 1, "2epoch+3": 2 * e + 3}.get(count, count)
    line, per = _line(ncv, periodic, bins)
    c = _walk(n, periodic, n + ncv)
    m1, m2 = P.MetaD(line, periodic=per), P.MetaD(line, periodic=per)
    # a grid that already holds something, through the other kernel
    for m in (m1, m2):
        m.deposit(_walk(3, periodic, 1))
    h1 = m1.deposit(c)
    h2 = np.concatenate([m2.deposit(x[None, :]) for x in c])
    assert np.array_equal(h1, h2)
    (v1, d1), (v2, d2) = m1.grid(), m2.grid()
    assert np.array_equal(v1, v2) and np.array_equal(d1, d2)


@pytest.mark.parametrize("ncv,periodic,bins", [k for k in CASES if k[0] <= 3])
def test_against_the_oracle(ncv, periodic, bins):
    import plumed2_amd as P

    line, per = _line(ncv, periodic, bins)
    c = _walk(300, periodic, 7)
    m = P.MetaD(line, periodic=per)
    h = m.deposit(c)
    lo = [-math.pi if p else -2.0 for p in periodic]
    hi = [math.pi if p else 2.0 for p in periodic]
    g = O.Grid(lo, hi, list(bins), [int(p) for p in periodic])
    oh = g.deposit_wt(c, [0.3] * ncv, 1.1, 6.0, 300 * KB)
    np.testing.assert_allclose(h, oh, rtol=1e-10)
    v, d = m.grid()
    assert np.max(np.abs(v - g.values())) <= 1e-10 * np.max(np.abs(g.values()))
    assert np.max(np.abs(d - g.derivs())) <= 1e-10 * np.max(np.abs(g.derivs()))


@pytest.mark.parametrize("at", [0, 3, 255, 256, 300])
@pytest.mark.parametrize("wt", [True, False])
def test_a_hill_outside_the_grid_ends_the_call(at, wt):
    import plumed2_amd as P

    line, per = _line(2, (False, False), (40, 33), wt)
    c = _walk(400, (False, False), 3)
    bad = c.copy()
    bad[at] = [5.0, 0.0]
    m1, m2 = P.MetaD(line, periodic=per), P.MetaD(line, periodic=per)
    with pytest.raises(P.Plumed2AmdError, match="outside the grid"):
        m1.deposit(bad)
    if at:
        m2.deposit(c[:at])
    assert np.array_equal(m1.grid()[0], m2.grid()[0])
    # the context stays usable
    assert np.array_equal(m1.deposit(c), m2.deposit(c))
