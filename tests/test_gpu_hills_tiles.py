"""Hills on grids far larger than their supports, where a deposition visits the
tiles around each hill and not those of the grid: bit for bit one call per hill
(every node receives the same FP64 additions in the same order), with supports
that cross tiles, wrap over a cut last tile and end at the walls."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _metad(periodic, bins, sigma):
    import plumed2_amd as P
    names = "abcd"[:len(bins)]
    return P.MetaD(f"m: METAD ARG={','.join(names)} SIGMA={','.join(str(s) for s in sigma)} HEIGHT=1.1 PACE=5 "
                   "BIASFACTOR=6 TEMP=300 "
                   f"GRID_MIN={','.join('-pi' if p else '-2' for p in periodic)} "
                   f"GRID_MAX={','.join('pi' if p else '2' for p in periodic)} GRID_BIN={','.join(str(b) for b in bins)}",
                   periodic={n: ("-pi", "pi") for n, p in zip(names, periodic) if p})


def _centres(n, periodic, seed):
    """clusters of hills, some of them at the walls or across the period"""
    rng = np.random.default_rng(seed)
    hi = np.where(periodic, math.pi, 2.0)
    at = rng.uniform(-1.0, 1.0, (7, len(periodic)))
    at[:4] = rng.choice([-1.0, 1.0], (4, len(periodic)))
    x = at[rng.integers(0, 7, n)] * hi + rng.normal(0, 0.1, (n, len(periodic)))
    return np.where(periodic, (x + math.pi) % (2 * math.pi) - math.pi, np.clip(x, -2.0, 1.9999))


# nodes of support to each side: ceil(3.54 sigma / spacing)
CASES = [((False,), (5000,), (0.01,)), ((True,), (5003,), (0.02,)),
         ((False, False), (203, 198), (0.04, 0.02)), ((True, True), (203, 192), (0.05, 0.02)),
         ((False, True), (400, 61), (0.01, 0.5)),  # a support of nearly the period on one CV
         ((False, True), (1100, 1000), (0.2, 0.3)),  # many tiles, supports that reach most of them
         ((True, False, True), (41, 38, 45), (0.1, 0.05, 0.07)),
         ((False, True, True, False), (21, 22, 23, 19), (0.05, 0.06, 0.07, 0.05))]


@pytest.mark.parametrize("periodic,bins,sigma", CASES)
@pytest.mark.parametrize("count", [5, 23, "epoch+6"])
def test_one_call_equals_hill_by_hill(periodic, bins, sigma, count):
    n = (1024 >> len(bins)) + 6 if count == "epoch+6" else count
    c = _centres(n, np.array(periodic), n + len(bins))
    m1, m2 = _metad(periodic, bins, sigma), _metad(periodic, bins, sigma)
    h1 = m1.deposit(c)
    h2 = np.concatenate([m2.deposit(x[None, :]) for x in c])
    assert np.array_equal(h1, h2)
    (v1, d1), (v2, d2) = m1.grid(), m2.grid()
    assert np.count_nonzero(v1) and np.array_equal(v1, v2) and np.array_equal(d1, d2)


def test_a_grid_of_more_tiles_than_a_launch_holds():
    """2^30 nodes (2^24 tiles of 64, one work-item a node and three more: 2^32)."""
    bins = (1 << 30,)
    m1, m2 = _metad((False,), bins, (1.0e-7,)), _metad((False,), bins, (1.0e-7,))
    rng = np.random.default_rng(4)
    c = 0.3 + np.cumsum(rng.normal(0, 1.0e-7, (1100, 1)), 0)
    assert np.array_equal(m1.deposit(c), np.concatenate([m2.deposit(c[k:k + 4]) for k in range(0, len(c), 4)]))
    at = c + rng.normal(0, 1.0e-7, c.shape)
    (b1, d1), (b2, d2) = m1.bias(at), m2.bias(at)
    assert np.any(b1 > 0.0) and np.array_equal(b1, b2) and np.array_equal(d1, d2)


def test_the_gaussian_is_good_to_a_rounding(monkeypatch):
    """One hill of height 1 at a node, arguments of the exponential exact: every
    node within 1.1 units in the last place of exp (a final rounding of half a unit,
    and two of a quarter in the reduced argument and the sum before it)."""
    import plumed2_amd as P

    monkeypatch.setenv("PLUMED_DP2CUTOFF_NOSTRETCH", "1")
    m = P.MetaD("m: METAD ARG=a SIGMA=1 HEIGHT=1 PACE=1 GRID_MIN=-4 GRID_MAX=4 GRID_BIN=32768")
    m.deposit(np.zeros((1, 1)))
    v, d = m.grid()
    x = -4.0 + np.arange(len(v)) / 4096.0
    e = np.exp(-0.5 * x.astype(np.longdouble) ** 2)
    near = 0.5 * x * x < 6.25
    ulp = np.spacing(e.astype(np.float64))
    assert not np.any(v[~near]) and np.count_nonzero(near) > 20000
    assert float(np.max(np.abs((v - e) / ulp)[near])) <= 1.1
    # the gradient: one rounding of the product more
    g = -x * e
    assert float(np.max(np.abs(d[:, 0] - g)[near])) <= 2.5 * np.spacing(1.0)
