"""Atoms whose coordinates are not numbers, or infinite, on the FP64 path: value
and pair count are those of the other atoms, the derivatives and the virial show
the same entries as no numbers as the oracle's (0 times the distance), and the
others equal the oracle's to 1e-12 of the largest, as on finite positions."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("na,nb", [(60, 0), (5, 90), (90, 1200), (1500, 0)])
@pytest.mark.parametrize("nl", ["", " NLIST NL_CUTOFF=0.9 NL_STRIDE=1"])
@pytest.mark.parametrize("sw", ["RATIONAL R_0=0.3 NN=6 MM=12 D_MAX=0.8", "RATIONAL R_0=0.3 NN=8 MM=16 D_MAX=0.8",
                                "RATIONAL R_0=0.3 NN=10 MM=20 D_MAX=0.8"])
def test_pairs(sw, nl, na, nb, bad):
    import plumed2_amd as P

    n = na + nb
    x = np.random.default_rng(n).uniform(0.0, (n / 33.4) ** (1 / 3), (n, 3))
    x[na // 2, 1] = bad
    act = P.Coordination(f"c: COORDINATION GROUPA=1-{na} " + (f"GROUPB={na + 1}-{n} " if nb else "")
                         + f"NOPBC SWITCH={{{sw}}}{nl}")
    v, d, w = act.calculate(x, np.eye(3))
    st = act.stats()
    assert st["path"] == 1
    good = np.delete(np.arange(n), na // 2)
    ov, od, ow, npair = O.coordination(O.Switch(sw), np.eye(3), x[good], na - 1, nb, use_pbc=False)
    assert st["contributing_pairs"] == npair and abs(v - ov) <= 1e-12 * abs(ov)
    if nl:  # such a pair is in no list
        assert np.max(np.abs(d[good] - od)) <= 1e-12 * np.max(np.abs(od)) and not np.any(d[na // 2])
        return
    _, od, ow, _ = O.coordination(O.Switch(sw), np.eye(3), x, na, nb, use_pbc=False)
    assert np.array_equal(np.isnan(d), np.isnan(od)) and np.any(np.isnan(od))
    assert np.array_equal(np.isnan(w), np.isnan(ow))
    ok = ~np.isnan(od)
    if np.any(ok):
        assert np.max(np.abs(d[ok] - od[ok])) <= 1e-12 * np.max(np.abs(od[ok]))
