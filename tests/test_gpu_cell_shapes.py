"""One context over cells of changing shape, whose column grids grow and shrink,
against a fresh context per cell: the same bits (atoms are ranked by key and
index, and every sum has a fixed order), and the oracle's pair counts."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SW = "RATIONAL R_0=0.2 NN=6 MM=12 D_MAX=0.4"
# tall to flat and back: the number of columns follows the face across c
CELLS = [(1.0, 1.0, 9.0), (1.2, 1.1, 7.0), (1.5, 1.5, 4.0), (1.8, 1.7, 3.0), (2.2, 2.1, 2.0), (2.6, 2.7, 1.3),
         (3.1, 3.1, 0.95), (1.0, 1.0, 9.0), (3.1, 3.1, 0.95), (2.2, 2.1, 2.0)]


@pytest.mark.parametrize("na,nb", [(300, 0), (120, 180), (40, 520), (2100, 0)])
def test_one_context_over_changing_cells(na, nb):
    import plumed2_amd as P

    n = na + nb
    k = (n / 300.0) ** (1.0 / 3.0)
    line = f"c: COORDINATION GROUPA=1-{na} " + (f"GROUPB={na + 1}-{n} " if nb else "") + f"SWITCH={{{SW}}}"
    act = P.Coordination(line)
    rng = np.random.default_rng(21)
    for step, edges in enumerate(CELLS):
        box = np.diag(np.array(edges) * k)
        x = rng.uniform(0.0, 1.0, (n, 3)) @ box
        v, d, w = act.calculate(x, box, step)
        st = act.stats()
        assert st["path"] == 0
        fresh = P.Coordination(line)
        fv, fd, fw = fresh.calculate(x, box, step)
        fresh.close()
        assert v == fv and np.array_equal(d, fd) and np.array_equal(w, fw), edges
        assert st["contributing_pairs"] == O.coordination(O.Switch(SW), box, x, na, nb)[3], edges


def test_rows_of_one_context_over_changing_cells():
    import torch
    import plumed2_amd as P

    n = 300
    rng = np.random.default_rng(22)
    wt = rng.normal(size=n)
    cn = P.CoordinationNumbers(SW, species=range(n))
    for edges in CELLS:
        box = np.diag(edges)
        x = torch.tensor(rng.uniform(0.0, 1.0, (n, 3)) @ box, dtype=torch.float64, device="cuda:0")
        got = cn(x, box, weights=wt)
        assert cn.action.stats()["path"] == 0
        fresh = P.CoordinationNumbers(SW, species=range(n))
        want = fresh(x, box, weights=wt)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), edges
