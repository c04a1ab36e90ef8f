"""The FP64 kernels (no cell, a cell narrower than twice the cut, no D_MAX)
against the FP64 oracle at the edges of their work split: wave and workgroup
remainders, one atom per workgroup up to 1,024 atoms and four above, one
thread per atom for many atoms against few, lists short and long.

Both sides sum at most ~1e4 FP64 terms per output, in another order:
1e4 * 2^-53 ~ 1e-12 of the sum of magnitudes, held to 1e-10."""
import numpy as np
import pytest

import oracle as O
from test_gpu_coordination import check

pytestmark = pytest.mark.gpu

SW = ["RATIONAL R_0=0.3", "RATIONAL R_0=0.35 NN=8 MM=16 D_MAX=1.6", "RATIONAL R_0=0.3 NN=8 MM=20", "EXP R_0=0.2 D_MAX=1.7"]
ORTHO = np.diag([2.9, 3.2, 3.05])
TRIC = np.array([[3.0, 0.0, 0.0], [0.4, 3.1, 0.0], [-0.3, 0.5, 2.9]])


def _line(na, nb, sw, extra=""):
    return (f"c: COORDINATION GROUPA=1-{na} " + (f"GROUPB={na + 1}-{na + nb} " if nb else "")
            + f"SWITCH={{{sw}}} {extra}")


@pytest.mark.parametrize("na,nb", [(1, 1), (2, 0), (63, 0), (257, 0), (1024, 0), (1025, 0), (1030, 3), (5, 1027),
                                   (4097, 64), (65, 4099), (2, 5000)])
@pytest.mark.parametrize("case", [(0, None), (1, ORTHO), (2, TRIC), (3, None)])
def test_all_pairs_split(na, nb, case):
    import plumed2_amd as P

    k, box = case
    n = na + nb
    x = np.random.default_rng(n).uniform(-0.5, 3.5, (n, 3))
    act = P.Coordination(_line(na, nb, SW[k], "" if box is not None else "NOPBC"))
    v, d, w = act.calculate(x, np.eye(3) if box is None else box)
    ov, od, ow, npair = O.coordination(O.Switch(SW[k]), np.eye(3) if box is None else box, x, na, nb,
                                       use_pbc=box is not None)
    check(v, d, w, ov, od, ow, 1e-10, 1e-10, 1e-10)
    st = act.stats()
    assert st["path"] == 1 and st["contributing_pairs"] == npair


@pytest.mark.parametrize("na,nb,mode", [(3, 0, "NLIST"), (259, 0, "NLISTCELLS"), (1500, 0, "NLIST"),
                                        (700, 2100, "NLIST"), (40, 2600, "NLISTCELLS"), (1, 700, "NLIST")])
@pytest.mark.parametrize("box", [ORTHO, TRIC, None])
def test_listed_pairs_split(na, nb, mode, box):
    import plumed2_amd as P

    n = na + nb
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 3.0, (n, 3))
    sw, cut = "RATIONAL R_0=0.3 D_MAX=1.2", 1.5
    act = P.Coordination(_line(na, nb, sw, f"{mode} NL_CUTOFF={cut} NL_STRIDE=3" + ("" if box is not None else " NOPBC")))
    b = ORTHO if box is None else box
    for step in range(4):
        if step % 3 == 0:
            pbc = O.Pbc(b)
            pairs = (O.nl_classic(pbc, box is not None, cut, x, na, nb) if mode == "NLIST" or box is None
                     else O.nl_cells(pbc, cut, x, na, nb))
        v, d, w = act.calculate(x, b, step=step)
        ov, od, ow, npair = O.coordination(O.Switch(sw), b, x, na, nb, use_pbc=box is not None, pairs=pairs)
        check(v, d, w, ov, od, ow, 1e-10, 1e-10, 1e-10)
        assert act.stats()["contributing_pairs"] == npair
        x = x + rng.normal(0.0, 0.01, x.shape)


@pytest.mark.parametrize("nrows,nenv", [(1, 1), (3, 65), (5, 700), (130, 64)])
def test_number_rows_split(nrows, nenv):
    import torch

    import plumed2_amd as P

    n = nrows + nenv
    x = np.random.default_rng(n).uniform(0.0, 2.5, (n, 3))
    sw = "RATIONAL R_0=0.3"
    cn = P.coordination_numbers_torch(sw, torch.tensor(x, device="cuda"), box=TRIC, species_a=range(nrows),
                                      species_b=range(nrows, n)).cpu().numpy()
    ref = O.coordination_numbers(O.Switch(sw), TRIC, x, species_a=range(nrows), species_b=range(nrows, n))
    assert np.max(np.abs(cn - ref)) <= 1e-10 * np.max(np.abs(ref))
