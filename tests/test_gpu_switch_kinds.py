"""Every switch type through the cluster pair kernel compiled for it (one and
two groups, derivatives), against the FP64 oracle, with D_0 > 0 (the flat part)
among them, and two atoms at one place where the switch has a gradient there
(TANH and Q with D_0 = 0 have a kink at zero distance).  Tolerances of the cluster path: the pair
terms are FP64 rounded to FP32 (2^-24 each, sums of at most ~500 a lane)."""
import numpy as np
import pytest

import oracle as O
from test_gpu_coordination import check

pytestmark = pytest.mark.gpu

KINDS = ["RATIONAL R_0=0.3 NN=8 MM=20 D_MAX=1.1", "RATIONAL R_0=0.25 NN=6 MM=10 D_0=0.1 D_MAX=1.0",
         "RATIONAL R_0=0.3 NN=7 MM=13 D_MAX=1.0", "RATIONAL R_0=0.3 NN=14 MM=28 D_MAX=1.0", "EXP R_0=0.2 D_0=0.1 D_MAX=1.0",
         "GAUSSIAN R_0=0.3 D_MAX=1.0", "GAUSSIAN R_0=1.0 D_MAX=1.1", "SMAP R_0=0.4 A=3 B=2 D_MAX=1.0",
         "CUBIC D_0=0.2 D_MAX=0.9", "TANH R_0=0.4 D_MAX=1.0", "COSINUS R_0=0.8 D_MAX=1.0",
         "Q R_0=0.3 BETA=20 LAMBDA=1.5 REF=0.3 D_MAX=1.0"]


@pytest.mark.parametrize("nb", [0, 400])
@pytest.mark.parametrize("sw", KINDS)
def test_switch_kind(sw, nb):
    import plumed2_amd as P

    n = 1500
    rng = np.random.default_rng(17)
    x = rng.uniform(0.0, 3.1, (n, 3))
    if not sw.startswith(("TANH", "Q ")):
        x[7] = x[1203]
    box = np.array([[3.1, 0.0, 0.0], [0.2, 3.0, 0.0], [-0.1, 0.25, 3.2]])
    groups = f"GROUPA=1-{n - nb}" + (f" GROUPB={n - nb + 1}-{n}" if nb else "")
    act = P.Coordination(f"c: COORDINATION {groups} SWITCH={{{sw}}}")
    v, d, w = act.calculate(x, box)
    ov, od, ow, npair = O.coordination(O.Switch(sw), box, x, n - nb, nb)
    check(v, d, w, ov, od, ow)
    st = act.stats()
    assert st["path"] == 0 and st["contributing_pairs"] == npair
