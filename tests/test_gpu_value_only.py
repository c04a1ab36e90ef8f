"""Value-only calls (no derivatives asked for) under every switch, groups apart
and groups that share atoms, against the FP64 oracle: values to 1e-6 as for the
calls with derivatives (FP64 terms rounded to FP32, FP64 sums), pair counts
equal; and such a call takes no longer than one with derivatives (5% for the
clock)."""
import numpy as np
import pytest

import oracle as O
from test_gpu_rows_speed import _time
from test_gpu_switch_kinds import KINDS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", ["one", "apart", "shared"])
@pytest.mark.parametrize("sw", KINDS)
def test_value_only(sw, groups):
    import torch
    import plumed2_amd as P

    n = 1500
    x = np.random.default_rng(19).uniform(0.0, 3.1, (n, 3))
    box = np.array([[3.1, 0.0, 0.0], [0.2, 3.0, 0.0], [-0.1, 0.25, 3.2]])
    na, lo = {"one": (n, n), "apart": (1100, 1100), "shared": (1100, 700)}[groups]
    req = np.concatenate([np.arange(na), np.arange(lo, n)])
    line = f"c: COORDINATION GROUPA=1-{na} " + (f"GROUPB={lo + 1}-{n} " if lo < n else "")
    act = P.Coordination(line + f"SWITCH={{{sw}}}")
    t = torch.tensor(x[req], dtype=torch.float64, device="cuda:0")
    v = torch.empty(1, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    act.calculate_device(t.data_ptr(), box, 0, v.data_ptr(), 0, 0)
    st = act.stats()
    ov, _, _, npair = O.coordination(O.Switch(sw), box, x[req], na, n - lo, absidx=req)
    assert st["path"] == 0 and st["contributing_pairs"] == npair
    torch.cuda.synchronize()
    assert abs(float(v) - ov) <= 1e-6 * abs(ov)


@pytest.mark.parametrize("sw", ["EXP R_0=0.1 D_MAX=0.8", "TANH R_0=0.3 D_MAX=0.8", "RATIONAL R_0=0.3 NN=6 MM=12 D_MAX=0.8"])
def test_no_slower_than_with_derivatives(sw):
    import torch
    import plumed2_amd as P

    n = 200000
    box = np.diag([(n / 33.4) ** (1 / 3)] * 3)
    x = torch.tensor(np.random.default_rng(20).uniform(0, box[0, 0], (n, 3)), dtype=torch.float64, device="cuda:0")
    v = torch.empty(1, dtype=torch.float64, device="cuda:0")
    act = P.Coordination(f"c: COORDINATION GROUPA=1-{n} SWITCH={{{sw}}}")
    act.set_stream(torch.cuda.current_stream().cuda_stream)
    full = _time(lambda: act.calculate_torch(x, box, 0))
    alone = _time(lambda: act.calculate_device(x.data_ptr(), box, 0, v.data_ptr(), 0, 0))
    assert alone <= 1.05 * full, (alone, full)
