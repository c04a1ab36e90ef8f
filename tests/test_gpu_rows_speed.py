"""Time of COORDINATIONNUMBER calls against calls of the same work in another
form, on the GPU's clock with margins of several times."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _time(f, calls=20):
    import torch
    for _ in range(3):
        f()
    best = float("inf")
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(calls):
            f()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) / calls)
    return best


def test_weighted_rows_of_groups_that_share_atoms():
    """Rows that are also environment atoms: no more than three times the call
    with the groups apart (a search per pair inside D_MAX takes 15 times it)."""
    import torch
    import plumed2_amd as P

    n, na = 30000, 3000
    box = np.diag([(n / 33.4) ** (1 / 3)] * 3)
    x = torch.tensor(np.random.default_rng(1).uniform(0, box[0, 0], (n, 3)), dtype=torch.float64, device="cuda:0")
    w = torch.ones(na, dtype=torch.float64, device="cuda:0")
    t = []
    for env in (range(n), range(na, n)):
        cn = P.CoordinationNumbers("RATIONAL R_0=0.3 NN=6 MM=12 D_MAX=1.2", species_a=range(na), species_b=env)
        t.append(_time(lambda: cn(x, box, weights=w)))
        assert cn.action.stats()["path"] == 0
        cn.close()
    assert t[0] <= 3.0 * t[1], t
