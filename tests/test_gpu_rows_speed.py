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


def test_many_rows_of_a_small_environment():
    """FP64 rows of 500,000 atoms: against one environment atom less than half
    of the time against 128 (a wave per row takes nearly the same for both)."""
    import ctypes as C
    import torch
    import plumed2_amd as P
    from plumed2_amd import _capi as A

    n = 500128
    sw = P.parse_switch("RATIONAL R_0=0.3 NN=6 MM=12 D_MAX=1.2")
    x = torch.tensor(np.random.default_rng(2).uniform(0, 24.0, (n, 3)), dtype=torch.float64, device="cuda:0")
    idx = torch.arange(n, dtype=torch.int32, device="cuda:0")
    cn = torch.empty(500000, dtype=torch.float64, device="cuda:0")
    s = torch.cuda.current_stream().cuda_stream

    def rows(nenv):
        A.check(A.lib().p2a_coordination_numbers_device(
            s, C.byref(sw), None, 0, n, 500000, idx.data_ptr(), nenv, idx.data_ptr() + 4 * 500000, x.data_ptr(),
            cn.data_ptr()))

    t = [_time(lambda: rows(k)) for k in (1, 128)]
    assert t[0] <= 0.5 * t[1], t


@pytest.mark.parametrize("nrows,nenv", [(1, 1), (999, 1), (1000, 1), (16001, 16), (15999, 16), (300, 129), (1 << 18, 3)])
def test_both_forms_of_the_rows_against_plain_torch(nrows, nenv):
    import torch
    import plumed2_amd as P

    rng = np.random.default_rng(nrows + nenv)
    x = torch.tensor(rng.uniform(0, 3.0, (nrows + nenv, 3)), dtype=torch.float64, device="cuda:0")
    got = P.coordination_numbers_torch("RATIONAL R_0=0.3 NN=6 MM=12 D_MAX=1.2 NOSTRETCH", x, None,
                                       species_a=range(nrows), species_b=range(nrows, nrows + nenv))
    r2 = ((x[:nrows, None] - x[None, nrows:]) ** 2).sum(-1)
    want = torch.where(r2 <= 1.2 ** 2, 1.0 / (1.0 + (r2 / 0.09) ** 3), 0.0).sum(1)
    # sums of at most 129 terms in [0, 1], each good to a few ulp
    assert torch.max(torch.abs(got - want)) <= 1e-13 * nenv
