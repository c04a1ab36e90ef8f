"""p2a_metad_forces_device against p2a_apply_force_device and
p2a_cdist_apply_force_device on cleared arrays (the same FP64 products and
sums: equal bit for bit), at group sizes around the workgroup, with atoms in
both groups and without a distance; and the centre distance at the sizes of
its trips (512 atoms of a group) against the oracle (1e-12, as the chain's
tests)."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n1,n2", [(2, 1, 1), (300, 255, 257), (5000, 513, 600), (1111, 0, 0)])
def test_forces_in_one_pass(n, n1, n2):
    import torch

    import plumed2_amd as P
    from plumed2_amd import _capi as A

    rng = np.random.default_rng(n)
    dev = torch.device("cuda")
    t = lambda *s: torch.tensor(rng.normal(size=s), device=dev)  # noqa: E731
    f, d, w, dd, wd = t(2), t(n, 3), t(3, 3), t(max(n1 + n2, 1), 3), t(3, 3)
    cd = None
    if n1:
        g1, g2 = rng.permutation(n)[:n1], rng.permutation(n)[:n2]
        cd = P.CenterDistance(n, g1, g2)
    s = torch.cuda.current_stream().cuda_stream
    p = lambda x: C.c_void_p(x.data_ptr())  # noqa: E731
    F, W = torch.full((n, 3), 7.0, device=dev, dtype=torch.float64), torch.full((3, 3), 7.0, device=dev, dtype=torch.float64)
    A.check(A.lib().p2a_metad_forces_device(C.c_void_p(s), n, p(f), p(d), p(w), cd._ctx if cd else None, p(dd), p(wd),
                                            p(F), p(W)))
    F0, W0 = torch.zeros_like(F), torch.zeros_like(W)
    A.check(A.lib().p2a_apply_force_device(C.c_void_p(s), n, p(f), p(d), p(w), p(F0), p(W0)))
    if cd:
        cd.apply_force_device(s, f.data_ptr() + 8, dd.data_ptr(), wd.data_ptr(), F0.data_ptr(), W0.data_ptr())
    assert torch.equal(F, F0) and torch.equal(W, W0)


@pytest.mark.parametrize("n1,n2", [(1, 1), (1, 700), (511, 512), (513, 1025), (64, 65)])
@pytest.mark.parametrize("masses", [False, True])
def test_center_distance_sizes(n1, n2, masses):
    import torch

    import plumed2_amd as P

    rng = np.random.default_rng(n1 + n2)
    n = n1 + n2
    box = np.array([[4.0, 0.0, 0.0], [0.5, 3.9, 0.0], [-0.4, 0.3, 4.2]])
    # two compact chains that cross the cell's faces
    x = np.concatenate([np.cumsum(rng.normal(0, 0.05, (k, 3)), axis=0) + o for k, o in ((n1, 0.1), (n2, 1.7))])
    x = x + rng.integers(-1, 2, (n, 3)) @ box
    m = rng.uniform(1.0, 16.0, n) if masses else None
    cd = P.CenterDistance(n, np.arange(n1), np.arange(n1, n), masses=m)
    v, d, w = (t.cpu().numpy() for t in cd.calculate_torch(torch.tensor(x, device="cuda"), box))
    ov, od, ow, _, _ = O.center_distance(box, x, np.arange(n1), np.arange(n1, n), masses=m)
    assert abs(v[0] - ov) <= 1e-12 * abs(ov)
    assert np.max(np.abs(d - od)) <= 1e-12 * np.max(np.abs(od))
    assert np.max(np.abs(w - ow)) <= 1e-12 * np.max(np.abs(ow))
