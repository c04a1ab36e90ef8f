"""Depositions captured into a HIP graph, replayed between eager depositions of
other lengths, and calls longer than the cells kept at once: bit for bit the
same hills through eager calls in shorter parts (every node and corner receives
the same FP64 additions in the same order)."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_hills import _line, _walk

pytestmark = pytest.mark.gpu


def _parts(m, c, n):
    return np.concatenate([m.deposit(c[k:k + n]) for k in range(0, len(c), n)])


def _same(m1, m2):
    (v1, d1), (v2, d2) = m1.grid(), m2.grid()
    return np.array_equal(v1, v2) and np.array_equal(d1, d2)


@pytest.mark.parametrize("warm", [True, False])
@pytest.mark.parametrize("ncv,periodic,bins,n", [(2, (False, False), (40, 33), 300), (2, (True, True), (50, 64), 17),
                                                 (4, (False, True, False, True), (9, 40, 11, 35), 70)])
def test_replayed_between_longer_calls(ncv, periodic, bins, n, warm):
    import torch
    import plumed2_amd as P
    from plumed2_amd import _capi as A

    line, per = _line(ncv, periodic, bins)
    m1, m2 = P.MetaD(line, periodic=per), P.MetaD(line, periodic=per)
    c = _walk(n, periodic, 5)
    ct = torch.tensor(c, dtype=torch.float64, device="cuda:0")
    ht = torch.zeros(n, dtype=torch.float64, device="cuda:0")
    s = torch.cuda.Stream()
    A.check(A.lib().p2a_metad_set_stream(m1._ctx, C.c_void_p(s.cuda_stream)))
    if warm:  # the workspace is there before the capture
        w = _walk(9, periodic, 6)
        assert np.array_equal(m1.deposit(w), _parts(m2, w, 1))
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        A.check(A.lib().p2a_metad_deposit_device(m1._ctx, n, C.c_void_p(ct.data_ptr()), C.c_void_p(ht.data_ptr())))
    # longer than everything before, and longer than the cells kept at once
    for k, more in enumerate((3, 66 * (1024 >> ncv) + 5, 40)):
        e = _walk(more, periodic, 7 + k)
        assert np.array_equal(m1.deposit(e), _parts(m2, e, 1000))
        scratch = [torch.full((1 << 18,), float("nan"), device="cuda:0") for _ in range(8)]
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(ht.cpu().numpy(), m2.deposit(c))
        assert _same(m1, m2)
        del scratch


@pytest.mark.parametrize("at", [None, 4095, 4096, 4161, 8200])
def test_calls_longer_than_the_cells_kept_at_once(at):
    import plumed2_amd as P

    ncv, periodic, bins = 4, (False, True, False, True), (9, 40, 11, 35)
    line, per = _line(ncv, periodic, bins)
    n = 2 * 64 * 64 + 64 + 3
    c = _walk(n, periodic, 8)
    m1, m2 = P.MetaD(line, periodic=per), P.MetaD(line, periodic=per)
    if at is None:
        assert np.array_equal(m1.deposit(c), _parts(m2, c, 999))
    else:
        bad = c.copy()
        bad[at, 0] = 5.0
        with pytest.raises(P.Plumed2AmdError, match="outside the grid"):
            m1.deposit(bad)
        _parts(m2, c[:at], 999)
    assert _same(m1, m2)
