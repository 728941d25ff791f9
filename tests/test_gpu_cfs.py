"""Converged fits split over lanes (cfs.hip): shared by a whole wave, one to a group, resumed from the
one-lane kernel, and the one-pass kernel all give the same parameters, counts and flags."""
import numpy as np
import pytest

import qcstorm as Q

pytestmark = pytest.mark.gpu


def _fit(ctx, K, d_rois, n, mode, init):
    import torch
    P = 5 * K + 1 if ctx.params.LocType == Q.LOCTYPE_AS3D else 3 * K + 2
    th = torch.full((n, P), -7.0, dtype=torch.float32, device="cuda")
    info = torch.full((n, 4), -7, dtype=torch.int32, device="cuda")
    ll = torch.zeros(n, dtype=torch.float64, device="cuda")
    ctx.cfit_dev(K, d_rois, n, mode, init, th, info, ll)
    torch.cuda.synchronize()
    return th, info, ll


# the second size of each model is past its line for whole launches of the split kernel
@pytest.mark.parametrize("loc,R,sizes", [(0, 7, (1, 5, 12001, 50000)), (0, 9, (28001,)), (0, 11, (3, 40001)), (1, 7, (12001,)),
                                         (1, 9, (2, 9000, 50000)), (1, 11, (1, 12001))])
def test_split_fits_match_bitwise(gpu, loc, R, sizes):
    import torch
    m = 499
    sp = Q.default_sim(width=R, height=R, astig=loc, n_per_unit_max=3, min_sep=1.0, max_sep=4.0, photons_min=300.0, photons_max=6000.0)
    rois, _ = Q.sim_rois_host(sp, 5200 + 10 * R + loc, m)
    rois[-3, :R * R] = 65535
    rois[-2, :R * R] = 0
    rois[-1, :R * R] = np.where(np.arange(R * R) == R + 1, 60000, 100)
    d = torch.from_numpy(rois.view(np.int16)).cuda()
    p = Q.default_params(QE=1.0, ROISize=R, LocType=loc, p1_XGY=-111.11, p1_XLY=-111.11)
    ctx, one = Q.Context(p), Q.Context(p)
    one.set_tuning(queue=0)
    prev = None
    for K in (1, 2, 3):
        mode = Q.CFIT_INIT_HEUR if K == 1 else Q.CFIT_INIT_ADD
        th, info, ll = _fit(ctx, K, d, m, mode, prev)
        th1, info1, ll1 = _fit(one, K, d, m, mode, prev)
        assert torch.equal(th.view(torch.int32), th1.view(torch.int32))
        assert torch.equal(info[:, :2], info1[:, :2])
        assert torch.equal(ll.view(torch.int64), ll1.view(torch.int64))
        for n in sizes:
            idx = torch.arange(n, device="cuda") % m
            t, i, l = _fit(ctx, K, d[idx].contiguous(), n, mode, prev[idx].contiguous() if prev is not None else None)
            assert torch.equal(t.view(torch.int32), th.view(torch.int32)[idx]), (K, n)
            assert torch.equal(i, info[idx]), (K, n)    # evaluation counts too
            assert torch.equal(l.view(torch.int64), ll.view(torch.int64)[idx]), (K, n)
        prev = th


def test_split_fits_pin_stop_and_flat_stop(gpu):
    """The opt-in stops count the same trials in every kernel."""
    import torch
    m = 300
    sp = Q.default_sim(width=9, height=9, astig=1, n_per_unit_max=3, min_sep=1.0, max_sep=4.0)
    rois, _ = Q.sim_rois_host(sp, 5301, m)
    d = torch.from_numpy(rois.view(np.int16)).cuda()
    p = Q.default_params(QE=1.0, ROISize=9, LocType=1, p1_XGY=-111.11, p1_XLY=-111.11)
    out = []
    for queue, rep in ((0, 1), (1, 1), (1, 40)):
        ctx = Q.Context(p)
        ctx.set_tuning(pin_stop=1, queue=queue)
        r = d.repeat(rep, 1).contiguous()
        prev = None
        for K in (1, 2, 3):
            prev, info, _ = _fit(ctx, K, r, m * rep, Q.CFIT_INIT_HEUR if K == 1 else Q.CFIT_INIT_ADD, prev)
        out.append((prev.view(torch.int32)[-m:].clone(), info[-m:, :2].clone()))
    assert (out[0][1][:, 1] & Q.CFIT_PINNED).any()
    for t, i in out[1:]:
        assert torch.equal(t, out[0][0]) and torch.equal(i, out[0][1])
