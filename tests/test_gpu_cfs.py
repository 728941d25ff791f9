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


# One wave per CU has 16,384 lanes on 256 CUs: a lane of the one-lane kernel runs three fits and more, in chunks from
# the queue, before the wave leaves its last ones; a group of the split kernel (elliptical K = 3) takes nine.
@pytest.mark.parametrize("loc,R,n", [(0, 7, 50001), (0, 7, 49000), (0, 7, 15001), (0, 9, 50001), (0, 11, 50001), (1, 7, 40001), (1, 9, 50001), (1, 11, 40001)])
def test_refilled_lanes_match_bitwise(gpu, loc, R, n):
    import torch
    m = 499
    sp = Q.default_sim(width=R, height=R, astig=loc, n_per_unit_max=3, min_sep=1.0, max_sep=4.0, photons_min=300.0, photons_max=6000.0)
    rois, _ = Q.sim_rois_host(sp, 5400 + 10 * R + loc, m)
    d = torch.from_numpy(rois.view(np.int16)).cuda()
    p = Q.default_params(QE=1.0, ROISize=R, LocType=loc, p1_XGY=-111.11, p1_XLY=-111.11)
    ctx, one = Q.Context(p), Q.Context(p)
    ctx.set_tuning(waves_per_cu=1)
    one.set_tuning(queue=0)
    idx = torch.arange(n, device="cuda") % m
    r = d[idx].contiguous()
    prev = None
    for K in (1, 2, 3):
        mode = Q.CFIT_INIT_HEUR if K == 1 else Q.CFIT_INIT_ADD
        th, info, ll = _fit(one, K, d, m, mode, prev)
        t, i, l = _fit(ctx, K, r, n, mode, prev[idx].contiguous() if prev is not None else None)
        assert torch.equal(t.view(torch.int32), th.view(torch.int32)[idx]), K
        assert torch.equal(i[:, :2], info[idx, :2]), K
        assert torch.equal(l.view(torch.int64), ll.view(torch.int64)[idx]), K
        assert bool((i[:, 2] <= info[idx, 2]).all()), K
        prev = th


@pytest.mark.parametrize("wpc", [0, 1])
def test_mixed_sizes_past_the_line_match_one_pass(gpu, wpc):
    """Three sizes in one launch of the one-lane kernel, each with its own queue and left fits."""
    import torch
    m = 300
    ctx = Q.Context(Q.default_params(QE=1.0, ROISize=7, PixelSize=100.0))
    ctx.set_tuning(waves_per_cu=wpc)
    sets, refs = [], []
    for R, n in ((7, 30001), (9, 20003), (11, 9007)):
        sp = Q.default_sim(width=R, height=R, n_per_unit_max=3, min_sep=1.0, max_sep=4.0, photons_min=500.0, photons_max=5000.0)
        d = torch.from_numpy(Q.sim_rois_host(sp, 5500 + R, m)[0].view(np.int16)).cuda()
        one = Q.Context(Q.default_params(QE=1.0, ROISize=R, PixelSize=100.0))
        one.set_tuning(queue=0)
        rl = torch.zeros((3 * m, 12), dtype=torch.float32, device="cuda")
        rs = torch.zeros(m, dtype=torch.int32, device="cuda")
        one.fit_mle_dev(d, m, 3, rl, rs)
        idx = torch.arange(n, device="cuda") % m
        sets.append((R, d[idx].contiguous(), n, torch.full((3 * n, 12), -7.0, device="cuda"), torch.full((n,), -7, dtype=torch.int32, device="cuda")))
        refs.append((rl.reshape(m, 36), rs, idx))
    ctx.fit_mle_mixed_dev(sets, 3)
    torch.cuda.synchronize()
    for (R, _, n, loc, sel), (rl, rs, idx) in zip(sets, refs):
        assert torch.equal(sel, rs[idx]), R
        assert torch.equal(loc.reshape(n, 36).view(torch.int32), rl[idx].view(torch.int32)), R
        assert (rs == 3).any() and (rs == 1).any()
