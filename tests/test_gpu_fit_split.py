"""Fits with an ROI split over a group of lanes: every group size the dispatch chooses gives the
oracle's rows bit for bit, at the smallest calls and on both sides of each line of the rule."""
import numpy as np
import pytest

import qcstorm as Q
import oracle_lib as O

pytestmark = pytest.mark.gpu


def _sample(R, loc, m, kmax):
    """m simulated ROI records, the last eight of them degenerate (they take the log's general form)."""
    sp = Q.default_sim(width=R, height=R, astig=loc, n_per_unit_max=kmax, min_sep=1.0, max_sep=3.0, photons_min=600, photons_max=6000)
    rois, _ = Q.sim_rois_host(sp, 4100 + 10 * R + loc, m)
    px = rois[:, :R * R]
    k = np.arange(R * R)
    px[-8] = 0
    px[-7] = 65535
    px[-6] = 100
    px[-5] = np.where(k == R * R // 2, 60000, 100)
    px[-4] = np.where(k % 2 == 0, 65535, 0)
    px[-3] = np.where(k % R == 0, 30000, 90)
    px[-2] = 100 + k
    px[-1] = np.where(k < R, 65535, 101)
    return rois, O.wle(rois, R, loc)


def _tiled(params, rois, wle, n, loc_cap):
    import torch
    m = len(rois)
    idx = torch.arange(n, device="cuda") % m
    d_r = torch.from_numpy(rois.view(np.int16)).cuda()[idx].contiguous()
    d_w = torch.from_numpy(wle).cuda()[idx].contiguous()
    loc = torch.full((loc_cap, 12), -3.0, dtype=torch.float32, device="cuda")
    rows = Q.Context(params).fit_dev(d_r, d_w, n, loc)
    torch.cuda.synchronize()
    return loc, rows, idx


ONE = [(0, 5, (24000, 24001, 64001, 240001)), (0, 7, (24000, 24001, 400001)), (1, 7, (24001, 200001)), (0, 9, (28001, 110001)),
       (1, 9, (28001, 110001)), (1, 5, (64001, 240001)), (0, 11, (28001,)), (1, 11, (28001,)), (0, 13, ()), (1, 13, ()), (0, 15, ()),
       (1, 15, ()), (0, 17, (20001,)), (1, 17, (20001,))]


@pytest.mark.parametrize("loc,R,lines", ONE)
def test_one_emitter_groups_bit_exact(gpu, loc, R, lines):
    import torch
    m = 151
    rois, wle = _sample(R, loc, m, 1)
    params = Q.default_params(QE=1.0, ROISize=R, LocType=loc, p1_XGY=-111.11, p1_XLY=-111.11)
    ref, _ = O.fit(params, rois, wle)
    ref = torch.from_numpy(ref.view(np.int32)).cuda()
    for n in (1, 17, m) + lines:
        got, rows, idx = _tiled(params, rois, wle, n, n)
        assert rows == n
        bad = (got.view(torch.int32) != ref[idx]).any(1).sum().item()
        assert bad == 0, (n, bad)


@pytest.mark.parametrize("loc,R,k", [(0, 5, 332), (0, 7, 332), (1, 7, 332), (0, 9, 663), (1, 9, 199), (0, 11, 663), (1, 11, 199), (0, 13, 3),
                                     (1, 13, 3)])
def test_cascade_groups_bit_exact(gpu, loc, R, k):
    """k copies of a sample (past the narrow group's line): each copy's rows, and k times its appended rows."""
    import torch
    m = 151
    rois, _ = _sample(R, loc, m, 3)
    rois[::3, R * R + 4] = 1    # the detector's multi flag
    wle = O.wle(rois, R, loc)
    params = Q.default_params(QE=1.0, ROISize=R, LocType=loc, MultiEmitterFitEn=1, p1_XGY=-111.11, p1_XLY=-111.11)
    ref, _ = O.fit(params, rois, wle)
    extra = len(ref) - m
    ref = torch.from_numpy(ref[:m].view(np.int32)).cuda()
    for c in (1, k):
        got, rows, idx = _tiled(params, rois, wle, c * m, 2 * c * m)
        assert rows == c * (m + extra)
        bad = (got[:c * m].view(torch.int32) != ref[idx]).any(1).sum().item()
        assert bad == 0, (c, bad)


@pytest.mark.parametrize("loc", [0, 1])
def test_fast_math_groups_agree(gpu, loc):
    """The hardware exp and log give the same rows for every group size."""
    import torch
    m = 151
    rois, wle = _sample(7, loc, m, 1)
    params = Q.default_params(QE=1.0, LocType=loc, FitMath=Q.MATH_FAST, p1_XGY=-111.11, p1_XLY=-111.11)
    ref = None
    for n in (m, 24001, 400001):
        got, _, idx = _tiled(params, rois, wle, n, n)
        if ref is None:
            ref = got.view(torch.int32).clone()
        assert torch.equal(got.view(torch.int32), ref[idx])


# both sides of the lines that calls with the hardware exp and log have of their own
FAST = [(0, 5, (8192, 8193, 16385, 32769)), (1, 5, (32769,)), (0, 7, (8193, 36001, 65537, 100001)), (1, 7, (36001, 65537)),
        (0, 9, (6000, 6001, 16385, 36001, 65537, 100001)), (1, 9, (6001, 16385, 200001)), (0, 13, (26000, 26001, 70003)),
        (1, 13, (26000, 26001))]


@pytest.mark.parametrize("loc,R,lines", FAST)
def test_fast_math_lines_agree(gpu, loc, R, lines):
    import torch
    m = 151
    rois, wle = _sample(R, loc, m, 1)
    params = Q.default_params(QE=1.0, ROISize=R, LocType=loc, FitMath=Q.MATH_FAST, p1_XGY=-111.11, p1_XLY=-111.11)
    ref, _, _ = _tiled(params, rois, wle, m, m)
    ref = ref.view(torch.int32)
    assert (ref[:, 0] != 0).sum().item() > m // 8   # the 5x5 window refuses most elliptical shapes (40 stay)
    for n in lines:
        got, rows, idx = _tiled(params, rois, wle, n, n)
        assert rows == n
        assert torch.equal(got.view(torch.int32), ref[idx]), n
