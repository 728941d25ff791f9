"""The scans, the row sort and the neighbour table at the edges of their launches, exactly as the oracle:
one-launch and two-launch scans and their tiles, one to four digits of the frame, rows at every digit's end,
bucket tables of the smallest and of larger sizes."""
import numpy as np
import pytest
import torch

import oracle_lib as O
import qcstorm as Q
from test_gpu_stats import _check
from test_gpu_stats import _rows as _stat_rows

pytestmark = pytest.mark.gpu


def _rows(n, seed, frames):
    rng = np.random.default_rng(seed)
    loc = rng.normal(0, 1, (n, 12)).astype(np.float32)
    loc[:, 0] = rng.choice([0.0, 0.5, 1.0, 1.5, 2.0, 400.0, np.nan], n)
    loc[:, 11] = rng.choice(frames, n)
    return loc


# 2048 rows are a tile of the sort, 4096 / 16384 items a tile of the two-launch / one-launch scan; the sort
# scans 256 counts a tile, so 131,072 rows (64 tiles) are the last with one launch
@pytest.mark.parametrize("n", [1, 63, 64, 65, 2047, 2048, 2049, 4097, 16383, 16384, 16385, 20481, 131072, 131073])
def test_rows_sorted_and_unsorted(gpu, n):
    loc = _rows(n, n, np.arange(1, 40))
    ctx = Q.Context(Q.default_params(ImageWidth=64, ImageHigh=64))
    d = torch.from_numpy(loc).cuda()
    out = torch.full_like(d, -7.0)
    m = ctx.compact_sorted_dev(d, n, 3, 30, out)
    ref = O.compact_sorted(loc, 3, 30)
    assert m == len(ref)
    np.testing.assert_array_equal(out[:m].cpu().numpy(), ref)
    assert bool((out[m:] == -7.0).all())
    out.fill_(-7.0)
    m = ctx.compact_dev(d, n, out)
    keep = loc[loc[:, 0] > 1.0]
    assert m == len(keep)
    np.testing.assert_array_equal(out[:m].cpu().numpy(), keep)
    assert bool((out[m:] == -7.0).all())


@pytest.mark.parametrize("first,end", [(0, 0), (5, 260), (5, 261), (-300, -45), (-300, 65235), (-300, 65236), (0, 1 << 24),
                                       (-(1 << 24), 1 << 24), (-(1 << 31), (1 << 31) - 1)])
def test_frame_digits(gpu, first, end):
    n = 5000
    mid = (first + end) // 2
    frames = np.array([first - 1, first, first + 1, first + 255, first + 256, mid, mid + 1, end - 256, end - 1, end, end + 1, np.nan,
                       np.inf, -np.inf], np.float64).astype(np.float32)
    loc = _rows(n, 3, frames)
    ctx = Q.Context(Q.default_params(ImageWidth=64, ImageHigh=64))
    d = torch.from_numpy(loc).cuda()
    out = torch.empty_like(d)
    m = ctx.compact_sorted_dev(d, n, first, end, out)
    # the oracle counts every frame of the range: past 2^25 of them its definition is written out here
    if end - first < 1 << 25:
        ref = O.compact_sorted(loc, first, end)
    else:
        with np.errstate(invalid="ignore"):
            fr = np.clip(np.nan_to_num(loc[:, 11].astype(np.float64), nan=0.0), -2.0**31, 2.0**31 - 1).astype(np.int64)
        keep = np.flatnonzero((np.trunc(np.nan_to_num(loc[:, 0])) > 1) & (fr >= first) & (fr <= end))
        ref = loc[keep[np.argsort(fr[keep], kind="stable")]]
    assert m == len(ref) and m > 0
    np.testing.assert_array_equal(out[:m].cpu().numpy(), ref)


# 256 buckets are the fewest; 512 rows are a work-group of the row pass, 16 molecules one of the neighbour pass
@pytest.mark.parametrize("n,nframes,dense", [(1, 1, False), (2, 1, True), (17, 2, True), (255, 3, True), (257, 4, True), (513, 5, False),
                                             (4099, 2, True), (16385, 500, True), (40000, 6, True)])
def test_stats_table(gpu, n, nframes, dense):
    p = Q.default_params(ImageWidth=333, ImageHigh=250)
    _check(p, _stat_rows(n, n, nframes, 333, 250, dense))


def test_stats_far_apart_frames(gpu):
    p = Q.default_params(ImageWidth=100, ImageHigh=64)
    loc = _stat_rows(700, 9, 5, 100, 64, True)
    loc[:, 11] = np.sort(np.random.default_rng(1).choice([-70000.0, -3.0, 0.0, 1.0, 123456.0], 700)).astype(np.float32)
    _check(p, loc)


# the neighbour pass takes 32,768 molecules a round: less than one, a little more than one, several
@pytest.mark.parametrize("n,lt", [(32000, 0), (34500, 0), (34500, 1), (120011, 0)])
def test_stats_rounds_of_the_neighbour_pass(gpu, n, lt):
    p = Q.default_params(ImageWidth=4000, ImageHigh=3000, LocType=lt)
    loc = _stat_rows(n, n + lt, 3, 4000, 3000, True)   # three frames: none is left out
    loc[:, 1:3] = np.clip(loc[:, 1:3], 5.5, [3994.0, 2994.0])
    got = _check(p, loc)
    assert got["density_total"] == n and got["density_n1"] > 0


# past 1,500,000 rows of more than 256 frames the last pass leaves the order and the rows are copied by it
@pytest.mark.parametrize("n", [1500000, 1500001])
@pytest.mark.parametrize("nf", [256, 257, 70000])
def test_rows_of_large_calls(gpu, n, nf):
    g = torch.Generator(device="cuda").manual_seed(nf)
    d = torch.rand((n, 12), generator=g, device="cuda")
    d[:, 0] = torch.randint(0, 5, (n,), generator=g, device="cuda").float()
    fr = torch.randint(0, nf + 2, (n,), generator=g, device="cuda")   # one before the first and one past the last
    d[:, 11] = fr.float()
    keep = torch.nonzero((d[:, 0] > 1) & (fr >= 1) & (fr <= nf)).flatten()
    ref = d[keep[torch.sort(fr[keep], stable=True).indices]]
    out = torch.full_like(d, -7.0)
    ctx = Q.Context(Q.default_params(ImageWidth=64, ImageHigh=64))
    m = ctx.compact_sorted_dev(d, n, 1, nf, out)
    assert m == len(keep)
    assert torch.equal(out[:m], ref)
    assert bool((out[m:] == -7.0).all())


# cells of fewer and of more molecules than a lane walks by itself (24), and both in one call
@pytest.mark.parametrize("lt", [0, 1])
@pytest.mark.parametrize("n,dense", [(400, False), (800, False), (900, True), (5000, False), (20000, True)])
def test_stats_dense_cells(gpu, n, dense, lt):
    W = 96
    p = Q.default_params(ImageWidth=W, ImageHigh=W, LocType=lt)
    rng = np.random.default_rng(n + lt)
    loc = _stat_rows(n, n + lt, 2, W, W, False)
    if dense:   # half of them within one cell's width
        loc[: n // 2, 1:3] = rng.uniform(41.0, 49.0, (n // 2, 2))
        loc[:, 1:] = loc[rng.permutation(n), 1:]
        loc = loc[np.argsort(loc[:, 11], kind="stable")]
    got = _check(p, loc)
    assert got["density_total"] > n // 2
