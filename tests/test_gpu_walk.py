"""The extraction's row walk at the edges of its strips, steps and value range, exactly as the oracle: widths around
multiples of 56 columns, heights around its steps and walk lengths, backgrounds from 0 to the top of uint16 (the
background term is a float sum that has to truncate as the integer one), few and many pixels at the threshold."""
import numpy as np
import pytest

import oracle_lib as O
import qcstorm as Q

pytestmark = pytest.mark.gpu


def _frames(W, H, nf, level, amp, noise, seed):
    rng = np.random.default_rng(seed)
    img = level + rng.normal(0, noise, (nf, H, W)) if noise >= 0 else rng.integers(0, 65536, (nf, H, W)).astype(float)
    yy, xx = np.mgrid[-3:4, -3:4]
    spot = np.exp(-(xx**2 + yy**2) / (2 * 1.2**2))
    for f in range(nf):
        for _ in range(max(2, W * H // 300)):
            x, y = rng.integers(0, W), rng.integers(0, H)
            x0, x1, y0, y1 = max(x - 3, 0), min(x + 4, W), max(y - 3, 0), min(y + 4, H)
            img[f, y0:y1, x0:x1] += amp * rng.uniform(0.1, 1.0) * spot[y0 - y + 3:y1 - y + 3, x0 - x + 3:x1 - x + 3]
    return np.clip(np.rint(img), 0, 65535).astype(np.uint16)


SIZES = [(13, 12, 1, 1), (55, 17, 2, 1), (56, 16, 3, 2), (57, 33, 2, 2), (64, 64, 2, 1), (111, 15, 5, 5), (112, 130, 1, 1), (113, 40, 4, 3),
         (169, 300, 2, 2), (224, 129, 3, 1)]
LEVELS = [(0.0, 900.0, 0.0), (100.0, 1500.0, 8.0), (30000.0, 9000.0, 60.0), (64000.0, 3000.0, 20.0), (2000.0, 65000.0, 30.0), (0.0, 0.0, -1.0)]


@pytest.mark.parametrize("loc,multi", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("W,H,nf,B", SIZES)
def test_walk_exact(gpu, W, H, nf, B, loc, multi):
    p = Q.default_params(QE=1.0, ImageWidth=W, ImageHigh=H, BatchedImageNum=B, LocType=loc, MultiEmitterFitEn=multi, ROISize=7)
    ctx = Q.Context(p)
    found = 0
    for k, (level, amp, noise) in enumerate(LEVELS):
        fr = _frames(W, H, nf, level, amp, noise, 100 * W + k)
        rois, wle, n, _ = O.extract(p, fr, start_frame=3, cap=20000)
        g_rois, g_wle, g_n = ctx.extract(fr, start_frame=3, cap=20000)
        assert g_n == n, (level, g_n, n)
        assert np.array_equal(g_rois, rois)
        assert np.array_equal(g_wle.view(np.uint32), wle.view(np.uint32))
        found += n
    assert found > 0 or W < 20


@pytest.mark.parametrize("R,multi,B", [(5, 0, 1), (7, 1, 2), (11, 1, 1), (17, 1, 2), (17, 0, 1)])
def test_list_exact(gpu, R, multi, B):
    """Windows across strip borders for the marks; nearest neighbours from next door to past the entries that a
    work-group keeps (a far spot in a wide frame that is crowded elsewhere), alone in a frame, and none."""
    W, H, nf = 4000, 60, 4
    rng = np.random.default_rng(R + multi)
    img = 200.0 + rng.normal(0, 6, (nf, H, W))
    yy, xx = np.mgrid[-4:5, -4:5]
    spot = np.exp(-(xx**2 + yy**2) / (2 * 1.3**2))

    def put(f, x, y, a):
        img[f, y - 4:y + 5, x - 4:x + 5] += a * spot

    for x in range(30, 2600, 11):
        for y in range(16, 46, 11):
            put(0, x + int(rng.integers(-1, 2)), y + int(rng.integers(-1, 2)), rng.uniform(2500, 5000))
    put(0, 3900, 30, 4000.0)
    put(2, 2000, 30, 4000.0)
    for x in range(50, 3900, 28):
        put(3, x, int(rng.integers(18, 42)), 3500.0)
        put(3, x + int(rng.integers(4, 8)), int(rng.integers(18, 42)), 2500.0)
    fr = np.clip(np.rint(img), 0, 65535).astype(np.uint16)
    p = Q.default_params(QE=1.0, ImageWidth=W, ImageHigh=H, BatchedImageNum=B, MultiEmitterFitEn=multi, ROISize=R)
    rois, wle, n, _ = O.extract(p, fr, start_frame=70000, cap=5000)
    ctx = Q.Context(p)
    for cap in (5000, 300):
        g_rois, g_wle, g_n = ctx.extract(fr, start_frame=70000, cap=cap)
        if cap == 5000:
            assert g_n == n and n > 700
            assert np.array_equal(g_rois, rois)
            assert np.array_equal(g_wle.view(np.uint32), wle.view(np.uint32))
        else:
            r2, w2, n2, _ = O.extract(p, fr, start_frame=70000, cap=cap)
            assert g_n == n2 and np.array_equal(g_rois, r2) and np.array_equal(g_wle.view(np.uint32), w2.view(np.uint32))
