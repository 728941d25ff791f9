"""Weight gradients of the warm-start network split over the batch's rows: batches of one ROI, of odd
sizes around the slices of 64 rows, and past one pass's 65,536 ROIs."""
import numpy as np
import pytest

import nn_ref as R
import qcstorm as Q
from qcstorm import warmstart as WS

pytestmark = pytest.mark.gpu


def _batch(n, seed):
    import torch
    rois, _ = WS.sim_dev(n, seed)
    lab = torch.zeros((n, 16), dtype=torch.float32, device="cuda")
    Q.Context(WS.params()).label_dev(rois, n, lab)
    torch.cuda.synchronize()
    return rois, lab


@pytest.mark.parametrize("n", [1, 7, 65, 301])
def test_gradient_of_odd_batches(gpu, n):
    net = Q.Net(seed=3)
    rois, lab = _batch(n, 40 + n)
    g, loss = net.grad_dev(WS.params(), rois, lab, n)
    w = net.params().astype(np.float64)
    out, cache = R.forward(w, rois.cpu().numpy().view(np.uint16))
    L, d = R.loss_grad(out, lab.cpu().numpy().astype(np.float64), cache["scale"], cache["bh"])
    ref = R.unpack(R.backward(cache, d))
    got = R.unpack(g.astype(np.float64))
    assert abs(loss - L) <= 2e-2 * max(abs(L), 1e-3)
    for k in ref:
        # bf16 roundings (2^-9 per operand) of up to four layers on the way back, as for the large batch
        assert np.linalg.norm(got[k] - ref[k]) <= 3e-2 * np.linalg.norm(ref[k]) + 1e-7, (k, n)


def test_gradient_over_two_passes(gpu):
    """The mean gradient of 65,536 + 17 ROIs is the weighted mean of its two passes'."""
    net = Q.Net(seed=4)
    n1, n2 = 65536, 17
    rois, lab = _batch(n1 + n2, 51)
    p = WS.params()
    g, loss = net.grad_dev(p, rois, lab, n1 + n2)
    g1, l1 = net.grad_dev(p, rois[:n1], lab[:n1], n1)
    g2, l2 = net.grad_dev(p, rois[n1:].contiguous(), lab[n1:].contiguous(), n2)
    ref = (n1 * g1.astype(np.float64) + n2 * g2) / (n1 + n2)
    # fp32 sums of the same terms; the per-ROI scale 1/n is rounded before the bf16 products (2^-9)
    assert np.linalg.norm(g - ref) <= 4e-3 * np.linalg.norm(ref)
    assert abs(loss - (n1 * l1 + n2 * l2) / (n1 + n2)) <= 1e-4 * abs(loss)
