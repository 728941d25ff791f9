"""The CRLB rows on both sides of the line between 16 lanes and one lane a row, and at the ends of a work-group,
exactly as the oracle: rows without a bound, values past the narrow range, the smallest and largest widths."""
import numpy as np
import pytest
import torch

import oracle_lib as O
import qcstorm as Q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lt,n", [(0, 1), (0, 3), (0, 5), (0, 64), (0, 90000), (0, 90001), (1, 1), (1, 4), (1, 67), (1, 110000), (1, 110001)])
def test_crlb_exact(gpu, lt, n):
    rng = np.random.default_rng(n + lt)
    loc = rng.normal(0, 1, (n, 12)).astype(np.float32)
    loc[:, 4:6] = rng.choice([0.05, 0.1001, 0.7, 1.3, 4.0, 9.99, 10.0], (n, 2)) * rng.choice([1.0, 0.999, 1.001], (n, 2))
    loc[:, 6] = 10.0 ** rng.uniform(-1, 6, n)
    loc[:, 7] = 10.0 ** rng.uniform(-1, 4, n)
    odd = rng.integers(0, n, max(1, n // 50))
    loc[odd, 6] = rng.choice([1e22, 1e30, np.inf, np.nan, -5.0], len(odd)).astype(np.float32)
    p = Q.default_params(LocType=lt)
    ref = O.crlb(p, loc)
    d = torch.from_numpy(loc).cuda()
    Q.Context(p).crlb_dev(d, n)
    torch.cuda.synchronize()
    got = d.cpu().numpy()
    ref = loc if ref is None else ref
    both_nan = np.isnan(got) & np.isnan(ref)
    assert np.array_equal(np.where(both_nan, 0, got.view(np.uint32)), np.where(both_nan, 0, ref.view(np.uint32)))
