"""The rows of top_k_rows_kernel: sixteen bytes at a time or not, threads' shares of 13 runs of four and of more, all large elements in the share of few threads, NaN,
infinities, zeros of both signs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rows,k", [(3, 1, 3), (4096, 2, 40), (4097, 1, 1024), (53248, 1, 40), (53252, 2, 500), (53251, 2, 40), (65536, 1, 1000)])
@pytest.mark.parametrize("case", ["any", "few threads", "one run", "nan", "infinite", "zeros"])
def test_candidates_in_order(agpu, dev, n, rows, k, case):
    import torch
    from async_gpu_amd import ops
    x = np.random.default_rng(n + k).standard_normal((rows, n)).astype(np.float32) * 3
    if case == "few threads":
        x[:, 20::4096] += 500.0
        x[:, 23::4096] = 700.0
        x[:, 4092::4096] = 700.0
    elif case == "one run":
        x[:, -7:] = 50.0
        x[:, :3] = 50.0
    elif case == "nan":
        x[:, 1::2] = np.nan
        x[-1, 2:] = np.nan
    elif case == "infinite":
        x[:, ::3] = -np.inf
        x[0, 2:] = -np.inf
        x[:, 1::97] = np.inf
    elif case == "zeros":
        x = np.minimum(x, np.float32(0))
        x[:, ::5] *= 0  # zeros of both signs: one value
    idx, val = ops.top_k(torch.from_numpy(x).to(dev), k, 0.7)
    idx, val = idx.cpu().numpy().view(np.uint32), val.cpu().numpy()
    scaled = x / np.float32(0.7)
    for r in range(rows):
        order = np.lexsort((np.arange(n), -np.where(np.isnan(scaled[r]), -np.inf, scaled[r]), np.isnan(scaled[r])))[:k]
        assert np.array_equal(idx[r], order) and np.array_equal(val[r], scaled[r][order], equal_nan=True), r
