"""Transposed CSR product (k_spmv_t) at the edges of its steps and parts, with the
zero values that a chunk of all candidates holds, against FP64.

Tolerance: a column is a sum of k float products in any order, each rounded once:
(k + 2) 2^-24 of the sum of their sizes.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(gpu_ctx_factory):
    return gpu_ctx_factory()


def _dev(a, dtype):
    return torch.as_tensor(np.asarray(a, dtype), device="cuda")


@pytest.mark.parametrize("lengths,n", [
    ([1], 1), ([0, 3, 0, 4, 5], 7), ([0, 0], 5),
    ([63, 64, 65, 255, 256, 257, 511, 512, 513], 600),
    ([2047, 2048, 2049, 0, 4095, 4097], 5000),       # several parts a row
    ([100000], 100000), ([7] * 5000, 300),
])
@pytest.mark.parametrize("zeros", [0.0, 0.95, 1.0])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-0.5, 1.5)])
def test_transposed(ctx, lengths, n, zeros, alpha, beta):
    from epetreco_amd.api import OP_T
    rng = np.random.default_rng(n)
    m = len(lengths)
    rp = np.concatenate([[0], np.cumsum(lengths)])
    col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lengths]).astype(np.int64)
    val = np.where(rng.random(col.size) < zeros, 0, rng.normal(size=col.size)).astype(np.float32)
    x = rng.normal(size=m).astype(np.float32)
    x[::7] = 0.0
    y0 = rng.normal(size=n).astype(np.float32)
    row = np.repeat(np.arange(m), lengths)
    p = val.astype(np.float64) * x[row]
    want = beta * y0.astype(np.float64)
    size, k = np.abs(want), np.bincount(col, minlength=n) + 1
    np.add.at(want, col, alpha * p)
    np.add.at(size, col, np.abs(alpha * p))
    y = ctx.csrmv(OP_T, m, n, alpha, _dev(val, np.float32), _dev(rp, np.int32),
                  _dev(col, np.int32), _dev(x, np.float32), beta, _dev(y0, np.float32))
    assert np.all(np.abs(y.cpu().numpy() - want) <= (k + 2) * 2.0 ** -24 * size + 1e-37)


def test_transposed_not_finite(ctx):
    """0 times an infinity is added as well."""
    from epetreco_amd.api import OP_T
    val = [0.0, 1.0, 0.0, np.inf, 0.0, np.nan]
    y = ctx.csrmv(OP_T, 2, 6, 1.0, _dev(val, np.float32), _dev([0, 2, 6], np.int32),
                  _dev(np.arange(6), np.int32), _dev([np.inf, 2.0], np.float32), 1.0,
                  _dev(np.ones(6), np.float32)).cpu().numpy()
    np.testing.assert_array_equal(y, np.float32([np.nan, np.inf, 1, np.inf, 1, np.nan]))
