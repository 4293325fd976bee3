"""Blocked multi-frame MLEM on few rows over many columns, where the forward product
has from one to hundreds of splits, against FP64.

Tolerance: every sum has at most k positive terms, each rounded once in the product
and at most k times in the sum, in any order: an iteration's image is off by at most
(k_row + k_column + 16) 2^-24 of itself, k_row = 200 and k_column = m, and two
iterations by twice that.  The image is compared voxel by voxel.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F", [2, 14, 33])
@pytest.mark.parametrize("m,n", [(1, 500), (3, 70001), (127, 30000), (130, 200000), (700, 40000)])
def test_few_rows(gpu_ctx_factory, oracle, m, n, F):
    from epetreco_amd.api import Matrix
    rng = np.random.default_rng(m + F)
    k = 200
    rp = np.arange(m + 1, dtype=np.int64) * k
    col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for _ in range(m)]).astype(np.int32)
    val = rng.uniform(0.1, 1.0, col.size).astype(np.float32)
    ctx = gpu_ctx_factory()
    A = Matrix.from_csr(ctx, torch.as_tensor(rp), torch.as_tensor(col), torch.as_tensor(val), n)
    A.attach_transpose()
    Y = rng.poisson(5.0, (m, F)).astype(np.float32) + 1.0
    s = A.colsum_f64().float()
    X0 = rng.uniform(0.5, 1.5, (n, F)).astype(np.float32)
    X = torch.as_tensor(X0, device="cuda")
    ll, _ = ctx.mlem(A, torch.as_tensor(Y, device="cuda"), s, X, 2)
    assert ctx.batched_config(A, F)["path"].startswith("blocked")
    want = oracle.mlem_f64_frames(m, n, val, rp, col, Y, s.cpu().numpy(), X0, 2)
    bar = 2 * (k + m + 16) * 2.0 ** -24
    assert np.all(np.abs(X.cpu().numpy() - want) <= bar * np.abs(want) + 1e-30)
    xr = X0.astype(np.float64)          # log-likelihood of the first image
    yh = np.add.reduceat(val[:, None] * xr[col], rp[:-1], axis=0)
    np.testing.assert_allclose(np.asarray(ll)[0], (Y * np.log(yh) - yh).sum(0),
                               atol=(k + 16) * 2.0 ** -24 * (Y + yh).sum())
