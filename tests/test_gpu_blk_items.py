"""Blocked multi-frame MLEM where partial sums of many splits are added for more
elements (rows times frames) than the card has lanes for a wavefront a SIMD, 65,536,
and for just fewer: by a thread and by 16 wavefronts.  Against FP64, voxel by voxel,
with the bound of test_gpu_blk_splits.py, (k_row + k_column + 16) 2^-24 an iteration."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [2000, 2100])
def test_many_splits(gpu_ctx_factory, oracle, m):
    from epetreco_amd.api import Matrix
    n, F, k = 120000, 32, 24
    rng = np.random.default_rng(m)
    rp = np.arange(m + 1, dtype=np.int64) * k
    step = n // k
    col = (np.arange(k) * step + rng.integers(0, step, (m, k))).astype(np.int32).reshape(-1)
    val = rng.uniform(0.1, 1.0, col.size).astype(np.float32)
    ctx = gpu_ctx_factory()
    A = Matrix.from_csr(ctx, torch.as_tensor(rp), torch.as_tensor(col), torch.as_tensor(val), n)
    A.attach_transpose()
    Y = rng.poisson(5.0, (m, F)).astype(np.float32) + 1.0
    s = A.colsum_f64().float()
    X0 = rng.uniform(0.5, 1.5, (n, F)).astype(np.float32)
    X = torch.as_tensor(X0, device="cuda")
    ctx.mlem(A, torch.as_tensor(Y, device="cuda"), s, X, 1)
    cfg = ctx.batched_config(A, F)
    assert cfg["path"].startswith("blocked") and cfg["forward"]["splits"] > 32, cfg
    want = oracle.mlem_f64_frames(m, n, val, rp, col, Y, s.cpu().numpy(), X0, 1)
    per_column = np.bincount(col, minlength=n).max()
    bar = (k + per_column + 16) * 2.0 ** -24
    assert np.all(np.abs(X.cpu().numpy() - want) <= bar * np.abs(want) + 1e-30)
