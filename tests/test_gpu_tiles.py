"""Back projection without a transposed copy, by tiles of 8,192 columns in LDS: sizes
about the tile's edge, row counts about the blocks', rows of few entries in a tile (16
lanes each) and of many (32 lanes), one entry a row and none.

Tolerance: an entry is rounded twice (its row's factor, its product), sums of a block
are FP64, and at most 2,048 blocks' sums, rounded once each, are added in FP32 (16
wavefronts, four sums each): 3 + 2048 / 64 + 20 roundings of 2^-24 of the sum of
magnitudes, 4e-6."""
import numpy as np
import pytest
import torch

from helpers import decoded, env_ctx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("n", [5, 8191, 8192, 8193, 40000])
@pytest.mark.parametrize("m,per_row", [(1, 4), (63, 5), (129, 1), (700, 30), (700, 600), (3000, 40)])
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_tiles(monkeypatch, storage, n, m, per_row, beta):
    import scipy.sparse as sp
    from epetreco_amd.api import OP_T, VAL_F16, Matrix
    ctx = env_ctx(monkeypatch, EPET_BP="tiled")
    rng = np.random.default_rng(n + m)
    k = min(per_row, n)
    counts = rng.integers(max(1, k // 2), k + 1, m)
    counts[m // 2] = 0
    col = np.concatenate([np.sort(rng.choice(n, c, replace=False)) for c in counts] + [[]]).astype(np.int32)
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    val = rng.uniform(0.1, 1.0, col.size).astype(np.float32)
    A = Matrix.from_csr(ctx, torch.as_tensor(rp), torch.as_tensor(col), torch.as_tensor(val), n)
    if storage == "f16":
        A = A.convert(VAL_F16)
    rp, col, val = decoded(A)
    K = sp.csr_matrix((val.astype(np.float64), col, rp), shape=(m, n)).T
    x = rng.normal(size=m).astype(np.float32)
    x[::7] = 0.0
    y0 = rng.normal(size=n).astype(np.float32)
    y = torch.as_tensor(y0, device="cuda")
    A.spmv(OP_T, torch.as_tensor(x, device="cuda"), y, alpha=1.5, beta=beta)
    want = 1.5 * (K @ x.astype(np.float64)) + beta * y0
    bar = 4e-6 * (1.5 * (abs(K) @ np.abs(x)) + abs(beta * y0)) + 1e-30
    assert np.all(np.abs(y.cpu().numpy() - want) <= bar)
