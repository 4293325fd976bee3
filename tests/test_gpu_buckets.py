"""The transposed copy placed by buckets of 8 columns (rows of 128 entries and more on
average) at its edges: a last bucket of 1 to 8 columns, buckets beyond the 6,144
entries that fit LDS, few rows and many, empty rows, rows longer than a workgroup.
The copy is compared entry by entry with SciPy's transpose through a back projection of
unit vectors' sums: small whole numbers, whose FP32 sums are exact."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,per_row", [(1, 300, 300), (3, 4096, 2000), (200, 1025, 400),
                                         (33, 1031, 200), (900, 1032, 300), (6500, 160, 150),
                                         (2000, 40007, 260), (700, 9000, 3000)])
@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_copy_by_buckets(gpu_ctx_factory, m, n, per_row, storage):
    from epetreco_amd.api import OP_T, VAL_F16, Matrix
    ctx = gpu_ctx_factory()
    rng = np.random.default_rng(m + n)
    counts = rng.integers(per_row // 2, per_row + 1, m)
    counts[rng.random(m) < 0.1] = 0
    counts[0] = per_row
    while counts.sum() < 128 * m:
        counts[np.argmin(counts)] = per_row
    rp = np.zeros(m + 1, np.int64)
    rp[1:] = np.cumsum(counts)
    col = np.concatenate([np.sort(rng.choice(n, int(k), replace=False)) for k in counts])
    val = np.float32(2.0) ** rng.integers(0, 3, col.size)
    val[rp[:-1][counts > 0]] = 4.0          # the row maximum a power of two: exact in FP16
    M = sp.csr_matrix((val.astype(np.float64), col, rp), shape=(m, n))
    A = Matrix.from_csr(ctx, torch.as_tensor(rp), torch.as_tensor(col.astype(np.int32)),
                        torch.as_tensor(val.astype(np.float32)), n)
    if storage == "f32":
        A.attach_transpose()
        for k in range(3):
            x = rng.integers(-4, 5, m).astype(np.float32)
            got = A.spmv(OP_T, torch.as_tensor(x, device="cuda")).cpu().numpy()
            assert np.array_equal(got, (M.T @ x).astype(np.float32))
    else:
        # an iteration with every voxel at 1 goes through the copy, scales folded in
        B = A.convert(VAL_F16).attach_transpose()
        y = rng.integers(1, 9, m).astype(np.float32)
        X = torch.ones(n, device="cuda")
        ctx.mlem(B, torch.as_tensor(y, device="cuda"), torch.ones(n, device="cuda"), X, 1)
        yh = M @ np.ones(n)
        c = M.T @ np.where(yh > 0, y / np.where(yh > 0, yh, 1), 0)
        c /= c.sum()
        np.testing.assert_allclose(X.cpu().numpy(), c, rtol=2e-5, atol=2e-7 * c.max())
