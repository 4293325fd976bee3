"""The transposed copy at its edges: column tiles (36,864 columns per tile of
counters), row blocks (16 rows and more), batches of 1,024 rows, rows with more
than 1,024 entries in a tile, empty rows and columns.  Back projections of small
whole numbers, whose FP32 sums are exact: equal, no tolerance."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(gpu_ctx_factory):
    return gpu_ctx_factory()


def _matrix(m, n, per_row, rng):
    rows, cols = [], []
    for r in range(m):
        k = 0 if r % 7 == 3 else min(n, rng.integers(1, 2 * per_row + 1))
        c = np.sort(rng.choice(n, k, replace=False))
        rows.append(np.full(k, r))
        cols.append(c)
    r, c = np.concatenate(rows), np.concatenate(cols)
    v = rng.integers(1, 8, len(r)).astype(np.float32)
    return sp.csr_matrix((v, (r, c)), shape=(m, n))


@pytest.mark.parametrize("m,n,per_row", [(1, 1, 1), (15, 5, 2), (17, 36863, 40), (300, 36864, 30),
                                         (300, 36865, 30), (2500, 80001, 20), (40, 80001, 900),
                                         (5000, 700, 100), (64, 40000, 4000)])
@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_back_projection_through_the_copy(ctx, m, n, per_row, storage):
    from epetreco_amd.api import OP_T, VAL_F16, Matrix
    rng = np.random.default_rng(m + n)
    M = _matrix(m, n, per_row, rng)
    if storage == "f16":     # a power of two as the row maximum keeps the stored values exact
        M.data = np.float32(2.0) ** rng.integers(0, 3, M.nnz)
    A = Matrix.from_csr(ctx, torch.as_tensor(M.indptr.astype(np.int64)), torch.as_tensor(M.indices),
                        torch.as_tensor(M.data), n)
    x = rng.integers(-4, 5, m).astype(np.float32)
    want = M.T.astype(np.float64) @ x
    if storage == "f32":
        A.attach_transpose()
        got = A.spmv(OP_T, torch.as_tensor(x, device="cuda")).cpu().numpy()
        assert np.array_equal(got, want.astype(np.float32))
    else:
        # one MLEM iteration goes through the copy with the row scale folded in
        B = A.convert(VAL_F16).attach_transpose()
        y = torch.as_tensor(np.abs(x) + 1, device="cuda")
        s = torch.ones(n, device="cuda")
        X = torch.full((n,), 1.0, device="cuda")
        ctx.mlem(B, y, s, X, 1)
        yh = M.astype(np.float64) @ np.ones(n)
        e = np.where(yh > 0, (np.abs(x) + 1) / np.where(yh > 0, yh, 1), 0)
        c = M.T.astype(np.float64) @ e
        c /= c.sum()
        np.testing.assert_allclose(X.cpu().numpy(), c, rtol=2e-5, atol=2e-7 * c.max())
