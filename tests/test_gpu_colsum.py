"""Column sums in FP64 (epet_matrix_colsum_f64): sums in LDS and atomics in memory,
at the edges of the column tiles and of the rule between the two, against NumPy.
Sums of at most 2,000 positive doubles in any order: rtol 2000 * 2^-53 < 3e-13."""
import numpy as np
import pytest
import torch

from helpers import decoded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("m,n,per_row", [
    (1, 1, 1), (2000, 7, 5),           # a few columns
    (900, 16384, 150), (900, 16385, 150), (300, 40000, 1200),   # one, two, three tiles
    (60, 16385, 150),                  # too few entries per column: atomics in memory
    (17, 200, 90),                     # fewer rows than a workgroup takes
])
def test_colsum(gpu_ctx_factory, storage, m, n, per_row):
    from epetreco_amd.api import VAL_BF16, VAL_F16, Matrix
    rng = np.random.default_rng(m + n)
    k = rng.integers(0, per_row + 1, m) if per_row > 1 else np.ones(m, int)
    k[-1] = per_row
    rp = np.zeros(m + 1, np.int64)
    rp[1:] = np.cumsum(k)
    col = np.concatenate([np.sort(rng.choice(n, int(c), replace=False)) for c in k]).astype(np.int32)
    val = rng.uniform(0.1, 1.0, col.size).astype(np.float32)
    ctx = gpu_ctx_factory()
    A = Matrix.from_csr(ctx, torch.as_tensor(rp), torch.as_tensor(col), torch.as_tensor(val), n)
    if storage != "f32":
        A = A.convert({"bf16": VAL_BF16, "f16": VAL_F16}[storage])
    _, dcol, dval = decoded(A)
    want = np.zeros(n)
    np.add.at(want, dcol, dval.astype(np.float64))
    np.testing.assert_allclose(A.colsum_f64().cpu().numpy(), want, rtol=3e-13)


def test_unordered_columns(gpu_ctx_factory):
    """Columns in any order and repeated: the atomics in memory take them."""
    from epetreco_amd.api import Matrix
    rng = np.random.default_rng(1)
    m, n, k = 300, 50, 40
    rp = np.arange(m + 1, dtype=np.int64) * k
    col = rng.integers(0, n, m * k).astype(np.int32)
    val = rng.uniform(0.1, 1.0, m * k).astype(np.float32)
    A = Matrix.from_csr(gpu_ctx_factory(), torch.as_tensor(rp), torch.as_tensor(col),
                        torch.as_tensor(val), n)
    want = np.zeros(n)
    np.add.at(want, col, val.astype(np.float64))
    np.testing.assert_allclose(A.colsum_f64().cpu().numpy(), want, rtol=3e-13)
