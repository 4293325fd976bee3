"""LDS-tiled single-frame products (k_rows_lds) at the edges of their split: rows
of 0 to many blocks of 64 chunks, empty tiles, one row, every storage, one and
several tiles, against FP64 on the stored values.

Tolerance: |y - y64| <= 2e-5 * (|alpha| |A| |x| + |beta y|) per row, the bar of
the other products.
"""
import numpy as np
import pytest
import torch

from helpers import decoded

pytestmark = pytest.mark.gpu


def _csr(rng, m, n, lengths):
    rp = np.zeros(m + 1, np.int64)
    rp[1:] = np.cumsum(np.minimum(lengths, n))
    col = np.concatenate([np.sort(rng.choice(n, size=int(k), replace=False))
                          for k in np.diff(rp)] or [np.zeros(0)]).astype(np.int32)
    val = rng.uniform(0.1, 1.0, col.size).astype(np.float32)
    return rp, col, val


def _lengths(kind, m, rng):
    if kind == "uneven":        # empty rows, single entries, chunk edges, long rows
        return rng.choice([0, 1, 7, 8, 9, 64, 511, 512, 513, 3000], size=m)
    if kind == "one_long":      # all entries in one row, many empty ones around it
        k = np.zeros(m, np.int64)
        k[m // 2] = 64 * m + 5
        return k                # (the LDS products need 64 entries per row)
    return np.full(m, 200)


SHAPES = [
    (1, 4097, "even"),             # one row, less than one window
    (333, 100, "even"),            # one tile, shorter than 128 KB
    (700, 32768, "uneven"),        # exactly one tile
    (700, 32769, "uneven"),        # a second tile of one column
    (500, 100001, "uneven"),       # four tiles
    (1000, 70000, "one_long"),     # windows of empty rows
    (3000, 40000, "even"),
]


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("m,n,kind", SHAPES)
def test_product(gpu_ctx_factory, storage, m, n, kind):
    import scipy.sparse as sp
    from epetreco_amd.api import OP_N, VAL_BF16, VAL_F16, Matrix
    rng = np.random.default_rng(m + n)
    lengths = _lengths(kind, m, rng)
    rp, col, val = _csr(rng, m, n, lengths)
    assert val.size >= 64 * m
    ctx = gpu_ctx_factory()
    A = Matrix.from_csr(ctx, torch.as_tensor(rp), torch.as_tensor(col), torch.as_tensor(val), n)
    if storage != "f32":
        A = A.convert({"bf16": VAL_BF16, "f16": VAL_F16}[storage])
    prp, pcol, pval = decoded(A)
    M = sp.csr_matrix((pval.astype(np.float64), pcol, prp), shape=(m, n))
    X = torch.as_tensor(rng.normal(size=n + 1).astype(np.float32), device="cuda")
    Y0 = rng.normal(size=m).astype(np.float32)
    # x aligned to 16 bytes and not
    for x, alpha, beta in ((X[:n], 1.0, 0.0), (X[1:], -0.5, 1.5)):
        y = torch.as_tensor(Y0, device="cuda")
        A.spmv(OP_N, x, y, alpha=alpha, beta=beta)
        xh = x.cpu().numpy().astype(np.float64)
        want = alpha * (M @ xh) + beta * Y0
        bar = 2e-5 * (abs(alpha) * (abs(M) @ np.abs(xh)) + abs(beta * Y0)) + 1e-30
        assert np.all(np.abs(y.cpu().numpy() - want) <= bar)


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("m,n,kind", SHAPES)
@pytest.mark.parametrize("projected", [True, False])
def test_back_projection(gpu_ctx_factory, storage, m, n, kind, projected):
    """Without a transposed copy (k_bp_tiled), before and after a forward product;
    weights of 0 and an infinity."""
    import scipy.sparse as sp
    from epetreco_amd.api import OP_N, OP_T, VAL_BF16, VAL_F16, Matrix
    rng = np.random.default_rng(m + n)
    rp, col, val = _csr(rng, m, n, _lengths(kind, m, rng))
    ctx = gpu_ctx_factory()
    A = Matrix.from_csr(ctx, torch.as_tensor(rp), torch.as_tensor(col), torch.as_tensor(val), n)
    if storage != "f32":
        A = A.convert({"bf16": VAL_BF16, "f16": VAL_F16}[storage])
    prp, pcol, pval = decoded(A)
    M = sp.csr_matrix((pval.astype(np.float64), pcol, prp), shape=(m, n)).T.tocsr()
    if projected:
        A.spmv(OP_N, torch.ones(n, device="cuda"))
    x = rng.normal(size=m).astype(np.float32)
    x[::5] = 0.0
    Y0 = rng.normal(size=n).astype(np.float32)
    for alpha, beta in ((1.0, 0.0), (-0.5, 1.5)):
        y = torch.as_tensor(Y0, device="cuda")
        A.spmv(OP_T, torch.as_tensor(x, device="cuda"), y, alpha=alpha, beta=beta)
        want = alpha * (M @ x.astype(np.float64)) + beta * Y0
        bar = 2e-5 * (abs(alpha) * (abs(M) @ np.abs(x)) + abs(beta * Y0)) + 1e-30
        assert np.all(np.abs(y.cpu().numpy() - want) <= bar)
    x[m // 2] = np.inf                # only the voxels of that row become infinite
    y = A.spmv(OP_T, torch.as_tensor(x, device="cuda")).cpu().numpy()
    row = pcol[prp[m // 2]:prp[m // 2 + 1]]
    hit = np.zeros(n, bool)
    hit[row[pval[prp[m // 2]:prp[m // 2 + 1]] > 0]] = True
    assert np.all(np.isinf(y[hit])) and np.all(np.isfinite(y[~hit]))
