"""The image update of MLEM at the edges of its split: images just within and just
beyond one workgroup's, frame counts that do not divide a workgroup, odd and even
iteration counts, stopped frames, with and without the transposed copy, against
the FP64 oracle (rel-L2 <= 1e-5, the bar of the other MLEM tests)."""
import numpy as np
import pytest
import torch

from helpers import decoded, rel_l2

pytestmark = pytest.mark.gpu


def _matrix(ctx, m, n, per_row, rng):
    from epetreco_amd.api import Matrix
    col = np.sort(np.argsort(rng.random((m, n)), axis=1)[:, :per_row], axis=1).astype(np.int32)
    val = rng.uniform(0.1, 1.0, (m, per_row)).astype(np.float32)
    rp = np.arange(m + 1, dtype=np.int64) * per_row
    return Matrix.from_csr(ctx, torch.as_tensor(rp), torch.as_tensor(col.ravel()),
                           torch.as_tensor(val.ravel()), n)


@pytest.mark.parametrize("n,F", [(1, 1), (63, 1), (16384, 1), (16385, 1), (20001, 1),
                                 (5461, 3), (5462, 3), (2340, 7), (2341, 7), (256, 64), (257, 64)])
@pytest.mark.parametrize("transposed", [True, False])
@pytest.mark.parametrize("niter", [1, 4])
def test_update(gpu_ctx_factory, oracle, n, F, transposed, niter):
    rng = np.random.default_rng(n + F)
    ctx = gpu_ctx_factory()
    A = _matrix(ctx, 200, n, min(n, 12), rng)
    if transposed:
        A.attach_transpose()
    Y = rng.poisson(6.0, (A.m, F)).astype(np.float32)
    X0 = rng.uniform(0.5, 1.5, (n, F)).astype(np.float32) / n
    s = A.colsum_f64().float()              # zero where a voxel has no entry
    shape = (lambda a: a[:, 0].copy()) if F == 1 else (lambda a: a)
    X = torch.as_tensor(shape(X0), device="cuda")
    ctx.mlem(A, torch.as_tensor(shape(Y), device="cuda"), s, X, niter)
    rp, col, val = decoded(A)
    want = oracle.mlem_f64_frames(A.m, A.n, val, rp, col, Y, s.cpu().numpy(),
                                  X0.astype(np.float64), niter)
    got = X.cpu().numpy().reshape(n, F)
    for f in range(F):
        assert rel_l2(got[:, f], want[:, f]) < 1e-5


@pytest.mark.parametrize("n", [300, 9000])
def test_stopped_frames_stay(gpu_ctx_factory, n):
    """A frame that meets the tolerance keeps its image while the others go on."""
    rng = np.random.default_rng(n)
    ctx = gpu_ctx_factory()
    A = _matrix(ctx, 200, n, 12, rng).attach_transpose()
    rp, col, val = decoded(A)
    Y = rng.poisson(6.0, (A.m, 3)).astype(np.float32)
    # the start's own projection: a fixed point where a voxel has entries (the others
    # go to zero in the first iteration), so it stops early
    Y[:, 1] = np.add.reduceat(val.astype(np.float64), rp[:-1]) / n
    s = A.colsum_f64().float()
    X = torch.full((n, 3), 1.0 / n, device="cuda")
    ll, iters = ctx.mlem(A, torch.as_tensor(Y, device="cuda"), s, X, 12, tol=1e-9)
    ref = torch.full((n, 3), 1.0 / n, device="cuda")
    ctx.mlem(A, torch.as_tensor(Y, device="cuda"), s, ref, 12)
    assert iters[0] == 12 and iters[2] == 12 and 2 <= iters[1] < 12
    short = torch.full((n, 3), 1.0 / n, device="cuda")
    ctx.mlem(A, torch.as_tensor(Y, device="cuda"), s, short, int(iters[1]))
    assert rel_l2(X[:, 1].cpu().numpy(), short[:, 1].cpu().numpy()) < 1e-6
    for f in (0, 2):
        assert rel_l2(X[:, f].cpu().numpy(), ref[:, f].cpu().numpy()) < 1e-6
