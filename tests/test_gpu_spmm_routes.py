"""Which kernels a multi-frame product runs on.  Forward products of a matrix with
bricks that the row kernel does faster stay there.  It adds in a fixed order, so the
route shows in the bits: equal to the same product in a context that allows the row
kernels only, or not.

Tolerance against FP64: the bar of the other products, rtol 2e-5 of the sum of
magnitudes."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import decoded, env_ctx

pytestmark = pytest.mark.gpu


def scan(gpu_ctx_factory, nx, ny, nz, nrays, rows, storage="f32"):
    """A matrix of `rows` neighbouring channels of a 13 x 13 segment scan, with its
    transposed copy."""
    from epetreco_amd.api import VAL_BF16, VAL_F16
    from epetreco_amd.geometry import MeasurementSetup, VoxelGrid
    d = 0.05 / max(nx, ny, nz)
    s = MeasurementSetup(-0.23, 0.23, 3, 13, 13, 13, 13, 120.0, 0.02, 0.004, 0.004)
    g = VoxelGrid(-d * nx / 2, -d * ny / 2, -d * nz / 2, d, d, d, nx, ny, nz)
    ctx = gpu_ctx_factory(setup=s, grid=g, nrays=nrays, seed=6)
    A = ctx.sm_build((s.nchannels // 3 + np.arange(rows)).astype(np.int32))
    if storage != "f32":
        A = A.convert({"bf16": VAL_BF16, "f16": VAL_F16}[storage])
    return ctx, A.attach_transpose()


def product(ctx, A, op, X):
    from epetreco_amd._lib import check, lib
    from epetreco_amd.api import OP_N
    Y = torch.empty((A.m if op == OP_N else A.n, X.shape[1]), device="cuda")
    check(lib().epet_matrix_spmm(ctx.handle, A.handle, op, X.shape[1], 1.0,
                                 ctypes.c_void_p(X.data_ptr()), 0.0, ctypes.c_void_p(Y.data_ptr())))
    return Y


def with_bricks(ctx, A):
    """Builds A's bricks, as MLEM of several frames does before it begins."""
    x = torch.full((A.n, 2), 1.0 / A.n, device="cuda")
    ctx.mlem(A, torch.ones(A.m, 2, device="cuda"), A.colsum_f64().float(), x, 1)
    assert ctx.batched_config(A, 2)["path"].startswith("bricks")


@pytest.mark.parametrize("F", [2, 3, 8, 16])
def test_small_products_stay_with_the_rows(gpu_ctx_factory, monkeypatch, F):
    from epetreco_amd.api import OP_N
    ctx, A = scan(gpu_ctx_factory, 16, 16, 16, 64, 9001)
    rows_only = env_ctx(monkeypatch, EPET_BATCHED="gather")
    with_bricks(ctx, A)
    X = torch.rand(A.n, F, device="cuda")
    for _ in range(3):
        assert torch.equal(product(ctx, A, OP_N, X), product(rows_only, A, OP_N, X))


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("F", [4, 11, 32, 33, 64])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-0.5, 1.5)])
def test_products_on_bricks(gpu_ctx_factory, storage, F, alpha, beta):
    """Products large enough for bricks, on a grid whose voxel blocks reach past its
    edges and rows that fill no last group."""
    import scipy.sparse as sp
    from epetreco_amd.api import OP_N, OP_T
    ctx, A = scan(gpu_ctx_factory, 51, 49, 53, 64, 6001, storage)
    with_bricks(ctx, A)
    rp, col, val = decoded(A)
    M = sp.csr_matrix((val.astype(np.float64), col, rp), shape=(A.m, A.n))
    rng = np.random.default_rng(F)
    for op, K, nin, nout in ((OP_N, M, A.n, A.m), (OP_T, M.T, A.m, A.n)):
        X = rng.normal(size=(nin, F)).astype(np.float32)
        Y0 = rng.normal(size=(nout, F)).astype(np.float32)
        Y = torch.as_tensor(Y0, device="cuda")
        A.spmm(op, torch.as_tensor(X, device="cuda"), Y, alpha=alpha, beta=beta)
        want = alpha * (K @ X.astype(np.float64)) + beta * Y0
        bar = 2e-5 * (abs(alpha) * (abs(K) @ np.abs(X)) + abs(beta * Y0)) + 1e-30
        assert np.all(np.abs(Y.cpu().numpy() - want) <= bar)


def test_streams_and_a_graph(gpu_ctx_factory, monkeypatch):
    """Calls on two streams share nothing; a captured call runs on the rows, and every
    replay gives the eager result."""
    from epetreco_amd._lib import check, lib
    from epetreco_amd.api import OP_N, Context
    ctx, A = scan(gpu_ctx_factory, 52, 52, 52, 64, 6001)
    rows_only = env_ctx(monkeypatch, EPET_BATCHED="gather")
    with_bricks(ctx, A)
    X = [torch.rand(A.n, 6, device="cuda") for _ in range(2)]
    want = [product(ctx, A, OP_N, x) for x in X]
    rows = product(rows_only, A, OP_N, X[0])
    torch.cuda.synchronize()
    assert not torch.equal(want[0], rows)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    ctxs = [Context(0, st) for st in streams]
    outs = [[torch.zeros(A.m, 6, device="cuda") for _ in range(20)] for _ in range(2)]
    torch.cuda.synchronize()
    for k in range(20):
        for i in range(2):
            check(lib().epet_matrix_spmm(ctxs[i].handle, A.handle, OP_N, 6, 1.0,
                                         ctypes.c_void_p(X[i].data_ptr()), 0.0,
                                         ctypes.c_void_p(outs[i][k].data_ptr())))
    torch.cuda.synchronize()
    for i in range(2):
        for o in outs[i]:
            assert torch.equal(o, want[i])
    g = torch.cuda.CUDAGraph()
    y = torch.zeros(A.m, 6, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=streams[0]):
        check(lib().epet_matrix_spmm(ctxs[0].handle, A.handle, OP_N, 6, 1.0,
                                     ctypes.c_void_p(X[0].data_ptr()), 0.0,
                                     ctypes.c_void_p(y.data_ptr())))
    for _ in range(3):
        y.fill_(7.0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, rows)


def test_values_written_in_place(gpu_ctx_factory):
    """Products after values were written through the matrix's own arrays are products of
    those values, bricks built or not."""
    from epetreco_amd._lib import check, lib
    from epetreco_amd.api import OP_N, OP_T
    ctx, A = scan(gpu_ctx_factory, 52, 52, 52, 64, 6001)
    with_bricks(ctx, A)
    X = {OP_N: torch.rand(A.n, 8, device="cuda"), OP_T: torch.rand(A.m, 8, device="cuda")}
    before = {op: product(ctx, A, op, x) for op, x in X.items()}
    val = A.arrays()[2]
    for factor in (2.0, 0.5):       # exact in FP32
        v = A.to_torch()[2] * factor
        check(lib().epet_memcpy_d2d(ctx.handle, ctypes.c_void_p(val), ctypes.c_void_p(v.data_ptr()),
                                    4 * A.nnz))
        for op, x in X.items():
            got, want = product(ctx, A, op, x), before[op] * (2.0 if factor == 2.0 else 1.0)
            assert (got - want).abs().max() <= 2e-5 * want.abs().max()
