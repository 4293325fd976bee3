"""Multi-frame MLEM on bricks (matrix-core steps of 64 rows by 16 columns) against
the blocked products and the FP64 oracle, on generated matrices: padded frame
counts 8, 16, 32 and 64 with full and ragged frames, all storages, grids whose
2x2x2 bricks reach past the edge, row counts that are no multiple of a group,
and steps more than half full.

Tolerances: both paths add FP32 products of at most a few thousand terms per
row in another order, so images agree to a few 1e-7 in relative 2-norm per
iteration; 3 iterations, bar 5e-6 (and 1e-5 against FP64).  Log-likelihoods are
FP64 sums of FP32 projections: 1e-6 relative.  A frame with an infinity or NaN
must come out like the blocked products' (same places, same finite values), and
the other frames must not notice."""
import numpy as np
import pytest
import torch

from helpers import decoded, env_ctx

pytestmark = pytest.mark.gpu


def _problem(gpu_ctx_factory, nx, ny, nz, nrays, na, every, storage, d=0.0033):
    from epetreco_amd.api import VAL_BF16, VAL_F16
    from epetreco_amd.geometry import MeasurementSetup, VoxelGrid
    s = MeasurementSetup(-0.23, 0.23, na, 5, 5, 5, 5, 180.0 / na, 0.02, 0.004, 0.004)
    g = VoxelGrid(-d * nx / 2, -d * ny / 2, -d * nz / 2, d, d, d, nx, ny, nz)
    ctx = gpu_ctx_factory(setup=s, grid=g, nrays=nrays, seed=2)
    A = ctx.sm_build(np.arange(0, s.nchannels, every, dtype=np.int32))
    if storage != "f32":
        A = A.convert({"bf16": VAL_BF16, "f16": VAL_F16}[storage])
    return ctx, A.attach_transpose()


def _run(ctx, A, Y, s, X0, niter, graph):
    X = X0.clone()
    ll, _ = ctx.mlem(A, Y, s, X, niter, use_graph=graph)
    return X.cpu().numpy(), ll


def _data(A, F, seed=0):
    rng = np.random.default_rng(seed)
    Y = torch.as_tensor(rng.poisson(4.0, (A.m, F)).astype(np.float32), device="cuda")
    X0 = torch.as_tensor(rng.uniform(0.5, 1.5, (A.n, F)).astype(np.float32) / A.n, device="cuda")
    return Y, A.colsum_f64().float(), X0


def _rel(a, b):
    return float(np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b))


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("F", [2, 8, 9, 16, 17, 32, 33, 64])
def test_frames(gpu_ctx_factory, oracle, monkeypatch, storage, F):
    ctx, A = _problem(gpu_ctx_factory, 15, 13, 17, 24, 6, 1, storage)
    Y, s, X0 = _data(A, F, F)
    X, ll = _run(ctx, A, Y, s, X0, 3, True)
    cfg = ctx.batched_config(A, F)
    assert cfg["path"].startswith("bricks"), cfg
    blocked = env_ctx(monkeypatch, EPET_BATCHED="blocked")
    Xb, llb = _run(blocked, A, Y, s, X0, 3, True)
    assert blocked.batched_config(A, F)["path"].startswith("blocked")
    rp, col, val = decoded(A)
    X64 = oracle.mlem_f64_frames(A.m, A.n, val, rp, col, Y.cpu().numpy(), s.cpu().numpy(),
                                 X0.cpu().numpy().astype(np.float64), 3)
    for f in range(F):
        assert _rel(X[:, f], Xb[:, f].astype(np.float64)) < 5e-6
        assert _rel(X[:, f], X64[:, f]) < 1e-5
    np.testing.assert_allclose(ll, llb, rtol=1e-6)
    Xe, lle = _run(ctx, A, Y, s, X0, 3, False)
    for f in range(F):
        assert _rel(Xe[:, f], X[:, f].astype(np.float64)) < 5e-6
    np.testing.assert_allclose(lle, ll, rtol=1e-6)


@pytest.mark.parametrize("nx,ny,nz,nrays,na,every", [(16, 16, 16, 8, 18, 1),     # thin steps
                                                     (4, 3, 5, 64, 3, 1),
                                                     (9, 9, 9, 128, 7, 3),
                                                     (31, 33, 29, 64, 6, 1)])
@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_shapes(gpu_ctx_factory, oracle, monkeypatch, nx, ny, nz, nrays, na, every, storage):
    F = 6
    d = 0.05 / max(nx, ny, nz)
    ctx, A = _problem(gpu_ctx_factory, nx, ny, nz, nrays, na, every, storage, d)
    Y, s, X0 = _data(A, F, 3)
    X, ll = _run(ctx, A, Y, s, X0, 3, True)
    rp, col, val = decoded(A)
    X64 = oracle.mlem_f64_frames(A.m, A.n, val, rp, col, Y.cpu().numpy(), s.cpu().numpy(),
                                 X0.cpu().numpy().astype(np.float64), 3)
    print(ctx.batched_config(A, F), flush=True)
    for f in range(F):
        assert _rel(X[:, f], X64[:, f]) < 1e-5


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("F", [8, 12, 30, 50])
def test_full_steps(gpu_ctx_factory, oracle, storage, F):
    """Wide segments over a few large voxels: rows that hold nearly every voxel, so
    that steps have more entries than are loaded ahead (512 of at most 1,024)."""
    from epetreco_amd.api import VAL_BF16, VAL_F16
    from epetreco_amd.geometry import MeasurementSetup, VoxelGrid
    s = MeasurementSetup(-0.23, 0.23, 30, 2, 2, 2, 2, 0.2, 0.02, 0.02, 0.02)
    g = VoxelGrid(-0.08, -0.01, -0.01, 0.01, 0.01, 0.01, 16, 2, 2)
    ctx = gpu_ctx_factory(setup=s, grid=g, nrays=256, seed=4)
    A = ctx.sm_build(None, m=s.nchannels)
    if storage != "f32":
        A = A.convert({"bf16": VAL_BF16, "f16": VAL_F16}[storage])
    A.attach_transpose()
    Y, sens, X0 = _data(A, F, 7)
    X, _ = _run(ctx, A, Y, sens, X0, 3, True)
    cfg = ctx.batched_config(A, F)
    assert cfg["path"].startswith("bricks") and cfg["forward"]["entries_per_step"] > 512, cfg
    rp, col, val = decoded(A)
    X64 = oracle.mlem_f64_frames(A.m, A.n, val, rp, col, Y.cpu().numpy(), sens.cpu().numpy(),
                                 X0.cpu().numpy().astype(np.float64), 3)
    for f in range(F):
        assert _rel(X[:, f], X64[:, f]) < 1e-5


@pytest.mark.parametrize("what", ["y inf", "y nan", "x inf", "x nan", "y huge"])
@pytest.mark.parametrize("F", [5, 16, 20, 40])
def test_not_finite(gpu_ctx_factory, monkeypatch, what, F):
    ctx, A = _problem(gpu_ctx_factory, 15, 13, 17, 24, 6, 1, "f32")
    Y, s, X0 = _data(A, F, 1)
    clean, _ = _run(ctx, A, Y, s, X0, 2, False)
    bad = {"inf": float("inf"), "nan": float("nan"), "huge": 3e38}[what.split()[1]]
    f = F - 2
    if what[0] == "y":
        Y[A.m // 2, f] = bad
    else:
        X0[A.n // 2, f] = bad
    X, ll = _run(ctx, A, Y, s, X0, 2, False)
    assert ctx.batched_config(A, F)["path"].startswith("bricks")
    blocked = env_ctx(monkeypatch, EPET_BATCHED="blocked")
    Xb, llb = _run(blocked, A, Y, s, X0, 2, False)
    for k in range(F):
        if k != f:
            assert _rel(X[:, k], clean[:, k].astype(np.float64)) < 5e-6
    assert np.array_equal(np.isnan(X[:, f]), np.isnan(Xb[:, f]))
    assert np.array_equal(np.isinf(X[:, f]), np.isinf(Xb[:, f]))
    ok = np.isfinite(Xb[:, f])
    np.testing.assert_allclose(X[ok, f], Xb[ok, f], rtol=1e-4, atol=1e-30)
    assert np.array_equal(np.isnan(ll), np.isnan(llb)) and np.array_equal(np.isinf(ll), np.isinf(llb))
    ok = np.isfinite(llb)
    np.testing.assert_allclose(ll[ok], llb[ok], rtol=1e-6)


@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("F", [2, 4, 8, 11, 32, 64])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-0.5, 1.5)])
def test_products(gpu_ctx_factory, storage, F, alpha, beta):
    """spmm on bricks (transposed copy attached) against FP64 on the stored values:
    rtol 2e-5 of the sum of magnitudes, the bar of the other products."""
    import scipy.sparse as sp
    from epetreco_amd.api import OP_N, OP_T
    ctx, A = _problem(gpu_ctx_factory, 15, 13, 17, 24, 6, 1, storage)
    rp, col, val = decoded(A)
    M = sp.csr_matrix((val.astype(np.float64), col, rp), shape=(A.m, A.n))
    A.spmm(OP_N, torch.zeros(A.n, 64, device="cuda"))   # enough work for the bricks to be built
    rng = np.random.default_rng(F)
    for op, K, nin, nout in ((OP_N, M, A.n, A.m), (OP_T, M.T, A.m, A.n)):
        X = rng.normal(size=(nin, F)).astype(np.float32)
        Y0 = rng.normal(size=(nout, F)).astype(np.float32)
        Y = torch.as_tensor(Y0, device="cuda")
        A.spmm(op, torch.as_tensor(X, device="cuda"), Y, alpha=alpha, beta=beta)
        want = alpha * (K @ X.astype(np.float64)) + beta * Y0
        bar = 2e-5 * (abs(alpha) * (abs(K) @ np.abs(X)) + abs(beta * Y0)) + 1e-30
        assert np.all(np.abs(Y.cpu().numpy() - want) <= bar)


def test_products_on_two_streams_and_in_a_graph(gpu_ctx_factory):
    """Calls on two streams share nothing; a captured call runs the kernels that
    need no working memory, and replays give the eager result."""
    from epetreco_amd.api import OP_N, OP_T, Context
    ctx, A = _problem(gpu_ctx_factory, 15, 13, 17, 24, 6, 1, "f32")
    A.spmm(OP_T, torch.zeros(A.m, 64, device="cuda"))
    X = [torch.rand(A.m, 6, device="cuda") for _ in range(2)]
    want = [A.spmm(OP_T, x).double() for x in X]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    ctxs = []
    for st in streams:
        with torch.cuda.stream(st):
            ctxs.append(Context(0, st))
    from epetreco_amd._lib import check, lib
    import ctypes
    outs = [[torch.zeros(A.n, 6, device="cuda") for _ in range(20)] for _ in range(2)]
    torch.cuda.synchronize()
    for k in range(20):
        for i in range(2):
            check(lib().epet_matrix_spmm(ctxs[i].handle, A.handle, OP_T, 6, 1.0,
                                         ctypes.c_void_p(X[i].data_ptr()), 0.0,
                                         ctypes.c_void_p(outs[i][k].data_ptr())))
    torch.cuda.synchronize()
    for i in range(2):
        for o in outs[i]:
            assert (o.double() - want[i]).norm() <= 1e-6 * want[i].norm()
    # captured
    g = torch.cuda.CUDAGraph()
    y = torch.zeros(A.n, 6, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=streams[0]):
        check(lib().epet_matrix_spmm(ctxs[0].handle, A.handle, OP_T, 6, 1.0,
                                     ctypes.c_void_p(X[0].data_ptr()), 0.0,
                                     ctypes.c_void_p(y.data_ptr())))
    for _ in range(3):
        y.fill_(7.0)
        g.replay()
        torch.cuda.synchronize()
        assert (y.double() - want[0]).norm() <= 1e-6 * want[0].norm()


@pytest.mark.parametrize("rows", [449, 456, 480, 511, 512])
@pytest.mark.parametrize("F", [8, 50])
def test_rows_that_fill_no_group(gpu_ctx_factory, oracle, rows, F):
    """Row counts that leave the last group of 64 partly empty: the ratios of the
    whole group are written, so the vector that holds them covers it."""
    from epetreco_amd.geometry import MeasurementSetup, VoxelGrid
    s = MeasurementSetup(-0.23, 0.23, 32, 2, 2, 2, 2, 0.2, 0.02, 0.02, 0.02)
    g = VoxelGrid(-0.08, -0.01, -0.01, 0.01, 0.01, 0.01, 16, 2, 2)
    ctx = gpu_ctx_factory(setup=s, grid=g, nrays=256, seed=4)
    A = ctx.sm_build(np.arange(rows, dtype=np.int32)).attach_transpose()
    Y, sens, X0 = _data(A, F, 7)
    X, _ = _run(ctx, A, Y, sens, X0, 3, False)
    assert ctx.batched_config(A, F)["path"].startswith("bricks")
    rp, col, val = decoded(A)
    X64 = oracle.mlem_f64_frames(A.m, A.n, val, rp, col, Y.cpu().numpy(), sens.cpu().numpy(),
                                 X0.cpu().numpy().astype(np.float64), 3)
    for f in range(F):
        assert _rel(X[:, f], X64[:, f]) < 1e-5
