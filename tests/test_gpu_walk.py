"""Generated rows at the edges of the ray walk, bit for bit against the oracle:
grids of 1 to 257 planes (one lane per plane, 64 per wavefront, up to 256), rays
parallel to one or two axes (segments without extent), windows beyond the
smallest sets of cells, and ray counts around a wavefront.  Equal bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(gpu_ctx_factory, oracle, setup, grid, nrays, channels, keep_zeros):
    ctx = gpu_ctx_factory(setup=setup, grid=grid, nrays=nrays, seed=3)
    lst = np.asarray(channels, np.int32)
    orp, ocol, oval = oracle.sm_rows(setup, grid, lst, nrays, 3, keep_zeros=keep_zeros)
    if keep_zeros:
        sme, vxl, cnl, n = ctx.getSystemMatrix(lst, len(ocol) + 8, keep_zeros=True)
        assert n == len(ocol)
        assert np.array_equal(cnl.cpu().numpy(), np.repeat(lst, np.diff(orp)))
        assert np.array_equal(vxl.cpu().numpy(), ocol)
        assert np.array_equal(sme.cpu().numpy(), oval)
    else:
        rp, col, val, _ = ctx.sm_build(lst).to_torch()
        assert np.array_equal(rp.cpu().numpy(), orp)
        assert np.array_equal(col.cpu().numpy(), ocol)
        assert np.array_equal(val.cpu().numpy(), oval)
    return len(ocol)


def _grid(nx, ny, nz, edge=0.05):
    from epetreco_amd.geometry import VoxelGrid
    d = edge / max(nx, ny, nz)
    return VoxelGrid(-d * nx / 2, -d * ny / 2, -d * nz / 2, d, d, d, nx, ny, nz)


def _setup(seg=(0.02, 0.004, 0.004), na=8, n=5):
    from epetreco_amd.geometry import MeasurementSetup
    return MeasurementSetup(-0.23, 0.23, na, n, n, n, n, 360.0 / na, *seg)


@pytest.mark.parametrize("keep_zeros", [False, True])
@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 2, 63), (63, 4, 5), (64, 3, 7), (5, 6, 65),
                                  (65, 33, 20), (20, 70, 31), (128, 5, 6), (9, 5, 129),
                                  (256, 4, 3), (257, 3, 4)])
def test_grids(gpu_ctx_factory, oracle, dims, keep_zeros):
    s = _setup()
    rng = np.random.default_rng(sum(dims))
    chan = np.sort(rng.choice(s.nchannels, 24, replace=False))
    _check(gpu_ctx_factory, oracle, s, _grid(*dims), 7, chan, keep_zeros)


@pytest.mark.parametrize("keep_zeros", [False, True])
@pytest.mark.parametrize("seg", [(0.02, 0.0, 0.004), (0.02, 0.004, 0.0), (0.02, 0.0, 0.0),
                                 (0.0, 0.004, 0.004), (0.0, 0.0, 0.0)])
@pytest.mark.parametrize("n", [16, 40])
def test_axis_parallel_rays(gpu_ctx_factory, oracle, seg, n, keep_zeros):
    s = _setup(seg, na=4, n=3)     # angles of 90 degrees: rays along x and along z
    chan = np.arange(0, s.nchannels, 5)
    _check(gpu_ctx_factory, oracle, s, _grid(n, n, n), 5, chan, keep_zeros)


@pytest.mark.parametrize("nrays", [1, 2, 63, 64, 65, 256])
def test_ray_counts(gpu_ctx_factory, oracle, nrays):
    s = _setup()
    chan = np.arange(11, s.nchannels, 601)
    _check(gpu_ctx_factory, oracle, s, _grid(30, 28, 33), nrays, chan, False)


@pytest.mark.parametrize("seg", [0.002, 0.006, 0.012, 0.03])
def test_wide_windows(gpu_ctx_factory, oracle, seg):
    # windows from a few hundred to beyond 32,768 cells
    s = _setup((0.02, seg, seg), na=5, n=2)
    chan = np.arange(0, s.nchannels, 3)
    _check(gpu_ctx_factory, oracle, s, _grid(60, 60, 60), 96, chan, False)
