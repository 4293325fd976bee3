"""The candidate test on squares: lengths in metres, and scaled so far down and up that
the squares leave the range in which they decide and the root and quotient do; grids
whose voxel centres lie at the candidate radius of a channel along an axis, within a
few roundings of it.  Rows bit for bit the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(gpu_ctx_factory, oracle, setup, grid, channels, keep_zeros):
    ctx = gpu_ctx_factory(setup=setup, grid=grid, nrays=6, seed=5)
    lst = np.asarray(channels, np.int32)
    orp, ocol, oval = oracle.sm_rows(setup, grid, lst, 6, 5, keep_zeros=keep_zeros)
    if keep_zeros:
        val, col, row, n = ctx.getSystemMatrix(lst, len(ocol) + 8, keep_zeros=True)
        assert n == len(ocol)
        assert np.array_equal(row.cpu().numpy(), np.repeat(lst, np.diff(orp)))
    else:
        rp, col, val, _ = ctx.sm_build(lst).to_torch()
        assert np.array_equal(rp.cpu().numpy(), orp)
    assert np.array_equal(col.cpu().numpy(), ocol)
    assert np.array_equal(val.cpu().numpy(), oval)


def _setup(scale, na, n):
    from epetreco_amd.geometry import MeasurementSetup
    return MeasurementSetup(-0.23 * scale, 0.23 * scale, na, n, n, n, n, 360.0 / na,
                            0.02 * scale, 0.004 * scale, 0.004 * scale)


@pytest.mark.parametrize("keep_zeros", [False, True])
@pytest.mark.parametrize("scale", [2.0 ** -30, 1.0, 2.0 ** 26])
def test_scales(gpu_ctx_factory, oracle, scale, keep_zeros):
    from epetreco_amd.geometry import VoxelGrid
    d = 0.0025 * scale
    s = _setup(scale, 8, 5)
    g = VoxelGrid(-10 * d, -9 * d, -8.5 * d, d, d, d, 20, 18, 17)
    _check(gpu_ctx_factory, oracle, s, g, np.arange(3, s.nchannels, 151), keep_zeros)


@pytest.mark.parametrize("keep_zeros", [False, True])
@pytest.mark.parametrize("ulps", [-40, -3, -1, 0, 1, 2, 5, 40])
def test_centres_at_the_radius(gpu_ctx_factory, oracle, ulps, keep_zeros):
    """One head segment a side: the centre line is the x axis, and the grid's first
    row of centres lies at y = -R (R depends on the voxel, whose size stays)."""
    from epetreco_amd.geometry import VoxelGrid
    s = _setup(1.0, 4, 1)
    d = 0.001
    R = 0.5 * (np.sqrt(0.02 ** 2 + 2 * 0.004 ** 2) + np.sqrt(3.0) * d)
    oy = -R * (1.0 + ulps * 2.0 ** -23) - 0.5 * d
    g = VoxelGrid(-20 * d, oy, -0.5 * d, d, d, d, 40, 30, 1)
    _check(gpu_ctx_factory, oracle, s, g, np.arange(s.nchannels), keep_zeros)
