"""Memory that freed matrices leave with the library goes back to the driver when
asked for: free memory after a matrix of some 400 MB was built, transposed and closed
is what it was before, to 32 MB."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_release_cached(gpu_ctx_factory):
    from epetreco_amd.geometry import MeasurementSetup, VoxelGrid
    s = MeasurementSetup(-0.23, 0.23, 3, 13, 13, 13, 13, 120.0, 0.02, 0.004, 0.004)
    g = VoxelGrid(-0.026, -0.026, -0.026, 0.001, 0.001, 0.001, 52, 52, 52)
    ctx = gpu_ctx_factory(setup=s, grid=g, nrays=64, seed=2)
    lst = (s.nchannels // 3 + np.arange(20000)).astype(np.int32)

    def use():
        A = ctx.sm_build(lst).attach_transpose()
        taken = 16 * A.nnz
        A.close()
        return taken

    use()                     # the context's own working memory
    ctx.release_cached()
    before = _free()
    taken = use()
    assert _free() < before - taken // 2
    ctx.release_cached()
    assert _free() >= before - (32 << 20)
    use()                     # and the memory is there again
