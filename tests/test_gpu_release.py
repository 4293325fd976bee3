"""Device memory that the library keeps.

Memory that freed matrices leave with the library goes back to the driver when
asked for: free memory after a matrix of some 400 MB was built, transposed and closed
is what it was before, to 32 MB."""
import ctypes

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


def test_blocks_freed_outside(gpu_ctx_factory):
    """A block from epet_malloc that the caller frees with hipFree, a smaller one of the
    caller's own at its address, and that one freed with epet_free: the next epet_malloc of
    the first size must not be handed the small one.  (No memory is touched.)"""
    from epetreco_amd._lib import check, lib
    ctx = gpu_ctx_factory()
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipFree.argtypes = [ctypes.c_void_p]
    hip.hipMemGetAddressRange.argtypes = [ctypes.POINTER(ctypes.c_void_p),
                                          ctypes.POINTER(ctypes.c_size_t), ctypes.c_void_p]
    big = 48 << 20
    met = 0
    for small in (4 << 20, 24 << 20, 40 << 20, (46 << 20) + 4096, 47 << 20, big - (64 << 10), big - 4096, big - 512):
        p, q, r = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
        check(lib().epet_malloc(ctx.handle, ctypes.byref(p), big))
        assert hip.hipFree(p) == 0
        assert hip.hipMalloc(ctypes.byref(q), small) == 0
        met += q.value == p.value
        check(lib().epet_free(ctx.handle, q))
        check(lib().epet_malloc(ctx.handle, ctypes.byref(r), big))
        base, size = ctypes.c_void_p(), ctypes.c_size_t()
        assert hip.hipMemGetAddressRange(ctypes.byref(base), ctypes.byref(size), r) == 0
        assert base.value == r.value and size.value >= big
        check(lib().epet_free(ctx.handle, r))
        ctx.release_cached()
    print("same address in", met, "of 8", flush=True)
