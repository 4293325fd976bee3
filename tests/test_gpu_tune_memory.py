"""What tuning the splits of bricks leaves behind: the partial sums of the splits that
are kept, and not those of the splits that were tried.

60,000 rows of 64 frames may be split 64 times by their steps, 983 MB of partial
sums.  A first run with 2 frames builds the bricks; what 64 frames then keep beyond
it is their two gathered vectors and those partial sums, to 32 MB."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_partial_sums_kept(gpu_ctx_factory):
    from epetreco_amd.geometry import MeasurementSetup, VoxelGrid
    s = MeasurementSetup(-0.23, 0.23, 6, 13, 13, 13, 13, 60.0, 0.02, 0.004, 0.004)
    g = VoxelGrid(-0.026, -0.026, -0.026, 0.001, 0.001, 0.001, 52, 52, 52)
    ctx = gpu_ctx_factory(setup=s, grid=g, nrays=64, seed=2)
    A = ctx.sm_build((s.nchannels // 3 + np.arange(60000)).astype(np.int32)).attach_transpose()
    sens = A.colsum_f64().float()
    y = torch.ones(A.m, 64, device="cuda")
    x = torch.full((A.n, 64), 1.0 / A.n, device="cuda")
    y2, x2 = y[:, :2].contiguous(), x[:, :2].contiguous()
    before = x.clone()

    def free():
        ctx.release_cached()
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    ctx.mlem(A, y2, sens, x2, 1)
    f2 = free()
    ctx.mlem(A, y, sens, x, 1)
    kept = f2 - free()
    cfg = ctx.batched_config(A, 64)
    assert cfg["path"].startswith("bricks")
    print(kept >> 20, "MB kept,", cfg, flush=True)
    m, n = (A.m + 63) // 64 * 64, (A.n + 63) // 64 * 64
    parts = [0 if k == 1 else k for k in (cfg["forward"]["splits"], cfg["back_projection"]["splits"])]
    assert kept <= 64 * 4 * (m + n + parts[0] * m + parts[1] * n) + (32 << 20)
    # and the shapes for 2 frames still run, without being tuned again
    assert ctx.batched_config(A, 2)["path"].startswith("bricks")
    x.copy_(before)
    ctx.mlem(A, y, sens, x, 1)
    assert torch.isfinite(x).all()
