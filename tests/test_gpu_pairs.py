"""The sort's scan of pairs at the edges of its quads and wavefronts, in arrays that
start at any element, against numpy.  Whole numbers: equal, no tolerance."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(gpu_ctx_factory):
    return gpu_ctx_factory()


def _dev(a, dtype):
    return torch.as_tensor(np.asarray(a, dtype), device="cuda")


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 255, 256, 257, 1027, 8195])
@pytest.mark.parametrize("start", [0, 1, 2, 3])     # arrays need not lie on 16 bytes
def test_pairs_out_of_order_anywhere(ctx, n, start):
    rng = np.random.default_rng(n)
    key = np.sort(rng.choice(200 * 300, n, replace=False))
    val = rng.random(n).astype(np.float32)
    for at in sorted({-1, 0, n // 2, *(q for q in (2, 3, 254, 255, 256, 1022, 1023) if q < n - 1), n - 2}):
        k = key.copy()
        if 0 <= at < n - 1:
            k[[at, at + 1]] = k[[at + 1, at]]
        row, col = k // 300 - 100, k % 300 - 150
        t = [_dev(np.concatenate([np.zeros(start), a]), d)[start:]
             for a, d in ((val, np.float32), (row, np.int32), (col, np.int32))]
        ctx.cooSort(*t)
        o = np.argsort(k, kind="stable")
        for got, a in zip(t, (val, row, col)):
            assert np.array_equal(got.cpu().numpy(), a[o])
