"""COO helpers at their edges, against numpy: row counting over runs of equal
ids (spans of 1024 entries, 64 per step) and the sort's in-order shortcut.
Whole numbers: equal, no tolerance."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(gpu_ctx_factory):
    return gpu_ctx_factory()


def _i32(a):
    return torch.as_tensor(np.asarray(a, np.int32), device="cuda")


def _rows(kind, n, m, rng):
    if kind == "sorted":
        return np.sort(rng.integers(0, m, n))
    if kind == "one":
        return np.full(n, m - 1)
    if kind == "alternating":
        return np.arange(n) % 2 * (m - 1)
    if kind == "runs":       # runs of 1..200 equal ids in any order
        out = np.repeat(rng.integers(0, m, n), rng.integers(1, 200, n))
        return out[:n]
    return rng.integers(0, m, n)


@pytest.mark.parametrize("kind", ["sorted", "one", "alternating", "runs", "random"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 70001])
def test_row_pointers(ctx, kind, n):
    m = 37
    r = _rows(kind, n, m, np.random.default_rng(n))
    got = ctx.convertCoo2Csr(_i32(r), m).cpu().numpy()
    want = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=m))])
    assert np.array_equal(got, want)


@pytest.mark.parametrize("at", [0, 63, 64, 1024, 4999])
@pytest.mark.parametrize("bad", [-1, 37])
def test_row_id_out_of_range_is_refused(ctx, at, bad):
    from epetreco_amd.api import EpetError
    r = np.full(5000, 5)
    r[at] = bad
    with pytest.raises(EpetError):
        ctx.convertCoo2Csr(_i32(r), 37)


@pytest.mark.parametrize("n", [2, 255, 256, 257, 5000])
@pytest.mark.parametrize("swap", ["none", "first", "last", "equal"])
def test_sort_of_pairs_in_order(ctx, n, swap):
    rng = np.random.default_rng(n)
    key = np.sort(rng.choice(200 * 300, n, replace=False))
    row, col = key // 300 - 100, key % 300 - 150      # negative ids among them
    val = rng.random(n).astype(np.float32)
    if swap == "first":
        row[[0, 1]], col[[0, 1]] = row[[1, 0]], col[[1, 0]]
    elif swap == "last":
        row[[-2, -1]], col[[-2, -1]] = row[[-1, -2]], col[[-1, -2]]
    elif swap == "equal":
        row[1], col[1] = row[0], col[0]
    tv = torch.as_tensor(val, device="cuda")
    tr, tc = _i32(row), _i32(col)
    ctx.cooSort(tv, tr, tc)
    o = np.lexsort((col, row))
    assert np.array_equal(tr.cpu().numpy(), row[o])
    assert np.array_equal(tc.cpu().numpy(), col[o])
    assert np.array_equal(tv.cpu().numpy(), val[o])
