"""Softmax's quotients where they go through one reciprocal a row and where they do not: rows of two live elements, whose sum
is the same in any order, along rows and across them (a kernel that divides)."""
import numpy as np
import pytest

from ngraph_amd import hipq as H


@pytest.mark.gpu
@pytest.mark.parametrize("n", [4, 7, 64, 128, 197, 384])
def test_rows_and_columns_give_the_same_quotients(gpu_lib, n):
    print("[case] softmax quotients", n, flush=True)
    gaps = np.concatenate([np.linspace(0, 110, 1500), np.linspace(69.0, 69.6, 400), np.linspace(87, 104, 600), np.random.default_rng(3).uniform(0, 20, 500)]).astype(np.float32)
    x = np.full((gaps.size, n), -np.inf, np.float32)
    rows = np.arange(gaps.size)
    top = (rows * 7) % n
    x[rows, (top + 1 + rows % (n - 1)) % n] = 3.0 - gaps  # beside the largest, not on it
    x[rows, top] = 3.0
    along = H.softmax(x, (1,))
    across = H.softmax(np.ascontiguousarray(x.T), (0,)).T
    assert np.array_equal(along.view(np.uint32), np.ascontiguousarray(across).view(np.uint32))
    assert (along[along > 0] < 2.0**-100).any() and np.all(along[:, :].max(axis=1) >= 0.5)


@pytest.mark.gpu
def test_rows_without_a_sum(gpu_lib):
    print("[case] softmax without a sum", flush=True)
    x = np.random.default_rng(5).standard_normal((6, 128)).astype(np.float32)
    x[1, 5], x[2, 9], x[3], x[4, 1:] = np.inf, np.nan, -np.inf, -np.inf
    got = H.softmax(x, (1,))
    assert np.isnan(got[1:4]).all() and np.isfinite(got[[0, 4, 5]]).all() and got[4, 0] == 1.0 and not got[4, 1:].any()
