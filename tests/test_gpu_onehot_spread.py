"""onehot-mfma on books whose values differ in scale inside a vector or between
neighbouring vectors, against rows of B that are zero opposite the large ones:
the outputs are sums of the small values alone, and as exact as without the
large ones."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import run_plan, say

pytestmark = pytest.mark.gpu


def _mixed(group, kind, shift):
    """(A's codes, mixed book, book with its large values zero, B's codes, book)."""
    from oracle import vq4_numpy as o
    m, n, k = 1280, 16 * 8 * group, 256
    rng = np.random.default_rng([group, shift])
    book = rng.standard_normal((16, group)).astype(np.float32)
    idx = rng.integers(0, 16, (m, k // group))
    large = np.zeros((16, group), bool)
    zero_rows = np.zeros(k, bool)
    if kind == "lone":                    # one place of every vector
        large[:, 5] = True
        zero_rows[5::group] = True
    elif kind == "single":                # all but one value of the only vector used
        large[:] = True
        large[3, 5] = False
        idx[:] = 3
        zero_rows[:] = True
        zero_rows[5::group] = False
    elif kind == "half":                  # half the places
        large[:, ::2] = True
        zero_rows[::2] = True
    else:                                 # every other vector of a row
        large[8:] = True
        idx %= 8
        idx[:, 1::2] += 8
        zero_rows.reshape(-1, group)[1::2] = True
    mixed, small = book.copy(), book.copy()
    mixed[large] *= np.float32(2.0 ** shift)
    small[large] = 0
    b_idx = rng.integers(1, 16, (k, n // group))
    b_idx[zero_rows] = 0
    b_book = (rng.standard_normal((16, group)) * 0.02).astype(np.float32)
    b_book[0] = 0
    return ((m, n, k), o.pack_indices(idx.reshape(-1)), mixed, small,
            o.pack_indices(b_idx.reshape(-1)), b_book)


@pytest.mark.parametrize("group", [16, 32])
@pytest.mark.parametrize("kind", ["lone", "half", "vectors", "single"])
@pytest.mark.parametrize("shift", [0, 3, 6, 10, 14, 17, 20, 30, 90])
def test_small_values_keep_their_bits(vqdev, group, kind, shift):
    """Both products have the same exact value, and the error of the one without
    large values is that of FP32 sums; twice it leaves room for another order. A
    single small value met alone is held to 2^-17 of itself."""
    from oracle import vq4_numpy as o
    (m, n, k), a, mixed, small, b, b_book = _mixed(group, kind, shift)
    words = (2, m, n, k, group, 16, 0, 0)
    assert vqdev.path_name(words) == "onehot-mfma"
    exact = (o.decode(a, small, m * k, group).reshape(m, k).astype(np.float64)
             @ o.decode(b, b_book, k * n, group).reshape(k, n).astype(np.float64))
    errors = []
    for book in (small, mixed):
        say("onehot spread", group, kind, shift)
        out, status = run_plan(vqdev, words, (a, book, b, b_book), 4 * m * n, np.float32)
        assert status == 0
        errors.append(np.linalg.norm(out.reshape(m, n) - exact) / np.linalg.norm(exact))
    assert errors[1] <= (2.0 ** -17 if kind == "single" else 2 * errors[0]), errors


@pytest.mark.parametrize("m", [1153, 1280])
@pytest.mark.parametrize("k", [32, 64, 288, 544])
@pytest.mark.parametrize("group", [16, 32])
@pytest.mark.parametrize("spread", [12, 20])
def test_wide_books_at_odd_sizes(vqdev, m, k, group, spread):
    """The bf16 form where the digit kernel leaves a book to it: rows that end
    inside a block, k of one 32-block to more than a pass of it."""
    from oracle import vq4_numpy as o
    n = 20 * 8 * group
    rng = np.random.default_rng([m, k, group])
    book = rng.standard_normal((16, group)).astype(np.float32)
    book[3:, 1::2] *= np.float32(2.0 ** spread)
    a = o.pack_indices(rng.integers(0, 16, m * k // group))
    b = o.pack_indices(rng.integers(0, 16, k * n // group))
    b_book = (rng.standard_normal((16, group)) * 0.02).astype(np.float32)
    words = (2, m, n, k, group, 16, 0, 0)
    assert vqdev.path_name(words) == "onehot-mfma"
    say("onehot wide book", m, n, k, group, spread)
    out, status = run_plan(vqdev, words, (a, book, b, b_book), 4 * m * n, np.float32, fill=0xFF)
    assert status == 0
    exact = (o.decode(a, book, m * k, group).reshape(m, k).astype(np.float64)
             @ o.decode(b, b_book, k * n, group).reshape(k, n).astype(np.float64))
    top = np.abs(exact).max(axis=1, keepdims=True)
    assert (np.abs(out.reshape(m, n) - exact) <= 1e-5 * top).all()
