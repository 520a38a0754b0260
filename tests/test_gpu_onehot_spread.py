"""onehot-mfma on large grids, where six-bit digits hold A's book or, where its
values differ too much in scale inside a vector or between neighbouring
vectors, three bf16 terms: edges of the digit kernel's rule and blocks, and
products whose rows of B are zero opposite the large values, so that the outputs
are sums of the small ones alone and as exact as without the large ones."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import image, run_plan, say

pytestmark = pytest.mark.gpu


def _rows(rng, m):
    """Rows to check: the first and last of the blocks' edges and some others."""
    edge = [r for r in (0, 31, 32, 63, 64, 127, 128, m - 129, m - 128, m - 65, m - 64, m - 1) if 0 <= r < m]
    return np.unique(np.concatenate([edge, rng.integers(0, m, 40)]))


def _exact(a, b, rows, m, n, k, group):
    from oracle import vq4_numpy as o
    return (o.decode(*a, m * k, group).reshape(m, k)[rows].astype(np.float64)
            @ o.decode(*b, k * n, group).reshape(k, n).astype(np.float64))


def _check(vqdev, a, b, rng, m, n, k, group):
    words = (2, m, n, k, group, 16, 0, 0)
    assert vqdev.path_name(words) == "onehot-mfma"
    out, status = run_plan(vqdev, words, (*a, *b), 4 * m * n, np.float32, fill=0xFF)
    assert status == 0
    rows = _rows(rng, m)
    out, exact = out.reshape(m, n), _exact(a, b, rows, m, n, k, group)
    top = np.abs(exact).max(axis=1, keepdims=True)
    assert (np.abs(out[rows] - exact) <= 1e-5 * top).all()
    assert np.isfinite(out).all()


# m, n, k, group on both sides of the rule's lines (64 rows; 256 blocks of 64 rows from k
# = 1024, or 512 at group 16; 544 from 512; 896 below), rows one past a block and one
# short, k of one 32-block and of odd and even numbers of them
SHAPES = [(129, 86 * 128, 2080, 16), (128, 128 * 128, 2048, 16), (127, 129 * 128, 2080, 16),
          (64, 270 * 128, 2048, 16), (65, 130 * 128, 2048, 16), (129, 86 * 256, 2080, 32),
          (257, 52 * 128, 544, 16), (1153, 14 * 256, 1056, 32), (1089, 31 * 256, 544, 32),
          (1089, 30 * 256, 512, 32), (2177, 26 * 128, 288, 16), (2177, 25 * 128, 224, 16),
          (1024, 112 * 128, 256, 16), (2175, 27 * 256, 32, 32), (2177, 32 * 256, 96, 32),
          (2113, 32 * 256, 64, 32)]


@pytest.mark.parametrize("m,n,k,group", SHAPES)
def test_products(vqdev, m, n, k, group):
    rng = np.random.default_rng([m, n, k])
    say("onehot large grid", m, n, k, group)
    _check(vqdev, image(rng, m * k, group), image(rng, k * n, group, 0.02), rng, m, n, k, group)


@pytest.mark.parametrize("group,k", [(16, 288), (16, 544), (32, 32), (32, 64), (32, 288), (32, 544)])
@pytest.mark.parametrize("m", [2113, 2177])
@pytest.mark.parametrize("spread", [12, 20])
def test_wide_books_at_odd_sizes(vqdev, m, k, group, spread):
    """The bf16 terms where the digit kernel leaves a book to them."""
    from oracle import vq4_numpy as o
    n = 32 * 8 * group
    rng = np.random.default_rng([m, k, group])
    book = rng.standard_normal((16, group)).astype(np.float32)
    book[3:, 1::2] *= np.float32(2.0 ** spread)
    say("onehot wide book", m, n, k, group, spread)
    a = (o.pack_indices(rng.integers(0, 16, m * k // group)), book)
    _check(vqdev, a, image(rng, k * n, group, 0.02), rng, m, n, k, group)


def _mixed(group, kind, shift):
    """(sizes, A's codes, mixed book, book with its large values zero, B's codes, book)."""
    from oracle import vq4_numpy as o
    m, n, k = 2113, 32 * 8 * group, 256
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
@pytest.mark.parametrize("shift", [0, 3, 6, 10, 14, 20, 90])
def test_small_values_keep_their_bits(vqdev, group, kind, shift):
    """Both products have the same exact value, and the error of the one without
    large values is that of FP32 sums; twice it leaves room for another order. A
    single small value met alone is held to 2^-17 of itself."""
    (m, n, k), a, mixed, small, b, b_book = _mixed(group, kind, shift)
    words = (2, m, n, k, group, 16, 0, 0)
    assert vqdev.path_name(words) == "onehot-mfma"
    rows = _rows(np.random.default_rng(shift), m)
    exact = _exact((a, small), (b, b_book), rows, m, n, k, group)
    errors = []
    for book in (small, mixed):
        say("onehot spread", group, kind, shift)
        out, status = run_plan(vqdev, words, (a, book, b, b_book), 4 * m * n, np.float32)
        assert status == 0
        errors.append(np.linalg.norm(out.reshape(m, n)[rows] - exact) / np.linalg.norm(exact))
    assert errors[1] <= (2.0 ** -17 if kind == "single" else 2 * errors[0]), errors
