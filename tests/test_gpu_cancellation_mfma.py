"""Cancellation-heavy operands on the products that sum on 6-bit digits, Gram
tables, code counts and bf16 terms.

Inner indices (or whole groups of them) come in pairs x, -x(1 + eps) against equal
rows of B, so that every output is eps times smaller than the sum of magnitudes
that flows through it. No FP32 order holds 1e-5 of max|y| here. Each output is held
to gamma_N sum_k |x_k w_k|, N the roundings that its path makes on the way:

* onehot-mfma on digits: 6 a 64-step of k into a code's sum, each of terms that
  add to at most |x| (1 + 2^-4) in magnitude (balanced digits), then 17;
* gram-mfma: 3 a pair of groups on digits, whose instructions lose up to 2^-24 of
  their block scales (at most 2^4 times an entry's terms), and the slices' sums;
* joint-mfma: whole counts, then 33 of the two products with the books;
* the general products: 6 a 16-step of k of terms of at most |x| (1 + 2^-7), and the
  slices' sums.
"""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import run_plan, say

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _gamma(roundings):
    return roundings * U / (1 - roundings * U)


# path, m, n, k, group, flags, roundings of a sum (times its terms' excess)
CASES = [
    ("onehot-mfma", 257, 130 * 128, 2048, 16, 0, (6 * 2048 / 64) * (1 + 2 ** -4) + 17),
    ("onehot-mfma", 1089, 16 * 256, 4096, 32, 0, (6 * 4096 / 64) * (1 + 2 ** -4) + 17),
    ("gram-mfma", 96, 512, 14336, 32, 2, 3 * 448 / 2 * 2 ** 4 + 64),
    ("gram-mfma", 70, 300, 4096, 8, 2, 3 * 512 / 2 * 2 ** 4 + 64),
    ("joint-mfma", 256, 512, 4096, 16, 1, 33),
    ("joint-mfma", 128, 256, 250, 32, 1, 33),
    ("general", 64, 1600, 4096, 16, 0, (6 * 4096 / 16) * (1 + 2 ** -7) + 64),
    ("general", 64, 800, 4096, 32, 3, (6 * 4096 / 16) * (1 + 2 ** -7) + 64)]


@pytest.mark.parametrize("path,m,n,k,group,flags,roundings", CASES)
@pytest.mark.parametrize("eps", [1e-1, 1e-2, 1e-3])
def test_within_the_bound_of_its_sums(vqdev, path, m, n, k, group, flags, roundings, eps):
    from oracle import vq4_numpy as o
    words = (2, m, n, k, group, 16, flags, 0)
    assert vqdev.path_name(words) == path
    rng = np.random.default_rng([m, n, k, int(1 / eps)])
    book = np.empty((16, group), np.float32)
    book[0::2] = rng.standard_normal((8, group))
    book[1::2] = (-book[0::2].astype(np.float64) * (1 + eps)).astype(np.float32)
    b_book = (rng.standard_normal((16, group)) * 0.02).astype(np.float32)
    # A's vectors: along k (pairs of groups) or, stored k x m, along m (pairs of rows)
    if flags & 1:
        a_idx = 2 * rng.integers(0, 8, (k, m // group))
        a_idx[1::2] = a_idx[0::2] + 1
    else:
        a_idx = 2 * rng.integers(0, 8, (m, k // group))
        a_idx[:, 1::2] = a_idx[:, 0::2] + 1
    pair = 1 if flags & 1 else group     # inner indices apart
    if flags & 2:                        # B stored n x k, its vectors along k
        b_idx = rng.integers(0, 16, (n, k // group))
        b_idx[:, 1::2] = b_idx[:, 0::2]
        if flags & 1:                    # pairs of rows inside a vector: equal neighbours
            b_book[:, 1::2] = b_book[:, 0::2]
    else:
        b_idx = rng.integers(0, 16, (k, n // group)).reshape(k // (2 * pair), 2, pair, n // group)
        b_idx[:, 1] = b_idx[:, 0]
    a, b = o.pack_indices(a_idx.reshape(-1)), o.pack_indices(b_idx.reshape(-1))
    say("cancellation", path, m, n, k, group, flags, eps)
    out, status = run_plan(vqdev, words, (a, book, b, b_book), 4 * m * n, np.float32, fill=0xFF)
    assert status == 0
    x = o.decode(a, book, m * k, group).astype(np.float64)
    w = o.decode(b, b_book, n * k, group).astype(np.float64)
    x = x.reshape(k, m).T if flags & 1 else x.reshape(m, k)
    w = w.reshape(n, k).T if flags & 2 else w.reshape(k, n)
    exact, sizes = x @ w, np.abs(x) @ np.abs(w)
    error = np.abs(out.reshape(m, n) - exact)
    say(f"max|y| {np.abs(exact).max():.3g} of {sizes.max():.3g}, err/max|y| "
        f"{error.max() / np.abs(exact).max():.2e}, of the bound {(error / (_gamma(roundings) * sizes)).max():.3f}")
    assert (error <= _gamma(roundings) * sizes).all()
