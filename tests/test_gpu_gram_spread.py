"""gram-mfma where entries of one Gram table differ in scale by more than its
rows and columns do: outputs that meet the small ones alone keep their bits."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import run_plan, say

pytestmark = pytest.mark.gpu

# the most that three bf16 terms a Gram entry, summed over 537 groups in one
# slice of k, were off (2-norm, books of normal entries: 4e-7 to 7.5e-7), twice
SUMS = 1.5e-6


@pytest.mark.parametrize("group", [8, 16, 32])
@pytest.mark.parametrize("m,n", [(20, 300), (96, 257)])
@pytest.mark.parametrize("shift", [0, 1, 2, 3, 4, 6, 8, 12, 20, 40, 90])
def test_small_entries_keep_their_bits(vqdev, group, m, n, shift):
    """Entries 0 to 7 of A's book hold 1 at a place where B's entries 0 to 7 are
    zero, and values 2^-shift of the other entries' elsewhere. Even rows and even
    columns use those entries alone, so that their outputs meet Gram entries that
    are small in their rows and in their columns."""
    from oracle import vq4_numpy as o
    k = 537 * group
    rng = np.random.default_rng([group, m, shift])
    book = rng.standard_normal((16, group)).astype(np.float32)
    book[:8] *= np.float32(2.0 ** -shift)
    book[:8, 0] = 1
    b_book = rng.standard_normal((16, group)).astype(np.float32)
    b_book[:8, 0] = 0
    idx, b_idx = rng.integers(0, 8, (m, k // group)), rng.integers(0, 8, (n, k // group))
    idx[1::2] += 8
    b_idx[1::2] += 8
    a, b = o.pack_indices(idx.reshape(-1)), o.pack_indices(b_idx.reshape(-1))
    words = (2, m, n, k, group, 16, 2, 0)
    assert vqdev.path_name(words) == "gram-mfma"
    exact = (o.decode(a, book, m * k, group).reshape(m, k).astype(np.float64)
             @ o.decode(b, b_book, n * k, group).reshape(n, k).T.astype(np.float64))
    say("gram spread", group, m, n, shift)
    out, status = run_plan(vqdev, words, (a, book, b, b_book), 4 * m * n, np.float32, fill=0xFF)
    assert status == 0
    out = out.reshape(m, n)
    for r in (0, 1):
        for c in (0, 1):
            want = exact[r::2, c::2]
            error = np.linalg.norm(out[r::2, c::2] - want) / np.linalg.norm(want)
            say(f"rows {r} columns {c}: {error:.2e}")
            assert error <= SUMS


@pytest.mark.parametrize("group", [8, 16, 32])
@pytest.mark.parametrize("m,n,k_groups", [(1, 1, 2047), (33, 255, 1023), (64, 256, 1001), (129, 513, 65)])
def test_wide_tables_at_odd_sizes(vqdev, group, m, n, k_groups):
    """The bf16 terms at the edges of their blocks, passes and slices of k."""
    from oracle import vq4_numpy as o
    k = k_groups * group
    rng = np.random.default_rng([group, m, n])
    book = rng.standard_normal((16, group)).astype(np.float32)
    book[:, 1:] *= np.float32(2.0 ** -20)
    b_book = rng.standard_normal((16, group)).astype(np.float32)
    b_book[:8, 0] = 0
    a = o.pack_indices(rng.integers(0, 16, m * k_groups))
    b = o.pack_indices(rng.integers(0, 16, n * k_groups))
    words = (2, m, n, k, group, 16, 2, 0)
    say("gram wide", group, m, n, k)
    vqdev.device.set_policy(2)
    try:
        assert vqdev.path_name(words) == "gram-mfma" or m * n * k < 1 << 22
        out, status = run_plan(vqdev, words, (a, book, b, b_book), 4 * m * n, np.float32, fill=0xFF)
    finally:
        vqdev.device.set_policy(0)
    assert status == 0
    x = o.decode(a, book, m * k, group).reshape(m, k).astype(np.float64)
    w = o.decode(b, b_book, n * k, group).reshape(n, k).astype(np.float64)
    # FP32 sums of k / group entries: at most one rounding each, of the sum of
    # the entries' magnitudes
    bound = 3 * k_groups * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T)
    assert (np.abs(out.reshape(m, n) - x @ w.T) <= bound).all()
