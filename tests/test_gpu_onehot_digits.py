"""onehot-mfma at sizes that the six-bit digits and the bf16 terms share between
them (packed A, k a multiple of 32; test_gpu_onehot_spread.py has the line): rows
around the 128-row blocks, an odd number of 32-element blocks of k, book entries of
any magnitude."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import image, run_plan, say

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _exact(ops, m, n, k, group):
    from oracle import vq4_numpy as o
    a = o.decode(ops[0], ops[1], m * k, group).reshape(m, k).astype(np.float64)
    return a @ o.decode(ops[2], ops[3], k * n, group).reshape(k, n).astype(np.float64)


def _check(vqdev, ops, m, n, k, group):
    words = (2, m, n, k, group, 16, 0, 0)
    assert vqdev.path_name(words) == "onehot-mfma"
    say("onehot digits", m, n, k, group)
    out, status = run_plan(vqdev, words, ops, 4 * m * n, np.float32, fill=0xFF)
    assert status == 0
    out, exact = out.reshape(m, n), _exact(ops, m, n, k, group)
    top = np.abs(exact).max(axis=1, keepdims=True)
    assert (np.abs(out - exact) <= TOL * top).all()


# m, n, k, group: one row past a block, one short, k of a single 32-block, odd
# and even numbers of them, code words that start inside a word of the row
@pytest.mark.parametrize("m,n,k,group", [
    (129, 80 * 256, 32, 32), (255, 80 * 256, 96, 32), (1281, 16 * 256, 288, 32),
    (257, 56 * 128, 64, 16), (640, 32 * 128, 160, 16), (127, 112 * 128, 2080, 16)])
def test_products(vqdev, m, n, k, group):
    rng = np.random.default_rng([m, n, k])
    _check(vqdev, image(rng, m * k, group) + image(rng, k * n, group, 0.02), m, n, k, group)


@pytest.mark.parametrize("group", [16, 32])
@pytest.mark.parametrize("a_scale,b_scale", [(1.0, 0.02), (1e30, 1e-30), (1e-30, 1e30), (0.0, 1.0)])
def test_rows_and_books_of_any_magnitude(vqdev, group, a_scale, b_scale):
    """Even rows of A use entries 2^-24 below the others' and keep the bar
    against their own largest output."""
    from oracle import vq4_numpy as o
    m, n, k = 1280, 16 * 8 * group, 256
    rng = np.random.default_rng(group)
    book = (rng.standard_normal((16, group)) * a_scale).astype(np.float32)
    book[:8] *= np.float32(2.0 ** -24)
    idx = rng.integers(8, 16, (m, k // group))
    idx[0::2] -= 8
    _check(vqdev, (o.pack_indices(idx.reshape(-1)), book) + image(rng, k * n, group, b_scale), m, n,
           k, group)


@pytest.mark.parametrize("group", [16, 32])
@pytest.mark.parametrize("case", ["nan_a", "inf_b", "overflow"])
def test_status(vqdev, group, case):
    m, n, k = 1280, 16 * 8 * group, 64
    rng = np.random.default_rng(group)
    ops = [*image(rng, m * k, group), *image(rng, k * n, group, 0.02)]
    if case == "nan_a":
        ops[1][11, 3] = np.nan
    elif case == "inf_b":
        ops[3][2, 0] = np.inf
    else:
        ops[1][:], ops[3][:] = 3e19, 3e19
    say("onehot digits status", group, case)
    assert run_plan(vqdev, (2, m, n, k, group, 16, 0, 0), ops, 4 * m * n, np.float32)[1] == 1
