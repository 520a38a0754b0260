"""The 256/192-row tiling of onehot-mfma, which large grids with k an odd
multiple of 16 take: rows around both block sizes against float64."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import image, run_plan, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1024, 112 * 128, 16), (1024, 112 * 128, 272), (2048, 56 * 128, 48)])
def test_products(vqdev, m, n, k):
    from oracle import vq4_numpy as o
    group = 16
    rng = np.random.default_rng([m, n, k])
    a, b = image(rng, m * k, group), image(rng, k * n, group, 0.02)
    words = (2, m, n, k, group, 16, 0, 0)
    assert vqdev.path_name(words) == "onehot-mfma"
    say("onehot mixed", m, n, k)
    out, status = run_plan(vqdev, words, a + b, 4 * m * n, np.float32, fill=0xFF)
    assert status == 0
    exact = (o.decode(*a, m * k, group).reshape(m, k).astype(np.float64)
             @ o.decode(*b, k * n, group).reshape(k, n).astype(np.float64))
    top = np.abs(exact).max(axis=1, keepdims=True)
    assert (np.abs(out.reshape(m, n) - exact) <= 1e-5 * top).all()
