"""The error of onehot-mfma's sums for few rows: no larger than that of the
fixed-point bins, which serve the same products with fewer rows."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import image, run_plan, say

pytestmark = pytest.mark.gpu

# 2-norm of the difference from float64 over the result's, of the bins with 4 and
# 5 rows on 4096 x 14336: 1.08e-7 to 1.20e-7 at groups 8, 16 and 32, dense and packed
BINS = 1.2e-7


@pytest.mark.parametrize("m,n,k,group,dense", [
    (5, 14336, 4096, 32, True), (8, 14336, 4096, 32, True), (8, 14336, 4096, 32, False),
    (4, 14336, 4096, 32, False), (9, 4096, 4096, 8, True), (16, 4096, 4096, 16, True),
    (33, 4096, 4096, 16, False), (128, 4096, 4096, 32, True), (128, 4096, 4096, 32, False)])
def test_error(vqdev, m, n, k, group, dense):
    from alelyon_compute_kit.vq import VQArray
    from oracle import vq4_numpy as o
    rng = np.random.default_rng([m, k, group, dense])
    words = (2, m, n, k, group, 16, 0, 0)
    b = image(rng, k * n, group, 0.02)
    w = o.decode(*b, k * n, group).reshape(k, n).astype(np.float64)
    say("onehot sums", m, n, k, group, dense)
    if dense:
        assert vqdev.dense_path_name(words) == "onehot-mfma"
        x = rng.standard_normal((m, k)).astype(np.float32)
        out = vqdev.matmul_dense(x, VQArray((k, n), group, *b))
    else:
        assert vqdev.path_name(words) == "onehot-mfma"
        a = image(rng, m * k, group)
        x = o.decode(*a, m * k, group).reshape(m, k)
        out, status = run_plan(vqdev, words, a + b, 4 * m * n, np.float32)
        assert status == 0
    exact = x.astype(np.float64) @ w
    error = np.linalg.norm(out.reshape(m, n) - exact) / np.linalg.norm(exact)
    say(f"error {error:.2e}")
    assert error <= BINS
