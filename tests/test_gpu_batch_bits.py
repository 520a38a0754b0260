"""A product has the same bits alone and in a batch: its path, its slices of k and
their order are chosen from the product, also where the batch's size changes
whether the slices run side by side or in one block."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import image, run_plan, say

pytestmark = pytest.mark.gpu


# general: below and above 2^22 multiply-adds and k = 160, few and many slices, all
# tile heights; gram: slices side by side, in pairs and walked, short and long k;
# joint: codes gathered and transposed by the pre-pass
@pytest.mark.parametrize("m,n,k,group,flags", [
    (64, 64, 100, 16, 0), (65, 130, 159, 8, 3), (100, 300, 1000, 16, 0), (33, 77, 4001, 8, 3),
    (20, 1000, 400, 32, 3), (300, 200, 700, 16, 0),
    (33, 255, 16 * 1023, 16, 2), (64, 256, 8 * 601, 8, 2), (1, 300, 32 * 500, 32, 2),
    (128, 128, 300, 16, 1), (256, 128, 200, 32, 1), (64, 256, 96, 8, 1)])
@pytest.mark.parametrize("count", [2, 9, 40])
def test_batch_equals_singles(vqdev, m, n, k, group, flags, count):
    words = (2, m, n, k, group, 16, flags, 0)
    assert vqdev.path_name(words) == vqdev.path_name(words, count=count)
    rng = np.random.default_rng([m, n, k, flags])
    items = [image(rng, m * k, group) + image(rng, k * n, group, 0.02) for _ in range(count)]
    say("batch bits", vqdev.path_name(words), m, n, k, group, flags, count)
    ops = tuple(np.concatenate([item[s].reshape(-1) for item in items]) for s in range(4))
    out, status = run_plan(vqdev, words, ops, 4 * m * n * count, np.uint32, count=count)
    assert status == 0
    out = out.reshape(count, m * n)
    for i in {0, 1, count - 1}:
        single, status = run_plan(vqdev, words, items[i], 4 * m * n, np.uint32)
        assert status == 0
        np.testing.assert_array_equal(out[i], single)
