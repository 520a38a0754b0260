"""Decode on both sides of the output sizes (160 and 256 MiB) at which it changes
how it stores: a bit copy of the book's vectors."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import image, run_plan, say

pytestmark = pytest.mark.gpu

MIB = 1 << 18  # values in 1 MiB


@pytest.mark.parametrize("group", [8, 32])
@pytest.mark.parametrize("elements", [160 * MIB, 160 * MIB + 5, 256 * MIB, 256 * MIB + 3])
def test_decode(vqdev, group, elements):
    from oracle import vq4_numpy as o
    codes, book = image(np.random.default_rng([group, elements]), elements, group)
    say("decode stores", group, elements)
    out, status = run_plan(vqdev, (1, elements, 1, 1, group, 16, 0, 0), (codes, book), 4 * elements,
                           np.uint32)
    assert status == 0
    assert np.array_equal(out, o.decode(codes, book, elements, group).reshape(-1).view(np.uint32))
