"""Books with an entry far above the rest that no code uses: the product neither
overflows nor loses bits of the entries it does use."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import run_plan, say

pytestmark = pytest.mark.gpu


def _operands(rng, m, n, k, group, a_scale, a_extreme, b_scale, b_extreme):
    from oracle import vq4_numpy as o
    ops = []
    for count, scale, extreme in ((m * k, a_scale, a_extreme), (k * n, b_scale, b_extreme)):
        book = (rng.standard_normal((16, group)) * scale).astype(np.float32)
        book[15] = extreme
        ops += [o.pack_indices(rng.integers(0, 15, -(-count // group))), book]
    return ops


@pytest.mark.parametrize("m,n,k,group,flags,path", [
    (128, 64, 700, 16, 1, "joint-mfma"), (128, 192, 200, 32, 1, "joint-mfma"),
    (256, 128, 300, 8, 1, "joint-mfma"),
    (40, 100, 2000, 16, 3, "general"), (70, 130, 500, 8, 0, "general")])
@pytest.mark.parametrize("a_scale,a_extreme,b_scale,b_extreme", [
    (1.0, 1e30, 1.0, 1e10), (1e-10, 1e25, 1e5, 1e20), (1e-10, 1e30, 1.0, 1.0), (1.0, 1.0, 1e-12, 3e38),
    (1e10, 1e38, 1e-10, 1e38), (1e-20, 1e-20, 1e-15, 1e15)])
def test_unused_extremes(vqdev, oracle, m, n, k, group, flags, path, a_scale, a_extreme, b_scale, b_extreme):
    from oracle import vq4_numpy as o
    words = (2, m, n, k, group, 16, flags, 0)
    assert vqdev.path_name(words) == path
    rng = np.random.default_rng([m, n, k])
    ops = _operands(rng, m, n, k, group, a_scale, a_extreme, b_scale, b_extreme)
    say("book extremes", path, m, n, k, group, a_scale, a_extreme, b_scale, b_extreme)
    out, status = run_plan(vqdev, words, ops, 4 * m * n, np.float32, fill=0xFF)
    assert status == oracle.matmul(*ops, m, n, k, group, flags)[1] == 0
    a = o.decode(ops[0], ops[1], m * k, group).astype(np.float64)
    b = o.decode(ops[2], ops[3], k * n, group).astype(np.float64)
    a = a.reshape(k, m).T if flags & 1 else a.reshape(m, k)
    b = b.reshape(n, k).T if flags & 2 else b.reshape(k, n)
    exact = a @ b
    top = np.abs(exact).max(axis=1, keepdims=True)
    # FP32 results: half a unit of the smallest subnormal beside the usual bar
    assert (np.abs(out.reshape(m, n) - exact) <= 2e-6 * top + 2.0 ** -149).all()
