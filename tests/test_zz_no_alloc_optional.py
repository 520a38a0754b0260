"""ack_vq_noalloc on the paths that can do without a workspace (general, gram-mfma
and joint-mfma): ack_vq's bits whether their partial sums fit the handle's area,
do not (joint-mfma's transposed codes of 8 to 16 MiB) or are not needed,
and beside another handle's pending scratch work."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import image, say

pytestmark = pytest.mark.gpu

SHAPES = [(100, 300, 1000, 16, 0), (33, 77, 4001, 8, 3), (20, 1000, 400, 32, 3), (1024, 2050, 131, 16, 1),
          (1, 4096, 14336, 32, 2), (33, 255, 16 * 1023, 16, 2), (4, 600, 8 * 4099, 8, 2),
          (1024, 2048, 8 * 600, 8, 2),
          (128, 128, 300, 16, 1), (4096, 4096, 257, 16, 1), (128, 8192, 20000, 8, 1)]


class _Call:
    def __init__(self, device, ops, words):
        self.device, self.plan = device, np.asarray(words, "<u4").tobytes()
        self.bufs = [device.buffer(a.nbytes) for a in ops]
        for b, a in zip(self.bufs, ops):
            b.upload(a)
        self.out, self.status = device.buffer(4 * words[1] * words[2]), device.buffer(4)
        self.status.upload(np.zeros(1, np.uint32))

    def launch(self, entry):
        d = self.device
        with d.lock:
            return getattr(d.lib.cdll, entry)(d.handle, *(b.handle for b in self.bufs), self.out.handle,
                                              self.status.handle, self.plan, len(self.plan))

    def result(self):
        assert int(self.status.download(np.uint32)[0]) == 0
        return self.out.download(np.uint32)

    def free(self):
        for b in self.bufs + [self.out, self.status]:
            b.free()


@pytest.mark.parametrize("m,n,k,group,flags", SHAPES)
def test_the_same_bits(vqdev, m, n, k, group, flags):
    rng = np.random.default_rng([m, n, k])
    words = (2, m, n, k, group, 16, flags, 0)
    call = _Call(vqdev.device, image(rng, m * k, group) + image(rng, k * n, group, 0.02), words)
    try:
        results = []
        for entry in ("ack_vq", "ack_vq_noalloc"):
            say(entry, vqdev.path_name(words), m, n, k, group, flags)
            assert call.launch(entry) == 0
            results.append(call.result())
        np.testing.assert_array_equal(*results)
    finally:
        call.free()


@pytest.mark.parametrize("m,n,k,group,flags", [SHAPES[0], SHAPES[4], SHAPES[9]])
def test_accepted_beside_pending_scratch_work(vqdev, m, n, k, group, flags):
    """A handle's onehot-mfma work holds the scratch; the other handle's calls on
    these paths are accepted at once, give ack_vq's bits and take nothing from it."""
    from alelyon_compute_kit import ack
    rng = np.random.default_rng([m, n, k, 2])
    ops = image(rng, m * k, group) + image(rng, k * n, group, 0.02)
    long = (2, 512, 4096, 4096, 32, 16, 0, 0)
    assert vqdev.path_name(long) == "onehot-mfma"
    long_ops = image(rng, 512 * 4096, 32) + image(rng, 4096 * 4096, 32, 0.02)
    calls = []
    with ack.Device() as second:
        try:
            calls = [_Call(second, long_ops, long),
                     _Call(vqdev.device, ops, (2, m, n, k, group, 16, flags, 0))]
            holder, other = calls
            assert other.launch("ack_vq") == 0
            want = other.result()
            say("noalloc beside scratch work", m, n, k, group, flags)
            assert [holder.launch("ack_vq_noalloc") for _ in range(3)] == [0, 0, 0]
            assert other.launch("ack_vq_noalloc") == 0
            assert holder.launch("ack_vq_noalloc") == 0
            np.testing.assert_array_equal(other.result(), want)
            holder.result()
        finally:
            for call in calls:
                call.free()
