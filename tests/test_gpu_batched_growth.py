"""The batched full build with leaf stages that grow unevenly: 16 clouds make 624 leaf places necessary at the first
split (496 unused cloud nodes and 16 * 8 children), more than the first stage of the keys (608) and fewer than that of
the counts (640), so only the keys grow; the next level then needs 624 + 7 * (internal children) places."""

import numpy as np
import pytest

from test_gpu_batched import PlainClouds, _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("large", [1, 4, 13])
def test_batched_build_grows_both_stages(hip, large):
    print(f"batched growth, {large} of 16 clouds split twice", flush=True)
    rng = np.random.default_rng(large)
    sizes = np.array([600 if c < large else 20 for c in range(16)], dtype=np.int64)
    n, ngmax = int(sizes.sum()), 8
    x, y, z = (rng.random(n).astype(np.float32) for _ in range(3))
    h = np.full(n, 0.05, np.float32)
    boxes, buckets = [(0.0, 1.0)] * 16, np.full(16, 16, np.uint32)
    b = hip.Batched(sizes, [hip.make_box(lo, hi, np.float32) for lo, hi in boxes], buckets, curve=hip.HILBERT, ngmax=ngmax)
    b.set_particles(x, y, z, h)
    b.build()
    plain = PlainClouds(hip, sizes, boxes, buckets, hip.HILBERT, ngmax, x, y, z, h)
    plain.build()
    _compare(b, plain, "build")
