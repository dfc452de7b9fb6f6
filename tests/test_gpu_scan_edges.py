"""The exclusive scan behind the leaf layouts at the edges of its three forms: one tile of 4096, up to 1024 tiles (every
tile sums the partials before it), more (the partials are scanned in between); against numpy, exactly."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILE = 4096


@pytest.mark.parametrize("n", [1, 63, TILE - 1, TILE, TILE + 1, 255 * TILE + 7, 256 * TILE, 257 * TILE + 1, 1024 * TILE,
                               1024 * TILE + 1, 1030 * TILE - 5])
def test_scan_edges(hip, n):
    print(f"scan n {n}", flush=True)
    counts = np.random.RandomState(n % 1000).randint(0, 900, n).astype(np.uint32)
    layout = hip.leaf_layout(hip.DeviceArray.from_numpy(counts))
    want = np.concatenate([[0], np.cumsum(counts, dtype=np.uint64)]).astype(np.uint32)
    assert np.array_equal(layout.download(), want)


@pytest.mark.parametrize("kd", [np.uint32, np.uint64])
@pytest.mark.parametrize("levels", [0, 1, 2, 4])
def test_link_of_full_trees(hip, oracle, levels, kd):
    """Trees whose every leaf lies at one level: each level of the nodes starts where the previous one ends, and the
    levels below the leaves' hold none."""
    print(f"link, leaves at level {levels}, {np.dtype(kd).name}", flush=True)
    step = (1 << (63 if kd == np.uint64 else 30)) >> (3 * levels)
    leaves = (np.arange(8**levels + 1, dtype=np.uint64) * np.uint64(step)).astype(kd)
    want, got = oracle.build_octree(leaves), hip.build_octree(leaves)
    for k in ("prefixes", "childOffsets", "internalToLeaf", "leafToInternal", "levelRange"):
        assert np.array_equal(got[k], want[k]), k
