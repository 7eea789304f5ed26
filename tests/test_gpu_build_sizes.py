"""BVH builds at the sizes where their tiles end: leaf tiles of 1024 and 32768,
sort tiles of 1024 and 4096 keys, levels of one and of many blocks, equal keys.
Every triangle is in the tree once with its own vertices, and hits equal the
oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _soup(n, seed, same=False):
    rng = np.random.default_rng(seed)
    pos = (rng.uniform(0, 1, (n, 1, 3)) + rng.uniform(-0.02, 0.02, (n, 3, 3))).astype(np.float32)
    if same:
        pos[:] = pos[:1]     # one Morton key: the tree splits by index
    return np.arange(3 * n, dtype=np.int32).reshape(-1, 3), pos.reshape(-1, 3)


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    o = rng.uniform(-1.0, 2.0, (n, 3))
    d = rng.uniform(0, 1, (n, 3)) - o
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3] = o
    r[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 7] = 3.402823466e38
    return r


@pytest.mark.parametrize("method", ["sah", "greedy"])
@pytest.mark.parametrize("n,same", [(1, False), (2, False), (3, True), (4, False), (9, False), (1023, False),
                                    (1024, False), (1025, False), (1030, True), (4097, False), (32768, False),
                                    (32769, False), (40000, True), (262145, False), (1050000, False)])
def test_build(dev, orc, n, same, method):
    idx, pos = _soup(n, n, same)
    dev.set_bvh_collapse(method)
    try:
        dev.upload_scene(idx, pos)
        for _ in range(2):       # the second build reuses the first one's buffers
            st = dev.build()
    finally:
        dev.set_bvh_collapse("sah")
    nodes, tris, prims, depth = dev.bvh()
    assert np.array_equal(np.sort(prims), np.arange(n))
    assert np.array_equal(tris.reshape(-1, 3, 3), pos[idx[prims]])
    assert st["nodes"] == len(nodes) and st["depth"] == depth
    # every node but the root is some node's child, once
    inner = np.unpackbits(nodes[:, 15:16], axis=1).sum(axis=1)
    base = nodes[:, 16:20].copy().view("<u4")[:, 0].astype(np.int64)
    assert inner.sum() == len(nodes) - 1
    assert np.array_equal(np.cumsum(inner) - inner + 1, base)
    rays = _rays(500, n)
    assert np.array_equal(dev.intersect(rays).view(np.uint32), orc.Scene(idx, pos).intersect_fp32(rays).view(np.uint32))
