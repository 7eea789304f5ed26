"""BVH builds of few triangles, sorted in one workgroup: key counts around a
wave, a round of the workgroup and the largest such sort, with equal keys."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 64, 65, 1023, 1024, 1025, 7168, 7169, 8191, 8192, 8193])
@pytest.mark.parametrize("same", [False, True])
def test_build(dev, orc, n, same):
    rng = np.random.default_rng(n)
    at = rng.uniform(0, 1, (n, 1, 3))
    if same:
        at[n // 3:] = at[0]              # two thirds of the keys are equal
    pos = (at + rng.uniform(-0.02, 0.02, (n, 3, 3)) * (0.0 if same else 1.0)).astype(np.float32)
    pos[:, 1:] += np.float32(0.01) * np.eye(3, dtype=np.float32)[:2]
    idx = np.arange(3 * n, dtype=np.int32).reshape(-1, 3)
    dev.upload_scene(idx, pos.reshape(-1, 3))
    dev.build()
    nodes, tris, prims, depth = dev.bvh()
    assert np.array_equal(np.sort(prims), np.arange(n))
    assert np.array_equal(tris.reshape(-1, 3, 3), pos[prims])
    r = np.zeros((400, 8), np.float32)
    o = rng.uniform(-1.0, 2.0, (400, 3))
    d = pos[rng.integers(0, n, 400)].mean(axis=1) - o
    r[:, 0:3] = o
    r[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 7] = 3.402823466e38
    ref = orc.Scene(idx, pos.reshape(-1, 3)).intersect_fp32(r)
    assert np.array_equal(dev.intersect(r).view(np.uint32), ref.view(np.uint32))
