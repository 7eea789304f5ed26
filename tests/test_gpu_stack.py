"""The traversal stack past its LDS entries: large overlapping triangles make
every ray keep many children, so entries beyond the LDS part live in global
memory, pushed from both sides of the border.  Hits are compared with the
oracle's brute force, batched renders whose launch shape keeps 8 or 16 entries
in LDS with plain ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _soup(n, seed):
    """n random triangles of unit size in the unit cube."""
    rng = np.random.default_rng(seed)
    pos = (rng.uniform(0, 1, (n, 1, 3)) + rng.uniform(-0.5, 0.5, (n, 3, 3))).astype(np.float32).reshape(-1, 3)
    return np.arange(3 * n, dtype=np.int32).reshape(-1, 3), pos


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    o = rng.uniform(-1.5, 2.5, (n, 3))
    d = rng.uniform(0, 1, (n, 3)) - o
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3] = o
    r[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 7] = 3.402823466e38
    return r


@pytest.mark.parametrize("n", [64, 1000, 6000])
def test_deep_stacks_equal_brute_force(dev, orc, n):
    idx, pos = _soup(n, 70 + n)
    dev.upload_scene(idx, pos)
    dev.build()
    rays = _rays(3001, n)
    # near misses keep the whole stack: tfar ends before most hits
    rays[::3, 7] = 0.4
    ref = orc.Scene(idx, pos).intersect_fp32_brute(rays)
    hits, _ = dev.intersect_counters(rays)
    assert np.array_equal(hits.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(dev.intersect(rays).view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(dev.occluded(rays) >= 0, ref[:, 0] >= 0)


@pytest.mark.parametrize("variant", [0, 1, 2, 3])
def test_lds_stack_depths_equal_plain_frames(prt, variant):
    idx, pos = _soup(6000, 9)
    w, h, depth = 70, 41, 5
    cam = prt.camera_from_view([0.5, 0.5, 3.0], 0.0, 0.0, 0.7, w / h)
    with prt.HipDevice(0) as dev:
        dev.upload_scene(idx, pos)
        dev.build()
        dev.set_camera(cam)
        dev.init_frame(w, h)
        for _ in range(2):
            dev.render("diffuseHip", depth, 0.8)
        scene, _ = dev.batch_add_scene(idx, pos)
        dev.batch_set_jobs([dict(scene=scene, width=w, height=h, spp=2, max_depth=depth, albedo=0.8, camera=cam)])
        dev.batch_set_tuning(variant)
        dev.batch_render()
        assert np.array_equal(dev.batch_accum(0), dev.accum())
