"""The cooperative tail of every persistent launch: a wave with at most 8 rays
or paths left goes on with 8 lanes per path, in the middle of a ray, and a
small launch is traced that way from its start.  Item counts around the borders
(one path, one group, one wave, a share of 8 for every wave, the largest small
launch of each mode, host queries answered in place) against lane-by-lane
launches, and the queries against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FLT_MAX = np.float32(3.402823466e38)


def _rays(n, seed, reach=FLT_MAX):
    rng = np.random.default_rng(seed)
    o = rng.uniform([-0.9, 0.25, -0.9], [0.9, 1.8, 0.9], (n, 3))
    d = rng.normal(size=(n, 3))
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3] = o
    r[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 7] = reach
    return r


@pytest.fixture(scope="module")
def scene(scenes, orc):
    mesh = scenes.scene_heightfield_boxes(1004, 24, 16)
    return mesh, orc.Scene(mesh.idx, mesh.pos)


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 63, 64, 65, 255, 257, 4097, 16384, 16385, 20011, 32768, 32769])
def test_queries(dev, scene, n):
    mesh, oracle = scene
    dev.upload_scene(mesh.idx, mesh.pos)
    dev.build()
    rays = _rays(n, n)
    rays[n // 2, 7] = -1.0                       # a dead ray among them
    ref = oracle.intersect_fp32(rays)
    short = _rays(n, n, 0.2)
    blocked = oracle.occluded_fp32(short) >= 0
    try:
        for tail in ("cooperative", "lanes"):
            dev.set_tail(tail)
            assert np.array_equal(dev.intersect(rays).view(np.uint32), ref.view(np.uint32))
            assert np.array_equal(dev.occluded(short) >= 0, blocked)
    finally:
        dev.set_tail("cooperative")


@pytest.mark.parametrize("size", [(1, 1), (3, 2), (8, 8), (9, 8), (65, 33), (256, 128), (256, 136),
                                  (383, 256), (385, 256)])
def test_renders(dev, prt, scene, size):
    mesh, _ = scene
    w, h = size
    cam = prt.camera_from_view([0.0, 1.9, 2.1], 0.75, 0.0, 0.9, w / h)
    dev.upload_scene(mesh.idx, mesh.pos)
    dev.build()
    dev.set_camera(cam)
    dev.init_frame(w, h)
    rgb = np.random.default_rng(3).uniform(0.1, 0.9, (mesh.tri_count, 3)).astype(np.float32)
    dldi = np.random.default_rng(4).normal(size=(h, w, 3)).astype(np.float32)
    with prt.HipDevice(0) as batch:
        sid, _ = batch.batch_add_scene(mesh.idx, mesh.pos)
        got = {}
        try:
            for tail in ("cooperative", "lanes"):
                dev.set_tail(tail)
                batch.set_tail(tail)
                out = []
                for renderer in ("primaryHip", "diffuseHip", "diffuse2Hip", "diffuseFastHip"):
                    dev.clear_frame()
                    rays = sum(dev.render(renderer, 6, 0.8)["ray"] for _ in range(3))
                    out += [dev.accum(), np.array(rays)]
                batch.batch_set_jobs([dict(scene=sid, width=w, height=h, spp=3, max_depth=6, albedo=0.8, camera=cam)])
                out += [np.array(batch.batch_render()["ray"]), batch.batch_accum(0)]
                dev.set_albedo(rgb)
                img, st = dev.render_albedo_image(0, 2, 6)
                grad, _ = dev.adjoint_albedo(0, 2, 6, dldi)
                got[tail] = (out + [img, np.array(st["ray"])], grad)
        finally:
            dev.set_tail("cooperative")
    for a, b in zip(got["cooperative"][0], got["lanes"][0]):
        assert np.array_equal(a, b)
    # the same terms added by atomics in another order: fp32 rounding of the
    # sum of at most 2 * 6 * w * h terms per triangle
    a, b = got["cooperative"][1].astype(np.float64), got["lanes"][1].astype(np.float64)
    assert np.abs(a - b).max() <= 1e-5 * max(1e-6, np.abs(b).max())
