"""Host arrays of every size class of the transfers: answered in place, one
chunk, two halves, a ring that wraps (2 MiB chunks, 6 slots).  A large query
equals the same rays asked in small parts; a frame read as floats agrees with
the same frame read as pixels, whose chunks end elsewhere."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3] = rng.uniform([-0.9, 0.3, -0.9], [0.9, 1.8, 0.9], (n, 3))
    d = rng.normal(size=(n, 3))
    r[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 7] = 3.402823466e38
    return r


@pytest.mark.parametrize("n", [32767, 32768, 32769, 65536, 65537, 131072, 131073, 262145, 900001])
def test_large_query_equals_small_ones(dev, scenes, n):
    mesh = scenes.scene_heightfield_box(1001, cells=32)
    dev.upload_scene(mesh.idx, mesh.pos)
    dev.build()
    rays = _rays(n, n)
    step = 20000
    hits = np.concatenate([dev.intersect(rays[k:k + step]) for k in range(0, n, step)])
    blocked = np.concatenate([dev.occluded(rays[k:k + step]) for k in range(0, n, step)]) >= 0
    assert np.array_equal(dev.intersect(rays).view(np.uint32), hits.view(np.uint32))
    assert np.array_equal(dev.occluded(rays) >= 0, blocked)


@pytest.mark.parametrize("w,h", [(1, 1), (128, 256), (361, 363), (362, 363), (1001, 777), (1920, 1080)])
def test_frame_read_as_floats_and_pixels(dev, prt, scenes, w, h):
    mesh = scenes.scene_heightfield_box(1001, cells=32)
    dev.upload_scene(mesh.idx, mesh.pos)
    dev.build()
    view = scenes.CONFIGS["heightfield_box_512"]["view"]
    dev.set_camera(prt.camera_from_view(view["pos"], view["angle_x"], view["angle_y"], view["fov_y"], w / h))
    dev.init_frame(w, h)
    dev.render("primaryHip")
    a, px = dev.accum(), dev.frame_bgr8()
    assert (a[..., 3] == 1.0).all()
    want = np.clip((a[..., :3].astype(np.float64) ** (1 / 2.2) * 255).astype(np.int64), 0, 255)
    got = np.stack([(px >> 16) & 255, (px >> 8) & 255, px & 255], -1)
    assert np.abs(got - want).max() <= 1     # fp32 powf against float64, before truncation


def test_indices_checked_in_parts(dev, scenes):
    """An index out of range is found wherever it stands, and the old scene stays."""
    mesh = scenes.scene_heightfield_box(1001, cells=512)      # 1.5 M indices: several parts
    dev.upload_scene(mesh.idx, mesh.pos)
    dev.build()
    rays = _rays(100, 1)
    before = dev.intersect(rays)
    for at, bad in ((0, -1), (262144, len(mesh.pos)), (mesh.idx.size - 1, 2 ** 31 - 1), (700001, -2 ** 31)):
        idx = mesh.idx.copy()
        idx.reshape(-1)[at] = bad
        with pytest.raises(RuntimeError, match="vertex index out of range"):
            dev.upload_scene(idx, mesh.pos)
        assert np.array_equal(dev.intersect(rays).view(np.uint32), before.view(np.uint32))
