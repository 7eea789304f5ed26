"""The adjoint's replay of recorded hits (max_depth <= 64) against the replay that
traces the path again (deeper): same rays, same gradient up to the order of the
atomic sums, with black and partly black albedos among them.  A path still
alive at depth 64 (caught inside a closed box) traces one ray more at 65, and
if that one escapes its 66 rays are replayed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,spp", [((8, 8), 1), ((64, 48), 1), ((256, 192), 2), ((400, 320), 3)])
@pytest.mark.parametrize("tail", ["cooperative", "lanes"])
def test_recorded_equals_traced_replay(prt, scenes, size, spp, tail):
    mesh = scenes.scene_heightfield_boxes(1004, 32, 24)
    w, h = size
    rng = np.random.default_rng(w)
    rgb = rng.uniform(0.1, 0.9, (mesh.tri_count, 3)).astype(np.float32)
    rgb[rng.uniform(size=mesh.tri_count) < 0.05] = 0.0
    rgb[rng.uniform(size=mesh.tri_count) < 0.05, 1] = 0.0
    dldi = rng.uniform(0.0, 1.0, (h, w, 3)).astype(np.float32)
    with prt.HipDevice(0) as dev:
        dev.set_tail(tail)
        dev.upload_scene(mesh.idx, mesh.pos)
        dev.build()
        dev.set_camera(prt.camera_from_view([0.0, 1.9, 2.1], 0.75, 0.0, 0.9, w / h))
        dev.init_frame(w, h)
        dev.set_albedo(rgb)
        recorded, rs = dev.adjoint_albedo(5, spp, 64, dldi)
        traced, ts = dev.adjoint_albedo(5, spp, 65, dldi)
        longer = dev.render_albedo_image(5, spp, 65)[1]["ray"] - dev.render_albedo_image(5, spp, 64)[1]["ray"]
    replayed_later = ts["ray"] - rs["ray"] - longer
    assert replayed_later >= 0 and replayed_later % 66 == 0
    # all terms are >= 0, so each sum of m terms is off by at most m ulps
    # of itself; no triangle gathers more than 2^13 terms of these sizes
    a, b = recorded.astype(np.float64), traced.astype(np.float64)
    assert np.abs(a - b).max() <= 2.0 ** -10 * b.max()
    assert (b[a > 0] > 0).all()      # the deeper paths only add terms
    assert np.abs(a - b).sum() <= 1e-5 * b.sum()
