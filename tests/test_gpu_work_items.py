"""How a persistent launch hands its work out: runs of 64 items dealt to 16
counters, the first run of each wave without one.  Item counts around the
borders (as many runs as waves, one more or less, runs that do not divide by
16, a last run of one item) against the oracle, and frames against the
wavefront pipeline, whose launches take their counts from the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(scenes, orc):
    mesh = scenes.scene_heightfield_boxes(1004, 24, 16)
    return mesh, orc.Scene(mesh.idx, mesh.pos)


@pytest.fixture(scope="module")
def answered(scene):
    _, oracle = scene
    rng = np.random.default_rng(7)
    r = np.zeros((4099, 8), np.float32)          # 4099 is prime: no run repeats another
    r[:, 0:3] = rng.uniform([-0.9, 0.25, -0.9], [0.9, 1.8, 0.9], (4099, 3))
    d = rng.normal(size=(4099, 3))
    r[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 7] = 3.402823466e38
    short = r.copy()
    short[:, 7] = 0.2
    return r, oracle.intersect_fp32(r), short, oracle.occluded_fp32(short) >= 0


@pytest.mark.parametrize("tail", ["cooperative", "lanes"])
@pytest.mark.parametrize("n", [1, 65, 1023, 1025, 32769, 65535, 65536, 65537, 65536 + 64 * 17 + 1, 131072, 131073,
                               196608, 196673, 262143, 262144, 262145, 262144 + 64 * 31 + 1, 700001])
def test_queries(dev, scene, answered, n, tail):
    mesh, _ = scene
    rays, hits, short, blocked = answered
    dev.upload_scene(mesh.idx, mesh.pos)
    dev.build()
    pick = np.arange(n) % 4099
    try:
        dev.set_tail(tail)
        assert np.array_equal(dev.intersect(rays[pick]).view(np.uint32), hits[pick].view(np.uint32))
        assert np.array_equal(dev.occluded(short[pick]) >= 0, blocked[pick])
    finally:
        dev.set_tail("cooperative")


@pytest.mark.parametrize("size", [(256, 256), (264, 256), (512, 256), (520, 264), (1023, 769), (1288, 1000)])
def test_frames(dev, prt, scene, size):
    mesh, _ = scene
    w, h = size
    dev.upload_scene(mesh.idx, mesh.pos)
    dev.build()
    dev.set_camera(prt.camera_from_view([0.0, 1.9, 2.1], 0.75, 0.0, 0.9, w / h))
    dev.init_frame(w, h)
    got = []
    try:
        for pipeline, ahead in (("wavefront", False), ("fused", False), ("fused", True)):
            dev.set_pipeline(pipeline)
            dev.set_lookahead(ahead)
            dev.clear_frame()
            rays = [dev.render("diffuseHip", 5, 0.8)["ray"] for _ in range(5)]
            got.append((dev.accum(), rays))
    finally:
        dev.set_pipeline("fused")
        dev.set_lookahead(True)
    for accum, rays in got[1:]:
        assert rays == got[0][1]
        assert np.array_equal(accum.view(np.uint32), got[0][0].view(np.uint32))


@pytest.mark.parametrize("variant", [0, 1, 2, 3])
@pytest.mark.parametrize("sizes", [[(1, 1)], [(8, 8), (9, 7)], [(64, 33), (3, 2), (31, 65)], [(256, 64), (128, 128)],
                                   [(256, 64), (129, 128)], [(256, 192), (257, 192)]])
def test_small_job_sets(dev, prt, scene, sizes, variant):
    mesh, _ = scene
    dev.upload_scene(mesh.idx, mesh.pos)
    dev.build()
    with prt.HipDevice(0) as batch:
        sid, _ = batch.batch_add_scene(mesh.idx, mesh.pos)
        cams = [prt.camera_from_view([0.0, 1.9, 2.1], 0.75, 0.0, 0.9, w / h) for w, h in sizes]
        batch.batch_set_tuning(variant)
        batch.batch_set_jobs([dict(scene=sid, width=w, height=h, spp=1, max_depth=5, albedo=0.8, camera=c)
                              for (w, h), c in zip(sizes, cams)])
        got = [batch.batch_render()["ray"] for _ in range(3)]     # as launched, captured, replayed
        ref = np.zeros(3, np.int64)
        for j, ((w, h), c) in enumerate(zip(sizes, cams)):
            dev.set_camera(c)
            dev.init_frame(w, h)
            dev.clear_frame()
            ref += [dev.render("diffuseHip", 5, 0.8)["ray"] for _ in range(3)]
            assert np.array_equal(batch.batch_accum(j).view(np.uint32), dev.accum().view(np.uint32))
        assert got == list(ref)
