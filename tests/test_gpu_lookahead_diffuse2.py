"""Frame lookahead of the diffuse2 renderer: the same images and ray counts per
frame as without it, at sizes around those where it starts, with paths that
stop between a shadow ray and the path's next, and across calls that break the
chain (another renderer, depth, camera or a cleared frame)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ready(dev, scenes):
    mesh = scenes.scene_heightfield_boxes(1004, 24, 16)
    dev.upload_scene(mesh.idx, mesh.pos)
    dev.build()
    return dev


def _frames(dev, prt, w, h, calls):
    out = []
    for ahead in (False, True):
        dev.set_lookahead(ahead)
        dev.set_camera(prt.camera_from_view([0.0, 1.9, 2.1], 0.75, 0.0, 0.9, w / h))
        dev.init_frame(w, h)
        dev.clear_frame()
        rays = []
        for renderer, depth, albedo in calls:
            rays.append(dev.render(renderer, depth, albedo)["ray"])
        out.append((dev.accum(), rays))
    dev.set_lookahead(True)
    return out


@pytest.mark.parametrize("depth", [0, 1, 6, 17])
@pytest.mark.parametrize("size", [(181, 182), (256, 136), (385, 256), (717, 405), (1288, 1000)])
def test_chain(ready, prt, size, depth):
    (a, ra), (b, rb) = _frames(ready, prt, *size, [("diffuse2Hip", depth, 0.8)] * 11)
    assert ra == rb
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_broken_chain(ready, prt):
    d2, d1 = ("diffuse2Hip", 5, 0.8), ("diffuseHip", 5, 0.8)
    calls = [d2, d2, d2, d2, d1, d1, d1, d1, d2, d2, d2, ("diffuse2Hip", 4, 0.8), ("diffuse2Hip", 4, 0.8), ("diffuse2Hip", 4, 0.7),
             ("diffuse2FastHip", 4, 0.7), d2, ("primaryHip", 0, 0.8), d2, d2, d2]
    (a, ra), (b, rb) = _frames(ready, prt, 500, 300, calls)
    assert ra == rb
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
