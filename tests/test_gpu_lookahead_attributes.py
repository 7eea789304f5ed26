"""Frame lookahead on a mesh with vertex normals and texture coordinates: the
same images and ray counts per frame as without it, for paths that are handed
over between shading frames that read the attributes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ready(prt, scenes):
    mesh = scenes.scene_smooth(1006, 16)
    with prt.HipDevice(0) as dev:
        dev.upload_scene(mesh.idx, mesh.pos)
        dev.set_attributes(mesh.normals, mesh.texcoords)
        dev.build()
        yield dev


@pytest.mark.parametrize("renderer", ["diffuseHip", "diffuse2Hip"])
@pytest.mark.parametrize("size", [(8, 8), (181, 182), (717, 405)])
def test_chain(ready, prt, scenes, size, renderer):
    view, (w, h) = scenes.SMOOTH_VIEW, size
    out = []
    for ahead in (False, True):
        ready.set_lookahead(ahead)
        ready.set_camera(prt.camera_from_view(view["pos"], view["angle_x"], view["angle_y"], view["fov_y"], w / h))
        ready.init_frame(w, h)
        rays = [ready.render(renderer, 6, 0.8)["ray"] for _ in range(9)]
        out.append((ready.accum(), rays))
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0].view(np.uint32), out[1][0].view(np.uint32))
