"""The depth pass's line spans at their edges: boxes around 64 lines and 64 pixels per line, tall
and wide, slivers, split large faces, unpacked candidate words in both line directions, and item
counts on both sides of the lines between 16, 4 and 1 lanes to a face.  Ids, barycentrics and
vertex normals bit-exact against the oracle."""
import pytest

from gvv_amd import scenes
from parity_util import run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tri", [((-2.0, -1.0, 0.0), (2.0, -1.0, 0.0), (0.0, 1.2, 0.0)),
                                 ((-0.9, -0.9, 0.0), (0.9, 0.88, 0.1), (0.9, 0.9, 0.0)),
                                 ((-1.5, 0.001, 0.0), (1.5, 0.0, 0.2), (1.5, 0.02, 0.0)),
                                 ((0.0, -1.5, 0.0), (0.013, 1.5, 0.1), (-0.01, 1.5, 0.0))])
@pytest.mark.parametrize("wh", [(1, 1), (16, 16), (17, 16), (63, 65), (64, 64), (129, 40), (300, 7), (7, 300), (500, 500),
                                (8300, 70), (70, 8300)])
def test_one_triangle(device, wh, tri):
    s = scenes.single_triangle(width=wh[0], height=wh[1], z_m=1.2, tri_m=tri)
    for tuning in ((16, 256), (16, 1 << 20)):
        run_parity(s, device, "vertexColor", "shaded", m2d=False, check_grads=False, tuning=tuning)


@pytest.mark.parametrize("level,views", [(4, 12), (4, 13), (5, 12), (5, 13)])
def test_lanes_per_face(device, level, views):
    """5,120 or 20,480 faces in 12 or 13 views: 61,440 / 66,560 / 245,760 / 266,240 items."""
    s = scenes.config0(width=96, height=80, level=level, n_cameras=views)
    run_parity(s, device, "vertexColor", "shaded", m2d=False, check_grads=False)
