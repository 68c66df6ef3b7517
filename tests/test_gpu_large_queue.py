"""The large-face queue filled by every lanes-per-face variant of the depth pass (16, 8, 2 and 1 lanes),
with small and large faces mixed and a last, partial group of 64 (view, face) items: every large face
queued once and none lost, so face ids, barycentrics and vertex normals are bit-exact against the
oracle; and the 1-lane variant on both sides of its 2,097,152 items."""
import pytest

from gvv_amd import scenes
from parity_util import run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views", [1, 3, 97, 330])
def test_mixed_sizes(device, views):
    """812 faces in 1, 3 (16 lanes), 97 (8 lanes) or 330 views (2 lanes)."""
    s = scenes.config1(width=90, height=80, cols=29, rows=14, n_cameras=views, tex_size=8, with_target=False)
    assert s.F == 812
    run_parity(s, device, "vertexColor", "shaded", m2d=False, check_grads=False, tuning=(16, 16))


@pytest.mark.parametrize("views", [102, 103])
def test_one_lane_per_face(device, views):
    """20,480 faces in 102 or 103 views: 2,088,960 items take 2 lanes to a face, 2,109,440 one."""
    s = scenes.config0(width=40, height=33, level=5, n_cameras=views)
    assert s.F == 20480
    run_parity(s, device, "vertexColor", "shaded", m2d=False, check_grads=False, tuning=(16, 16))
