"""The backward's slot flush: tiles of a few faces (corners of a vertex merged in LDS), tiles around the
32-face limit and past the slots, tile edges 8, 16 and 32, with and without colour terms, against the
oracle with the suite's gradient tolerances."""
import numpy as np
import pytest

from gvv_amd import scenes
from parity_util import run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("level,res", [(1, 64), (2, 50), (3, 64), (4, 72), (5, 40)])
def test_flush(device, level, res, tile):
    s = scenes.config0(width=res, height=res + 3, level=level, n_cameras=2)
    s.uv = np.random.Generator(np.random.PCG64(level)).uniform(
        0, 1, size=s.uv.shape).astype("float32")
    for albedo, shading, m2d in (("textured", "shaded", False), ("vertexColor", "shadeless", False),
                                 ("vertexColor", "shaded", True), ("foregroundMask", "shaded", True)):
        run_parity(s, device, albedo, shading, m2d=m2d, tuning=(tile, 256))
