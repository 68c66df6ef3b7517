"""Faces whose own binary32 errors reach past a fixed pre-test margin -- needles, vertices from 1 mm in
front of the camera and far off screen, long lenses, a scene far from the world's origin -- through
every pass that skips pixels by the pre-test (small boxes, boxes walked by a wavefront, the large-face
pass, the screen tiles): face ids, barycentrics and vertex normals bit-exact against the oracle."""
import numpy as np
import pytest

from gvv_amd import scenes
from parity_util import run_parity

pytestmark = pytest.mark.gpu


def hard_faces(kind, n=24, width=400, height=300, seed=1):
    rng = np.random.Generator(np.random.PCG64(seed))
    away = 3e5 if kind == "far" else 0.0
    focal = 12.0 if kind == "lens" else 1.2
    pos = np.array([1000.0 + away, 300.0 - away, -2000.0 + away])
    E = scenes.look_at(pos / scenes.MM, target_m=(pos + np.array([-0.3, -0.1, 0.6]) * 3000) / scenes.MM)
    K = scenes.pinhole(width, height, focal)
    R = np.asarray(E, np.float64).reshape(3, 4)[:, :3]
    f, cx, cy = K.reshape(3, 3)[0, 0], K.reshape(3, 3)[0, 2], K.reshape(3, 3)[1, 2]
    v = []
    for t in range(n):
        depth = rng.uniform(1000, 4000) * (10 if kind in ("lens", "far") else 1)
        px = rng.uniform([0, 0], [width, height], size=(3, 2)) * 1.4 - 0.2 * np.array([width, height])
        z = depth * (1 + 0.1 * rng.normal(size=3))
        if kind == "closeup":
            z = 5000.0 ** rng.uniform(0, 1, size=3)
        if kind == "offscreen":
            a = rng.uniform(0, 2 * np.pi)
            px[t % 3] = 30000.0 ** rng.uniform(0.7, 1.2) * np.array([np.cos(a), np.sin(a)])
            z[t % 3] = 3000.0 ** rng.uniform(0.1, 1)
        c = np.stack([(px[:, 0] - cx) / f * z, (px[:, 1] - cy) / f * z, z], 1)
        if kind == "needles":
            c[2] = c[0] + rng.uniform(0.2, 0.9) * (c[1] - c[0]) + 10.0 ** rng.uniform(-1.5, 0.3) * rng.normal(size=3)
        v.append(pos + c @ R)
    v = np.concatenate(v).astype(np.float32)
    s = scenes.single_triangle(width=width, height=height)
    s.faces = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    s.uv = np.tile(s.uv, (n, 1, 1))
    s.vpos, s.vcol = v[None], rng.uniform(0, 1, size=(1, 3 * n, 3)).astype(np.float32)
    s.extr, s.intr = np.asarray(E, np.float32).reshape(1, 1, 12), np.asarray(K, np.float32).reshape(1, 1, 9)
    s.meta = dict(name=f"hard {kind}")
    return s


@pytest.mark.parametrize("kind", ["needles", "closeup", "offscreen", "lens", "far"])
def test_hard_faces(device, kind):
    s = hard_faces(kind)
    for kw in (dict(tuning=(16, 16)), dict(tuning=(16, 1 << 20)), dict(depth_pass=1)):
        run_parity(s, device, "vertexColor", "shaded", m2d=False, check_grads=False, **kw)
