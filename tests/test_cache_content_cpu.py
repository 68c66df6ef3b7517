"""The renderer cache's key compares whole contents: meshes that agree in the values its hash samples and
differ elsewhere are different keys, and a key kept in the cache owns its values, so that a caller's
arrays may change after the call."""
import numpy as np
import pytest

from gvv_amd import renderer


def key(faces, tc):
    return renderer.cache_key(faces, tc, 1000, 1, 8, 8, "vertexColor", "shaded", 2, 2, False, 0, 0)


def arrays(n=3000):
    rng = np.random.default_rng(n)
    return rng.integers(0, 1000, n).astype(np.int32), rng.uniform(0, 1, 2 * n).astype(np.float32)


@pytest.mark.parametrize("n", [3, 63, 64, 65, 129, 3000])
def test_every_value_counts(n):
    faces, tc = arrays(n)
    k = key(faces, tc)
    assert k == key(faces.copy(), tc.copy()) and hash(k) == hash(key(faces.copy(), tc.copy()))
    for i in range(n):
        other = faces.copy()
        other[i] += 1
        assert key(other, tc) != k
    sampled = {j for j in range(0, 2 * n, max(1, 2 * n // 64))}
    for i in range(2 * n):
        other = tc.copy()
        other[i] += 1
        assert key(faces, other) != k
        if i not in sampled:            # the hash is the same: only the comparison tells them apart
            assert hash(key(faces, other)) == hash(k)


def test_kept_keys_own_their_values(monkeypatch):
    made = []

    class Fake:
        def __init__(self, faces, tc, *args):
            made.append((np.array(faces), np.array(tc)))

    monkeypatch.setattr(renderer, "Rasterizer", Fake)
    monkeypatch.setattr(renderer, "_cache", {})
    monkeypatch.setattr(renderer.torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(renderer, "_raw_stream", lambda index: 0)
    get = lambda f, t: renderer.get_rasterizer(f, t, 1000, 1, 8, 8, "vertexColor", "shaded")
    faces, tc = arrays()
    faces0, tc0 = faces.copy(), tc.copy()
    first = get(faces, tc)
    assert get(faces.copy(), tc.copy()) is first
    faces[17] += 1                       # off the hash's sample
    tc[1] += 1
    second = get(faces, tc)
    assert second is not first and len(made) == 2
    faces[:], tc[:] = faces0, tc0
    assert get(faces, tc) is first and get(faces.copy(), tc) is first
