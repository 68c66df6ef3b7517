"""The depth pass's pre-test, with the margin the kernels give each face, keeps every pixel that the exact
ray/triangle test accepts: needles, vertices from 1 mm in front of the camera and far off screen, long
lenses, wide images, scenes far from the world's origin (checked on the host with the kernels' own
header).  With the fixed margin alone pixels are lost in these classes, so the check resolves it."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "pretest_cover_check.hip")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_pretest_covers_exact_test(tmp_path):
    exe = str(tmp_path / "pretest_cover_check")
    r = subprocess.run([HIPCC, "-O2", "-std=c++17", "-ffp-contract=off", "-fhip-fp32-correctly-rounded-divide-sqrt",
                        "--offload-arch=gfx950", SRC, "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = subprocess.run([exe, "8000"], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0
    rows = [line.split() for line in out.stdout.splitlines()]
    classes = {r[0]: dict(zip(r[1::2], map(float, r[2::2]))) for r in rows}
    assert set(classes) == {"ordinary", "needles", "near", "closeup", "offscreen", "lens", "far"}
    for name, c in classes.items():
        assert c["accepted"] > 50_000, name
        assert c["missed"] == 0 and c["missed_px"] == 0, name
        # the device's 1-ulp reciprocals move a bound by far less than what is left of it
        assert c["share"] < 0.5, name
        assert c["on"] > 0.8 * c["faces"], name        # the pre-test is not won by switching it off
    assert classes["ordinary"]["on"] == classes["ordinary"]["faces"]
    # margins stay near the least, also where a vertex far off screen has an error of hundreds of px
    assert classes["ordinary"]["median"] < 0.05 and classes["near"]["median"] < 0.2
    assert classes["offscreen"]["median"] < 2.0
    for name in ("needles", "closeup", "offscreen", "lens", "far"):
        assert classes[name]["plain"] > 0, name        # what the fixed margin loses
