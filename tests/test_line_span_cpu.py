"""The depth pass's line spans keep every pixel that the exact ray/triangle test accepts (checked
on the host with the kernels' own header), and leave most of the rest out."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "line_span_check.hip")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_line_spans_cover_exact_test(tmp_path):
    exe = str(tmp_path / "line_span_check")
    r = subprocess.run([HIPCC, "-O2", "-std=c++17", "-ffp-contract=off", "-fhip-fp32-correctly-rounded-divide-sqrt",
                        "--offload-arch=gfx950", SRC, "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = subprocess.run([exe, "200000"], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0
    f = out.stdout.split()
    vals = dict(zip(f[0::2], f[1::2]))
    assert int(vals["boxes"]) > 50_000 and int(vals["accepted"]) > 1_000_000
    assert int(vals["missed"]) == 0
    # an accepted pixel stays inside every bound by most of the margin: the device's 1-ulp
    # reciprocal moves a bound by far less than what is left
    assert float(vals["slack"]) > 0.5 * float(vals["margin"])
    assert int(vals["kept"]) < 0.75 * int(vals["area"])
