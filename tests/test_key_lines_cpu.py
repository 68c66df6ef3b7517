"""The large-face pass walks rows, so that neighbouring candidates share lines of the visibility buffer:
the spans keep every pixel of the edge test, and tall boxes touch a fraction of the lines that their
columns would (checked on the host with the kernels' own header)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "key_lines_check.hip")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_large_faces_walk_rows(tmp_path):
    exe = str(tmp_path / "key_lines_check")
    r = subprocess.run([HIPCC, "-O2", "-std=c++17", "-ffp-contract=off", "--offload-arch=gfx950", SRC, "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = subprocess.run([exe, "3000"], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
    f = out.stdout.split()
    vals = dict(zip(f[0::2], map(int, f[1::2])))
    assert vals["passed"] > 1_000_000 and vals["missed"] == 0 and vals["tall"] > 500
    assert vals["row_lines"] < 0.4 * vals["side_lines"]
    kernel = open(os.path.join(HERE, "..", "gvv-differentiable-cuda-renderer_amd", "csrc", "gvv_forward.hip")).read()
    large = kernel[kernel.index("void raster_large_face("):kernel.index("__global__ void __launch_bounds__(64) k_raster_large(")]
    assert "bl.start_rows(" in large and "bl.start(" not in large
