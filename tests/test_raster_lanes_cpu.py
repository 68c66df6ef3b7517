"""The multi-mesh autotuner times the depth-pass variant that the runs take: the lanes per face of all
the meshes' items, and the one variant of a batched run (checked on the host with the kernels' own
header, and that both the runs and the trials ask it)."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "raster_lanes_check.hip")
CSRC = os.path.join(HERE, "..", "gvv-differentiable-cuda-renderer_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_lanes_of_runs_and_trials(tmp_path):
    exe = str(tmp_path / "raster_lanes_check")
    r = subprocess.run([HIPCC, "-O1", "-std=c++17", "-ffp-contract=off", "--offload-arch=gfx950", SRC, "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    rows = [tuple(map(int, line.split())) for line in
            subprocess.run([exe], capture_output=True, text=True, timeout=60, check=True).stdout.splitlines()]
    assert [lanes for _, lanes, _, _ in rows] == [16, 16, 8, 8, 2, 2, 1, 1]
    assert all(batched == only for _, _, batched, only in rows)
    multi = open(os.path.join(CSRC, "gvv_multi.hip")).read()
    assigned = re.findall(r"raster_items = (.*);", multi)
    assert len(assigned) == 2 and all(a.startswith("shared_raster_items(") and "m->batched" in a for a in assigned)
    forward = open(os.path.join(CSRC, "gvv_forward.hip")).read()
    assert "raster_body<kBatchedLanes>" in forward and "raster_lanes(p.raster_items)" in forward
