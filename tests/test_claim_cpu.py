"""The backward's slot flush adds every corner's terms to its own vertex whichever words of concurrent
LDS stores stay (checked on the host with the kernels' own header)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "claim_check.hip")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_corner_claims(tmp_path):
    exe = str(tmp_path / "claim_check")
    r = subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950", SRC, "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = subprocess.run([exe, "20000"], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0
    f = out.stdout.split()
    vals = dict(zip(f[0::2], map(int, f[1::2])))
    assert vals["one_word"] == 0
    assert vals["two_words"] > 0                 # the model does mix the words of an entry
    # the kernel stores entries of this type alone: one word, which a lane's store leaves whole
    assert vals["entry_bytes"] == 4
    kernel = open(os.path.join(HERE, "..", "gvv-differentiable-cuda-renderer_amd", "csrc", "gvv_backward.hip")).read()
    assert "claim_entry(" in kernel and "claim_target(" in kernel and "make_int2(" not in kernel
