"""The forward-rate kernels hold a path's 40 forwards and 40 adjoints in registers: none of them spills (the
compiler's own report of the ahead-of-time build, no device needed)."""
import os
import re
import subprocess
import sys

from conftest import ROOT


def test_no_scratch(tmp_path):
    sys.path.insert(0, os.path.join(ROOT, "sde-sim-rs_amd"))
    import build
    r = subprocess.run([build.HIPCC] + build.HIP_FLAGS + ["--cuda-device-only", "-S", "-o", str(tmp_path / "lmm.s"),
                       os.path.join(build.CSRC, "lmm_kernels.hip")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    found = re.findall(r"\.amdhsa_kernel (\S*sdesim_lmm\S*)\n(?:.*\n)*?\s*\.amdhsa_private_segment_fixed_size (\d+)",
                       (tmp_path / "lmm.s").read_text())
    assert len(found) == 8
    assert all(int(scratch) == 0 for _, scratch in found), found
