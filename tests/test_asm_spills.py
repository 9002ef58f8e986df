"""No form of the K-part GEMMs (unholy_amd/csrc/fp8_kpart.hip) spills vector registers: a reload inside the K loop waits for
every direct load in flight before it. Read from the metadata of the compiled assembly (no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_kpart_forms_do_not_spill(tmp_path):
    out = tmp_path / "fp8_kpart.s"
    csrc = os.path.join(ROOT, "unholy_amd", "csrc")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++20", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"), "-I", csrc, "--cuda-device-only", "-S",
                    os.path.join(csrc, "fp8_kpart.hip"), "-o", str(out)], check=True, capture_output=True)
    meta = re.findall(r"\.name:\s+(_Z\S*kpart_kernel\S*).*?\.vgpr_spill_count:\s+(\d+)", out.read_text(), re.S)
    assert len(meta) == 22
    assert [m for m in meta if int(m[1])] == []
