"""What the forward velocity sweep's instances (one cell a thread, compact and row tiles)
take of a SIMD's registers, from the compiler's own metadata: 8 waves of up to 80 scalar
and 64 vector registers fit."""
import os
import re
import shutil
import subprocess

import pytest

from elastic_fm_vp_vs_rho_amd import build


def test_velocity_sweep_leaves_a_simd_its_eight_waves(tmp_path):
    if not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")):
        pytest.skip("no hipcc")
    asm = tmp_path / "forward.s"
    flags = [f for f in build.HIPCC_FLAGS if f != "-fPIC"]
    subprocess.run([build._hipcc(), *flags, "--offload-device-only", "-S", "-I", build.INCLUDE, "-I", build.CSRC,
                    os.path.join(build.CSRC, "forward.hip"), "-o", str(asm)], check=True, capture_output=True, timeout=300)
    text = asm.read_text()
    meta = text[text.index("amdhsa.kernels:"):]
    seen = 0
    for k in re.split(r"\n  - ", meta)[1:]:
        name = re.search(r"\.name:\s+(\S+)", k)
        tile = name and re.search(r"k_velocityILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E", name.group(1))
        if not tile or tile.group(3) != "1" or tile.group(4) == "8":
            continue
        seen += 1
        value = lambda key: int(re.search(r"\.%s:\s+(\d+)" % key, k).group(1))
        assert value("sgpr_count") <= 80, name.group(1)
        assert value("vgpr_count") <= 64, name.group(1)
        assert value("private_segment_fixed_size") == 0 and value("sgpr_spill_count") == 0, name.group(1)
    assert seen == 8
