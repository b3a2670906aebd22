"""The attention kernels' copies from global memory to LDS, in the assembly
hipcc makes of them: every copy has m0 written right before it with the wait
state that asks for, and a scalar base that the scalar unit wrote.  (A base
written by the vector unit needs five wait states, which the compiler does not
add in front of inline asm.)"""
import os
import re
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flashengine.cpp_amd")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no HIP compiler")
def test_copies_have_their_wait_states(tmp_path):
    out = tmp_path / "attn.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-mcode-object-version=5", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + os.path.join(PKG, "..", "include"),
                    "-I" + os.path.join(PKG, "csrc"), "--cuda-device-only", "-S",
                    os.path.join(PKG, "csrc", "attn_kernels.hip"), "-o", str(out)],
                   check=True, timeout=300, stderr=subprocess.DEVNULL)
    before = ["", ""]
    copies = 0
    for line in out.read_text().splitlines():
        line = line.split(";")[0].strip()
        if not line or line.endswith(":") or line.startswith("."):
            continue
        m = re.match(r"global_load_lds_dwordx4 v\S+, (off|s\[\d+:\d+\])", line)
        if m:
            copies += 1
            assert re.match(r"s_mov_b32 m0, s\d+$", before[0]), (before, line)
            if m[1] == "off":
                assert before[1] == "s_nop 0", (before, line)
            else:
                assert before[1].startswith("s_mov_b64 " + m[1] + ", s["), (before, line)
        before = [before[1], line]
    assert copies > 1000
