"""The kernels that hold a long row in a block's registers (fused_rows.hip) are worth their lanes only while they do: a lane that
spills goes to memory for what it spilled, several times a row. The compiler says how much of that every kernel needs."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not present")


def test_rows_held_in_registers_are_not_spilled(tmp_path):
    out = tmp_path / "fused_rows.s"
    cmd = [HIPCC, "-O3", "-std=c++17", "-ffp-contract=off", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "cumo_amd", "csrc"),
           "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-S", "--cuda-device-only", "-x", "hip",
           os.path.join(ROOT, "cumo_amd", "csrc", "fused_rows.hip"), "-o", str(out)]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, cwd=str(tmp_path))
    assert p.returncode == 0, p.stdout[-2000:]
    kernels = re.findall(r"^\s*\.amdhsa_kernel (\S*fused_\S+)\n(.*?)\.end_amdhsa_kernel", out.read_text(), flags=re.S | re.M)
    scratch = {name: int(re.search(r"\.amdhsa_private_segment_fixed_size (\d+)", text).group(1)) for name, text in kernels}
    # softmax and layernorm of two types, two block sizes, two forms of access
    assert sum("fused_wide_rows_kernel" in name for name in scratch) == 16, sorted(scratch)
    assert not [name for name, size in scratch.items() if size], scratch
