"""Which results are written through the second-level cache (cumo_amd/csrc/store_form.h): the rules compared with a look at
every row of a result, and the instructions that the forms become."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_rules_against_every_row(tmp_path):
    exe = tmp_path / "store_form_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-o", str(exe), os.path.join(ROOT, "tests", "store_form_check.cpp")], check=True)
    p = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert p.returncode == 0 and int(p.stdout) == 8 * 11 * 7 * 5 * 2 * 3 * 2, p.stdout


def test_kernels_that_write_rows_ask_whether_they_may_be_written_through():
    """Windows included: a row's start alone does not decide."""
    asked = 0
    for name in ("ew_kernels.h", "fused_rows.hip", "scan.hip"):
        with open(os.path.join(ROOT, "cumo_amd", "csrc", name)) as f:
            for line in f:
                if "store_pieces(" in line and any(s in line for s in ("step", "+ oo")):
                    asked += 1
                    assert "p.through && store_pieces(" in line, line
    assert asked == 6


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not present")
def test_forms_in_assembly(tmp_path):
    """Written through: `sc1`; large results beside whole pieces: `nt`, and `nt sc1` where a kernel writes tiles of many rows,
    with the two wait states behind it that the compiler keeps for stores of its own."""
    out = tmp_path / "store_form_probe.s"
    cmd = [HIPCC, "-O3", "-std=c++17", "-I" + os.path.join(ROOT, "cumo_amd", "csrc"), "--offload-arch=gfx950", "-Xclang", "-target-feature",
           "-Xclang", "-packed-fp32-ops", "-S", "--cuda-device-only", "-x", "hip", os.path.join(ROOT, "tests", "store_form_probe.hip"), "-o", str(out)]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, cwd=str(tmp_path))
    assert p.returncode == 0, p.stdout[-2000:]
    text = out.read_text()
    for name, off_pieces in (("probe_store_cached", ""), ("probe_store_streamed", "nt"), ("probe_tile_cached", ""), ("probe_tile_streamed", "nt sc1")):
        body = re.search(r"^%s:[^\n]*\n(.*?)\.Lfunc_end" % name, text, flags=re.S | re.M).group(1)
        lines = [l.strip() for l in body.splitlines() if l.strip() and not l.strip().startswith((";", "."))]
        stores = [(i, l) for i, l in enumerate(lines) if l.startswith("global_store_dwordx4")]
        forms = {re.sub(r"\s*;.*", "", re.split(r"\]|off", l)[-1]).strip() for _, l in stores}
        assert forms == {"sc1", off_pieces}, (name, stores)
        for i, l in stores:
            if l.endswith("nt sc1"):
                assert lines[i + 1] == "s_nop 1", lines[i:i + 2]
