"""Which results are written through the second-level cache (cumo_amd/csrc/store_form.h): the rules compared with a look at
every row of a result."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


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
