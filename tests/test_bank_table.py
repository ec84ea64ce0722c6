# SPDX-License-Identifier: Apache-2.0
"""The HBM bank's device table without a GPU (tests/c/k3_bank_table.c): it follows admissions and
evictions, is sent only when it has changed, without a wait, and not at all for a caller that
needs the whole layer resident while it is not."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_bank_table(tmp_path):
    exe = str(tmp_path / "bank")
    subprocess.run(["gcc", "-std=c99", "-O1", "-g", "-Wall", "-Wextra", "-Werror",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "kimi-k3-in-c_amd", "csrc"),
                    os.path.join(ROOT, "tests", "c", "k3_bank_table.c"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
