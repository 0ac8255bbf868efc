"""The native conversion of update lines is optional: the library builds where
Python's headers are missing, and the package works without the module."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("make") is None, reason="needs make")
def test_build_without_python_headers(tmp_path):
    plan = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "ddp_amd", "csrc"), f"PYINC={tmp_path}"],
                          capture_output=True, text=True, check=True).stdout
    assert "libddp.so" in plan and "hostconv" not in plan


def test_package_without_the_module():
    code = ("import sys; sys.modules['ddp_amd._hostconv'] = None\n"
            "import ddp_amd\n"
            "a = ddp_amd._updates_array([(1, 2, 3, 4), [0, 5, 6, 0]])\n"
            "print([(x.flag, x.u, x.v, x.w) for x in a])")
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    assert out.stdout.strip() == "[(1, 2, 3, 4), (0, 5, 6, 0)]"
