"""Kernel attributes are asked for on every device that runs the kernel."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_once_per_device(tmp_path):
    exe = tmp_path / "per_device_test"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-o", str(exe),
                    str(ROOT / "tests" / "cpp" / "per_device_test.cpp")], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True)
    assert "per device ok" in out.stdout


def test_no_attribute_is_asked_for_once_per_process():
    """hipFuncSetAttribute acts on the current device: no source may keep its
    result in a static of the process."""
    for f in (ROOT / "randomfield_amd" / "csrc").iterdir():
        assert not re.search(r"static\s+(const\s+)?hipError_t\s+\w+\s*=", f.read_text()), f.name
