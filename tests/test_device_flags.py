"""The once-a-device flags that guard the kernels' LDS limits
(novann_amd/csrc/novaq_device_flags.h): a flag a device, and none lost when
threads set them at once; and no launcher keeps such a flag for the whole
process.  CPU only (built with g++)."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "novann_amd", "csrc")


def test_flags_from_several_threads(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "device_flags_run")
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-o", exe,
                    os.path.join(HERE, "native", "device_flags_run.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout


def test_lds_limits_are_raised_in_one_place():
    """hipFuncSetAttribute is called by allow_lds alone, and every launcher's
    flag is a DeviceFlags: none is a process-wide bool or size."""
    calls, flags = [], []
    for name in sorted(os.listdir(CSRC)):
        with open(os.path.join(CSRC, name)) as f:
            text = f.read()
        calls += [name] * text.count("hipFuncSetAttribute(")
        flags += re.findall(r"static (\w+) (?:lds_\w+|raised)\b", text)
    assert calls == ["novaq_internal.h"]
    assert flags and set(flags) == {"DeviceFlags"}
