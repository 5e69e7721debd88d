"""The library's device allocation (xitils_amd/csrc/device_memory.h) on a host
stand-in for HIP: what is kept between calls is bounded, safe with several
threads, and given back when any allocation runs out of memory."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CPP = os.path.join(ROOT, "tests", "cpp")


@pytest.mark.parametrize("flags", [["-fsanitize=address,undefined", "-fno-sanitize-recover=undefined"], ["-fsanitize=thread"]])
def test_kept_memory_is_given_back(tmp_path, flags):
    exe = str(tmp_path / "device_memory_check")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", *flags, "-I", os.path.join(CPP, "fake_hip"), "-o", exe,
                    os.path.join(CPP, "device_memory_check.cpp"), "-pthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("OK"), r.stdout[-2000:] + r.stderr[-4000:]
