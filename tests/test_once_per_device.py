"""CPU check of the helper behind settings that the runtime keeps per device."""
import ctypes as C
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_once_per_device(tmp_path):
    out = str(tmp_path / "libopd.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I", os.path.join(os.path.dirname(HERE), "slai_amd", "csrc"),
                           os.path.join(HERE, "native", "once_per_device.cpp"), "-o", out])
    assert C.CDLL(out).opd_check() == 0
