"""Host emulation of the mixed-radix register-pass transforms (chapsim1.0_amd/csrc/chs_fftg.h): the
header compiled with g++, a block's threads run as threads.  Every even length 2^a 3^b 5^c in
18 ... 256 (shorter ones are one pass, which the kernels leave to the LDS transforms) and the
longer ones' plan shapes, both radix orders, both directions, FP64 and FP32,
inputs and outputs in memory and in LDS, against a long-double DFT (error over the largest
coefficient < 1e-14 FP64, < 2e-6 FP32, the register plans' bounds)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def smooth(v):
    for p in (2, 3, 5):
        while v % p == 0:
            v //= p
    return v == 1


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ absent")
def test_mixed_radix_plans_match_dft(tmp_path):
    exe = tmp_path / "fftg_emu"
    subprocess.run(["g++", "-std=c++20", "-O1", "-pthread", os.path.join(HERE, "native", "fftg_emu.cpp"),
                    "-o", str(exe)], check=True)
    ns = [n for n in range(18, 257, 2) if smooth(n)] + [300, 486, 500, 512, 640]
    r = subprocess.run([str(exe)] + [str(n) for n in ns], capture_output=True, text=True, timeout=600)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.count(" ok") == len(ns)
