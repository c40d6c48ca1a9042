"""The FP64 quotients and square roots of the kernels whose starting value is the
hardware's estimate or a related reciprocal (recip, recip_near, rdivf, qsqrt_h in
cffc_amd/csrc/euler2d_state.hpp), on the host from any estimate that the
hardware may give (tests/native/recip_chain_check.cpp): equal to the IEEE operation
bit for bit."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "native", "recip_chain_check.cpp")


def test_quotients_and_roots_are_correctly_rounded(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    with open("/proc/cpuinfo") as f:
        if " fma " not in f.read():
            pytest.skip("needs a CPU with FMA")
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(
        "#include <math.h>\n#include <stdint.h>\n#define __host__\n#define __device__\n#define __constant__\n"
        "#define __forceinline__ inline\n")
    exe = str(tmp_path / "recip_chain_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-mfma", "-ffp-contract=off", "-w", "-I", str(tmp_path), "-o", exe, SRC],
                   check=True)
    r = subprocess.run([exe, "4000000"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
