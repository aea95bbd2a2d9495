"""The kernels' divisions by multiply-adds (bgf_arith.h) on the host against the divisions themselves: every
FP32 significand for the reciprocals, random and extreme operands for the fixed divisors."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_divisions_round_as_ieee(tmp_path):
    exe = str(tmp_path / "arith")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I", os.path.join(ROOT, "bg_flood_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "arith_main.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
