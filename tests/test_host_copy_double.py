"""Staged host copies (csrc/host_copy.hip) on a test double of HIP whose streams run nothing
before they are waited for: what a failing call leaves behind."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hp-multiphysics_amd", "csrc")


def test_slots_of_failed_copies(tmp_path):
    exe = str(tmp_path / "cases")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{HERE}/hip_double", f"-I{CSRC}", "-o", exe,
                    f"{HERE}/hip_double/host_copy_cases.cpp", "-x", "c++", f"{CSRC}/host_copy.hip"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
