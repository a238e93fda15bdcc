"""The choice of a token's experts (csrc/pm355_route.h), its own source compiled for the CPU (route_host.cpp)."""
import os
import shutil
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_experts_of_a_token(tmp_path):
    """1 .. 100 experts, with and without groups: ties, scores that underflow, and rows with NaN, infinities, or nothing but them - the experts named are always experts there are"""
    shutil.copy(os.path.join(HERE, "..", "prima_cpp_amd", "csrc", "pm355_route.h"), tmp_path)
    (tmp_path / "pm355_dense.h").write_text("")            # (what the header includes is the device's; the program defines what is used of it)
    exe = str(tmp_path / "route")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", str(tmp_path), os.path.join(HERE, "route_host.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
