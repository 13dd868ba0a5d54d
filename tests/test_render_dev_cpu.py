"""The render kernels' forms without a division, on the host: the gaussian's
divisions by constants round as the division for every significand, and the
column wrap is the remainder for every index."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_divisions_left_out(tmp_path):
    exe = str(tmp_path / "render_host")
    subprocess.run(["g++", "-std=c++17", "-O2", "-mfma", "-ffp-contract=off", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(ROOT, "tests", "render_host.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
