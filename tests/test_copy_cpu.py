"""Context::copy on the host, over a stand-in for the runtime (copy_host.cpp):
sizes around the pieces and the rule's limit, without pinned memory to have,
and from and to memory that the caller has pinned itself."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copy(tmp_path):
    exe = str(tmp_path / "copy_host")
    subprocess.run(["g++", "-std=c++17", "-O2", "-w", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "copy_host.cpp"),
                    os.path.join(ROOT, "blacktracer_amd", "csrc", "copy.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
