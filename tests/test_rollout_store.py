"""The rollout store (opencloth_amd/csrc/rollout_store.cpp) on the host, over a
stand-in for the HIP runtime: the two layouts, an arena that changes from one
to the other, and allocations that fail."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_layouts_and_failures(tmp_path):
    exe = str(tmp_path / "rollout_store")
    csrc = os.path.join(ROOT, "opencloth_amd", "csrc")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I", os.path.join(ROOT, "include"), "-I", csrc,
                    os.path.join(os.path.dirname(__file__), "cpp", "rollout_store.cpp"),
                    os.path.join(csrc, "rollout_store.cpp"), "-o", exe], check=True, capture_output=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert len(r.stdout.strip().splitlines()) == 9 * 7 + 7 + 1
