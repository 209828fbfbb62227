"""Device and pinned memory that cannot be had, and the two layouts of a
rollout's states: handles go on without it where they can, with the same bits,
and a call that fails leaves no error for the next one."""
import os
import subprocess

import pytest

from opencloth_amd.build import LIBDIR, ROOT
from tests.helpers import say

pytestmark = pytest.mark.gpu


def test_layouts_and_failed_allocations(tmp_path):
    exe = str(tmp_path / "failed_alloc")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), os.path.join(os.path.dirname(__file__), "cpp", "failed_alloc.cpp"),
                    "-o", exe, "-L", LIBDIR, "-lopencloth", "-L/opt/rocm/lib", "-lamdhip64", "-ldl",
                    f"-Wl,-rpath,{LIBDIR}", "-Wl,-rpath,/opt/rocm/lib"], check=True, capture_output=True, timeout=120)
    say("failed allocations")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    say(r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip().endswith("wrong 0") and len(r.stdout.strip().splitlines()) == 2 * (5 * 3 + 4 + 1) + 4 + 1
