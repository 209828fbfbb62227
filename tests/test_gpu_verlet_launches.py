"""The resident Verlet steps from inside (tests/cpp/verlet_resident.cpp): how a
call of many steps is split over launches, complete and incomplete teams of
blocks (the resident route is the one that runs: it refuses other cloths), and
what the calls say after a wait between blocks has ended without its word."""
import os
import subprocess

import pytest

from opencloth_amd.build import LIBDIR, ROOT
from tests.helpers import say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("verlet") / "verlet_resident")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "opencloth_amd", "csrc"),
                    os.path.join(os.path.dirname(__file__), "cpp", "verlet_resident.cpp"), "-o", exe, "-L", LIBDIR,
                    "-lopencloth", "-L/opt/rocm/lib", "-lamdhip64", "-ldl", f"-Wl,-rpath,{LIBDIR}",
                    "-Wl,-rpath,/opt/rocm/lib"], check=True, capture_output=True, timeout=120)
    return exe


def run(exe, what):
    say("verlet", what)
    r = subprocess.run([exe, what], capture_output=True, text=True, timeout=60)
    say(r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
    lines = r.stdout.strip().splitlines()
    assert lines[-1] == "wrong 0"
    return lines[:-1]


def test_long_calls_are_split(exe):
    assert len(run(exe, "launches")) == 2


def test_a_lost_state_is_reported_until_it_is_replaced(exe):
    assert len(run(exe, "lost")) == 1 + 2 * 5 + 1


def test_complete_and_incomplete_teams(exe):
    lines = run(exe, "teams")
    assert len(lines) == 6 * (7 * 3 + 1)
