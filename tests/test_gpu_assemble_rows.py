"""The assembly of cloths of up to 128 tiles (half tiles per block, sums per
row) where its blocks can go wrong: one row, a half tile alone or missing, the
largest tile count and the first beyond it; steps bit-exact against the FP32
oracle.  And a solve whose blocks could not all start, from the row sums."""
import os
import subprocess

import numpy as np
import pytest

from opencloth_amd import scenes
from opencloth_amd.build import LIBDIR, ROOT
from tests.helpers import oracle_params, say

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("nx,ny", [(3, 4), (64, 4), (64, 5), (67, 12), (130, 13), (21, 21), (512, 128), (512, 129),
                                   (3, 1024), (3, 1025)])
@pytest.mark.parametrize("warm", [True, False])
def test_steps_bitwise(nx, ny, warm):
    from oracle import Oracle
    from opencloth_amd.cloth import ImplicitCloth

    rng = np.random.default_rng(nx * 1000 + ny)
    X0 = scenes.grid_positions(nx, ny, 4.0, 0.0)
    X = (X0 + 2e-3 * rng.standard_normal(X0.shape)).astype(np.float32)
    V = (0.1 * rng.standard_normal(X0.shape)).astype(np.float32)
    pins = (rng.random(nx * ny) < 0.05).astype(np.uint8)
    p = scenes.StepParams(cg_max_iters=20, cg_tol=1e-4, cg_tol_mode=scenes.TOL_RELATIVE, warm_start=warm)
    sp = scenes.grid_springs(nx, ny, X0)
    say("assemble rows", nx, ny, warm)
    cl = ImplicitCloth(nx, ny, X, sp, pins, p, V)
    cl.step(3)
    Xr, Vr = Oracle(32).system(nx * ny, sp, pins).rollout(X, V, oracle_params(p, nx, ny), 3)[:2]
    Xg, Vg = cl.get_state()
    assert np.array_equal(bits(Xg), bits(Xr)) and np.array_equal(bits(Vg), bits(Vr))


@pytest.mark.parametrize("nx,ny,its,tol", [(200, 100, 15, 2), (200, 100, 40, 1), (512, 128, 6, 2)])
def test_partial_team(tmp_path, nx, ny, its, tol):
    exe = str(tmp_path / "resident_team_rows")
    cpp = os.path.join(os.path.dirname(__file__), "cpp")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "opencloth_amd", "csrc"), "-I", cpp,
                    os.path.join(cpp, "resident_team_rows.cpp"), "-o", exe, "-L", LIBDIR,
                    "-lopencloth", "-L/opt/rocm/lib", "-lamdhip64", f"-Wl,-rpath,{LIBDIR}", "-Wl,-rpath,/opt/rocm/lib"],
                   check=True, capture_output=True, timeout=120)
    say("resident team from rows", nx, ny, its, tol)
    r = subprocess.run([exe, str(nx), str(ny), str(its), str(tol)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    lines = r.stdout.strip().splitlines()
    assert len(lines) == 4
    for line in lines:
        it0, st0, it, st = (int(t) for t in line.split(":")[1].split()[:4])
        assert line.endswith("same 1") and (it, st) == (it0, st0), line
