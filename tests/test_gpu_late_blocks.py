"""The resident solve on a GPU that others use too: blocks that start after its
roll was closed take part (same bits as a complete team, in a fraction of the
time of the one block there was), and handles that step on streams of their
own give the bits that they give alone."""
import os
import subprocess

import numpy as np
import pytest

from opencloth_amd import scenes
from opencloth_amd.build import LIBDIR, ROOT
from tests.helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,its,tol", [(512, 512, 30, 2), (512, 300, 60, 1), (256, 250, 60, 2)])
def test_late_blocks_take_part(tmp_path, nx, ny, its, tol):
    exe = str(tmp_path / "late_blocks")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "opencloth_amd", "csrc"),
                    os.path.join(os.path.dirname(__file__), "cpp", "late_blocks.cpp"), "-o", exe, "-L", LIBDIR,
                    "-lopencloth", "-L/opt/rocm/lib", "-lamdhip64", f"-Wl,-rpath,{LIBDIR}", "-Wl,-rpath,/opt/rocm/lib"],
                   check=True, capture_output=True, timeout=120)
    say("late blocks", nx, ny, its, tol)
    r = subprocess.run([exe, str(nx), str(ny), str(its), str(tol)], capture_output=True, text=True, timeout=60)
    say(r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
    lines = r.stdout.strip().splitlines()
    assert len(lines) == 2
    us = []
    for line in lines:
        f = line.split(":")[1].split()
        assert f[0:2] == f[2:4] and f[5] == "1", line
        us.append(float(f[7]))
    if tol == 2:  # (a solve that converges is over before they come, or soon after)
        assert us[1] < us[0] / 2, lines


def test_handles_on_streams_of_their_own():
    from opencloth_amd.cloth import ImplicitCloth
    from opencloth_amd.hiptime import Stream, device_synchronize

    say("three handles, three streams")
    rng = np.random.default_rng(5)
    scene = []
    for nx, ny, its in ((512, 512, 12), (449, 289, 20), (130, 70, 40)):
        X0 = scenes.grid_positions(nx, ny, 4.0, 0.0)
        X = (X0 + 1e-4 * rng.standard_normal(X0.shape)).astype(np.float32)
        pins = np.zeros(nx * ny, np.uint8)
        pins[:nx] = 1
        scene.append((nx, ny, X, scenes.grid_springs(nx, ny, X0), pins,
                      scenes.StepParams(dt=1.0 / 120.0, cg_max_iters=its, cg_tol=0.0, cg_tol_mode=scenes.TOL_NONE)))
    alone, together = [], []
    for sc in scene:
        cl = ImplicitCloth(*sc)
        cl.step(24)
        alone.append(cl.get_state())
        cl.close()
    streams = [Stream() for _ in scene]
    handles = [ImplicitCloth(*sc) for sc in scene]
    device_synchronize()
    for cl, st in zip(handles, streams):
        cl.set_stream(st.handle)
    for _ in range(12):
        for cl in handles:
            cl.step(2)
    for cl in handles:
        together.append(cl.get_state())
        assert cl.sticky_status() == 0
    device_synchronize()
    for cl in handles:
        cl.close()
    for a, b in zip(alone, together):
        assert all(np.array_equal(p.view(np.uint32), q.view(np.uint32)) for p, q in zip(a, b))
