"""The tiled PBD solver's plan (opencloth_amd/csrc/pbd_plan.cpp) on the host:
over grids, ragged and random constraint lists a block's closure projects its
owned particles exactly as the colour-by-colour schedule does, and constraint
lists that reach too far, and positions without an order, are refused."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_closures_equal_the_colour_schedule(tmp_path):
    exe = str(tmp_path / "pbd_plan")
    csrc = os.path.join(ROOT, "opencloth_amd", "csrc")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O2", "-pthread", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I", os.path.join(ROOT, "include"), "-I", csrc,
                    os.path.join(os.path.dirname(__file__), "cpp", "pbd_plan.cpp"),
                    os.path.join(csrc, "pbd_plan.cpp"), "-o", exe], check=True, capture_output=True, timeout=240)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    lines = r.stdout.strip().splitlines()
    assert len(lines) == 6 * 4 * 3 + 6 + 6
    for line in lines:
        name, (ok, nb, wrong) = line.rsplit(" ", 3)[0], map(int, line.rsplit(" ", 3)[1:])
        assert wrong == 0 and ok == (not name.endswith("refused")) and (nb > 0) == ok, line
