"""CPU check of the nested-dissection plan.

nd_plan.h: tests/nd_plan_check.cpp executes the tree with dense complex<double>
fronts, following the gather semantics of the device kernels, on random complex
symmetric periodic 5-point operators (16 grids: square, ragged, elongated along
either side, as small as 4 x 4).  Dissection is a direct method, so the solve
must reach a relative residual below 1e-10; a dropped, doubled or misplaced
coupling fails by orders of magnitude."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_nd_plan_is_a_direct_solver(tmp_path):
    exe = tmp_path / "nd_plan_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "fdfd.jl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "nd_plan_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    lines = out.stdout.strip().splitlines()
    assert len(lines) == 16
    assert out.returncode == 0, "\n".join(l for l in lines if "FAIL" in l)
