"""What the FULL kernels alone use, checked on the CPU: their knot search by one
entry a bucket against upper_bound (interp.h:40), in FP32 through the offset
formed from the float's bits, and the shared-memory regions of the Black-Scholes
barrier's rows and of the split Sobol table."""
import json
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_full_layout(tmp_path):
    exe = str(tmp_path / "full_layout_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    os.path.join(ROOT, "tests", "cpp", "full_layout_check.cpp"), "-o", exe], check=True)
    out = json.loads(subprocess.run([exe], capture_output=True, text=True, check=True).stdout)
    assert out["grids"] > 500 and out["probes"] > 1_000_000, out
    assert out["wrong"] == 0 and out["outside"] == 0, out
    assert out["regions"] > 200 and out["bad"] == 0, out
