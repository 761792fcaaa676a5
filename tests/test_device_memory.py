"""The engine's device memory, on the CPU: the library's objects linked with
stand-ins for the HIP calls that count allocations on a device of a chosen size
and run no kernel (tests/cpp/device_memory.cpp).  cf_aad_footprint bounds what a
call takes; a call that needs what earlier ones keep gets it; a call whose
larger choice does not fit takes the smaller one; tables whose upload failed are
uploaded again; and itemized risk shares its sweeps by what they cost."""
import json
import os
import shutil
import subprocess

import pytest

from compfinance_amd import build as _build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "compfinance_amd", "_build")
FP64, FP32, CHECKPOINT, RECOMPUTE = 0, 1, 0, 1


@pytest.fixture(scope="module")
def device(tmp_path_factory):
    objs = [os.path.join(BUILD, name + ".o") for _, name, _ in _build.SOURCES]
    if not all(os.path.exists(o) for o in objs) or not shutil.which("g++"):
        pytest.skip("library objects not built (python -m compfinance_amd.build)")
    tmp = tmp_path_factory.mktemp("device_memory")
    src, obj, exe = os.path.join(ROOT, "tests", "cpp", "device_memory.cpp"), str(tmp / "main.o"), str(tmp / "main")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-c", src, "-o", obj],
                   check=True)
    subprocess.run(["g++", "-o", exe, obj] + objs + ["-lpthread"], check=True)

    def run(*args):
        out = subprocess.run([exe] + [str(a) for a in args], capture_output=True, text=True, timeout=120, check=True)
        return json.loads(out.stdout)

    return run


@pytest.mark.parametrize("paths", [4096, (1 << 18) + 1, 1 << 20, 5 << 20])
@pytest.mark.parametrize("mode", [CHECKPOINT, RECOMPUTE])
@pytest.mark.parametrize("precision", [FP64, FP32])
def test_footprint_bounds_the_call(device, precision, mode, paths):
    """To the rounding of each buffer to 256 bytes, and the sums that the
    synchronous calls keep in host memory."""
    r = device("footprint", precision, mode, paths)
    assert r["rc"] == 0 and r["used"] > 0
    assert r["used"] <= r["footprint"] <= r["used"] + (1 << 20)


def test_several_slots_only_beside_the_other_buffers(device):
    r = device("tight", FP64, CHECKPOINT, (1 << 24) + 1)
    assert r["rc"] == 0 and r["launches"] > 0, r


def test_one_slot_when_the_device_is_fuller_than_it_says(device):
    r = device("short")
    assert r["rc"] == 0 and r["launches"] > 0, r


@pytest.mark.parametrize("scenario", [("held", FP32, CHECKPOINT, 1 << 25), ("server",), ("itemized",),
                                      ("itemized", FP64, CHECKPOINT, 1 << 22), ("points",)])
def test_kept_buffers_are_given_back(device, scenario):
    r = device(*scenario)
    assert r["rc0"] == 0 and r["rc"] >= 0, r
    assert r["used"] < r["before"]


def test_itemized_falls_back(device):
    r = device("itemized_short")
    assert r["rc"] == 1 + 30 * 36 and r["launches"] > 0, r


@pytest.mark.parametrize("calls,paths,shared", [(2, 1 << 14, True), (3, 1 << 14, True), (3, 1 << 20, False),
                                                (4, 1 << 20, True)])
def test_few_calls_on_many_paths_are_swept_by_the_payoff(device, calls, paths, shared):
    """A forward and its sums, then a sweep and its sums by the payoff, or the
    four kernels of the shared sweeps."""
    r = device("itemized_calls", FP64, CHECKPOINT, paths, calls)
    assert r["rc"] > 0 and r["launches"] == (6 if shared else 2 + 2 * calls), r


@pytest.mark.parametrize("failing", [1, 2])
def test_a_failed_upload_is_done_again(device, failing):
    """An itemized call uploads two tables, those of the plan and its own."""
    r = device("upload", FP64, CHECKPOINT, 4096, failing)
    assert r["rc0"] < 0 and r["rc"] > 0, r
    assert r["before"] == failing                      # (the first call ended at the failing upload)
    assert r["uploads"] - r["before"] == 3 - failing   # the second did it again, and those after it
