"""The kernels that one lambda evaluation launches, per precision and patch
size, on the CPU (tests/launch_probe.cpp stands in for the launches): rows of
the patches are formed by k_rows in FP32 alone, where a buffer for them is
there."""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_DIR = os.path.join(os.path.dirname(HERE), "pgure-svt_amd", "pguresvt")
ROCM = "/opt/rocm"


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists(os.path.join(LIB_DIR, "libpgsvt.so")):
        pytest.skip("no g++ or no built library")
    exe = str(tmp_path_factory.mktemp("probe") / "launch_probe")
    cmd = ["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + ROCM + "/include",
           os.path.join(HERE, "launch_probe.cpp"), "-o", exe, "-L" + LIB_DIR, "-lpgsvt", "-L" + ROCM + "/lib",
           "-lamdhip64", "-Wl,-rpath," + LIB_DIR + ":" + ROCM + "/lib"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    return [l.split() for l in r.stdout.splitlines()]


@pytest.mark.parametrize("bits", [32, 64])
def test_rows_are_formed_in_fp32_alone(lines, bits):
    seen = 0
    for patch, frames, b, rows, status, *kernels in lines:
        if int(b) != bits:
            continue
        seen += 1
        case = (patch, frames, b, rows, status, kernels)
        formed = [k for k in kernels if "k_rows" in k]
        if bits == 64:
            assert not formed, case
            # patches above 4 x 4 write their rows in k_eval
            want = "k_round_prep" if int(patch) <= 4 else "k_eval"
            assert len(kernels) == 1 and want in kernels[0] and status == "0", case
        elif rows == "1":
            assert len(formed) == 1 and len(kernels) == 2 and status == "0", case
        else:  # nowhere to put the rows: refused, not written to a null address
            assert not formed and status != "0", case
    assert seen == 12
