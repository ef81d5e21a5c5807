"""The backend's host side on the CPU: backend.cpp compiled over a stand-in for
the HIP runtime whose streams run as late as the calls allow
(host_backend/hip/hip_runtime.h) and kernels that only move rows. Each scenario
is one process, under AddressSanitizer and UBSan."""

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HERE = ROOT / "tests" / "host_backend"
CSRC = ROOT / "plamo-3-translate.c_amd" / "csrc"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ is not available")


@pytest.fixture(scope="module")
def host_backend(tmp_path_factory):
    out = tmp_path_factory.mktemp("host_backend")
    flags = ["-g", "-O1", "-w", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
             "-D__HIP_PLATFORM_AMD__"]
    parts = ["hooks", "checkpoint", "synthetic"]
    lines = [["gcc", "-std=c11", *flags, "-I/opt/rocm/include", "-c", str(CSRC / f"{p}.c"), "-o",
              str(out / f"{p}.o")] for p in parts]
    exe = out / "host_backend"
    lines.append(["g++", "-std=c++17", *flags, f"-I{HERE}", "-o", str(exe),
                  str(HERE / "host_backend.cpp"), *[str(out / f"{p}.o") for p in parts],
                  "-lpthread", "-lm"])
    for line in lines:
        r = subprocess.run(line, capture_output=True, text=True, timeout=300)
        if r.returncode and "sanitizer" in r.stderr.lower():
            pytest.skip("the host compiler has no sanitizer runtime")
        assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("scenario", [
    # A step on full windows after the host edited them: the rows it moves are
    # still being uploaded.
    "edited_window", "edited_window_pageable",
    # Every launch of such a step failing in turn.
    "failed_launch", "failed_launch_pageable",
    # A single full window among layers whose windows are not full.
    "lone_window",
    # An allocation that fits only without the prompts' weight fragments.
    "fragments_make_room",
])
def test_host_side(host_backend, scenario):
    r = subprocess.run([str(host_backend), scenario], capture_output=True, text=True, timeout=120,
                       env={"ASAN_OPTIONS": "detect_leaks=1"})
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr[-3000:]
