"""The bookkeeping of the chunk calls' device scratch, on the host: a g++ build of saragossa_amd/csrc/scratch.h with
tests/native/scratch.cpp under AddressSanitizer + UBSan, over a device that only counts."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_what_a_captured_launch_holds_stays(tmp_path):
    exe = tmp_path / "scratch"
    build = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wextra", "-Werror", "-fsanitize=address,undefined",
                            "-fno-sanitize-recover=undefined", "-I" + os.path.join(ROOT, "saragossa_amd", "csrc"),
                            os.path.join(ROOT, "tests", "native", "scratch.cpp"), "-o", str(exe)],
                           capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and run.stdout.strip().endswith("ok"), (run.stdout, run.stderr[-2000:])
