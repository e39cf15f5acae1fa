"""The three bf16 terms of an f32 factor, on the host: a g++ build of saragossa_amd/csrc/f32_terms.h with
tests/native/f32_terms.cpp, which bounds what the six products that the f32 chunk kernel keeps leave out."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_kept_products_are_as_exact_as_f32_ones(tmp_path):
    exe = tmp_path / "f32_terms"
    build = subprocess.run(["g++", "-std=c++17", "-O2", "-I" + os.path.join(ROOT, "saragossa_amd", "csrc"),
                            os.path.join(ROOT, "tests", "native", "f32_terms.cpp"), "-o", str(exe)],
                           capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and run.stdout.strip().endswith("ok"), run.stdout
