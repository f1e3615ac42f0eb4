"""The order of training samples on the CPU: tests/sample_order_check.cpp compares
it with its definition and checks that its table stays within 2 MB, however many
samples there are."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_sample_order_and_its_memory(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "sample_order_check")
    src = os.path.join(HERE, "sample_order_check.cpp")
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", src, "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "wrong 0 table_bytes 2097152", r.stdout
