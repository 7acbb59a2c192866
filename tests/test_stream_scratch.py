"""Ordering of the flash key-split scratch, on the CPU: tests/cpp/test_stream_scratch.cpp compiled with
the pool's source and stand-ins for the HIP calls."""

import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(REPO, "scicompute-attention_amd", "src")


def test_stream_scratch_orders_every_use_of_a_buffer(tmp_path):
    exe = str(tmp_path / "stream_scratch")
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-I" + os.path.join(REPO, "include"), "-I" + SRC,
                    os.path.join(REPO, "tests", "cpp", "test_stream_scratch.cpp"),
                    os.path.join(SRC, "runtime", "scratch_pool.cpp"),
                    os.path.join(SRC, "api", "status.cpp"), "-o", exe, "-pthread"], check=True)
    proc = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    print(proc.stdout)
    assert proc.returncode == 0, proc.stdout + proc.stderr
