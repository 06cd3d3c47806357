"""The policy for scratch that a call can do without (final184_amd/csrc/scratch.hpp), compiled
with g++ and run on the host: growth, limit, refused sizes, and no block freed too early."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_scratch_policy(tmp_path):
    exe = str(tmp_path / "scratch_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=address,undefined",
                    os.path.join(ROOT, "tests", "cpp", "scratch_test.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "SCRATCH OK" in out.stdout
