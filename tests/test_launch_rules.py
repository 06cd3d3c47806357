"""The host's launch sizes (final184_amd/csrc/launch_rules.hpp), compiled with g++ and run on
the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_launch_rules(tmp_path):
    exe = str(tmp_path / "launch_rules_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=address,undefined",
                    os.path.join(ROOT, "tests", "cpp", "launch_rules_test.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "LAUNCH RULES OK" in out.stdout
