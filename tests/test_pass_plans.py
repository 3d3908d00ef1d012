"""The planner of D2Q9 passes, compiled for the host (no GPU): run lengths and
tiles (tests/native/pass_plans.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_splits_and_tiles(tmp_path):
    exe = str(tmp_path / "pass_plans")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-fsanitize=undefined",
                        "-fno-sanitize-recover=all", "-o", exe, os.path.join(HERE, "native", "pass_plans.cpp")],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "pass plans: ok" in r.stdout, r.stdout + r.stderr[-3000:]
