"""The persistent minimizer's host side on the CPU (tests/cpp/team_plan_check.cpp): team sizes on devices
and partitions with fewer CUs, a batch's plan, and the room for teams that wait for each other."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_team_plan(tmp_path):
    exe = str(tmp_path / "team_plan_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-pthread", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "team_plan_check.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
