"""The rules of the create-time races (opt-fft_amd/csrc/race.hpp) on the CPU, over a simulated
clock: a kernel whose first launches are late is not dropped for it, near-ties go to the earlier
one, a kernel that fails to launch ends nothing, and a mixed plan's race costs what it did with
fewer presets."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_race_rules(tmp_path):
    exe = tmp_path / "race_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "opt-fft_amd", "csrc"),
                    "-o", str(exe), os.path.join(ROOT, "tests", "race", "race_check.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.split()[-1] == "OK", r.stdout + r.stderr
