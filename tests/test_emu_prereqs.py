"""The emulator builds follow every source that they are compiled from: a changed launcher or kernel
header must not leave an old library to the CPU tests."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")
CSRC = "../../opt-fft_amd/csrc"


def _prerequisites(target):
    r = subprocess.run(["make", "-C", EMU, "-pnq", target], capture_output=True, text=True, timeout=60)
    for line in r.stdout.splitlines():
        if line.startswith(target + ":") and ":=" not in line:
            return {os.path.normpath(p) for p in line.split(":", 1)[1].split()}
    raise AssertionError(r.stdout + r.stderr)


@pytest.mark.parametrize("target", ["libfft3d_emu.so", "emu_asan"])
def test_every_header_is_a_prerequisite(target):
    pre = _prerequisites(target)
    want = {f for f in os.listdir(EMU) if f.endswith(".hpp")}
    want |= {os.path.normpath(os.path.join(CSRC, f)) for f in os.listdir(os.path.join(EMU, CSRC))
             if f.endswith(".hpp")}
    assert not want - pre, sorted(want - pre)
