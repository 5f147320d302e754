"""The exact fits' workspace, shared by the meshes of a context, on the CPU
build of the library with AddressSanitizer (tests/emu/drive_workspace.py)."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "emu"))

from test_emu_cpu import _asan  # noqa: E402


@pytest.mark.skipif(_asan() is None, reason="g++ with AddressSanitizer not available")
@pytest.mark.parametrize("what", ["threads", "refused", "large"])
def test_emulated_workspace(what):
    import build as emu_build

    emu_build.build()
    env = dict(os.environ, LD_PRELOAD=_asan(), ASAN_OPTIONS="detect_leaks=0", EMU_POISON="1")
    p = subprocess.run([sys.executable, os.path.join(HERE, "emu", "drive_workspace.py"), what], env=env,
                       capture_output=True, text=True, timeout=600)
    print(p.stdout[-3000:])
    print(p.stderr[-3000:])
    assert p.returncode == 0 and "ALL PASS" in p.stdout
