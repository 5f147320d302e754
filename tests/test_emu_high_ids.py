"""Patch ids of 2^30 and more in the expansion queue (the meshes accepted have
up to 2^31 - 1 patches), on the CPU build of the kernels: tests/emu/high_ids.cpp."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "emu"))

from test_emu_cpu import _asan  # noqa: E402


@pytest.mark.skipif(_asan() is None, reason="g++ with AddressSanitizer not available")
def test_patch_id_of_31_bits(tmp_path):
    import build as emu_build

    lib = emu_build.build()
    out = os.path.dirname(lib)
    exe = str(tmp_path / "high_ids")
    subprocess.check_call(emu_build.CXX + ["-I", os.path.join(HERE, "emu", "include"), "-I", os.path.join(out, "src"),
                                           "-I", os.path.join(emu_build.ROOT, "include"),
                                           os.path.join(HERE, "emu", "high_ids.cpp"), lib, "-Wl,-rpath," + out, "-o", exe])
    p = subprocess.run([exe], env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0", EMU_POISON="1"),
                       capture_output=True, text=True, timeout=120)
    print(p.stdout, p.stderr[-3000:])
    assert p.returncode == 0 and "PASS" in p.stdout
