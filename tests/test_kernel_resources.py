"""What the exact fits of the device-counted lists compile to for gfx950
(csrc/k_exact.hip, k_exact_fit): sets of up to 96 rows at two waves per SIMD
without scratch, for expanded sets and for refits.  At one wave per SIMD the
fits of an undistorted box's grown sets take 1.7 times as long."""
import os
import re
import shutil
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "core_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def _resources(source, kernel):
    """[{mangled name, VGPRs, ScratchSize, Occupancy}] of a source's kernels."""
    p = subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-device-only", "-O3", "-std=c++17",
                        "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-c",
                        os.path.join(SRC, source), "-o", os.devnull, "-Rpass-analysis=kernel-resource-usage"],
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-3000:]
    out = []
    for part in p.stderr.split("Function Name: ")[1:]:
        if kernel in part.split()[0]:
            num = lambda what: int(re.search(what + r"[^:]*: (\d+)", part).group(1))
            out.append({"name": part.split()[0], "scratch": num("ScratchSize"), "waves": num("Occupancy")})
    return out


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_grown_sets_two_waves():
    fits = _resources("k_exact.hip", "k_exact_fit")
    assert fits and all(f["scratch"] == 0 for f in fits), fits
    for mode in ("ILi10ELi1E", "ILi10ELi2E", "ILi4ELi1E", "ILi4ELi2E"):  # terms; expanded sets, refits
        assert any(f["waves"] >= 2 for f in fits if mode in f["name"]), (mode, fits)
