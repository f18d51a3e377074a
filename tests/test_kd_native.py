"""The trace kernel's kd predicates by per-beam bounds
(beamtrace2007_amd/csrc/kd_pred.h) compiled for the host and compared with the
reference's arithmetic on random and borderline beams
(tests/native/kd_parity.cpp). No device is used."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not shutil.which(HIPCC) and not os.path.exists(HIPCC), reason="hipcc not available")
def test_kd_bounds_decide_as_the_reference_arithmetic(tmp_path):
    exe = tmp_path / "kd_parity"
    src = os.path.join(ROOT, "tests", "native", "kd_parity.cpp")
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-O2", "-ffp-contract=off",
                    "-fno-fast-math", "-Wno-unused-function", src, "-o", str(exe)], check=True,
                   capture_output=True, timeout=300)
    out = subprocess.run([str(exe), "400000"], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    word, cases, share = out.stdout.split()
    assert word == "ok" and cases == "400000"
    assert float(share) < 2e-3  # the band is 2.4e-5 of a distance wide: a few comparisons in 10^4 at most
