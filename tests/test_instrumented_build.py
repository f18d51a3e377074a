"""The instrumented build (-DBTG_PHASE_CYCLES: trace-loop clocks per region,
btg_run_info.phaseCycles) compiles: its macros add arguments and statements
that the ordinary build leaves out. No device is used."""
import os
import shutil
import subprocess

import pytest

from beamtrace2007_amd.build import DEVICE_FLAGS, HERE, HIPCC
from conftest import ROOT


@pytest.mark.skipif(not shutil.which(HIPCC) and not os.path.exists(HIPCC), reason="hipcc not available")
def test_phase_clock_build_compiles():
    flags = [f for f in DEVICE_FLAGS if f != "-shared"]
    out = subprocess.run([HIPCC, *flags, "-fsyntax-only", "-DBTG_PHASE_CYCLES", "-I", os.path.join(ROOT, "include"),
                          os.path.join(HERE, "csrc", "engine.hip")], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr[-4000:]
