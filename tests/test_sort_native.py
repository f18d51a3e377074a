"""The canonical list's sort (beamtrace2007_amd/csrc/poly_order.h) compiled for
the host: lists with NaN and infinite corners, zeros of both signs and equal
polygons keep every polygon once, in order (tests/native/sort_parity.cpp). No
device is used."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not shutil.which(HIPCC) and not os.path.exists(HIPCC), reason="hipcc not available")
def test_every_place_of_a_canonical_list_is_taken_once(tmp_path):
    exe = tmp_path / "sort_parity"
    src = os.path.join(ROOT, "tests", "native", "sort_parity.cpp")
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-O2", "-ffp-contract=off",
                    "-fno-fast-math", "-Wno-unused-function", "-I", os.path.join(ROOT, "include"), src, "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe), "2000"], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok 2000")
