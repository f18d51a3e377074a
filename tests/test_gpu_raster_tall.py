"""Rasterization around the workgroup's 256 polygons and the row count at which
a polygon goes to the launch for tall ones (32): against the host rasterizer,
bit for bit."""
import numpy as np
import pytest

from conftest import load_scene
from test_gpu_raster import host_raster, renderer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 256, 257, 2000])
@pytest.mark.parametrize("rows", [31.0, 32.0, 33.0, 300.0, 0.0])
def test_rows_and_blocks(require_gpu, n, rows):
    """rows: height of every polygon in pixels (0: all sizes mixed)."""
    from beamtrace2007_amd.gpu import POLY_DTYPE
    from beamtrace2007_amd.host import camera
    W, H = 257, 311
    sp = load_scene("room")[3]
    cam = camera(sp["view"], W, H)
    hw, hh = float(cam[12]), float(cam[13])
    g = np.random.Generator(np.random.PCG64(n * 1000 + int(rows)))
    p = np.zeros(n, POLY_DTYPE)
    h = np.full(n, rows) if rows else g.choice([0.4, 1, 3, 20, 32, 33, 100, 700], n)
    w = g.choice([0.5, 2, 9, 70, 400], n)
    cx, cy = g.uniform(-10, W + 10, n), g.uniform(-10, H + 10, n)
    four = g.random(n) < 0.6
    for k, (sx, sy) in enumerate([(-1, -1), (1, -1), (1, 1), (-1, 1)]):
        x = cx + sx * w / 2 + g.uniform(-0.2, 0.2, n) * w
        y = cy + sy * h / 2
        p["x"][:, k] = (x / W * 2 - 1) * hw
        p["y"][:, k] = (y / H * 2 - 1) * hh
    for f in ("x", "y"):
        p[f][:, 3] = np.where(four, p[f][:, 3], p[f][:, 2])
    p["n"] = np.where(four, 4, 3)
    p["tri"] = g.permutation(n).astype(np.int32) - (n > 255)  # one filtered out (tri -1)
    print(f"raster {n} polygons of {rows} rows", flush=True)
    r = renderer("room")
    for shadow in (False, True):
        want = host_raster(cam, W, H, p if shadow else p[p["tri"] >= 0], shadow)
        assert np.array_equal(r.raster(cam, W, H, p, shadow), want)
