"""Rasterization where its split of the work changes: lists from one polygon to
the lengths at which a workgroup takes 8, 16 and 256 of them, spans around the
widths from which eight lanes and the whole wave write them, polygons around the row count that
sends them to the second launch, and so many of those that they are cut into
fewer slices. Against the host rasterizer, bit for bit."""
import numpy as np
import pytest

from conftest import load_scene
from test_gpu_raster import host_raster, renderer

pytestmark = pytest.mark.gpu


def boxes(cam, W, H, n, rows, width, seed):
    """n quads of about rows x width pixels (0: all sizes mixed), some over the image's edges."""
    from beamtrace2007_amd.gpu import POLY_DTYPE
    hw, hh = float(cam[12]), float(cam[13])
    g = np.random.Generator(np.random.PCG64(seed))
    h = np.full(n, float(rows)) if rows else g.choice([0.5, 1, 5, 31, 32, 33, 64, 65, 200], n)
    w = np.full(n, float(width)) if width else g.choice([0.5, 1, 3, 4, 5, 6, 15, 16, 17, 31, 32, 33, 64, 65, 200], n)
    cx, cy = g.uniform(-5, W + 5, n), g.uniform(-5, H + 5, n)
    p = np.zeros(n, POLY_DTYPE)
    for k, (sx, sy) in enumerate([(-1, -1), (1, -1), (1, 1), (-1, 1)]):
        x = cx + sx * w / 2 + g.uniform(-0.1, 0.1, n) * w
        y = cy + sy * h / 2
        p["x"][:, k] = (x / W * 2 - 1) * hw
        p["y"][:, k] = (y / H * 2 - 1) * hh
    p["n"] = 4
    p["tri"] = g.permutation(n)
    return p


@pytest.mark.parametrize("n,rows,width", [(1, 0, 0), (7, 30, 90), (8, 0, 0), (9, 0, 0), (255, 32, 4), (1000, 33, 5),
                                          (8192, 3, 6), (8193, 0, 0), (16500, 0, 3), (70000, 2, 5), (3000, 40, 1),
                                          (6000, 70, 2), (9000, 65, 9),
                                          (500, 8, 16), (500, 8, 32)])
def test_lists_rows_and_widths(require_gpu, n, rows, width):
    from beamtrace2007_amd.host import camera
    W, H = 301, 259
    cam = camera(load_scene("room")[3]["view"], W, H)
    p = boxes(cam, W, H, n, rows, width, n + rows + width)
    print(f"raster {n} polygons of {rows} x {width}", flush=True)
    r = renderer("room")
    for shadow in (False, True):
        assert np.array_equal(r.raster(cam, W, H, p, shadow), host_raster(cam, W, H, p, shadow))
