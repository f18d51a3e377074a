"""Canonical polygon lists are sorted on the device: the same polygons as the
device's own order gives, in the reference's order (triangle, corner count,
corners, area), at lengths around the sort's blocks of 256 and runs."""
import numpy as np
import pytest

from conftest import load_scene

pytestmark = pytest.mark.gpu


def key(p):
    k = [int(p["tri"]), int(p["n"])]
    for i in range(int(p["n"])):
        k += [float(p["x"][i]), float(p["y"][i])]
    return tuple(k + [float(p["area"])])


@pytest.mark.parametrize("name,W,H,tile", [("analytic", 1, 1, 8), ("analytic", 16, 16, 1), ("analytic", 32, 8, 1),
                                           ("analytic", 33, 8, 1), ("room", 32, 32, 2), ("plant", 64, 48, 8),
                                           ("atrium", 96, 64, 16)])
def test_canonical_lists_are_in_order(require_gpu, name, W, H, tile):
    from beamtrace2007_amd.gpu import GpuRenderer
    from beamtrace2007_amd.host import camera
    s, a, k, sp = load_scene(name)
    cam = camera(sp["view"], W, H)
    r = GpuRenderer(s)
    try:
        ordered, _ = r.primary(cam, W, H, tile=tile, canonical=True)
        as_is, _ = r.primary(cam, W, H, tile=tile, canonical=False)
        shadow, _ = r.point_shadows(cam, W, H, as_is, sp["point_light"], canonical=True)
        shadow_as_is, _ = r.point_shadows(cam, W, H, ordered, sp["point_light"], canonical=False)
    finally:
        r.close()
    print(f"{name} {W}x{H} tile {tile}: {len(ordered)} and {len(shadow)} polygons", flush=True)
    for x, y in ((ordered, as_is), (shadow, shadow_as_is)):
        assert len(x) == len(y)
        keys = [key(p) for p in x]
        assert keys == sorted(keys)
        assert sorted(p.tobytes() for p in x) == sorted(p.tobytes() for p in y)
