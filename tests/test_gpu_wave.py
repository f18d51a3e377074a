"""The fused trace-and-split kernel at the sizes where its dealing, stacks and
rounds change: a single root, fewer roots than waves, one heavy root whose
sub-beams spread over many waves and rounds, more roots than the device has
lanes (rounds of separate launches first), and queues so small that roots find
no room and are traced again. Against the oracle, bit for bit, as the other
parity tests."""
import numpy as np
import pytest

from conftest import check_soft, load_scene
from refpy import Oracle, canon

pytestmark = pytest.mark.gpu

COUNTERS = ("kdSteps", "leafVisits", "triTests", "splits", "beams", "fiveSplits", "climbs")


@pytest.mark.parametrize("name,W,H,tile", [("analytic", 1, 1, 8), ("room", 8, 8, 8), ("room", 65, 63, 8),
                                           ("atrium", 64, 64, 64), ("analytic", 520, 513, 1)])
def test_primary_and_point_polygons(require_gpu, name, W, H, tile):
    from beamtrace2007_amd.gpu import GpuRenderer, polys_to_dict
    from beamtrace2007_amd.host import camera
    s, a, k, sp = load_scene(name)
    cam = camera(sp["view"], W, H)
    print(f"{name} {W}x{H} tile {tile}", flush=True)
    r, o = GpuRenderer(s), Oracle(a, k)
    try:
        gp, info = r.primary(cam, W, H, tile=tile)
        op = o.primary(cam, W, H, tile=tile)
        assert np.array_equal(canon(polys_to_dict(gp)), canon(op))
        if info["killed_roots"] == 0:
            assert [info["stats"][c] for c in COUNTERS] == [op["stats"][c] for c in COUNTERS]
        gs, _ = r.point_shadows(cam, W, H, gp, sp["point_light"])
        assert np.array_equal(canon(polys_to_dict(gs)), canon(o.point(cam, W, H, op, sp["point_light"])))
    finally:
        r.close()


@pytest.mark.parametrize("name,W,H,opts", [("plant", 1, 1, {}), ("room", 9, 7, {}), ("plant", 24, 24, {"capacity": 1024}),
                                           ("plant", 40, 24, {"budget": 64, "capacity": 2048}),
                                           ("analytic", 520, 513, {})])
def test_soft_shadows(require_gpu, name, W, H, opts):
    from beamtrace2007_amd.gpu import GpuRenderer
    from beamtrace2007_amd.host import camera
    s, a, k, sp = load_scene(name)
    cam = camera(sp["view"], W, H)
    print(f"soft {name} {W}x{H} {opts}", flush=True)
    r = GpuRenderer(s)
    try:
        r.set_options(**opts)
        g = r.soft_shadows(cam, W, H, sp["area_light"], exact=True)
    finally:
        r.close()
    check_soft(g, Oracle(a, k).soft(cam, W, H, sp["area_light"], exact=True))
