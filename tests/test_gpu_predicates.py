"""Beams for which the kd predicates by per-beam bounds never decide, so that the
trace takes the reference's arithmetic at every node: a scene with a triangle
beyond the coordinates the bounds are used for, and tiles with a corner whose
direction has components of 1e-20. Beside them ordinary views. Polygons against
the oracle bit for bit, and every counter: no root of these may be abandoned."""
import numpy as np
import pytest

from conftest import load_scene
from refpy import Oracle, canon

pytestmark = pytest.mark.gpu

COUNTERS = ("kdSteps", "leafVisits", "triTests", "splits", "beams", "rootBeams", "fiveSplits", "climbs")


def wide_scene(a):
    """The scene and a triangle of 2e9 at 1.5e15 (its neighbouring floats are 1.3e8 apart)."""
    from beamtrace2007_amd.host import Scene
    far = np.full((3, 3), 1.5e15, np.float32)
    far[1, 0] += 2e9
    far[2, 1:] += 2e9
    n = len(a["pos"])
    s = Scene.from_arrays(np.concatenate([a["pos"], far]),
                          np.concatenate([a["tris"], [[n, n + 1, n + 2]]]).astype(np.uint32))
    s.build_kd(0.4)
    return s


def axis_camera(view, tiny):
    """Along the view's main axis, off it by `tiny`: where the tiles' corners meet in the middle of the image, two
    components of the direction are `tiny`, and one of them along the middle row and column."""
    eye, target = np.array(view[:3]), np.array(view[3:6])
    axis = int(np.argmax(np.abs(target - eye)))
    cam = np.zeros(14, np.float32)
    cam[0:3] = eye
    cam[3:6] = tiny
    cam[3 + axis] = np.sign(target[axis] - eye[axis])
    cam[6 + (axis + 1) % 3] = 1
    cam[9 + (axis + 2) % 3] = 1
    cam[12:14] = 0.6, 0.45
    return cam


@pytest.mark.parametrize("kind,tiny", [("wide", None), ("axis", 1e-20), ("axis", -1e-30), ("room", None),
                                       ("conference", None)])
def test_polygons_and_counters(require_gpu, kind, tiny):
    from beamtrace2007_amd.gpu import GpuRenderer, polys_to_dict
    from beamtrace2007_amd.host import camera
    s, a, _, sp = load_scene("conference" if kind == "conference" else "room")
    if kind == "wide":
        s = wide_scene(a)
    W, H = 64, 48
    cam = axis_camera(sp["view"], tiny) if kind == "axis" else camera(sp["view"], W, H)
    print(f"predicates {kind} {tiny}", flush=True)
    o = Oracle(s.arrays(), s.kd_arrays())
    r = GpuRenderer(s)
    try:
        gp, gi = r.primary(cam, W, H, tile=8)
        op = o.primary(cam, W, H, tile=8)
        gs, si = r.point_shadows(cam, W, H, gp, sp["point_light"])
        os_ = o.point(cam, W, H, op, sp["point_light"])
    finally:
        r.close()
    assert len(op["n"]) > 400 and len(os_["n"]) > 40
    for g, i, want in ((gp, gi, op), (gs, si, os_)):
        assert i["killed_roots"] == 0
        assert np.array_equal(canon(polys_to_dict(g)), canon(want))
        assert [i["stats"][c] for c in COUNTERS] == [want["stats"][c] for c in COUNTERS]
