"""Primary rays where their stack of pending kd-tree children leaves LDS (more
than 12 entries): triangles whose sizes and distances to a corner span eight
octaves, seen from that corner, so that the tree is a deep chain along the
rays. At partial tiles and at one pixel; against the oracle, as the other
parity tests."""
import numpy as np
import pytest

from conftest import check_soft
from refpy import Oracle

IN_LDS = 12


def corner_scene(n=2000, octaves=8):
    from beamtrace2007_amd.host import Scene
    rng = np.random.default_rng(3)
    r = 8 * 2.0 ** (-octaves * rng.random((n, 1, 1)))
    pos = np.abs(r * rng.random((n, 1, 3)) + r * rng.normal(0, 0.06, (n, 3, 3)))
    s = Scene.from_arrays(pos.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(n, 3))
    s.build_kd(0.4)
    return s


def corner_camera(W, H):
    from beamtrace2007_amd.host import camera
    return camera(np.array([-0.03, -0.02, -0.025, 4, 4, 4, 0, 1, 0, 60], np.float32), W, H)


def most_pending(kd, o, d):
    """The most far children that a ray through the tree holds at once, hits aside."""
    split, data = kd["nodes"]["split"], kd["nodes"]["data"]
    with np.errstate(divide="ignore"):
        ends = np.sort(np.stack([(kd["bounds"][:3] - o) / d, (kd["bounds"][3:] - o) / d]), axis=0)
    node, t0, t1 = 0, max(0.0, ends[0].max()), ends[1].min()
    if t0 > t1:
        return 0
    stack, most = [], 0
    while True:
        while data[node] & 3 != 3:
            a, s, far = int(data[node] & 3), float(split[node]), int(data[node] >> 2)
            first, second = (node + 1, far) if o[a] < s else (far, node + 1)
            tp = (s - o[a]) / d[a]
            node = first
            if 0 < tp <= t1:
                if tp < t0:
                    node = second
                else:
                    stack.append((second, tp, t1))
                    t1 = tp
        most = max(most, len(stack))
        if not stack:
            return most
        node, t0, t1 = stack.pop()


def test_the_corner_scene_needs_the_deep_entries():
    kd, cam = corner_scene().kd_arrays(), corner_camera(33, 19).astype(np.float64)
    rays = [(cam[3:6] + cam[6:9] * ((2 * (x + 0.5) / 33 - 1) * cam[12]) + cam[9:12] * ((2 * (y + 0.5) / 19 - 1) * cam[13]))
            for y in range(19) for x in range(33)]
    assert sum(most_pending(kd, cam[:3], d) > IN_LDS for d in rays) >= 8


@pytest.mark.gpu
@pytest.mark.parametrize("W,H", [(33, 19), (1, 1), (16, 16), (130, 67)])
def test_deep_ray_stacks(require_gpu, W, H):
    from beamtrace2007_amd.gpu import GpuRenderer
    s, cam = corner_scene(), corner_camera(W, H)
    light = np.array([3, 9, 3, 1, 0, 0, 0, 0, 1], np.float32)
    print(f"rays {W}x{H}", flush=True)
    r = GpuRenderer(s)
    try:
        g = r.soft_shadows(cam, W, H, light, exact=True)
    finally:
        r.close()
    check_soft(g, Oracle(s.arrays(), s.kd_arrays()).soft(cam, W, H, light, exact=True))
