"""Roots that a first run abandons for want of queue room (it reserves at most 128
records per root): a light behind a grid of small triangles, so that every root
holds hundreds of sub-beams at once and the queue overflows. They are traced
again with their budget reserved, which admits capacity / budget of them at
once; results against the oracle, as the other parity tests."""
import numpy as np
import pytest

from conftest import check_soft
from refpy import Oracle

pytestmark = pytest.mark.gpu

CAPACITY = 65536


def grid_scene(n: int = 16):
    from beamtrace2007_amd.host import Scene
    floor = np.array([[[-50, 0, -50], [50, 0, -50], [50, 0, 50]], [[-50, 0, -50], [50, 0, 50], [-50, 0, 50]]])
    rng = np.random.default_rng(7)
    c = (np.stack(np.meshgrid(np.arange(n), np.arange(n)), -1).reshape(-1, 2) + 0.5) / n * 4 - 2
    t = np.zeros((n * n, 3, 3))
    for k, (dx, dz) in enumerate([(-1, -0.7), (1, -0.6), (0.1, 0.9)]):
        t[:, k, 0] = c[:, 0] + 1.2 / n * dx
        t[:, k, 1] = 9.5 + 0.1 * rng.random(n * n)
        t[:, k, 2] = c[:, 1] + 1.2 / n * dz
    pos = np.concatenate([floor, t]).reshape(-1, 3).astype(np.float32)
    s = Scene.from_arrays(pos, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3))
    s.build_kd(0.4)
    return s


@pytest.mark.parametrize("budget,passes", [(1024, 1), (220, 2)])
def test_roots_without_room(require_gpu, budget, passes):
    """Budget 1024: no root goes over it, one retry holds them all. Budget 220: some do; they wait for a second
    retry with the larger budget."""
    from beamtrace2007_amd.gpu import GpuRenderer
    from beamtrace2007_amd.host import camera
    s = grid_scene()
    W = H = 32
    cam = camera(np.array([0, 5, 0.1, 0, 0, 0, 0, 0, 1, 40], np.float32), W, H)
    light = np.array([0, 10, 0, 4, 0, 0, 0, 0, 4], np.float32)
    print(f"roots without room, budget {budget}", flush=True)
    r = GpuRenderer(s)
    try:
        r.set_options(budget=budget, capacity=CAPACITY)
        g = r.soft_shadows(cam, W, H, light, exact=True)
    finally:
        r.close()
    info = g["info"]
    print({k: info[k] for k in ("rounds", "max_queue", "killed_roots", "retry_passes")}, flush=True)
    assert info["killed_roots"] > 0
    assert info["retry_passes"] == passes
    if passes == 1:
        # with 32 budgets reserved for each root, 65536 / 32768 = 2 of them would run at once, a round or more
        # for every two; 64 at once take a few chains of rounds
        assert info["rounds"] < info["killed_roots"] / 2
    check_soft(g, Oracle(s.arrays(), s.kd_arrays()).soft(cam, W, H, light, exact=True))
