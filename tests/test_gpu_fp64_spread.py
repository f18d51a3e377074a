"""FP64 cells where the number of lanes that work in each wave changes: an image
of one pixel, of fewer pixels than waves, of a few lanes per wave, each alone
and in one batch that has more pixels than the device has lanes. Results are
per-pixel fixed-point sums, so they agree bit for bit."""
import numpy as np
import pytest

from conftest import load_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,sizes", [("room", [(1, 1), (9, 7), (33, 31), (64, 65), (288, 256)]),
                                        ("plant", [(1, 1), (7, 9), (24, 24)])])
def test_images_alone_and_in_a_batch(require_gpu, name, sizes):
    from beamtrace2007_amd.gpu import GpuRenderer
    from beamtrace2007_amd.host import camera, camera_d
    s, _, _, sp = load_scene(name)
    jobs = [{"scene": 0, "cam": camera(sp["view"], W, H), "cam_d": camera_d(sp["view"], W, H), "W": W, "H": H,
             "light": sp["area_light"]} for W, H in sizes]
    r = GpuRenderer(s)
    try:
        r.set_options(precision=2)
        print(f"FP64 {name} {sizes}", flush=True)
        batch, _ = r.soft_batch(jobs, exact=True)
        for j, b in zip(jobs, batch):
            a = r.soft_shadows(j["cam"], j["W"], j["H"], j["light"], exact=True, cam_d=j["cam_d"])
            for f in ("tri", "vis", "E", "Eu"):
                assert np.array_equal(a[f], b[f]), (j["W"], j["H"], f)
    finally:
        r.close()
