"""FP64 images of more pixels than are traced together (2^22): the same bits
wherever the boundary between two parts falls, in scenes whose roots all fit the
first level and in one whose cells go through all three (atrium)."""
import numpy as np
import pytest

from conftest import load_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,W,H,first", [("room", 2048, 2048, 1), ("analytic", 2049, 2051, 33),
                                            ("room", 3001, 3000, 800), ("atrium", 2049, 2049, 40)])
def test_parts_of_a_large_image(require_gpu, name, W, H, first):
    """The image alone, and after another image of first x first pixels that moves the boundary."""
    from beamtrace2007_amd.gpu import GpuRenderer
    from beamtrace2007_amd.host import camera, camera_d
    s, _, _, sp = load_scene(name)
    jobs = [{"scene": 0, "cam": camera(sp["view"], w, h), "cam_d": camera_d(sp["view"], w, h), "W": w, "H": h,
             "light": sp["area_light"]} for w, h in ((first, first), (W, H))]
    r = GpuRenderer(s)
    try:
        r.set_options(precision=2)
        print(f"FP64 parts {name} {W}x{H} after {first}x{first}", flush=True)
        both, _ = r.soft_batch(jobs, exact=True)
        alone, _ = r.soft_batch(jobs[1:], exact=True)
        small, _ = r.soft_batch(jobs[:1], exact=True)
    finally:
        r.close()
    for a, b in ((both[1], alone[0]), (both[0], small[0])):
        for f in ("tri", "vis", "E", "Eu"):
            assert np.array_equal(a[f], b[f]), f
    # every part is traced: the lit share of the last rows is that of the rows above them
    lit = (alone[0]["vis"] > 0).mean(axis=1)
    assert lit[-1] > 0.5 * lit[-40]
