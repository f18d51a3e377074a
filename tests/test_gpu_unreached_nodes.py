"""Kd-trees with nodes that no descent reaches: their parent links are checked
for range only, so they may name each other in a circle or a node further on.
Such scenes are accepted, trace as the same scene without those nodes, and hold
no ancestor lists for them."""
import numpy as np
import pytest

from conftest import load_scene

pytestmark = pytest.mark.gpu


class Padded:
    """A scene whose node arrays end in nodes that nothing refers to."""

    def __init__(self, scene, extra):
        self.s, k = scene, dict(scene.kd_arrays())
        n = len(k["nodes"])
        nodes = np.zeros(len(extra), k["nodes"].dtype)
        for i, (data, _) in enumerate(extra):
            nodes[i] = (0.0, data(n), 0)
        k["nodes"] = np.concatenate([k["nodes"], nodes])
        k["parent"] = np.concatenate([k["parent"], np.array([p(n) for _, p in extra], np.uint32)])
        k["nodeBox"] = np.concatenate([k["nodeBox"], np.zeros((len(extra), 6), np.float32)])
        self.k = k

    def arrays(self):
        return self.s.arrays()

    def kd_arrays(self):
        return self.k


LEAF = 3
EXTRA = {
    # two leaves and a third that name each other
    "circle": [(lambda n: LEAF, lambda n: n + 1), (lambda n: LEAF, lambda n: n + 2), (lambda n: LEAF, lambda n: n)],
    # a leaf that names itself, and one that names the last node
    "self": [(lambda n: LEAF, lambda n: n), (lambda n: LEAF, lambda n: n + 2), (lambda n: LEAF, lambda n: 0)],
    # an inner node of its own with its two leaves
    "tree": [(lambda n: (n + 2) << 2, lambda n: n), (lambda n: LEAF, lambda n: n), (lambda n: LEAF, lambda n: n)],
}


@pytest.mark.parametrize("kind", sorted(EXTRA))
def test_unreached_nodes_change_nothing(require_gpu, kind):
    from beamtrace2007_amd.gpu import GpuRenderer
    from beamtrace2007_amd.host import camera
    s, _, _, sp = load_scene("room")
    W, H = 33, 21
    cam = camera(sp["view"], W, H)
    print(f"unreached nodes: {kind}", flush=True)
    out, sizes = [], []
    for scene in (s, Padded(s, EXTRA[kind])):
        r = GpuRenderer(scene)
        try:
            p, _ = r.primary(cam, W, H, tile=8)
            g = r.soft_shadows(cam, W, H, sp["area_light"], exact=True)
            second = r.add_scene(scene)  # after another scene's nodes
            b, _ = r.soft_batch([{"scene": second, "cam": cam, "W": W, "H": H, "light": sp["area_light"]}], exact=True)
            sizes.append((r.scene_bytes(0), r.scene_bytes(second)))
        finally:
            r.close()
        out.append([p.tobytes()] + [x[f].tobytes() for x in (g, b[0]) for f in ("tri", "vis", "E", "Eu")])
    assert out[0] == out[1]
    node_bytes = 12 + 24 + 4  # node, box and parent link
    assert all(y == x + len(EXTRA[kind]) * node_bytes for x, y in zip(*sizes))
