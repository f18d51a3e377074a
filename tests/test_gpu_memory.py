"""Calls on a device that has room for their queues and outputs but not for the
buffers that only make them faster: they go on without those, with the same
results. Each case runs in a process of its own, in which the library's hipMalloc
is one with a limit (tests/native/alloc_limit.c), once without and once with it."""
import ctypes
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


class Limit:
    """The process's hipMalloc (only in the processes that this module starts)."""

    def __init__(self, path):
        self.lib = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
        self.lib.alloc_limit.argtypes = [ctypes.c_size_t]
        self.lib.alloc_refuse.argtypes = [ctypes.c_int, ctypes.c_size_t]

    def bytes(self, n):
        self.lib.alloc_limit(n)

    def refuse(self, sizes):
        for i, n in enumerate(sizes):
            self.lib.alloc_refuse(i, n)

    def refusals(self):
        return self.lib.alloc_refusals()


def setup(name, W, H, **options):
    from beamtrace2007_amd.gpu import GpuRenderer
    from beamtrace2007_amd.host import camera
    from conftest import load_scene
    s, _, _, sp = load_scene(name)
    r = GpuRenderer(s)
    if options:
        r.set_options(**options)
    return r, camera(sp["view"], W, H), sp


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def wave_stacks(limit):
    """The wave stacks (100 KB for each of 2048 waves) in passes of every kind."""
    W, H = 70, 45
    def run(limited):
        if limited:
            limit.bytes(100 << 20)  # the queues of this capacity and the output lists are smaller
        r, cam, sp = setup("room", W, H, capacity=65536)
        p, _ = r.primary(cam, W, H, tile=8)
        q, _ = r.point_shadows(cam, W, H, p, sp["point_light"])
        out = [p, q]
        for precision in (0, 1):
            r.set_options(precision=precision)
            g = r.soft_shadows(cam, W, H, sp["area_light"], exact=True)
            out += [g[f] for f in ("tri", "vis", "E", "Eu")]
        r.close()
        return out
    return run


def ancestor_lists(limit, name, **options):
    """Climbs by parent links: a scene without its leaves' ancestor lists (8 B per leaf and level), which its bytes
    then don't count. Images, lists and counters."""
    from conftest import load_scene
    nodes = load_scene(name)[2]["nodes"]
    depth = np.zeros(len(nodes), np.int64)
    for i in np.flatnonzero(nodes["data"] & 3 != 3):  # children follow their parent
        depth[i + 1] = depth[nodes["data"][i] >> 2] = depth[i] + 1
    size = 8 * int(depth[nodes["data"] & 3 == 3].sum())
    W, H = 75, 50
    def run(limited):
        if limited:
            limit.refuse([size])
        r, cam, sp = setup(name, W, H, **options)
        p, i = r.primary(cam, W, H, tile=16)
        q, j = r.point_shadows(cam, W, H, p, sp["point_light"])
        out, infos = [p, q], [i, j]
        for precision in (0, 1):
            r.set_options(precision=precision)
            g = r.soft_shadows(cam, W, H, sp["area_light"], exact=True)
            out += [g[f] for f in ("tri", "vis", "E", "Eu")]
            infos.append(g["info"])
        assert all(i["killed_roots"] == 0 for i in infos)
        # a float sum over waves, in whatever order they end, is the one counter that may differ
        counters = [{k: v for k, v in i["stats"].items() if k != "droppedArea"} for i in infos]
        out.append(np.array([list(c.values()) for c in counters]))
        out.append(r.scene_bytes(0) + (size if limited else 0))
        r.close()
        return out
    return run


def lists(limit, **options):
    """Canonical polygon lists where nothing can be allocated beyond what the passes hold: sorted, and with a small
    budget (roots traced again) filtered, on the host."""
    W = H = 48
    def run(limited):
        r, cam, sp = setup("plant", W, H)
        p, _ = r.primary(cam, W, H, tile=16, canonical=False)
        r.point_shadows(cam, W, H, p, sp["point_light"], canonical=False)
        if options:
            r.set_options(**options)
        if limited:
            limit.bytes(1)
        p, info = r.primary(cam, W, H, tile=16)
        q, info2 = r.point_shadows(cam, W, H, p, sp["point_light"])
        assert len(p) > 256 and len(q) > 256  # more than a block of the device's sort
        for i in (info, info2):
            assert (i["retry_passes"] > 0) == bool(options)
        r.close()
        return [p, q]
    return run


def fp64_pools(limit, gib):
    """FP64 soft shadows with room for the pools of half or a quarter of the waves that fill the device."""
    W, H = 40, 30
    def run(limited):
        if limited:
            limit.bytes(int(gib * (1 << 30)))
        r, cam, sp = setup("room", W, H, precision=2)
        g = r.soft_shadows(cam, W, H, sp["area_light"], exact=True)
        r.close()
        return [g[f] for f in ("tri", "vis", "E", "Eu")]
    return run


def fp64_lists(limit):
    """An FP64 image of more than 2^22 pixels without room for the cell lists of 2^22 (17 entries of 8 B a pixel)."""
    W = H = 2049
    def run(limited):
        if limited:
            limit.refuse([64 + (17 << 22) * 8])
        r, cam, sp = setup("room", W, H, precision=2)
        g = r.soft_shadows(cam, W, H, sp["area_light"], exact=True)
        r.close()
        return [g[f] for f in ("tri", "vis", "E", "Eu")]
    return run


CASES = {"wave_stacks": wave_stacks,
         "ancestors_atrium": lambda limit: ancestor_lists(limit, "atrium"),
         "ancestors_plant": lambda limit: ancestor_lists(limit, "plant", leaf_cap=1),
         "sorted_lists": lists,
         "filtered_lists": lambda limit: lists(limit, primary_budget=4, budget=4),
         "fp64_lists": fp64_lists, "fp64_half": lambda limit: fp64_pools(limit, 2.0),
         "fp64_quarter": lambda limit: fp64_pools(limit, 1.0)}


@pytest.mark.gpu
@pytest.mark.parametrize("case", sorted(CASES))
def test_calls_go_on_without(require_gpu, tmp_path, case):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    shim = str(tmp_path / "alloc_limit.so")
    subprocess.run([cc, "-shared", "-fPIC", "-O1", os.path.join(HERE, "native", "alloc_limit.c"), "-o", shim, "-ldl"],
                   check=True, capture_output=True, timeout=60)
    print(f"without room: {case}", flush=True)
    out = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), shim, case], capture_output=True, text=True,
                         timeout=100)
    assert out.returncode == 0, out.stdout[-2000:] + out.stderr[-2000:]
    assert out.stdout.splitlines()[-1] == "ok"


if __name__ == "__main__":
    sys.path.insert(0, HERE)
    import conftest  # noqa: F401  (the repository's root on the path)
    lim = Limit(sys.argv[1])
    run = CASES[sys.argv[2]](lim)
    want = run(False)
    assert lim.refusals() == 0
    got = run(True)
    print("allocations refused:", lim.refusals(), flush=True)
    assert lim.refusals() > 0
    assert same(want, got)
    print("ok", flush=True)
