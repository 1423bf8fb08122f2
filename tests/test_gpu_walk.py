"""The ray walk of small launches (eight lanes a ray, one axis of the step per
lane, the next leaf read ahead) against the walk of large ones (two lanes a
ray): the same rays alone and repeated into a large batch, with equal hits and
equal cell and test counts."""
import numpy as np
import pytest

import radgpu
from edge_scenes import edge_scenes
from radgpu import scenes

pytestmark = pytest.mark.gpu


def _scene(kind):
    if kind in ("room", "hall"):
        return scenes.room_scene(3) if kind == "room" else scenes.hall_scene(2, n_boxes=12, box_h=3.5, wall_h=14.0)
    if kind in ("far", "turned"):  # coordinates that round; no wall along an axis
        sc = scenes.patch_room(4, 700)
        p = sc.p.astype(np.float64)
        if kind == "turned":
            c, s = np.cos(0.4), np.sin(0.4)
            p = p @ np.array([[c, s, 0], [-s, c, 0], [0, 0, 1]]) @ np.array([[1, 0, 0], [0, c, s], [0, -s, c]])
        else:
            p = p * 0.7 + [10000.3, -777.7, 0.1]
        return scenes.Scene(p.astype(np.float32), sc.frgb, sc.brgb)
    return edge_scenes()[kind]


@pytest.mark.parametrize("n", [1, 7, 3000])
@pytest.mark.parametrize("fma", ["1", "0"])
@pytest.mark.parametrize("kind", ["room", "hall", "far", "turned", "room_zero_area"])
def test_few_rays_equal_many(kind, fma, n):
    print(kind, fma, n, flush=True)
    with radgpu.Engine("-triangle", "20000", "-quiet", "1", "-fma", fma) as eng:
        eng.set_scene(_scene(kind)).prepare_host().upload()
        rec, g = eng.records()
        rng = np.random.default_rng(17)
        live = np.nonzero(rec["parent"] >= 0)[0]
        rays = np.zeros(n, radgpu.RAY_DTYPE)
        i, j = rng.choice(live, n), rng.choice(live, n)
        rays["p"] = rec["p"][i, rng.integers(0, 3, n)]
        rays["v"] = rec["c"][j] - rays["p"]
        rays["ban"] = rec["parent"][i]
        k = np.arange(n) % 8
        mid = (g[:3] + (g[3:] - g[:3]) * rng.random((n, 3))).astype(np.float32)
        d = rng.normal(size=(n, 3)).astype(np.float32)
        rays["p"][k >= 3], rays["v"][k >= 3] = mid[k >= 3], d[k >= 3]  # inside, anywhere
        rays["ban"][k >= 3] = -1
        rays["v"][k == 4, 2] = 0  # along planes and along an axis
        rays["v"][k == 5, 1:] = 0
        rays["v"][k == 6, 1] *= np.float32(1e-7)  # too slow along an axis to step there
        rays["p"][k == 7] = g[3:] + np.float32(1)  # outside
        few = eng.cast(rays)
        many = eng.cast(np.tile(rays, 400000 // n + 1))
    for a, b in zip(few, many):
        assert np.array_equal(np.tile(a, 400000 // n + 1), b)
