"""Segment visibility of the explicit matrix (the grid of segindex.h, the walls
left out of it, the walk in Z-order) against a test of every original: the
whole matrix, bit for bit, on scenes that take each rule to its edge."""
import numpy as np
import pytest

import oracle_lib as ol
import radgpu
from radgpu import scenes

pytestmark = pytest.mark.gpu


def _rotate(sc, angles):
    R = np.eye(3)
    for k, t in enumerate(angles):
        c, s = np.cos(t), np.sin(t)
        M = np.eye(3)
        i, j = (k + 1) % 3, (k + 2) % 3
        M[i, i], M[i, j], M[j, i], M[j, j] = c, -s, s, c
        R = M @ R
    return (sc.p.astype(np.float64) @ R.T).astype(np.float32)


def _scene(kind):
    if kind.startswith("room"):
        # walls left out; 64 to 8 rows of a tile per block
        return scenes.patch_room(3, int(kind[4:]))
    if kind == "moved":  # coordinates whose thirds and differences round
        sc = scenes.patch_room(4, 500)
        return scenes.Scene((sc.p * np.float32(0.7) + np.float32([1000.3, -77.7, 0.1])).astype(np.float32), sc.frgb, sc.brgb)
    if kind == "rotated":  # no triangle is left out
        sc = scenes.patch_room(5, 500)
        return scenes.Scene(_rotate(sc, (0.3, 0.5, 0.7)), sc.frgb, sc.brgb)
    if kind == "turned":  # walls along one axis only
        sc = scenes.patch_room(6, 500)
        return scenes.Scene(_rotate(sc, (0.0, 0.0, 0.4)), sc.frgb, sc.brgb)
    if kind == "hall":  # yawed boxes, most segments blocked
        return scenes.hall_scene(2, n_boxes=12, box_h=3.5, wall_h=14.0)
    if kind == "slivers":  # no cull radius
        sc = scenes.patch_room(7, 400)
        p = sc.p.copy()
        inner = np.abs(p - p.mean(axis=(0, 1))).max(axis=(1, 2)) < 4
        p[inner, 2] = p[inner, 0] + (p[inner, 1] - p[inner, 0]) * np.float32(0.5) + np.float32(1e-3)
        return scenes.Scene(p, sc.frgb, sc.brgb)
    if kind == "plane":  # one flat sheet: every triangle on the least and the greatest coordinate
        sc = scenes.patch_room(8, 600)
        k = (sc.p[:, :, 2] == 0).all(axis=1)
        return scenes.Scene(sc.p[k], sc.frgb[k], sc.brgb[k])
    raise KeyError(kind)


@pytest.mark.parametrize("kind", ["room64", "room200", "room700", "moved", "rotated", "turned", "hall", "slivers", "plane"])
@pytest.mark.parametrize("fma", ["1", "0"])
def test_matrix_equals_test_of_every_original(kind, fma):
    sc = _scene(kind)
    n = sc.n
    opts = ["-triangle", str(n), "-quiet", "1", "-fma", fma]
    print(kind, n, flush=True)
    with radgpu.Engine(*opts) as eng, radgpu.LinearSystem(n) as lin:
        eng.set_scene(sc).prepare_host().upload()
        lin.from_scene(eng)
        F = lin.matrix()
        rays = eng.counters()["rays"]
    o = ol.Oracle(*(opts + ["-jobs", "16"]))
    o.load(sc)
    o.build_tree()
    o.init_radiosity()
    o.prepartition()
    i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    pairs = np.stack([i.ravel(), j.ravel()], axis=1).astype(np.int32)
    want = o.ff_centroid(pairs, ol.VIS_BRUTE).reshape(n, n)
    open_ = o.ff_centroid(pairs, ol.VIS_NONE).reshape(n, n)
    # rows are scaled where their double sum exceeds 1: compare which entries
    # are non-zero, and their values up to that scale (two roundings)
    assert np.array_equal(F != 0, want != 0)
    s = want.astype(np.float64).sum(axis=1)
    scaled = want.astype(np.float64) / np.maximum(s, 1.0)[:, None]
    assert np.all(np.abs(F - scaled) <= 3 * 2.0 ** -24 * np.abs(scaled))
    assert rays * 2 >= int((open_ != 0).sum())
