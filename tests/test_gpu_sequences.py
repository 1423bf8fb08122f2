"""Calls on one engine that follow each other where a later one meets what an
earlier one left (slots, grids and buffers made for another size), and the
matrix of scenes at the edge of what its index is made for."""
import numpy as np
import pytest

import oracle_lib as ol
import radgpu
from radgpu import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fma", ["1", "0"])
@pytest.mark.parametrize("pieces", [(2,), (1, 3)])
def test_matrix_after_splits(pieces, fma):
    """-variant v3 adds slots to a scene that the upload had whole: the matrix
    of all of them (300 rows), which entries are open and their values, against a test of every
    original."""
    opts = ["-variant", "v3", "-adapt_area", "0.5", "-converge", "300", "-delta_ff", "5e-6", "-quiet", "1", "-fma", fma,
            "-triangle", "50000"]
    sc = scenes.v3_room(4, 1.05)
    with radgpu.Engine(*opts) as eng:
        eng.set_scene(sc).prepare_host().upload()
        n0 = len(eng.records()[0])
        assert n0 == sc.n
        with radgpu.LinearSystem(n0) as lin:
            lin.from_scene(eng)
        o = ol.Oracle(*(opts + ["-jobs", "16"]))
        o.load(sc)
        o.build_tree()
        o.init_radiosity()
        o.prepartition()
        n = n0
        for k in pieces:
            assert eng.shoot(k)[0] == k
            rec, _ = eng.records()
            o.iterate(k)
            assert rec.tobytes() == o.dump()[0].tobytes()
            assert len(rec) > n
            n = len(rec)
            print(fma, pieces, n0, "->", n, flush=True)
            with radgpu.LinearSystem(n) as lin:
                lin.from_scene(eng)
                F = lin.matrix()
            rows = np.sort(np.random.default_rng(n).choice(n, 300, replace=False))
            pairs = np.stack([np.repeat(rows, n), np.tile(np.arange(n), len(rows))], axis=1).astype(np.int32)
            want = o.ff_centroid(pairs, ol.VIS_BRUTE).reshape(len(rows), n)
            F = F[rows]
            assert np.array_equal(F != 0, want != 0)
            s = want.astype(np.float64).sum(axis=1)
            scaled = want.astype(np.float64) / np.maximum(s, 1.0)[:, None]
            # a row's scale and its product are rounded once each
            assert np.all(np.abs(F - scaled) <= 3 * 2.0 ** -24 * np.abs(scaled))
    with radgpu.Engine(*opts) as eng:  # first asked for after the splits: refused, as ever
        eng.set_scene(sc).prepare_host().upload()
        eng.shoot(pieces[0])
        n = len(eng.records()[0])
        with radgpu.LinearSystem(n) as lin, pytest.raises(radgpu.RadError, match="did not split"):
            lin.from_scene(eng)


@pytest.mark.parametrize("n", [2000, 8192])
@pytest.mark.parametrize("vis", ["segment", "reference"])
def test_matrix_between_shots(n, vis):
    """A matrix asked for between two runs of shots, whose replayed graph names
    the engine's buffers: the same records as without it, and the counters of
    both; a second upload counts from zero."""
    sc = scenes.patch_room(3, n)

    def counts(opts, shots, matrices):
        with radgpu.Engine("-triangle", str(n), "-quiet", "1", "-converge", "60", *opts) as eng, radgpu.LinearSystem(n) as lin:
            eng.set_scene(sc).prepare_host().upload()
            for k in range(2):
                if shots:
                    assert eng.shoot(16)[0] == 16
                for _ in range(matrices[k]):
                    lin.from_scene(eng, vis)
            c, rec = eng.counters(), eng.records()[0].tobytes()
            eng.upload()
            assert not any(eng.counters().values())
        return c, rec

    plain, want = counts((), True, (0, 0))
    only, _ = counts((), False, (1, 1))
    assert plain["rays"] > 0 and only["rays"] > 0
    for opts in ((), ("-graph", "1")):
        print(n, vis, opts, flush=True)
        both, rec = counts(opts, True, (1, 1))
        assert rec == want
        assert all(both[k] == plain[k] + only[k] for k in both)


@pytest.mark.parametrize("off", [1e4, 1e6])
def test_matrix_far_from_the_origin(off):
    """Coordinates that round by a cell of the segment grid or more: which
    entries are open, against a test of every original."""
    sc = scenes.patch_room(5, 700)
    p = (sc.p.astype(np.float64) + [off, -off / 3, 0.1]).astype(np.float32)
    opts = ["-triangle", str(sc.n), "-quiet", "1"]
    sc = scenes.Scene(p, sc.frgb, sc.brgb)
    with radgpu.Engine(*opts) as eng, radgpu.LinearSystem(sc.n) as lin:
        eng.set_scene(sc).prepare_host().upload()
        lin.from_scene(eng)
        F = lin.matrix()
    o = ol.Oracle(*(opts + ["-jobs", "16"]))
    o.load(sc)
    o.build_tree()
    o.init_radiosity()
    o.prepartition()
    i, j = np.meshgrid(np.arange(sc.n), np.arange(sc.n), indexing="ij")
    want = o.ff_centroid(np.stack([i.ravel(), j.ravel()], axis=1).astype(np.int32), ol.VIS_BRUTE)
    assert np.array_equal(F != 0, want.reshape(sc.n, sc.n) != 0)
