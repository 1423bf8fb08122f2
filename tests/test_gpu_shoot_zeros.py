"""Radiosities that start as -0 (a negative -light times a component of 0): the
first received +0 makes them +0, whether the vertex sees the source or not; the
whole TriStore against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle_lib as ol
import radgpu
from radgpu import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [300, 2121, 8193])
@pytest.mark.parametrize("emission,opts", [
    ((255, -300, 0), ["-converge", "60"]),  # (-255, 300, -0): shot as any light
    ((255, 0, 0), ["-converge", "-1000000"]),  # (-255, -0, -0): shot under a negative threshold
], ids=["two", "one"])
@pytest.mark.parametrize("more", [[], ["-select", "low", "-fma", "0"], ["-graph", "1"], ["-parallel_src", "3"]],
                         ids=lambda o: "".join(o[:2]) or "plain")
def test_negative_zero_emission(n, emission, opts, more):
    if "low" in more and "60" not in opts:
        pytest.skip("the reference's MaxDeltaRad takes no source of negative energy")
    sc = scenes.patch_room(3, n)
    brgb = np.zeros_like(sc.brgb)
    brgb[::7] = emission
    sc = scenes.Scene(sc.p, sc.frgb, brgb)
    opts = ["-triangle", str(n), "-quiet", "1", "-light", "-1"] + opts + more
    print(n, opts, flush=True)
    with radgpu.Engine(*opts) as eng:
        eng.set_scene(sc).prepare_host().upload()
        before = eng.records()[0]["accB"]
        assert (np.signbit(before) & (before == 0)).any()
        got = [eng.shoot(k)[0] for k in (1, 2, 8)]
        rec, _ = eng.records()
    o = ol.Oracle(*((opts[:-2] if "-graph" in opts else opts) + ["-jobs", "16"]))
    o.load(sc)
    o.build_tree()
    o.init_radiosity()
    o.prepartition()
    o.iterate(11)
    orec, _ = o.dump()
    assert got == [1, 2, 8]
    assert np.array_equal(np.signbit(rec["accB"]), np.signbit(orec["accB"]))
    assert rec.tobytes() == orec.tobytes()
