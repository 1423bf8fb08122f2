"""One source per iteration on scenes whose rays all fit the machine at once
(selection, form factors and rays in one launch, the next key beside the last):
against the oracle up to the last scene of that kind (8192 slots) and the first
past it, with calls of odd and even length, replayed graphs and a threshold
that keeps shot sources candidates."""
import numpy as np
import pytest

import oracle_lib as ol
import radgpu
from radgpu import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 2121, 8192, 8193])
@pytest.mark.parametrize("opts", [["-select", "high"], ["-select", "low", "-fma", "0"], ["-converge", "-1"],
                                  ["-graph", "1"], ["-parallel_src", "3"]], ids=lambda o: "".join(o[:2]))
def test_iterations_match_oracle(n, opts):
    sc = scenes.patch_room(3, n)
    brgb = np.zeros_like(sc.brgb)
    brgb[::37] = (255, 180, 90)
    sc = scenes.Scene(sc.p, sc.frgb, brgb)
    opts = ["-triangle", str(n), "-quiet", "1", "-converge", "60"] + opts
    pieces = [1, 2, 1, 16, 9] if "-graph" in opts else [1, 2, 1, 5, 2]
    print(n, opts, flush=True)
    with radgpu.Engine(*opts) as eng:
        eng.set_scene(sc).prepare_host().upload()
        got = [eng.shoot(k)[0] for k in pieces]
        rec, _ = eng.records()
    o = ol.Oracle(*((opts[:-2] if "-graph" in opts else opts) + ["-jobs", "16"]))
    o.load(sc)
    o.build_tree()
    o.init_radiosity()
    o.prepartition()
    o.iterate(sum(pieces))
    orec, _ = o.dump()
    assert len(rec) == n and got == pieces
    assert rec.tobytes() == orec.tobytes()
