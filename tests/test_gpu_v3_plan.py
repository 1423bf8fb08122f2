"""-variant v3 with the samples of a pass drawn ahead and its splits written
together, against the oracle's ordered walk: the whole TriStore bit for bit,
and with it the position in rand()'s sequence, where the plan reaches its
edges: samples that depart early and often, more samples than are drawn ahead
(one receiver's, or a pass's), a pool that fills within a pass, receivers split
without a sample, no sample at all, 0 and 1 passes of few shots."""
import numpy as np
import pytest

import oracle_lib as ol
import radgpu
from radgpu import scenes

pytestmark = pytest.mark.gpu

CASES = {
    "coarse": (1.25, ["-delta_ff", "5e-6"], 12),
    "departures": (1.25, ["-delta_ff", "1e-3", "-sample_area", "0.05"], 12),
    "departures_late": (1.05, ["-delta_ff", "3e-3", "-sample_area", "0.004"], 6),
    "one_sample": (1.25, ["-delta_ff", "1e-3", "-sample_area", "0.6"], 12),
    "no_sample": (1.25, ["-delta_ff", "1e-3", "-sample_area", "2"], 12),
    "groups": (1.25, ["-delta_ff", "1", "-sample_area", "0.03"], 4),  # 16 to 33 points each
    "past_the_plan": (1.25, ["-delta_ff", "1", "-sample_area", "0.0007"], 2),  # a pass's
    "one_past_the_plan": (1.25, ["-delta_ff", "1e-2", "-sample_area", "0.00004", "-adapt_area", "0.78"], 1),  # a receiver's
    "past_and_departures": (1.25, ["-delta_ff", "2e-3", "-sample_area", "0.0005"], 2),
}


def _solve(name, extra=()):
    cell, opts, shots = CASES[name]
    opts = ["-variant", "v3", "-adapt_area", "0.5", "-converge", "300", "-quiet", "1"] + opts + list(extra)
    if "-triangle" not in extra:
        opts += ["-triangle", "50000"]
    sc = scenes.v3_room(4, cell)
    print(name, extra, sc.n, flush=True)
    with radgpu.Engine(*opts) as eng:
        eng.set_scene(sc).prepare_host().upload()
        n0 = len(eng.records()[0])
        got = sum(eng.shoot(k)[0] for k in (1, shots))
        rec, _ = eng.records()
    o = ol.Oracle(*(opts + ["-jobs", "1"]))
    o.load(sc)
    o.build_tree()
    o.init_radiosity()
    o.prepartition()
    o.iterate(1 + shots)
    orec, _ = o.dump()
    return got, 1 + shots, n0, rec, orec


@pytest.mark.parametrize("fma", ["1", "0"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_planned_passes_equal_the_ordered_walk(name, fma):
    got, want, n0, rec, orec = _solve(name, ("-fma", fma))
    print(name, "slots", n0, "->", len(rec), flush=True)
    assert got == want
    assert len(rec) == len(orec) and rec.tobytes() == orec.tobytes()


@pytest.mark.parametrize("spare", [0, 3, 4, 5, 6, 7, 8, 9, 10, 11, 40])
def test_pool_fills_within_a_pass(spare):
    with radgpu.Engine("-quiet", "1", "-adapt_area", "0.5", "-triangle", "50000") as eng:
        n0 = len(eng.set_scene(scenes.v3_room(4, 1.25)).prepare_host().upload().records()[0])
    for name in ("coarse", "departures"):
        got, want, _, rec, orec = _solve(name, ("-triangle", str(n0 + spare)))
        assert got == want
        assert len(rec) == len(orec) and rec.tobytes() == orec.tobytes()
