"""Calls on one handle from several threads at once (a ctypes call lets go of the
interpreter lock): each one's answer is the one it has alone.  Column and ray
counts differ, so that buffers kept between calls are shared and outgrown."""
import threading

import numpy as np
import pytest

import radgpu
from radgpu import scenes

pytestmark = pytest.mark.gpu


def _at_once(jobs, rounds):
    """Runs the jobs in a thread each, rounds times; their answers' first
    difference from what they give alone, or None."""
    alone = [job() for job in jobs]
    gate, wrong = threading.Barrier(len(jobs)), []

    def work(k):
        gate.wait(60)
        for _ in range(rounds):
            if not all(np.array_equal(a, b) for a, b in zip(jobs[k](), alone[k])):
                wrong.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join(100)
        assert not t.is_alive()
    return wrong


def test_solves_on_one_system():
    n = 1500
    rng = np.random.default_rng(5)
    F = rng.random((n, n), np.float32) * np.float32(1.8 / n)

    def data(nrhs):
        return rng.uniform(0.2, 0.7, (n, nrhs)), rng.random((n, nrhs))

    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        (r1, e1), (r3, e3), (r40, e40) = data(1), data(3), data(40)
        jobs = [lambda: (lin.gather(r3, e3, tol=1e-9, max_outer=30, sweeps=5)[0],),
                lambda: (lin.gather(r40, e40, tol=1e-9, max_outer=30, sweeps=5)[0],),
                lambda: lin.adjoint(r1, e1, e1, tol=1e-9, max_outer=30, sweeps=5)[:2],
                lambda: (lin.multiply(e40, "f32"),),
                lambda: (lin.multiply(e3, "bf16"),),
                lambda: (lin.shoot(r3, e3, max_shots=200)[0],)]
        assert _at_once(jobs, 20) == []


def test_casts_on_one_engine():
    with radgpu.Engine("-triangle", "20000", "-quiet", "1") as eng:
        eng.set_scene(scenes.room_scene(1)).prepare_host().upload()
        rec, _ = eng.records()
        rng = np.random.default_rng(7)
        live = np.nonzero(rec["parent"] >= 0)[0]

        def rays(n):
            r = np.zeros(n, radgpu.RAY_DTYPE)
            i, j = rng.choice(live, n), rng.choice(live, n)
            r["p"] = rec["p"][i, rng.integers(0, 3, n)]
            r["v"] = rec["c"][j] - r["p"]
            r["ban"] = rec["parent"][i]
            return r

        jobs = [lambda r=rays(n): eng.cast(r) for n in (100, 3000, 40000, 90000)]
        jobs.append(lambda r=rays(5000): eng.cast_static(r))
        assert _at_once(jobs, 20) == []
