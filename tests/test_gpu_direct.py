"""Arrays that kernels read and write in pinned memory themselves against the
copies larger ones take, around the sizes where the calls change over (768 KB,
and 1 MB for a call's arrays together)."""
import numpy as np
import pytest

import radgpu
from radgpu import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def room():
    with radgpu.Engine("-triangle", "20000", "-quiet", "1") as eng:
        eng.set_scene(scenes.room_scene(1)).prepare_host().upload()
        rec, _ = eng.records()
        rng = np.random.default_rng(3)
        live = np.nonzero(rec["parent"] >= 0)[0]
        n = 60000
        rays = np.zeros(n, radgpu.RAY_DTYPE)
        i, j = rng.choice(live, n), rng.choice(live, n)
        rays["p"] = rec["p"][i, rng.integers(0, 3, n)]
        rays["v"] = rec["c"][j] - rays["p"]
        rays["ban"] = rec["parent"][i]
        yield eng, rays, eng.cast(rays)


@pytest.mark.parametrize("n", [1, 63, 1000, 23700, 23831, 23832, 24576, 24577, 40000])
@pytest.mark.parametrize("static", [False, True])
def test_casts_of_every_size_agree(room, n, static):
    eng, rays, ref = room
    if static and n > radgpu.CAST_STATIC_MAX:
        pytest.skip("more than a static cast takes")
    print(n, static, flush=True)
    for first in (0, 60000 - n):
        got = (eng.cast_static if static else eng.cast)(rays[first:first + n])
        for a, b in zip(got, ref):
            assert np.array_equal(a, b[first:first + n])


@pytest.mark.parametrize("n,nrhs", [(1024, 48), (1025, 48), (2048, 64), (2049, 64), (300, 3)])
def test_solves_around_the_line(n, nrhs):
    """The residual in FP64 of a solve to 1e-10 (its last place is the norm's)."""
    print(n, nrhs, flush=True)
    rng = np.random.default_rng(n)
    F = (rng.random((n, n)) / n).astype(np.float32)
    F64 = F.astype(np.float64)
    rho, E = rng.uniform(0.2, 0.7, (n, nrhs)), rng.random((n, nrhs))
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        for _ in range(2):  # the second one over the first one's buffers
            B, _ = lin.gather(rho, E, prec="f16", tol=1e-10, max_outer=60, sweeps=6)
            assert np.linalg.norm(E + rho * (F64 @ B) - B) <= 1.01e-10 * np.linalg.norm(E)
        if nrhs == 3:
            dE, drho, _ = lin.adjoint(rho, B, E, tol=1e-10, max_outer=60, sweeps=6)
            assert np.linalg.norm(E + F64.T @ (rho * dE) - dE) <= 1.01e-10 * np.linalg.norm(E)
            assert np.abs(drho - dE * (F64 @ B)).max() <= 1e-12 * np.abs(drho).max()


@pytest.mark.parametrize("n,nrhs", [(300, 3), (900, 48), (1000, 48), (1024, 48), (1025, 48), (1400, 48)])
def test_reference_copied_beside_direct_inputs(n, nrhs):
    """A solve's B does not depend on the values it is compared with, whose copy
    shares the pinned memory with inputs that no kernel has read yet."""
    print(n, nrhs, flush=True)
    rng = np.random.default_rng(n)
    F = (rng.random((n, n)) / n).astype(np.float32)
    rho, E = rng.uniform(0.2, 0.7, (n, nrhs)), rng.random((n, nrhs))
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        B, _ = lin.gather(rho, E, prec="f16", tol=1e-10, max_outer=60, sweeps=6)
        C, info = lin.gather(rho, E, prec="f16", tol=1e-10, max_outer=60, sweeps=6, Bref=B, target=1e-6)
    assert np.array_equal(B, C) and info["err"] == 0.0
