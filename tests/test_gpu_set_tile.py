"""Tiles of the low-precision sweep that a program sets itself: every one of
the documented ones, and what the tuner answers, at the sizes where a chunk of
the split holds the fewest k-blocks; the solves' residual in FP64."""
import numpy as np
import pytest

import radgpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [200, 1000, 1024, 4000])
@pytest.mark.parametrize("nrhs", [1, 20, 64, 100, 192])
@pytest.mark.parametrize("prec", ["f16", "bf16"])
def test_every_tile_is_taken_and_solves(n, nrhs, prec):
    print(n, nrhs, prec, flush=True)
    rng = np.random.default_rng(n + nrhs)
    F = rng.random((n, n), np.float32) * np.float32(1.8 / n)  # rows sum to about 0.9
    F64 = F.astype(np.float64)
    rho, E = rng.uniform(0.2, 0.7, (n, nrhs)), rng.random((n, nrhs))
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        tiles = [(rt, sk) for rt in (1, 2, 4) for sk in (1, 2, 4, 8)]
        tuned = lin.autotune(nrhs, prec)
        assert tuned in tiles
        for rt, sk in tiles + [tuned]:
            lin.set_tile(nrhs, prec, rt, sk)
            B, info = lin.gather(rho, E, prec=prec, tol=1e-9, max_outer=40, sweeps=5)
            r = E + rho * (F64 @ B) - B
            # the solver's own residual and this one differ by rounding in float64 only
            assert np.linalg.norm(r) <= 1e-9 * np.linalg.norm(E) + 1e-12 * np.linalg.norm(B), (rt, sk)
        for bad in ((3, 1), (1, 3), (8, 1), (1, 16), (0, 0)):
            with pytest.raises(radgpu.RadError):
                lin.set_tile(nrhs, prec, *bad)


@pytest.mark.parametrize("nrhs", [65, 129])
def test_rule_with_a_partly_filled_last_column_tile(nrhs):
    n = 8193
    print(n, nrhs, flush=True)
    rng = np.random.default_rng(n)
    k = 8
    U, W = rng.random((n, k), np.float32), rng.random((k, n), np.float32)
    F = (U / (U @ W.sum(1)).max()) @ W
    rho, E = rng.uniform(0.2, 0.7, (n, nrhs)), rng.random((n, nrhs))
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        B, _ = lin.gather(rho, E, prec="f16", tol=1e-10, max_outer=60, sweeps=6)
    FB = np.concatenate([F[i:i + 1024].astype(np.float64) @ B for i in range(0, n, 1024)])
    assert np.linalg.norm(E + rho * FB - B) <= 1.01e-10 * np.linalg.norm(E)
