"""The tile rule of wide solves (more than 64 columns) at the matrix sizes where
it changes over: a solve without tuning against the one with the tuner's tile,
and the residual in FP64."""
import numpy as np
import pytest

import radgpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 1024, 1280, 1281, 4096, 4097, 8193])
@pytest.mark.parametrize("nrhs", [65, 128, 129, 192])
def test_rule_against_tuner(n, nrhs):
    if n > 5000 and nrhs not in (128, 192):
        pytest.skip("the narrower of each kernel at the largest size")
    print(n, nrhs, flush=True)
    rng = np.random.default_rng(n)
    k = 8
    U, W = rng.random((n, k), np.float32), rng.random((k, n), np.float32)
    F = (U / (U @ W.sum(1)).max()) @ W
    rho, E = rng.uniform(0.2, 0.7, (n, nrhs)), rng.random((n, nrhs))
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        B, _ = lin.gather(rho, E, prec="f16", tol=1e-10, max_outer=60, sweeps=6)
        lin.autotune(nrhs, "f16")
        T, _ = lin.gather(rho, E, prec="f16", tol=1e-10, max_outer=60, sweeps=6)
    FB = np.zeros_like(B)
    for i in range(0, n, 1024):
        FB[i:i + 1024] = F[i:i + 1024].astype(np.float64) @ B
    assert np.linalg.norm(E + rho * FB - B) <= 1.01e-10 * np.linalg.norm(E)
    # either is within 1e-10 / 0.3 of the solution
    assert np.linalg.norm(B - T) <= 7e-10 * np.linalg.norm(E)
