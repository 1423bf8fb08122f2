"""The element-wise kernels of the gathering solves at the line between one and
eight rows per thread (2^19 elements, rows that are no multiple of eight), and
the low-precision copy of a matrix whose largest entry is where the scan for it
could miss it, against FP64 on the CPU.  The solves stop at a relative residual
of 1e-10 with reflectances up to 0.7, so the result is within 1e-10 / 0.3."""
import numpy as np
import pytest

import radgpu

pytestmark = pytest.mark.gpu


def _fixed_point(A, b, steps=90):  # b + A x: 0.7^90 is below 2e-14
    x = b.copy()
    for _ in range(steps):
        x = b + A(x)
    return x


@pytest.mark.parametrize("n,nrhs", [(2730, 192), (2731, 192), (5462, 96), (5465, 96), (10923, 48)])
def test_line_between_one_and_eight_rows(n, nrhs):
    print(n, nrhs, n * nrhs >= 1 << 19, flush=True)
    rng = np.random.default_rng(n)
    k = 24  # a low-rank matrix: the reference costs n k per product
    U, W = rng.random((n, k)), rng.random((k, n))
    scale = 1.0 / (U @ W.sum(1)).max()
    F = ((U * scale) @ W).astype(np.float32)
    F64 = F.astype(np.float64)
    rho, E = rng.uniform(0.2, 0.7, (n, nrhs)), rng.random((n, nrhs))
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        for prec in ("f16", "bf16"):
            B, info = lin.gather(rho, E, prec=prec, tol=1e-10, max_outer=60, sweeps=6)
            r = E + rho * (F64 @ B) - B
            assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(E)


@pytest.mark.parametrize("n", [1, 3, 100, 700, 1500])
@pytest.mark.parametrize("where", ["first", "last", "middle", "all"])
def test_largest_entry_sets_the_scale(n, where):
    rng = np.random.default_rng(n)
    F = (rng.random((n, n)) * (1e-5 / n)).astype(np.float32)
    i, j = {"first": (0, 0), "last": (n - 1, n - 1), "middle": (n // 2, n // 3), "all": (0, 0)}[where]
    F[i, j] = 0.9
    if where == "all":
        F[:] = 0.9 / n
    rho, E = rng.uniform(0.2, 0.7, (n, 3)), rng.random((n, 3))
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        B, _ = lin.gather(rho, E, prec="f16", tol=1e-10, max_outer=60, sweeps=6)
    ref = _fixed_point(lambda x: rho * (F.astype(np.float64) @ x), E)
    assert np.abs(B - ref).max() <= 4e-10 * np.abs(ref).max() * np.sqrt(n * 3)
