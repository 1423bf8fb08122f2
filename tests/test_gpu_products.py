"""The device products of the explicit-matrix solvers at the edges of their
tiles and dispatch rules, against plain float64."""
import numpy as np
import pytest

import radgpu

pytestmark = pytest.mark.gpu
U64 = 2.0 ** -53


# rows per block 8, 16 or 32 (one rule on the padded size): one patch, around
# 256 rows, four waves per row group (up to 8192 and 9216), one (8192), two
# (12288)
@pytest.mark.parametrize("n", [1, 255, 257, 7900, 8001, 9000, 12100])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 4])
def test_f64_product_few_columns(n, nrhs):
    rng = np.random.default_rng(n + nrhs)
    F = rng.random((n, n), np.float32)
    X = rng.standard_normal((n, nrhs))
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        Y = lin.multiply(X, "f32")
    F64 = F.astype(np.float64)
    # any order of summation stays within (n + 1) u of the sum of magnitudes; the reference's own order likewise
    assert (np.abs(Y - F64 @ X) <= 2 * (n + 1) * U64 * (F64 @ np.abs(X))).all()
