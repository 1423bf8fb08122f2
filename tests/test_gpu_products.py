"""The device products of the explicit-matrix solvers at the edges of their
tiles and dispatch rules, against plain float64."""
import os
import sys

import numpy as np
import pytest

import radgpu

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import linear as lo  # noqa: E402

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


# sweeps at the edges of the tile rule (16, 32, 64 and 128 or 32 rows a block:
# padded sizes up to 4096, 8192, 16384, beyond) and ragged ends; the solution
# satisfies the system in float64
@pytest.mark.parametrize("n,nrhs", [(1, 1), (17, 3), (256, 16), (4096, 3), (4097, 17), (8193, 3), (8193, 33), (16500, 1),
                                    (16500, 17)])
@pytest.mark.parametrize("prec", ["f16", "bf16"])
def test_gather_tile_rule(n, nrhs, prec):
    rng = np.random.default_rng(n)
    F = rng.random((n, n), np.float32) * np.float32(1.8 / n)  # rows sum to about 0.9
    rho = rng.uniform(0.2, 0.7, (n, nrhs))
    E = rng.uniform(0.0, 1.0, (n, nrhs))
    tol = 1e-9
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        B, info = lin.gather(rho, E, prec=prec, tol=tol, max_outer=40, sweeps=5)
    assert info["rel_res"] <= tol
    r = E + rho * (F.astype(np.float64) @ B) - B
    # the solver's own residual and this one differ by rounding in float64 only
    assert np.linalg.norm(r) <= tol * np.linalg.norm(E) + 1e-12 * np.linalg.norm(B)


# plain shooting in one block (every patches-per-thread and column form, the
# ragged ends, equal powers) and past its limits, bit for bit
@pytest.mark.parametrize("n,nrhs", [(1, 1), (63, 2), (1024, 1), (1025, 3), (2049, 3), (4097, 5), (5000, 3), (8192, 3), (8193, 3),
                                    (1500, 12), (1024, 16), (1025, 16), (3000, 6), (12288, 1), (12289, 1)])
def test_shooting_bits(n, nrhs):
    rng = np.random.default_rng(n + nrhs)
    F = rng.random((n, n), np.float32) * np.float32(1.6 / n)
    rho = rng.uniform(0.2, 0.8, (n, nrhs))
    E = np.where(rng.random((n, 1)) < 0.1, np.round(rng.uniform(0, 4, (n, nrhs))), 0.0)  # many ties
    shots = 150
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        B, info = lin.shoot(rho, E, max_shots=shots)
    want, _, src = lo.shoot32(F, rho, E, np.ones(n), shots)
    assert info["outer"] == len(src)
    assert np.array_equal(B.astype(np.float32), want)


# batches on each side of the residual's and the sweep's size rules (8192 and
# 16384 padded rows), one scene above all; tolerances met and missed
@pytest.mark.parametrize("sizes", [[1], [256, 257, 1, 40], [700] * 11, [1500] * 12, [8200, 64]])
@pytest.mark.parametrize("prec", ["f16", "bf16"])
def test_batch_size_rules(sizes, prec):
    rng = np.random.default_rng(len(sizes))
    tol = 1e-10
    with radgpu.SceneBatch(sizes) as b:
        Fs = [rng.random((n, n), np.float32) * np.float32(1.8 / n) for n in sizes]
        for s, F in enumerate(Fs):
            b.set_matrix(s, F)
        total = sum(sizes)
        rho = rng.uniform(0.2, 0.7, (total, 3))
        E = rng.uniform(0.0, 1.0, (total, 3))
        E[-64:] = 0.0  # the last scene starts converged where that is all of it
        B, rel, info = b.solve(rho, E, prec=prec, graph=True, tol=tol, outer=20, sweeps=5)
        Bs, rels, _ = b.solve(rho, E, prec=prec, graph=False, tol=tol, outer=20, sweeps=5)
        assert np.array_equal(B, Bs) and np.array_equal(rel, rels)
        assert info["above_tol"] == 0 and np.all(rel <= tol)
        o = 0
        for n, F in zip(sizes, Fs):
            r = E[o:o + n] + rho[o:o + n] * (F.astype(np.float64) @ B[o:o + n]) - B[o:o + n]
            assert np.linalg.norm(r) <= tol * np.linalg.norm(E[o:o + n]) + 1e-12 * np.linalg.norm(B[o:o + n])
            o += n
        # two refinements do not reach it
        _, rel2, info2 = b.solve(rho, E, prec=prec, graph=True, tol=1e-14, outer=2, sweeps=2)
        lit = [i for i, n in enumerate(sizes) if E[sum(sizes[:i]):sum(sizes[:i + 1])].any()]
        assert info2["above_tol"] == len(lit) and np.all(rel2[lit] > 1e-14)


# the FP64 MFMA product at each of its tiles: one, two and four column tiles,
# 64, 128 and 256 rows a block, split-K 1 to 8, ragged ends
@pytest.mark.parametrize("n,nrhs", [(1, 5), (250, 16), (300, 17), (300, 40), (1024, 64), (2049, 192), (4100, 30), (4100, 64),
                                    (4096, 192), (7900, 65), (9000, 16), (8192, 129)])
def test_f64_product_many_columns(n, nrhs):
    rng = np.random.default_rng(n + nrhs)
    F = rng.random((n, n), np.float32)
    X = rng.standard_normal((n, nrhs))
    with radgpu.LinearSystem(n) as lin:
        lin.set_matrix(F)
        Y = lin.multiply(X, "f32")
    F64 = F.astype(np.float64)
    assert (np.abs(Y - F64 @ X) <= 2 * (n + 1) * U64 * (F64 @ np.abs(X))).all()
