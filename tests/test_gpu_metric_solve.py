"""The density-fitting solves on the device around the 64 unknowns of a step: one block, full and ragged
last blocks, several blocks, against scipy's on the same right-hand side.

The fitted functions lie apart, the metric's condition number is below 1e4: 1e-11 of the largest
element (1e4 times FP64 rounding, 1e-12, and the sums over up to 260 functions)."""
import numpy as np
import pytest
import scipy.linalg

from serenity_amd import workloads as W, xc

pytestmark = pytest.mark.gpu


def engine(ctx, naux):
    Z, X = W.water_chain(1)
    b = xc.BasisController.from_file("DEF2-SVP", Z, X)
    r = np.random.default_rng(naux)
    k = int(np.ceil(naux ** (1 / 3)))
    at = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:naux] * 1.5 - 0.75 * (k - 1)
    a = xc.BasisController(np.zeros(naux), np.ones(naux), np.ones(naux), at, r.uniform(0.8, 1.2, naux), np.ones(naux))
    return b, xc.DensityFittedCoulomb(ctx, b, a, threshold=0.0)


@pytest.mark.parametrize("naux", [1, 63, 64, 65, 128, 200, 257])
def test_solves_match_scipy(ctx, naux):
    b, jc = engine(ctx, naux)
    assert jc._resident and np.linalg.cond(jc.metric) < 1e4
    for seed in (1, 2):
        R = np.random.default_rng(seed).standard_normal((b.nao, b.nao))
        P = R + R.T
        ref = jc.matrix(scipy.linalg.cho_solve(jc._cho, jc.rhs(P)))
        J = jc.coulomb(P)
        assert J.flags.f_contiguous and np.abs(J - ref).max() < 1e-11 * np.abs(ref).max()
    jc._release()


def test_a_density_that_is_not_finite_is_refused(ctx):
    b, jc = engine(ctx, 70)
    P = np.eye(b.nao)
    good = jc.coulomb(P)
    for bad in (np.nan, np.inf):
        Q = P.copy()
        Q[1, 1] = bad
        with pytest.raises(ValueError, match="infs or NaNs"):
            jc.coulomb(Q)
        assert np.abs(jc.coulomb(P) - good).max() < 1e-12 * np.abs(good).max()
    jc._release()
