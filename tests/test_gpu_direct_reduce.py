"""Matrices of up to 512 AOs get F and the energy from the row reduce itself, larger ones from the
finalize and the sum: both sides of the limit and the smallest, restricted, with F in place of P,
unrestricted and packed, FP64 and FP32 with its rounding term.

FP64 against the oracle to 1e-9 and the forms against each other to 1e-12 (sums of a few thousand terms
below 1 each in another order); FP32 to 2e-5 of the largest element and 1e-5 of the energy."""
import numpy as np
import pytest

from oracle import oracle as O
from serenity_amd import xc

pytestmark = pytest.mark.gpu


def system(nao, nblocks=7):
    """nao s shells of one primitive on a helix, and points around it."""
    t = 0.9 * np.arange(nao)
    X = np.stack([6.0 * np.cos(0.3 * t), 6.0 * np.sin(0.3 * t), 0.05 * t], 1)
    b = xc.BasisController(np.zeros(nao), np.ones(nao), np.ones(nao), X, 0.4 + 0.01 * (np.arange(nao) % 17),
                           np.full(nao, 0.5))
    rng = np.random.default_rng(nao)
    npts = 128 * nblocks - 5
    pts = X[rng.integers(0, nao, npts)] + rng.standard_normal((npts, 3))
    grid = xc.GridController(pts[np.argsort(pts[:, 2])], np.full(npts, 0.02))
    C = rng.standard_normal((nao, max(1, nao // 8))) / np.sqrt(nao)
    return b, grid, np.asfortranarray(2.0 * C @ C.T)


def resident(ctx, pot, P, in_place):
    n = len(P)
    dP = ctx.alloc(8 * n * n)
    dF = dP if in_place else ctx.alloc(8 * n * n)
    ctx.upload(dP, P.ravel(order="F"))
    E = pot.build_device(dP, dF)
    F = np.zeros(n * n)
    ctx.download(F, dF)
    ctx.free(dP)
    if not in_place:
        ctx.free(dF)
    return F.reshape(n, n, order="F"), E


@pytest.mark.parametrize("nao", [1, 17, 511, 512, 513])
@pytest.mark.parametrize("functional", ["LDA", "PBE"])
def test_both_sides_of_the_limit(ctx, nao, functional):
    b, grid, P = system(nao)
    F, E, _, _ = O.fock_build(b, grid.points, grid.weights, P, functional)
    bf = xc.BasisFunctionOnGridController(ctx, b, grid, keep_fp32=True)
    for prec in ("FP64", "FP32"):
        pot = xc.FuncPotential(bf, functional, prec)
        G = pot.getMatrix(P)
        assert np.array_equal(G, G.T)
        if prec == "FP64":
            assert np.abs(G - F).max() < 1e-9 and abs(pot.getEnergy() - E) < 1e-9 * max(1.0, abs(E))
        else:
            assert np.abs(G - F).max() < 2e-5 * np.abs(F).max() and abs(pot.getEnergy() - E) < 1e-5 * abs(E)
        for in_place in (False, True):
            H, e = resident(ctx, pot, P, in_place)
            assert np.abs(H - G).max() < 1e-12 and abs(e - pot.getEnergy()) < 1e-12 * max(1.0, abs(E))
        Fa, Fb = pot.getMatrixUnrestricted(0.5 * P, 0.5 * P)
        tol = 1e-9 if prec == "FP64" else 2e-5 * np.abs(F).max()
        assert np.abs(Fa - F).max() < tol and np.abs(Fb - F).max() < tol
        assert abs(pot.getEnergy() - E) < (1e-9 if prec == "FP64" else 1e-5) * max(1.0, abs(E))
    bf._release()


@pytest.mark.parametrize("sizes", [(1, 17, 512), (17, 513)])
@pytest.mark.parametrize("prec", ["FP64", "FP32"])
def test_packed(ctx, sizes, prec):
    made, alone = [], []
    for n in sizes:
        b, grid, P = system(n)
        bf = xc.BasisFunctionOnGridController(ctx, b, grid, keep_fp32=True)
        pot = xc.FuncPotential(bf, "PBE", prec)
        alone.append((pot.getMatrix(P), pot.getEnergy()))
        dP, dF = ctx.alloc(8 * n * n), ctx.alloc(8 * n * n)
        ctx.upload(dP, P.ravel(order="F"))
        made.append((n, bf, pot, dP, dF))
    E = xc.fock_build_packed([m[2] for m in made], [m[3] for m in made], [m[4] for m in made])
    for (n, bf, pot, dP, dF), (F, e0), e in zip(made, alone, E):
        G = np.zeros(n * n)
        ctx.download(G, dF)
        assert np.abs(G.reshape(n, n, order="F") - F).max() < 1e-12
        assert abs(e - e0) < 1e-12 * max(1.0, abs(e0))
        ctx.free(dP)
        ctx.free(dF)
        bf._release()
