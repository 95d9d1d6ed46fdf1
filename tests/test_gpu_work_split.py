"""The contractions at the edges of their work split: blocks whose AO count lies on either side of a
16-column sub-tile, of a density pass (96 columns), of a workgroup shape of the Fock kernel (64,
128, 160, 192 AOs) and of a 128-row panel; hydrogen rows give every count (5 AOs per atom in
def2-SVP, all of them near the grid).

FP64 against the oracle to 1e-9 (the bar of the parity tests); FP32 to 2e-5 of the largest element
(2^-24 relative to the largest terms of a sum)."""
import numpy as np
import pytest

from oracle import oracle as O
from serenity_amd import xc

pytestmark = pytest.mark.gpu


def hydrogens(k):
    """k hydrogens on a jittered ring of 2 bohr: every AO is significant in every block."""
    rng = np.random.default_rng(k)
    a = 2.0 * np.pi * np.arange(k) / k
    return np.ones(k, dtype=np.int32), np.stack([2 * np.cos(a), 2 * np.sin(a), rng.uniform(-0.3, 0.3, k)], 1)


@pytest.mark.parametrize("functional", ["LDA", "PBE"])
@pytest.mark.parametrize("atoms", [3, 4, 6, 7, 12, 13, 19, 20, 25, 26, 32, 33, 38, 39, 52])
def test_every_block_width(ctx, atoms, functional):
    Z, X = hydrogens(atoms)  # 5 atoms AOs: 15, 20, 30, 35, 60, 65, 95, 100, 125, 130, 160, 165, 190, 195, 260
    b = xc.BasisController.from_file("DEF2-SVP", Z, X)
    rng = np.random.default_rng(atoms)
    pts = rng.normal(0.0, 1.5, (1000, 3))  # 8 blocks, the last one short
    grid = xc.GridController(pts, rng.uniform(0.0, 0.05, 1000))
    C = rng.standard_normal((b.nao, 4)) / np.sqrt(b.nao)
    P = C @ C.T
    F, E, _, _ = O.fock_build(b, grid.points, grid.weights, P, functional)
    bf = xc.BasisFunctionOnGridController(ctx, b, grid, 128, 1e-9, 1, keep_fp32=True)
    assert bf.stats()[0] == b.nao * bf.getNBlocks()
    scale = max(1.0, np.abs(F).max())
    for precision, tol in (("FP64", 1e-9), ("FP32", 2e-5), ("MIXED", 2e-5)):
        pot = xc.FuncPotential(bf, functional, precision)
        for _ in range(2):  # the second mixed build carries the first one's dense blocks
            G = pot.getMatrix(P)
            assert np.abs(G - F).max() < tol * scale, precision
            assert abs(pot.getEnergy() - E) < tol * max(1.0, abs(E)), precision
    bf._release()


@pytest.mark.parametrize("atoms", [4, 20, 39])  # one, two and three column passes
def test_density_form_of_any_matrix(ctx, atoms):
    """Without gradient terms only the symmetric part of the matrix counts, alone and packed; the
    antisymmetric part adds rounding of its size to rho (1e-12 of the oracle's scale is left to it)."""
    Z, X = hydrogens(atoms)
    b = xc.BasisController.from_file("DEF2-SVP", Z, X)
    rng = np.random.default_rng(atoms)
    grid = xc.GridController(rng.normal(0.0, 1.5, (700, 3)), rng.uniform(0.0, 0.05, 700))
    C = rng.standard_normal((b.nao, 4)) / np.sqrt(b.nao)
    P = C @ C.T
    A = rng.standard_normal(P.shape) / b.nao
    bf = xc.BasisFunctionOnGridController(ctx, b, grid, 128, 1e-9, 1)
    pot = xc.FuncPotential(bf, "LDA", "FP64")
    F, E, _, _ = O.fock_build(b, grid.points, grid.weights, P, "LDA")
    G = pot.getMatrix(P + A - A.T)
    scale = max(1.0, np.abs(F).max())
    assert np.abs(G - F).max() < 1e-9 * scale and abs(pot.getEnergy() - E) < 1e-9 * max(1.0, abs(E))
    n = b.nao
    dP, dF = ctx.alloc(8 * n * n), ctx.alloc(8 * n * n)
    ctx.upload(dP, np.asfortranarray(P + A - A.T).ravel(order="F"))
    for _ in range(3):  # eager, captured, replayed
        e = xc.fock_build_packed([pot], [dP], [dF])
        H = np.zeros(n * n)
        ctx.download(H, dF)
        assert np.abs(H.reshape(n, n) - F).max() < 1e-9 * scale and abs(e[0] - E) < 1e-9 * max(1.0, abs(E))
    ctx.free(dP)
    ctx.free(dF)
    bf._release()


@pytest.mark.parametrize("functional", ["LDA", "PBE"])
@pytest.mark.parametrize("atoms", [3, 4, 13, 19, 20, 39])
def test_gradient_at_every_pass_width(ctx, atoms, functional):
    """15 to 195 AOs a block: one to three column passes, even and odd sub-tile counts."""
    Z, X = hydrogens(atoms)
    b = xc.BasisController.from_file("DEF2-SVP", Z, X)
    rng = np.random.default_rng(atoms)
    grid = xc.GridController(rng.normal(0.0, 1.5, (700, 3)), rng.uniform(0.0, 0.05, 700))
    C = rng.standard_normal((b.nao, 4)) / np.sqrt(b.nao)
    P = C @ C.T
    G, E = O.xc_gradient(b, grid.points, grid.weights, P, functional, b.getAtomIndicesOfBasis(), atoms)
    bf = xc.BasisFunctionOnGridController(ctx, b, grid, 128, 1e-9, 2)
    pot = xc.FuncPotential(bf, functional, "FP64")
    for _ in range(2):
        assert np.abs(pot.getGeomGradients(P) - G).max() < 1e-9 * max(1.0, np.abs(G).max())
        assert abs(pot.getEnergy() - E) < 1e-9 * max(1.0, abs(E))
    bf._release()
