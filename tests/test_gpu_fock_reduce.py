"""The row reduce of the Fock sub-tiles at the edges of its work split: rows whose entries are fewer
or more than the lane groups of a workgroup, segments shorter than one lane's four columns and longer
than a group's step, blocks of a few points, and both group widths (the wide one is taken from a mean
of 256 AOs per block on).

FP64 against the oracle to 1e-9 (the bar of the parity tests); the integer-sum form and the FP64
additions to 1e-12 of each other (rounding of sums of a few thousand terms below 1 each)."""
import numpy as np
import pytest

from oracle import oracle as O
from serenity_amd import workloads as W, xc

pytestmark = pytest.mark.gpu

CASES = [
    ("one-block", W.water_chain(1), "DEF2-SVP", 100, 128),       # every row: a single entry
    ("one-point-blocks", W.water_chain(1), "DEF2-SVP", 70, 1),   # 70 entries a row
    ("small-blocks", W.alkane(3), "DEF2-SVP", 6000, 7),          # more entries than lane groups
    ("narrow", W.alkane(8), "DEF2-SVP", 20000, 128),
    ("wide", W.water_cluster(3, 3, 3), "DEF2-TZVP", 6000, 128),  # mean n_b above 256 around the centre
]


@pytest.mark.parametrize("name,geometry,basis,npts,block", CASES, ids=[c[0] for c in CASES])
def test_reduce_matches_oracle(ctx, name, geometry, basis, npts, block):
    Z, X = geometry
    b = xc.BasisController.from_file(basis, Z, X)
    full = xc.molecular_grid(Z, X, accuracy=2)
    near = np.arange(npts)
    if name == "wide":  # the points around the cluster's centre, in grid order
        near = np.sort(np.argsort(np.linalg.norm(full.points - X.mean(0), axis=1))[:npts])
    grid = xc.GridController(full.points[near], full.weights[near])
    P = W.synthetic_density(b.overlap(), W.n_electrons(Z) // 2, seed=2)
    F, E, _, _ = O.fock_build(b, grid.points, grid.weights, P, "PBE", block_size=block)
    det = xc.Context(0)
    det.set_deterministic(True)
    got = []
    for c in (ctx, det):
        bf = xc.BasisFunctionOnGridController(c, b, grid, block, 1e-9, 1, keep_fp32=True)
        if name == "wide":
            assert bf.stats()[0] > 256 * bf.getNBlocks()
        pot = xc.FuncPotential(bf, "PBE", "FP64")
        G = pot.getMatrix(P)
        assert abs(pot.getEnergy() - E) < 1e-9 * max(1.0, abs(E))
        assert np.abs(G - F).max() < 1e-9
        assert np.array_equal(G, G.T)
        low = xc.FuncPotential(bf, "PBE", "FP32").getMatrix(P)
        got.append((G, low))
        bf._release()
    det.close()
    assert np.abs(got[0][0] - got[1][0]).max() < 1e-12
    assert np.abs(got[0][1] - got[1][1]).max() < 1e-12
    # FP32 contraction: 2^-24 relative to the largest terms of an element's sum
    assert np.abs(got[0][1] - F).max() < 2e-5 * np.abs(F).max()
