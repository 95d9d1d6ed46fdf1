"""Non-additive builds on cached densities around the 32 entries that one launch's lists hold: as many
subsystems as fit, one more, and several lists' worth; densities and energies new for all, for
one, and for none of them.

The direct build forms the same sums in the same order: equal energies, and F to 1e-13 (FP64 additions
in another order)."""
import numpy as np
import pytest

from serenity_amd import xc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nenv", [0, 1, 31, 32, 33, 66])
def test_cached_build_at_the_list_limit(ctx, nenv):
    rng = np.random.default_rng(nenv)
    pts = rng.uniform(-4.0, 4.0, (391, 3))
    grid = xc.GridController(pts, np.full(len(pts), 0.3))
    bfs, dPs = [], []
    for i in range(1 + nenv):
        Z, X = np.array([8 if i == 0 else 1], dtype=np.int32), rng.uniform(-3.0, 3.0, (1, 3))
        b = xc.BasisController.from_file("DEF2-SVP", Z, X)
        C = rng.standard_normal((b.nao, 2))
        bfs.append(xc.BasisFunctionOnGridController(ctx, b, grid))
        d = ctx.alloc(8 * b.nao * b.nao)
        ctx.upload(d, (0.1 * C @ C.T).ravel(order="F"))
        dPs.append(d)
        bfs[-1].update_density(d)
    n = bfs[0].getNBasisFunctions()
    dF = ctx.alloc(8 * n * n)
    for func in ("PBE", "LDA"):
        pot = xc.NAddFuncPotential(bfs[0], bfs[1:], func)
        F = np.zeros(n * n)
        E = pot.build_device(dPs[0], dPs[1:], dF)
        ctx.download(F, dF)
        for fresh in (range(len(bfs)), [nenv], []):
            for i in fresh:
                bfs[i].update_density(dPs[i])
            ctx.upload(dF, np.full(n * n, 7.0))
            e = pot.build_cached(dF)
            G = np.zeros(n * n)
            ctx.download(G, dF)
            assert e == E
            assert np.abs(G - F).max() < 1e-13
    for d in dPs + [dF]:
        ctx.free(d)
