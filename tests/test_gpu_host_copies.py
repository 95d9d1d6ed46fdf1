"""Host matrices on their way through the pinned ring: below and above one piece (1 MiB), more than the
ring holds, several matrices per call.  The resident forms take the same kernels on the same numbers:
densities equal bit for bit, F to 1e-13 (FP64 additions in another order)."""
import numpy as np
import pytest

from serenity_amd import xc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nao", [3, 362, 363, 725, 1030])
def test_host_and_resident_forms_agree(ctx, nao):
    rng = np.random.default_rng(nao)
    X = np.stack([0.8 * np.arange(nao), rng.uniform(-1, 1, nao), rng.uniform(-1, 1, nao)], 1)
    b = xc.BasisController(np.zeros(nao), np.ones(nao), np.ones(nao), X, rng.uniform(0.3, 0.6, nao), np.full(nao, 0.5))
    pts = X[rng.integers(0, nao, 600)] + rng.standard_normal((600, 3))
    bf = xc.BasisFunctionOnGridController(ctx, b, xc.GridController(pts, np.full(600, 0.05)))
    pot = xc.FuncPotential(bf, "PBE", "FP64")
    mats = []
    for _ in range(2):
        C = rng.standard_normal((nao, 4))
        mats.append(np.asfortranarray(C @ C.T / nao))
    d = [ctx.alloc(8 * nao * nao) for _ in range(4)]
    for x, m in zip(d, mats):
        ctx.upload(x, m.ravel(order="F"))
    E0 = pot.build_device(d[0], d[2])
    F0 = np.zeros(nao * nao)
    ctx.download(F0, d[2])
    F0 = F0.reshape(nao, nao, order="F")
    for _ in range(2):
        F = pot.getMatrix(mats[0])
        assert np.abs(F - F0).max() < 1e-13 and abs(pot.getEnergy() - E0) < 1e-13 * max(1.0, abs(E0))
        Fa, Fb = pot.getMatrixUnrestricted(mats[0], mats[1])
        Ga, Gb = pot.getMatrixUnrestricted(mats[1], mats[0])
        assert np.abs(Fa - Gb).max() < 1e-13 and np.abs(Fb - Ga).max() < 1e-13
    for x in d:
        ctx.free(x)
    bf._release()
