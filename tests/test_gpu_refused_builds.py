"""A host build of a controller whose server build is in flight is refused before it touches the
controller's density matrix: the server's result is that of the matrix it was given."""
import numpy as np
import pytest

from serenity_amd import xc
from serenity_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graphs", [False, True])
@pytest.mark.parametrize("precision", ["FP64", "FP32", "MIXED"])
def test_refused_build_leaves_the_server_build_alone(ctx, precision, use_graphs):
    Z, X = W.alkane(8)
    b = xc.BasisController.from_file("DEF2-TZVP", Z, X)
    g = xc.molecular_grid(Z, X)
    nocc = W.n_electrons(Z) // 2
    P, other = (W.synthetic_density(b.overlap(), nocc, seed=k) for k in (1, 2))
    bf = xc.BasisFunctionOnGridController(ctx, b, g, 128, 1e-9, 1, keep_fp32=True)
    pot = xc.FuncPotential(bf, "PBE", precision)
    F0, E0 = pot.getMatrix(P), pot.getEnergy()
    srv = xc.Server(ctx, nslots=1, use_graphs=use_graphs)
    for _ in range(3):
        t = srv.submit(bf, "PBE", precision, P)
        with pytest.raises(xc.XCError, match="in flight"):
            pot.getMatrix(other)
        with pytest.raises(xc.XCError, match="in flight"):
            pot.getMatrixUnrestricted(0.5 * other, 0.5 * other)
        F, E = srv.wait(t)
        assert np.abs(F - F0).max() < 1e-10 and abs(E - E0) < 1e-10
    srv._release()
    bf._release()
