"""Packed FP64 builds without gradient terms on a deterministic context: every system's density is
summed as in its build alone, whatever it is packed with, so F is the same bit for bit.  The sizes
lie on both sides of the 96 AOs up to which a density is one column pass."""
import numpy as np
import pytest

from serenity_amd import xc
from serenity_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dctx():
    c = xc.Context(0)
    c.set_deterministic(True)
    yield c
    c.close()


@pytest.fixture(scope="module")
def systems(dctx):
    out = []
    for k, ((Z, X), name, nao) in enumerate(((W.water_chain(1), "DEF2-SVP", 24), (W.water_chain(4), "DEF2-SVP", 96),
                                             (W.water_chain(3), "DEF2-TZVP", 129), (W.water_chain(5), "DEF2-SVP", 120))):
        b = xc.BasisController.from_file(name, Z, X)
        assert b.nao == nao
        g = xc.molecular_grid(Z, X, accuracy=2)
        P = W.synthetic_density(b.overlap(), W.n_electrons(Z) // 2, seed=k + 3)
        bf = xc.BasisFunctionOnGridController(dctx, b, g, 128, 1e-9, 1)
        dP, dF = dctx.alloc(8 * nao * nao), dctx.alloc(8 * nao * nao)
        dctx.upload(dP, np.asfortranarray(P))
        out.append(dict(bf=bf, n=nao, dP=dP, dF=dF))
    yield out
    for s in out:
        dctx.free(s["dP"])
        dctx.free(s["dF"])
        s["bf"]._release()


def _matrix(dctx, s):
    F = np.zeros((s["n"], s["n"]), order="F")
    dctx.download(F, s["dF"])
    return F


@pytest.mark.parametrize("functional", ["LDA", "TF"])
@pytest.mark.parametrize("members", [(0, 1), (0, 1, 2), (2, 1), (2, 3), (0, 1, 2, 3)])
def test_packed_equals_alone_bitwise(dctx, systems, members, functional):
    pack = [systems[i] for i in members]
    alone = []
    for s in pack:
        xc.FuncPotential(s["bf"], functional, "FP64").build_device(s["dP"], s["dF"])
        alone.append(_matrix(dctx, s))
    for rep in range(3):  # eager, captured, replayed
        for s in pack:
            dctx.upload(s["dF"], np.full((s["n"], s["n"]), 7.0))
        xc.fock_build_packed([xc.FuncPotential(s["bf"], functional, "FP64") for s in pack], [s["dP"] for s in pack],
                             [s["dF"] for s in pack])
        for s, Fa in zip(pack, alone):
            assert np.array_equal(_matrix(dctx, s), Fa), (members, functional, rep, s["n"])
