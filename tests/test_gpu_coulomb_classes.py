"""The J engine's class-specialised meetings (wavefronts of 64 pairs or auxiliary primitives of one
angular momentum) against the host's analytic 3-centre integrals, at the edges of their work split:
classes of fewer than, exactly and more than 64 members, lanes shared between pairs (f and g
auxiliary functions), and centres so far apart that the Boys argument leaves its table.

Tolerance 1e-11 relative to the largest element, as for the host comparison of test_gpu_coulomb.py:
sums of at most 1e5 terms of FP64 rounding (1e-16 each) stay two orders below."""
import numpy as np
import pytest

from serenity_amd import scf, workloads as W, xc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = xc.Context(0)
    yield c
    c.close()


def hydrogens(k, spacing):
    """k hydrogen atoms on a line: every class has a multiple of k members."""
    X = np.zeros((k, 3))
    X[:, 2] = spacing * np.arange(k)
    return np.ones(k, dtype=np.int32), X


CASES = [
    ("H1", "DEF2-SVP", hydrogens(1, 1.4), True),
    ("H2-far", "DEF2-SVP", hydrogens(2, 40.0), True),
    ("H16", "DEF2-SVP", hydrogens(16, 1.5), True),
    ("H17-cart", "DEF2-TZVP", hydrogens(17, 3.0), False),
    ("ethane", "DEF2-TZVP", W.alkane(2), True),
    ("water5", "DEF2-TZVP", W.water_chain(5), True),
    ("propane-cart", "DEF2-SVP", W.alkane(3), False),
]


@pytest.mark.parametrize("name,basis,geometry,spherical", CASES, ids=[c[0] for c in CASES])
def test_classes_match_host_integrals(ctx, name, basis, geometry, spherical):
    Z, X = geometry
    b = xc.BasisController.from_file(basis, Z, X, spherical=spherical)
    a = xc.BasisController.from_file("RI_J_WEIGEND", Z, X, spherical=spherical)
    r = np.random.default_rng(3).standard_normal((b.nao, b.nao))
    P = r + r.T
    c = np.random.default_rng(4).standard_normal(a.nao)
    B3, _ = scf.ri_j_integrals(b, a, 0.0)
    b_ref = B3 @ scf.pack_density(P)
    J_ref = scf.unpack_symmetric(B3.T @ c, b.nao)
    jc = xc.DensityFittedCoulomb(ctx, b, a, threshold=0.0)
    for _ in range(2):  # the second call finds the first one's sums in its buffers
        assert np.abs(jc.rhs(P) - b_ref).max() < 1e-11 * np.abs(b_ref).max()
        assert np.abs(jc.matrix(c) - J_ref).max() < 1e-11 * np.abs(J_ref).max()
    jc._release()
