"""What a call does where the device has no room for what makes it faster gives the same results."""
import numpy as np
import pytest

from serenity_amd import xc
from serenity_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_coulomb_with_the_solves_on_the_host(ctx):
    """J = B^T M^-1 B p with M^-1 on the device and on the host: the metric of RI_J_WEIGEND has a
    condition of about 1e6 here, which moves J by at most its square root times FP64 rounding times
    the 200 functions' sums (2e-11 of the largest element)."""
    Z, X = W.water_chain(2)
    b = xc.BasisController.from_file("DEF2-SVP", Z, X)
    jc = xc.DensityFittedCoulomb(ctx, b, xc.BasisController.from_file("RI_J_WEIGEND", Z, X))
    P = W.synthetic_density(b.overlap(), W.n_electrons(Z) // 2)
    J = jc.coulomb(P)
    jc._resident = False
    host = jc.coulomb(P)
    assert np.abs(J - host).max() < 2e-11 * np.abs(host).max()
    bad = P.copy()
    bad[0, 0] = np.nan
    for resident in (True, False):
        jc._resident = resident
        with pytest.raises(ValueError, match="infs or NaNs"):
            jc.coulomb(bad)
    jc._release()
