"""DensityFittedCoulomb refuses arrays of the wrong size before the library reads them."""
import numpy as np
import pytest

from serenity_amd import xc


def _bare(resident, n=3, naux=4):
    """An object without a device handle: the library would answer "null argument"."""
    jc = object.__new__(xc.DensityFittedCoulomb)
    jc.handle, jc.n, jc.naux, jc._resident, jc._cho = None, n, naux, resident, None
    return jc


@pytest.mark.parametrize("shape", [(2, 2), (4, 4), (3, 2), (8,), (0,), ()])
@pytest.mark.parametrize("call", ["rhs", "coulomb resident", "coulomb host"])
def test_density_of_another_size_is_refused(shape, call):
    jc = _bare("resident" in call)
    with pytest.raises(xc.XCError, match="basis has 3 functions"):
        getattr(jc, call.split()[0])(np.zeros(shape))


@pytest.mark.parametrize("shape", [(3,), (5,), (4, 4), (0,)])
def test_coefficients_of_another_number_are_refused(shape):
    with pytest.raises(xc.XCError, match="auxiliary basis has 4 functions"):
        _bare(False).matrix(np.zeros(shape))


@pytest.mark.parametrize("shape", [(3, 3), (9,)])
def test_density_of_the_right_size_reaches_the_library(shape):
    for jc, f in ((_bare(True), "coulomb"), (_bare(False), "rhs")):
        with pytest.raises(xc.XCError, match="null argument"):
            getattr(jc, f)(np.zeros(shape))
