"""DensityFittedCoulomb refuses arrays of the wrong size before the library reads them, and
keeps the metric's solves on the host only where the device has no room for its factor."""
import numpy as np
import pytest

from serenity_amd import _lib, xc


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


class _Library:
    """The calls of DensityFittedCoulomb without a device: every one succeeds but those given."""

    def __init__(self, message, **codes):
        self.message, self.codes = message, codes

    def xc_last_error(self):
        return self.message.encode()

    def __getattr__(self, name):
        def call(*args):
            if name == "xc_ri_metric":
                np.ctypeslib.as_array(args[-1], shape=(4, 4))[:] = np.eye(4)
            return self.codes.get(name, 0)
        return call


def _engine(monkeypatch, message="", **codes):
    class Basis:
        nao = 4

        def as_args(self):
            return ()

    class Context:
        def _register(self, obj):
            pass

    library = _Library(message, **codes)
    monkeypatch.setattr(_lib, "lib", lambda: library)
    monkeypatch.setattr(xc, "_DeviceBasis", lambda ctx, basis: type("", (), dict(handle=None)))
    return xc.DensityFittedCoulomb(Context(), Basis(), Basis())


@pytest.mark.parametrize("code", [1, 2, 4, 5])
def test_only_a_lack_of_room_keeps_the_solves_on_the_host(monkeypatch, code):
    assert _engine(monkeypatch)._resident
    assert not _engine(monkeypatch, xc_coulomb_set_metric=_lib.XC_ERR_MEMORY)._resident
    with pytest.raises(xc.XCError, match="a copy failed"):
        _engine(monkeypatch, "a copy failed", xc_coulomb_set_metric=code)


def test_only_a_right_hand_side_that_is_not_finite_is_a_value_error(monkeypatch):
    with pytest.raises(ValueError, match="infs or NaNs"):
        _engine(monkeypatch, "array must not contain infs or NaNs", xc_coulomb_build=5).coulomb(np.zeros((4, 4)))
    with pytest.raises(xc.XCError, match="bad_alloc"):
        _engine(monkeypatch, "std::bad_alloc", xc_coulomb_build=5).coulomb(np.zeros((4, 4)))
