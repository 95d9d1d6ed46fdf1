"""What a call does where the device has no room for what makes it faster gives the same results."""
import ctypes as C
import subprocess
import sys

import numpy as np
import pytest

from common import REPO
from serenity_amd import _lib, xc
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


# A refused call ends the recording of its stream for good, so this runs in a process of its own.
REFUSED = """
import ctypes as C
from serenity_amd import xc
c = xc.Context(0)
c.free(c.alloc(1 << 20))  # kept for reuse
assert C.CDLL("libamdhip64.so").hipStreamBeginCapture(C.c_void_p(c.stream), 1) == 0  # thread-local mode
for nbytes in (3 << 30, 1 << 20):
    try:
        c.alloc(nbytes)
        print("got", nbytes)
    except xc.XCError as e:
        print("code", e.code)
"""


def test_a_device_error_is_not_a_lack_of_memory(ctx):
    """An allocation that the runtime refuses (while the stream is recorded) is XC_ERR_DEVICE, and the
    blocks kept for reuse stay; one beyond the device is XC_ERR_MEMORY."""
    r = subprocess.run([sys.executable, "-c", REFUSED], cwd=REPO, capture_output=True, text=True, timeout=60)
    assert r.stdout.split("\n")[:2] == ["code 2", "got %d" % (1 << 20)], (r.stdout, r.stderr)
    with pytest.raises(xc.XCError) as e:
        ctx.alloc(1 << 46)
    assert e.value.code == 3


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("functional", ["LDA", "PBE"])
def test_first_unrestricted_device_build_recorded(ctx, functional, precision):
    """The first unrestricted device build of a controller whose spin buffers exist is recorded into a
    graph: it allocates nothing, and every replay, with other builds between, gives the eager result
    (sums of a few thousand terms in another order: 1e-12)."""
    hip = C.CDLL("libamdhip64.so")
    Z, X = W.water_chain(2)
    b = xc.BasisController.from_file("DEF2-SVP", Z, X)
    g = xc.molecular_grid(Z, X, accuracy=2)
    n, P = b.nao, W.synthetic_density(b.overlap(), W.n_electrons(Z) // 2)
    Pa, Pb = np.asfortranarray(0.6 * P), np.asfortranarray(0.4 * P)
    bf = xc.BasisFunctionOnGridController(ctx, b, g, 128, 1e-9, 1, keep_fp32=True)
    xc.NAddFuncPotential(bf, [], functional, precision).getMatrixUnrestricted(Pa, Pb, [], [])  # the spin buffers
    d = [ctx.alloc(8 * n * n) for _ in range(4)]
    ctx.upload(d[0], Pa)
    ctx.upload(d[1], Pb)
    ctx.synchronize()
    stream, graph, run = C.c_void_p(ctx.stream), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 1) == 0  # thread-local mode
    rc = _lib.lib().xc_fock_build_unrestricted_device(bf.handle, _lib.FUNCTIONALS[functional],
                                                      _lib.PRECISIONS[precision], 1e-11, *d, None)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0 and rc == 0
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    pot = xc.FuncPotential(bf, functional, precision)
    E = C.c_double()
    for swap in (False, True, False):
        ctx.upload(d[0], Pb if swap else Pa)
        ctx.upload(d[1], Pa if swap else Pb)
        assert hip.hipGraphLaunch(run, stream) == 0
        _lib.check(_lib.lib().xc_last_energy(ctx.handle, C.byref(E)))
        F = [np.zeros((n, n), order="F") for _ in range(2)]
        for f, p in zip(F, d[2:]):
            ctx.download(f, p)
        ref = pot.getMatrixUnrestricted(*((Pb, Pa) if swap else (Pa, Pb)))
        for f, r in zip(F, ref):
            assert np.abs(f - r).max() < 1e-12 * max(1.0, np.abs(r).max())
        assert abs(E.value - pot.getEnergy()) < 1e-12 * abs(E.value)
    hip.hipGraphExecDestroy(run)
    hip.hipGraphDestroy(graph)
    for p in d:
        ctx.free(p)
    bf._release()


@pytest.mark.parametrize("recorded", [False, True])
def test_second_spin_scratch_is_given_back(recorded):
    """An allocation beyond the device (refused) takes back the scratch with which a controller runs both
    spins at once; the builds after it run one spin after the other and give the same matrices.  A
    controller whose build is recorded in a graph keeps its scratch, and the graph its result."""
    hip = C.CDLL("libamdhip64.so")
    c = xc.Context(0)
    Z, X = W.water_chain(3)
    b = xc.BasisController.from_file("DEF2-SVP", Z, X)
    g = xc.molecular_grid(Z, X, accuracy=3)
    n, P = b.nao, W.synthetic_density(b.overlap(), W.n_electrons(Z) // 2)
    Pa, Pb = np.asfortranarray(0.6 * P), np.asfortranarray(0.4 * P)
    bf = xc.BasisFunctionOnGridController(c, b, g, 128, 1e-9, 1)
    pot = xc.FuncPotential(bf, "PBE", "FP64")
    xc.NAddFuncPotential(bf, [], "PBE", "FP64").getMatrixUnrestricted(Pa, Pb, [], [])  # the spin buffers
    d = [c.alloc(8 * n * n) for _ in range(4)]
    c.upload(d[0], Pa)
    c.upload(d[1], Pb)
    before = c.memory_in_use()
    ref = pot.getMatrixUnrestricted(Pa, Pb)
    E = pot.getEnergy()
    both = c.memory_in_use()
    assert both > before
    stream, graph, run = C.c_void_p(c.stream), C.c_void_p(), C.c_void_p()
    if recorded:
        c.synchronize()
        assert hip.hipStreamBeginCapture(stream, 1) == 0
        rc = _lib.lib().xc_fock_build_unrestricted_device(bf.handle, 1, 0, 1e-11, *d, None)
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0 and rc == 0
        assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    with pytest.raises(xc.XCError):
        c.alloc(1 << 46)
    kept = c.memory_in_use()
    assert kept == both if recorded else before <= kept < both
    for _ in range(2):
        F = pot.getMatrixUnrestricted(Pa, Pb)
        assert c.memory_in_use() == kept
        for f, r in zip(F, ref):
            assert np.abs(f - r).max() < 1e-12 * max(1.0, np.abs(r).max())
        assert abs(pot.getEnergy() - E) < 1e-12 * abs(E)
        if recorded:
            assert hip.hipGraphLaunch(run, stream) == 0
            c.synchronize()
            for p, r in zip(d[2:], ref):
                f = np.zeros((n, n), order="F")
                c.download(f, p)
                assert np.abs(f - r).max() < 1e-12 * max(1.0, np.abs(r).max())
    if recorded:
        hip.hipGraphExecDestroy(run)
        hip.hipGraphDestroy(graph)
    for p in d:
        c.free(p)
    c.close()
