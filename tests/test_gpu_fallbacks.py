"""What a call does where the device has no room for what makes it faster gives the same results."""
import subprocess
import sys

import numpy as np
import pytest

from common import REPO
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
