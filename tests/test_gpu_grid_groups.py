"""The SSF partition with the atoms over 8 or 16 lanes per candidate (one thread per candidate from 513
atoms on): the device grid equals the host's bit for bit at the edges of the lane groups and of the
LDS limit, and with atoms far enough apart that most cells vanish."""
import numpy as np
import pytest

from serenity_amd import workloads as W, xc

pytestmark = pytest.mark.gpu


def line(n, step):
    """n H atoms along a line (bohr), every third raised."""
    x = np.arange(n)
    return np.ones(n, dtype=np.int32), np.stack([step * x, 0.7 * (x % 3), 0.1 * (x % 2)], 1)


CASES = [("1", line(1, 1.0)), ("2", line(2, 1.4)), ("8", line(8, 1.4)), ("9", line(9, 1.4)), ("16", line(16, 1.4)),
         ("17", line(17, 1.4)), ("33-apart", line(33, 9.0)), ("waters", W.water_chain(7)),
         ("512", line(512, 4.0)), ("513", line(513, 4.0))]


@pytest.mark.parametrize("name,geometry", CASES, ids=[c[0] for c in CASES])
def test_device_grid_equals_host(ctx, name, geometry):
    Z, X = geometry
    host = xc.molecular_grid(Z, X, accuracy=1)
    dev = xc.molecular_grid(Z, X, accuracy=1, ctx=ctx)
    assert np.array_equal(host.points, dev.points)
    assert np.array_equal(host.weights, dev.weights)
