"""Reductions that fold in their producer's last block (at most 64 blocks of 1024
elements) against the same sums in two launches (hpcgx_dot_noalloc): the grouping
is the same, so the bits are.  Lengths around one element, one block, the last
one-launch length and the first two-launch one; the calls alternate, so each finds
the ticket as the one before left it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 63, 255, 1024, 1025, 33000, 65536, 65537, 110000]


def test_one_launch_same_bits_as_two(hip):
    rng = np.random.default_rng(31)
    P = hip.Problem(48)
    x = hip.DeviceArray.from_host(rng.uniform(-1, 1, P.m))
    y = hip.DeviceArray.from_host(rng.uniform(-1, 1, P.m))
    for _ in range(3):
        for n in LENGTHS + LENGTHS[::-1]:
            assert P.dot(x, y, n) == hip.dot_noalloc(x, y, n), n
            got = P.fused_waxpby_dot(0.125, x, y, n)
            assert got == hip.dot_noalloc(y, y, n), n
            assert P.residual(x, y, n) == (np.abs(x.host()[:n] - y.host()[:n]).max() if n else 0.0), n
    # what is not a number stays so
    v = rng.uniform(-1, 1, P.m)
    v[5], v[40000] = np.nan, np.inf
    z = hip.DeviceArray.from_host(v)
    assert np.isnan(P.dot(z, z, 1000)) and np.isnan(P.dot(z, z))
    v[5] = 0.0
    z.upload(v)
    assert P.dot(z, z, 1000) == hip.dot_noalloc(z, z, 1000) and P.dot(z, z) == np.inf
    P.close()
