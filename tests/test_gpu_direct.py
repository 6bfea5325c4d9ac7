"""The FP64 direct sum at the sizes where its split changes (64 targets per
workgroup; the sources over 16 waves up to 32,768 bodies and over 4 above, and
in two halves below 131,008 bodies, one where a half would be too short), for
single systems and batches whose systems share waves, against the oracle's
direct sum.  Tolerance: sums of n terms in different orders, each term a few
ulp: relative to the sum of the terms' magnitudes the difference is below
n 2^-53 by a wide margin; 1e-12 of the largest acceleration and potential.
"""
import numpy as np
import pytest

import oracle_lib as orc
from next_amd import ic
from next_amd.nbx import MODE_PHYSICS, PREC_FP64, Engine

pytestmark = pytest.mark.gpu


def check(a, pot, p, eps, tg):
    ad, pd = orc.direct_subset(p.x, p.y, p.z, p.m, eps, tg.astype(np.int64))
    assert np.max(np.abs(a[tg] - ad)) <= 1e-12 * max(np.max(np.abs(ad)), 1e-300)
    assert np.max(np.abs(pot[tg] - pd)) <= 1e-12 * max(np.max(np.abs(pd)), 1e-300)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 4095, 4097, 8193, 32768, 32769, 65537, 131008, 131009,
                               524287, 524289])
def test_sizes(n):
    p = ic.plummer(n, seed=n, virial=None)
    with Engine(mode=MODE_PHYSICS, precision=PREC_FP64, eps=0.01) as e:
        e.upload(p)
        a, pot = e.direct()
    tg = np.arange(n) if n <= 4096 else np.random.Generator(np.random.PCG64(1)).choice(n, 64, False)
    check(a, pot, p, 0.01, tg)


def test_batch_shares_waves():
    ps = [ic.plummer(n, seed=n, virial=None) for n in (1, 5, 64, 63, 700, 2, 130)]
    with Engine(mode=MODE_PHYSICS, precision=PREC_FP64, eps=0.01) as e:
        e.upload_batch(ps)
        e.accel()
        a, pot = e.direct()
    at = 0
    for p in ps:
        check(a[at:at + len(p)], pot[at:at + len(p)], p, 0.01, np.arange(len(p)))
        at += len(p)


def test_no_softening_and_far_bodies():
    """eps = 0: bodies at one point have an infinite potential and no defined
    force, others are finite; a distance whose square overflows adds nothing."""
    x = np.array([0.0, 0.0, 1.0, 1e200])
    z = np.zeros(4)
    p = ic.Particles(x, z, z, z, z, z, np.ones(4), np.zeros(4, np.int32))
    with Engine(eps=0.0) as e:
        e.upload(p)
        a, pot = e.direct()
    assert pot[0] == -np.inf and pot[1] == -np.inf and np.isnan(a[0, 0]) and np.isnan(a[1, 0])
    assert np.allclose(a[2], [-2.0, 0.0, 0.0], rtol=1e-15, atol=0) and np.isclose(pot[2], -2.0, rtol=1e-15)
    assert np.array_equal(a[3], np.zeros(3)) and abs(pot[3]) < 1e-150
