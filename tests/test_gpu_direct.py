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


def test_one_pair_is_as_accurate_as_a_square_root_and_a_divide():
    """2,000 systems of two bodies against 64-bit mantissas.  Coordinate
    differences are exact.  In u = 2^-53: r^2 + eps^2 takes four roundings, 2 u in
    1/r; 1/r itself is within 1.25 u (1.38e-16; a correctly rounded root and
    divide 1.5 u); the potential one product more, 4.25 u; the force 1/r three
    times, 9.75 u, three products and the sum, 13.75 u.  (One Newton step on the
    hardware's estimate is off by up to 37 u.)"""
    u = 2.0 ** -53
    rng = np.random.Generator(np.random.PCG64(23))
    ps = []
    for _ in range(2000):
        c = np.round(rng.uniform(-4.0, 4.0, (3, 2)) * 2 ** 20) / 2 ** 20
        z = np.zeros(2)
        ps.append(ic.Particles(*c, z, z, z, rng.uniform(0.5, 2.0, 2), np.zeros(2, np.int32)))
    eps = 0.01
    with Engine(mode=MODE_PHYSICS, precision=PREC_FP64, eps=eps) as e:
        e.upload_batch(ps)
        a, pot = e.direct()
    worst = [0.0, 0.0]
    L = np.longdouble
    for k, p in enumerate(ps):
        for i in (0, 1):
            d = [L(v[1 - i]) - L(v[i]) for v in (p.x, p.y, p.z)]
            r2 = sum(v * v for v in d) + L(eps) * L(eps)
            ri, m = 1 / np.sqrt(r2), L(p.m[1 - i])
            worst[0] = max(worst[0], float(abs(L(pot[2 * k + i]) / (-m * ri) - 1)))
            for q in range(3):
                if d[q] != 0:
                    worst[1] = max(worst[1], float(abs(L(a[2 * k + i, q]) / (m * ri * ri * ri * d[q]) - 1)))
    print(f"pair: potential {worst[0] / u:.2f} u, force {worst[1] / u:.2f} u", flush=True)
    assert worst[0] <= 4.25 * u and worst[1] <= 13.75 * u


@pytest.mark.parametrize("others", [[], [3], [1500], [40000], [140000, 7]])
def test_alone_and_in_a_batch(others):
    """How a launch splits the sources follows from its size (16 waves or 4, one
    half or two); a system's forces, potentials and energies do not."""
    ps = [ic.plummer(n, seed=n, virial=None) for n in (1, 2, 31, 33, 700, 1999)]
    with Engine(mode=MODE_PHYSICS, precision=PREC_FP64, eps=0.01) as e:
        e.upload_batch(ps + [ic.plummer(n, seed=n, virial=None) for n in others])
        a, pot = e.direct()
        energy = e.energy_systems(direct=True)
    at = 0
    for k, p in enumerate(ps):
        with Engine(mode=MODE_PHYSICS, precision=PREC_FP64, eps=0.01) as f:
            f.upload(p)
            b, bpot = f.direct()
            assert np.array_equal(a[at:at + len(p)], b) and np.array_equal(pot[at:at + len(p)], bpot), len(p)
            assert np.array_equal(energy[k], f.energy_systems(direct=True)[0]), len(p)
        at += len(p)
