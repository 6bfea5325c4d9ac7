"""The softening floor of dark-matter targets (octree.h:146-148),
2 size / (m/mi)^0.333333333, to the accuracy of a correctly rounded one.

Pairs of a heavy dark-matter body and a light source in opposite octants of
their root: at theta 0 the heavy body's force comes from the source's leaf
alone, and the floor exceeds every other length, so the force is
m d / (r^2 + floor^2)^1.5 and carries three times the floor's error.

Tolerance: 1/sqrt in the walk is the hardware's estimate and one Newton step,
relative error at most 4.2e-15 and 3.5e-16 in the root mean square (measured over
its mantissas), cubed in the force: 1.26e-14 and 1.05e-15.  The floor is right to
2 u (u = 2^-53; rounding of the powers, of the quotient and of the product,
carried along), cubed 6 u; eps^2 + r^2 is rounded once, 1.5 u in the force; three
products 3 u: 10.5 u = 1.2e-15 at most, below 4 u = 4.4e-16 in the root mean
square.  Together at most 1.4e-14, and 1.14e-15 in the root mean square, so half
of the pairs are within 1.6e-15 (sqrt 2 of that): 1.5e-14 for the largest error
and 2e-15 for the median.  A power whose logarithm is carried in 32 bits is off
by up to 7e-15 for masses between 1e-30 and 1e30 and by 3e-14 beyond, three
times that in the force.
"""
from decimal import Decimal, getcontext

import numpy as np
import pytest

import oracle_lib as orc
from next_amd import ic
from next_amd.nbx import Engine

pytestmark = pytest.mark.gpu

getcontext().prec = 50
POWER = Decimal(0.333333333)


def exact(p, size):
    """Force of body 1 on body 0 along x, floor alone as softening."""
    d = [Decimal(b) - Decimal(a) for a, b in ((p.x[0], p.x[1]), (p.y[0], p.y[1]), (p.z[0], p.z[1]))]
    m, mi = Decimal(p.m[1]), Decimal(p.m[0])
    floor = 2 * Decimal(size) / (POWER * (m / mi).ln()).exp()
    r2 = sum(x * x for x in d)
    assert floor > 100 * r2.sqrt()
    s = r2 + floor * floor
    return float(m * d[0] / (s * s.sqrt()))


@pytest.mark.parametrize("light,heavy", [((-6, 0), (8, 12)), ((-30, -10), (0, 30)), ((-40, 0), (60, 150)),
                                         ((-200, -180), (-140, -120))])
def test_floor_of_a_pair(light, heavy):
    rng = np.random.Generator(np.random.PCG64(17))
    ps = []
    for _ in range(200):
        c = rng.uniform(0.2, 1.0, 3)
        m = np.array([10.0 ** rng.uniform(*heavy), 10.0 ** rng.uniform(*light)])
        z = np.zeros(2)
        ps.append(ic.Particles(*(np.array([-c[k], c[k]]) for k in range(3)), z, z, z, m, np.array([1, 0], np.int32)))
    with Engine(theta=0.0) as e:
        e.upload_batch(ps)
        a = e.accel()
    err = []
    for k, p in enumerate(ps):
        want = exact(p, orc.root(p.x, p.y, p.z)[3] / 2)      # leaves one level below the root
        err.append(abs(a[2 * k, 0] - want) / abs(want))
    print(f"masses 1e{light} and 1e{heavy}: max {max(err):.2e} median {np.median(err):.2e}", flush=True)
    assert max(err) <= 1.5e-14 and np.median(err) <= 2e-15
