"""The sort of small systems (one launch up to 16,384 bodies, in place of the
nearly-sorted path up to 4,096) at the edges of its range and of a workgroup:
leaf order and keys against the oracle's, bit for bit, with bodies that share
the whole first key word (ordered by the second), on a first build and on the
builds of some steps.
"""
import numpy as np
import pytest

import oracle_lib as orc
from next_amd import ic
from next_amd.nbx import Engine

pytestmark = pytest.mark.gpu


def with_clumps(n, seed):
    """A Plummer sphere with a few clumps of bodies within 1e-9 of each other."""
    p = ic.plummer(n, seed=seed, virial=None)
    rng = np.random.Generator(np.random.PCG64(seed))
    for k in range(0, n - 5, max(n // 7, 6)):
        for a in (p.x, p.y, p.z):
            a[k:k + 4] = a[k] + rng.normal(size=4) * 1e-9
        for a in (p.vx, p.vy, p.vz):
            a[k:k + 4] = a[k]
    p.m[:] = 1e-14                     # negligible forces: the clumps stay together
    return p


def same_tree(e):
    x, y, z, *_ = e.download()
    t = e.debug_tree()
    o = orc.tree(x, y, z, np.full(len(x), 1e-14))
    for key in ("perm", "depth", "leaf", "body", "cmask"):
        assert np.array_equal(t[key], o[key]), key


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 4095, 4096, 4097, 16383, 16384, 16385])
def test_order(n):
    with Engine(theta=0.7, adaptive_dt=False) as e:
        e.upload(with_clumps(n, n))
        same_tree(e)
        e.run(1e-3, 3)
        same_tree(e)
