"""The upward pass in units of bodies (reference mode up to 393,216 bodies):
whole node tables against the oracle's, bit for bit, at the sizes where the
number of units changes (at most 768 bodies each, one unit up to 1,230), with
clumps whose chains of cells make a unit too large for LDS, with several systems
in a context, and at both sides of the size where a launch per depth takes over.
"""
import numpy as np
import pytest

import oracle_lib as orc
from next_amd import ic
from next_amd.nbx import Engine

pytestmark = pytest.mark.gpu


def same_tables(p, theta=0.7):
    with Engine(theta=theta) as e:
        e.upload(p)
        t = e.debug_tree()
    o = orc.tree(p.x, p.y, p.z, p.m)
    for key in ("depth", "leaf", "body", "cmask", "perm", "geo", "mass", "com", "q"):
        assert np.array_equal(t[key], o[key]), key


@pytest.mark.parametrize("n", [1, 2, 3, 767, 1535, 1536, 1537, 2304, 5000])
def test_unit_counts(n):
    same_tables(ic.plummer(n, seed=n, virial=None))


@pytest.mark.parametrize("n", [1200, 4000])
def test_units_too_large_for_lds(n):
    """Pairs 1e-9 apart share about 30 digits: a chain of 30 cells per pair."""
    p = ic.uniform_sphere(n, seed=n)
    rng = np.random.Generator(np.random.PCG64(n))
    k = np.arange(0, n // 3 * 2, 2)
    for a in (p.x, p.y, p.z):
        a[k + 1] = a[k] + rng.normal(size=len(k)) * 1e-9
    p.m[::11] = 0.0
    same_tables(p)


@pytest.mark.parametrize("n", [262144, 262145])
def test_both_sides_of_the_largest(n):
    same_tables(ic.plummer(n, seed=2, virial=None))


@pytest.mark.parametrize("n", [1230, 1231, 2305, 3073, 16385])
def test_units_of_equal_length(n):
    same_tables(ic.plummer(n, seed=n, virial=None))


@pytest.mark.parametrize("n", [393216, 393217])
def test_both_sides_of_512_units(n):
    same_tables(ic.plummer(n, seed=2, virial=None))


def test_systems_share_units():
    """Forces of systems of very different sizes in one context (units and the
    nodes beyond them hold several systems) equal each system's alone."""
    ps = [ic.plummer(n, seed=n, virial=None) for n in (1, 3000, 5, 800, 40, 9000, 1535, 2)]
    with Engine(theta=0.5) as e:
        e.upload_batch(ps)
        e.run(1e-3, 2)
        got = [e.download_system(s) for s in range(len(ps))]
    for s, p in enumerate(ps):
        with Engine(theta=0.5) as f:
            f.upload(p)
            f.run(1e-3, 2)
            assert np.array_equal(got[s], f.download()), s


def test_more_systems_than_workgroups():
    """Nodes beyond their units are worked off by at most 512 workgroups, and
    systems of up to half a unit have none: systems on both sides of that, and
    beyond the 512th, among many tiny ones."""
    small, large = ic.plummer(2, seed=1, virial=None), [ic.plummer(n, seed=n, virial=None) for n in
                                                       (3000, 383, 384, 385, 386, 5000, 770)]
    ps = [large[5]] + [small] * 600 + large + [small] * 500 + [large[0]]
    with Engine(theta=0.5) as e:
        e.upload_batch(ps)
        e.run(1e-3, 2)
        got = {k: e.download_system(k) for k in [0, 1, 600, 1100, len(ps) - 1] + list(range(601, 608))}
    for k, state in got.items():
        with Engine(theta=0.5) as f:
            f.upload(ps[k])
            f.run(1e-3, 2)
            assert np.array_equal(state, f.download()), k
