"""The reference-mode walk at the sizes where its group width changes.

The walk puts 64 / width lanes on each target of a group of `width` bodies;
the width follows the system's size and theta (8 for 896 to 4,096 bodies up to
theta 0.32; 16 below theta 0.35, up to 524,288 bodies below 0.4, 98,304 below
0.45, 20,480 up to 0.5 and 1,500 up to 0.55; else 32 up to 1,500 bodies, and up
to 196,608 between 0.4 and 0.8; else, and up to 64 bodies, 64).
Accelerations against the oracle's walk (octree.h:133-179) at the edges of
those ranges and of a group, with dark-matter targets (octree.h:146-148).
Tolerance: the accelerations' own, median <= 1e-12 and 99th percentile <=
1e-10 relative (the terms are the same, their order and the last bits of the
square roots differ: a few ulp each).
"""
import numpy as np
import pytest

import oracle_lib as orc
from next_amd import ic
from next_amd.nbx import Engine, NbxError

pytestmark = pytest.mark.gpu


def check(p, theta, what):
    with Engine(theta=theta) as e:
        e.upload(p)
        a = e.accel()
    n = len(p)
    tg = np.arange(n) if n <= 8192 else np.unique(np.concatenate(
        [np.arange(128), n - 1 - np.arange(128), np.random.Generator(np.random.PCG64(5)).choice(n, 4096, False)]))
    ao = orc.accel_subset(p.x, p.y, p.z, p.m, p.type, theta, tg.astype(np.int64))
    d = np.linalg.norm(ao, axis=1)
    err = np.linalg.norm(a[tg] - ao, axis=1) / np.where(d > 0, d, 1.0)
    print(f"{what}: median {np.median(err):.2e} p99 {np.percentile(err, 99):.2e} max {err.max():.2e}", flush=True)
    assert np.median(err) <= 1e-12 and np.percentile(err, 99) <= 1e-10


@pytest.mark.parametrize("theta", [0.0, 0.3, 0.5, 0.9])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 63, 64, 65, 257, 4095])
def test_small(n, theta):
    check(ic.plummer(n, seed=n, virial=None, type_fraction_dm=0.3), theta, f"n={n} theta={theta}")


@pytest.mark.parametrize("n,theta", [(4096, 0.5), (4097, 0.5), (98304, 0.39), (98305, 0.4), (98305, 0.39),
                                     (196608, 0.5), (196609, 0.5), (196609, 0.39), (4096, 0.32), (4097, 0.32),
                                     (4096, 0.33), (98304, 0.44), (98304, 0.45), (20480, 0.5), (20481, 0.5),
                                     (20480, 0.56), (196609, 0.56)])
def test_width_edges(n, theta):
    check(ic.plummer(n, seed=3, virial=None, type_fraction_dm=0.1), theta, f"n={n} theta={theta}")


@pytest.mark.parametrize("n,theta,width", [(64, 0.3, 64), (65, 0.3, 16), (895, 0.32, 16), (896, 0.32, 8),
                                           (1500, 0.55, 16), (1501, 0.55, 32), (1500, 0.56, 32), (1500, 0.95, 32),
                                           (1501, 0.8, 32), (1501, 0.81, 64), (20480, 0.51, 32), (196608, 0.81, 64),
                                           (524288, 0.35, 16), (524289, 0.35, 64), (524289, 0.34, 16)])
def test_widths(n, theta, width):
    p = ic.plummer(n, seed=8, virial=None, type_fraction_dm=0.1)
    with Engine(theta=theta) as e:
        e.upload(p)
        assert e.debug_groups()[1].max() == min(n, width)
    check(p, theta, f"n={n} theta={theta}")


@pytest.mark.parametrize("theta", [0.0, 0.05, 0.3, 0.7])
@pytest.mark.parametrize("scale", [1e-12, 1e-9, 1e-7, 1e17, 1e18, 1e20, 1e60])
def test_lengths_outside_fp32(scale, theta):
    """Metres instead of scale lengths, say: the squares of lengths, against
    which the opening test's band is kept, leave FP32's range."""
    p = ic.plummer(1500, seed=12, virial=None, type_fraction_dm=0.2)
    for a in (p.x, p.y, p.z):
        a *= scale
    check(p, theta, f"scale={scale} theta={theta}")


@pytest.mark.parametrize("theta", [0.0, 0.5])
def test_lengths_outside_fp32_in_a_batch(theta):
    ps = []
    for k, scale in enumerate((1.0, 1e20, 1e-9, 1e20, 1.0)):
        p = ic.plummer(700 + k, seed=k, virial=None)
        for a in (p.x, p.y, p.z):
            a *= scale
        ps.append(p)
    with Engine(theta=theta) as e:
        e.upload_batch(ps)
        a = e.accel()
    at = 0
    for p in ps:
        with Engine(theta=theta) as f:
            f.upload(p)
            assert np.array_equal(a[at:at + len(p)], f.accel())
        at += len(p)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_positions_that_are_not_finite(bad):
    p = ic.plummer(100, seed=1, virial=None)
    p.y[57] = bad
    with Engine(theta=0.5) as e:
        e.upload(p)
        with pytest.raises(NbxError):
            e.accel()


@pytest.mark.parametrize("lo,hi", [(-30, 30), (-3, 3), (200, 210), (-210, -200)])
def test_dark_matter_masses(lo, hi):
    """Masses over many orders of magnitude (zero among them): the softening
    floor's power of the mass ratio."""
    rng = np.random.Generator(np.random.PCG64(11))
    p = ic.plummer(600, seed=4, virial=None, type_fraction_dm=0.5)
    p.m[:] = 10.0 ** rng.uniform(lo, hi, len(p))
    p.m[::37] = 0.0
    # a zero-mass dark-matter target divides by its mass (octree.h:146): its floor is zero
    check(p, 0.5, f"masses 1e{lo}..1e{hi}")


@pytest.mark.parametrize("n", [200003, 1 << 20])
def test_sums_of_wide_groups(n):
    """A lane that has a target to itself adds up to some thousand terms, the
    distant nodes of the whole group first.  Against 64-bit mantissas, the median
    error may exceed that of NEXT's own FP64 walk by 30 % (1/sqrt by a Newton
    step where NEXT's is correctly rounded); in one running sum from far to near it
    did by 46 %, summed list by list it does by 3 to 12."""
    p = ic.uniform_sphere(n, seed=1)
    with Engine(theta=0.5) as e:
        e.upload(p)
        a = e.accel()
    tg = np.random.Generator(np.random.PCG64(1)).choice(n, 4096, False).astype(np.int64)
    hi, lo = orc.accel_subset_ext(p.x, p.y, p.z, p.m, p.type, 0.5, tg)
    scale = np.linalg.norm(hi, axis=1)
    mine, nexts = (np.median(np.linalg.norm((v - hi) - lo, axis=1) / scale)
                   for v in (a[tg], orc.accel_subset(p.x, p.y, p.z, p.m, p.type, 0.5, tg)))
    print(f"n={n}: median error {mine:.2e}, NEXT's {nexts:.2e}", flush=True)
    assert mine <= 1.3 * nexts


def test_theta_changes_the_width():
    """A context whose theta moves across the width rule gives the forces of
    a fresh context at that theta."""
    p = ic.plummer(100000, seed=6, virial=None)
    with Engine(theta=0.5) as e:
        e.upload(p)
        e.accel()
        e.set_theta(0.35)
        a = e.accel()
        e.set_theta(0.5)
        b = e.accel()
    for theta, got in ((0.35, a), (0.5, b)):
        with Engine(theta=theta) as f:
            f.upload(p)
            assert np.array_equal(got, f.accel())


def test_setting_theta_allocates_nothing():
    """nbx_set_theta marks; the next evaluation brings the group table up to
    date, captured runs included."""
    ps = [ic.plummer(n, seed=n, virial=None) for n in (200003, 5000)]
    with Engine(theta=0.5, adaptive_dt=False) as e:
        e.set_graph(1)
        e.upload_batch(ps)
        e.run(1e-4, 4)
        held = e.device_bytes()
        e.set_theta(0.35)               # four times as many groups for the first system
        assert e.device_bytes() == held
        e.run(1e-4, 4)
        got = e.download()
    with Engine(theta=0.5, adaptive_dt=False) as f:
        f.upload_batch(ps)
        for theta in (0.5, 0.35):
            f.set_theta(theta)
            for _ in range(4):
                f.step(1e-4)
        assert np.array_equal(got, f.download())


@pytest.mark.parametrize("sizes", [[1, 20481], [20481, 1, 1, 1], [20480, 20481], [5, 70, 30000, 3, 21000, 600], [25000] + [9] * 40])
def test_batch_of_mixed_widths(sizes):
    """The group table of a batch whose widths differ is cut by bodies: every
    system gets its forces alone, bit for bit."""
    ps = [ic.plummer(n, seed=k, virial=None, type_fraction_dm=0.2) for k, n in enumerate(sizes)]
    with Engine(theta=0.5) as e:
        e.upload_batch(ps)
        a = e.accel()
    at = 0
    for p in ps:
        with Engine(theta=0.5) as f:
            f.upload(p)
            assert np.array_equal(a[at:at + len(p)], f.accel())
        at += len(p)


@pytest.mark.parametrize("sizes", [[1], [1000], [20481], [1, 20481], [5, 70, 30000, 3, 21000, 600], [25000] + [9] * 40])
def test_group_table(sizes):
    """The groups the walk works through cover each body once, inside one
    system, in runs of that system's width, before and after theta moves it."""
    ps = [ic.plummer(n, seed=k, virial=None) for k, n in enumerate(sizes)]
    with Engine(theta=0.5) as e:
        e.upload_batch(ps)
        for theta in (0.5, 0.3, 0.9):
            e.set_theta(theta)
            first, count, sys_ = e.debug_groups()
            order = np.argsort(first)
            assert np.array_equal(first[order], np.concatenate([[0], np.cumsum(count[order])[:-1]]))
            assert count.sum() == sum(sizes)
            at = 0
            for s, n in enumerate(sizes):
                c = count[sys_ == s]
                assert c.sum() == n and np.all((first[sys_ == s] >= at) & (first[sys_ == s] + c <= at + n))
                width = {(1000, 0.5): 16, (20481, 0.5): 32, (20481, 0.3): 16, (30000, 0.5): 32}.get((n, theta))
                if width is not None:
                    assert c.max() == width and np.sum(c < width) <= 1, (n, theta)
                at += n
