"""Physics-mode walk: launches of few groups (up to 1,280, or 768 in FP64, or some
thousand of larger systems; not systems below 128 bodies) have further waves that
evaluate the lists, others one wave per group.  Both add the same terms in the
same order, so a system's results are the same bits alone (few groups) and
beside a large system that takes the launch over every such number.
"""
import numpy as np
import pytest

from next_amd import ic
from next_amd.nbx import MODE_PHYSICS, PREC_FP64, PREC_MIXED, Engine

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 5, 33, 64, 65, 129, 700, 5000]
LARGE = 700000


def run(ps, precision, alpha, steps):
    with Engine(theta=0.5, eps=0.01, mode=MODE_PHYSICS, precision=precision, adaptive_dt=False, alpha=alpha) as e:
        e.upload_batch(ps)
        a = e.accel()
        pot = e.potential()
        groups = len(e.debug_groups()[0])
        e.run(1e-3, steps)
        return groups, np.concatenate([a, pot[:, None], np.stack(e.download(), 1)], 1)


@pytest.mark.parametrize("precision,alpha", [(PREC_MIXED, 0.0), (PREC_FP64, 0.0), (PREC_MIXED, 1e-3)])
def test_same_bits_alone_and_beside_a_large_system(precision, alpha):
    ps = [ic.plummer(n, seed=n, virial=None) for n in SIZES]
    groups, got = run(ps + [ic.plummer(LARGE, seed=1, virial=None)], precision, alpha, 2)
    assert groups > 10240
    at = 0
    for p in ps:
        few, alone = run([p], precision, alpha, 2)
        assert few < 10240 * 4 // 5 - 64
        assert np.array_equal(got[at:at + len(p)], alone), len(p)
        at += len(p)


@pytest.mark.parametrize("precision", [PREC_MIXED, PREC_FP64])
@pytest.mark.parametrize("copies,group_size", [(1, 64), (60, 64), (1, 32), (60, 32), (60, 16)])
def test_same_bits_in_batches_of_any_width(copies, group_size, precision):
    """The choice follows the mean size of the systems, the number of groups and
    their size: small systems alone, beside copies of themselves and beside one
    that lifts the mean."""
    ps = [ic.plummer(n, seed=n, virial=None) for n in (127, 128, 700, 4100)]
    kw = dict(theta=0.5, eps=0.01, mode=MODE_PHYSICS, precision=precision, adaptive_dt=False, group_size=group_size)
    with Engine(**kw) as e:
        e.upload_batch(ps * copies + [ic.plummer(40000, seed=2, virial=None)])
        a, pot = e.accel(), e.potential()
    at = 0
    for p in ps:
        with Engine(**kw) as f:
            f.upload(p)
            assert np.array_equal(a[at:at + len(p)], f.accel()), len(p)
            assert np.array_equal(pot[at:at + len(p)], f.potential()), len(p)
        at += len(p)
