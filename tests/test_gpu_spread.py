"""A batch that does not fill the device is spread over it with a part of each
block's lane groups at work.  The part is chosen by the batch's size: at the sizes
around its steps every condition must end where it ends in a large batch, bit for
bit and with the same counts (a condition's integration uses its own group only).
"""
import numpy as np
import pytest

import accelerint_amd as acc
from accelerint_amd import mechanism as M

pytestmark = pytest.mark.gpu


@pytest.fixture
def session():
    acc.lib()
    yield acc
    acc.cleanup()


def run(mech, y0, P, precision):
    num = y0.shape[1]
    acc.set_kinetics(mech)
    acc.set_precision(precision)
    acc.set_abort_on_error(False)
    acc.initialize(num, 0)
    y = y0.copy(order="C")
    acc.integrate(num, 0.0, 1e-6, 1e-6, y, P[:num])
    out = y, acc.get_status(num), acc.get_counters(num)
    acc.cleanup()
    return out


@pytest.mark.parametrize("precision", [acc.PRECISION_FP64, acc.PRECISION_MIXED])
@pytest.mark.parametrize("n,groups", [(14, 8), (54, 4)])
def test_every_condition_of_a_small_batch(session, n, groups, precision):
    cus = 256  # compute units of the MI355X: the rule's steps lie at multiples of the resident blocks, 1 to 4 per unit
    mech = M.network(n)
    sizes = sorted({1, 2, groups - 1, groups, groups + 1} | {cus * m + d for m in (1, 2, 4) for d in (-1, 0, 1)})
    if n == 14:
        sizes += [8 * cus + 1, groups * 4 * cus]
    y0, P = M.initial_conditions(mech, max(sizes), seed=n)
    y, codes, counts = run(mech, y0, P, precision)
    assert (codes == 0).all()
    for num in sizes:
        ys, cs, ns = run(mech, y0[:, :num], P, precision)
        assert np.array_equal(ys, y[:, :num]), num
        assert np.array_equal(cs, codes[:num]) and np.array_equal(ns, counts[:num]), num
