"""The kinetics callbacks' packed tables at the edges of their layout: reaction
counts around the lanes of a group and around the passes of the rate loop, species
lists of no entry, of a whole batch and of one more, and empty slots anywhere in
a side.  dydt and the Jacobian against the oracle's.
"""
import dataclasses

import numpy as np
import pytest

import accelerint_amd as acc
from accelerint_amd import mechanism as M

pytestmark = pytest.mark.gpu

# 14 states: 16-lane groups; 54 and 112 states: 64-lane groups, two reactions per pass
SIZES = [(14, 1), (14, 15), (14, 16), (14, 17), (14, 27), (54, 1), (54, 63), (54, 64), (54, 65), (54, 127), (54, 128),
         (54, 129), (54, 193), (112, 1), (112, 129)]


@pytest.fixture
def session():
    acc.lib()
    yield acc
    acc.cleanup()


def first_reactions(n, nr):
    """The network's first nr reactions, every second one with its empty slots first."""
    m = M.network(n)
    slots = m.slots[:nr].copy()
    for j in range(0, nr, 2):
        for lo in (0, 3):
            side = slots[j, lo:lo + 3]
            slots[j, lo:lo + 3] = np.concatenate([side[side < 0], side[side >= 0]])
    return dataclasses.replace(m, nr=nr, slots=slots, lnA=m.lnA[:nr].copy(), beta=m.beta[:nr].copy(),
                               EaR=m.EaR[:nr].copy())


@pytest.mark.parametrize("n,nr", SIZES)
def test_callbacks_of_partial_networks(session, oracle_lib, n, nr):
    mech = first_reactions(n, nr)
    num = 5
    y0, P = M.initial_conditions(mech, num, seed=7 * n + nr)
    acc.set_kinetics(mech)
    acc.set_abort_on_error(False)
    acc.initialize(num, 0)
    dy, jac = acc.eval_callbacks(num, 0.0, y0, P)
    om = oracle_lib.Mechanism.kinetics(mech)
    for c in range(num):
        fo = oracle_lib.dydt(om, 0.0, P[c], y0[:, c])
        Jo = oracle_lib.jacobian(om, 0.0, P[c], y0[:, c])
        # the bars of the full networks' callback tests: rounding of the sums
        assert np.allclose(dy[:, c], fo, rtol=1e-11, atol=1e-12 * np.abs(fo).max())
        scale = np.abs(Jo).max(1, keepdims=True)
        assert (np.abs(jac[c] - Jo) <= 1e-11 * scale).all()


def test_longest_list_is_whole_batches():
    """The sizes above hold lists on both sides of a whole batch of eight entries."""
    rests = set()
    for n, nr in SIZES:
        s = first_reactions(n, nr).slots
        rests |= {sum(int(k in row) for row in s) % 8 for k in range(n - 1)}
    assert {0, 1, 7} <= rests
