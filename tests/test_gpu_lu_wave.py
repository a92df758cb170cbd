"""Pivot search of the one-wavefront LU (order 54) and of the 16-lane groups' LU
(order 14, four matrices a wavefront) and of the panels of the blocked LU (order
112, two rows a lane) on candidates that agree in their leading 32 bits: the search compares those first and the rest only among
the rows that attain the maximum.  Interchanges must be the oracle's dgetrf /
zgetrf ones: the largest magnitude wins whichever bits decide it, and equal
magnitudes go to the first row in LAPACK's current order.
"""
import numpy as np
import pytest

import accelerint_amd as acc

pytestmark = pytest.mark.gpu

STEPS = [(54, 0), (54, 1), (54, 17), (54, 52), (14, 0), (14, 1), (14, 5), (14, 12),
         (112, 0), (112, 15), (112, 16), (112, 47), (112, 64), (112, 110)]


@pytest.fixture
def session():
    acc.lib()
    yield acc
    acc.cleanup()


def embedded(rng, N, k, column):
    """Order-N matrix whose step-k candidates are `column` (N - k values): a
    well-separated leading block first, rows of it shuffled so that the steps
    before k have interchanged rows."""
    a = np.zeros((N, N))
    for i in range(k):
        a[i, i] = 64.0  # exact elimination: the block below it is zero
    a[k:, k:] = 0.25 * rng.standard_normal((N - k, N - k))
    a[k:, k] = column
    a[:k, k:] = rng.standard_normal((k, N - k))
    rows = rng.permutation(N)
    return a[rows]


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("N,k", STEPS)
def test_low_bits_decide(session, oracle_lib, N, k, cplx):
    rng = np.random.default_rng(90 + k)
    mats = []
    for spread in (1, 3, 40, 1, 2):  # how many candidates share each value
        c = 1.0 + (rng.permutation(N - k) // spread) * 2.0 ** -50
        mats.append(embedded(rng, N, k, c * rng.choice([-1.0, 1.0], N - k)))
    a = np.array(mats)
    if cplx:  # pure real and pure imaginary candidates of one magnitude rule
        a = a * np.where(rng.random((len(mats), N, 1)) < 0.5, 1.0, 1.0j)
    _, ipiv, info = acc.factor_test(a, acc.PRECISION_FP64)
    f = oracle_lib.zgetrf if cplx else oracle_lib.dgetrf
    assert (info == 0).all()
    for m in range(len(mats)):
        assert np.array_equal(ipiv[m], f(a[m])[1])


@pytest.mark.parametrize("N,k", STEPS)
def test_equal_candidates_fp32(session, oracle_lib, N, k):
    rng = np.random.default_rng(190 + k)
    a = embedded(rng, N, k, rng.choice([-1.0, 1.0], N - k))
    a = a.astype(np.float32).astype(np.float64)[None]
    _, ipiv, info = acc.factor_test(a, acc.PRECISION_MIXED)
    assert info[0] == 0
    # the steps up to k are exact in FP32; later ones round
    assert np.array_equal(ipiv[0][:k + 1], oracle_lib.dgetrf(a[0])[1][:k + 1])
