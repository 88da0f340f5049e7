"""GPU parity of small products on 16 x 16 and 32 x 32 tiles whose wavefronts share the k range: every
form against float64 and against the plain form's bits, at the edges of the tiles and of k."""
import ctypes

import numpy as np
import pytest

from gpu_util import Gpu, assert_bits_equal, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return Gpu()


def _rand(shape, seed):
    return np.random.default_rng(seed).standard_normal(shape).astype(np.float32)


def _product(gpu, form, A, B, *mid, out=None):
    """A (m, k) times B (k, n) through mnv_sgemm_<form>, without workspace; NaN where nothing is stored."""
    (m, k), n = A.shape, B.shape[1]
    a = gpu.up(np.ascontiguousarray(A if "tn" in form else A.T).reshape(-1))
    b = gpu.up(np.ascontiguousarray(B if "nt" in form else B.T).reshape(-1))
    c = gpu.up(np.full(m * n, np.nan, np.float32))
    args = [a.p, b.p] + list(mid[:1]) + [c.p, m, n, k] + list(mid[1:]) + [None, ctypes.c_size_t(0)]
    gpu.call("mnv_sgemm_" + form, *args)
    return gpu.down(c).reshape(n, m).T


# one value; tiles short by and past one row and column; k of less than a fetch, one more or less than 32, the waves' ranges
# unequal or empty; tall and wide; 32 x 32 tiles with four and with eight wavefronts
SHAPES = [(1, 1, 1), (15, 17, 3), (16, 16, 32), (17, 33, 31), (33, 15, 33), (100, 7, 257), (5, 300, 1023), (1, 40, 64), (40, 1, 129),
          (257, 255, 783), (10, 256, 256), (784, 256, 255), (513, 511, 509), (1421, 284, 487), (37, 3000, 300), (3001, 50, 402)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_small_products_in_every_form(gpu, m, n, k):
    say("small product", m, n, k)
    v = [ctypes.c_int() for _ in range(3)]
    assert gpu.L.mnv_sgemm_nn_plan(m, n, k, ctypes.c_size_t(0), *[ctypes.byref(x) for x in v]) == 0
    assert [x.value for x in v] == [64, 1, 1] and gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k) == 0
    A, B = _rand((m, k), m + k), _rand((k, n), n)
    got = _product(gpu, "nn", A, B)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    # each wavefront adds at most k products one by one: k roundings of 2^-24 of sums within |A||B|
    assert np.all(np.abs(got - A64 @ B64) <= (k + 8) * 2.0 ** -24 * (np.abs(A64) @ np.abs(B64)))
    assert_bits_equal(_product(gpu, "nt", A, B).ravel(), got.ravel(), "B transposed")
    assert_bits_equal(_product(gpu, "tn", A, B, None).ravel(), got.ravel(), "A transposed")
    bias, gate = _rand((m, 1), 3), _rand((m, n), 4)
    db, dg = gpu.up(bias.reshape(-1)), gpu.up(np.ascontiguousarray(gate.T).reshape(-1))
    biased = got + bias
    assert_bits_equal(_product(gpu, "nn_bias", A, B, db.p, 1).ravel(), np.where(biased > 0, biased, np.float32(0)).ravel(), "bias, ReLU")
    assert_bits_equal(_product(gpu, "nn_relu_bwd", A, B, dg.p).ravel(), np.where(gate > 0, got, np.float32(0)).ravel(), "gate")


@pytest.mark.parametrize("m,n,k", [(17, 18, 37), (70, 35, 257)])
def test_infinities_stay_in_their_rows_and_columns(gpu, m, n, k):
    """What lies past the end of a row, a column or k of an operand is never multiplied into the result."""
    A, B = _rand((m, k), 1), _rand((k, n), 2)
    A[2, k - 1], A[m - 1, 0], B[0, n - 1], B[k - 1, 1] = np.inf, np.nan, np.inf, np.nan
    with np.errstate(invalid="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
    for form, mid in (("nn", ()), ("nt", ()), ("tn", (None,))):
        got = _product(gpu, form, A, B, *mid)
        assert np.array_equal(np.isfinite(got), np.isfinite(want)), form
        assert np.array_equal(np.isnan(got), np.isnan(want)), form
