"""Products that leave grouped 64 x 64 tiles for 128 x 128 ones in bf16 parts: which do, and their parity against float64
with the queried workspace, with part of it and without."""
import ctypes

import numpy as np
import pytest

from minerva_amd import capi


def _plan(m, n, k, ws):
    v = [ctypes.c_int() for _ in range(3)]
    assert capi.lib().mnv_sgemm_nn_plan(m, n, k, ctypes.c_size_t(ws), *[ctypes.byref(x) for x in v]) == 0
    return tuple(x.value for x in v)


# 17 to 63 tiles of 128 x 128, ragged in every extent; 65 and more
MOVED = [(1340, 599, 3458), (2500, 200, 2048), (2048, 300, 3000), (341, 3956, 1002), (2177, 1155, 3047)]
# at most 16 tiles; one grouped tile per CU; ranges of under 20 us; ranges that gain nothing, or too little
STAY = [(200, 1000, 4099), (500, 500, 3000), (1000, 256, 4096), (4096, 256, 4096), (3312, 73, 1235), (143, 2058, 1764),
        (797, 3646, 888), (423, 3418, 592)]
# the k ranges of the grouped tiles; in parts with as many, or few more, sums of positive terms were less exact
RANGES = [(2177, 1155, 3047, 1), (2408, 1161, 2681, 1), (2871, 1084, 1927, 1), (3803, 2309, 2023, 1), (2048, 300, 3000, 3)]


@pytest.mark.parametrize("m,n,k", MOVED)
def test_products_weighed_against_the_parts(m, n, k):
    assert _plan(m, n, k, capi.lib().mnv_sgemm_nn_workspace_bytes(m, n, k))[0::2] == (128, 1)


@pytest.mark.parametrize("m,n,k", STAY)
def test_products_that_stay_on_small_tiles(m, n, k):
    assert _plan(m, n, k, 1 << 40)[0] == 64


@pytest.mark.parametrize("m,n,k,grouped", RANGES)
def test_parts_have_at_least_twice_the_ranges_of_the_grouped_tiles(m, n, k, grouped):
    """Whatever is lent; without a workspace there are no ranges, and the grouped tiles stay."""
    full = capi.lib().mnv_sgemm_nn_workspace_bytes(m, n, k)
    for ws in (0, 4 * m * n, full // 2, full, 1 << 40):
        rows, ranges, _ = _plan(m, n, k, ws)
        assert rows == 64 or (ws and ranges >= 2 * grouped), ws


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,grouped", RANGES)
def test_sums_of_positive_terms_are_as_exact_as_on_the_grouped_tiles(m, n, k, grouped):
    """Their distance from float64 (2-norm, relative) is that of 4 * grouped sums of k / (4 * grouped) positive terms,
    rounded at each: the squares of the partial sums of all add up to k / 48 / grouped^2 of the whole sum's.  A rounding
    is 0.4247 * 2^-24 of its value where logarithms are evenly spread; a tenth, and the additions of the ranges, on top."""
    from gpu_util import Gpu, say
    gpu = Gpu()
    rng = np.random.default_rng(k)
    A, B = rng.random((m, k), np.float32), rng.random((k, n), np.float32)
    exact = A.astype(np.float64) @ B.astype(np.float64)
    ws = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k)
    say("positive terms", m, n, k, "plan", _plan(m, n, k, ws))
    a, b = gpu.up(np.ascontiguousarray(A.T).reshape(-1)), gpu.up(np.ascontiguousarray(B.T).reshape(-1))
    c, scratch = gpu.empty(m * n), gpu.empty(max(1, ws // 4))
    gpu.call("mnv_sgemm_nn", a.p, b.p, c.p, m, n, k, scratch.p, ctypes.c_size_t(ws))
    error = np.linalg.norm(gpu.down(c).reshape(n, m).T.astype(np.float64) - exact) / np.linalg.norm(exact)
    assert error <= 1.1 * 0.4247 * 2.0 ** -24 * np.sqrt(k / 48 / grouped ** 2 + 4 * grouped / 3 + 1)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", MOVED)
def test_weighed_products_against_float64(m, n, k):
    from gpu_util import Gpu, say
    gpu = Gpu()
    rng = np.random.default_rng(k)
    A, B = rng.standard_normal((m, k), np.float32), rng.standard_normal((k, n), np.float32)
    # sums of k products round at most k times, by 2^-24 of sums within |A||B|; the parts leave out 3 x 2^-25 of a product
    exact = A.astype(np.float64) @ B.astype(np.float64)
    bound = (k + 8) * 2.0 ** -24 * (np.abs(A) @ np.abs(B)).astype(np.float64)
    a, b = gpu.up(np.ascontiguousarray(A.T).reshape(-1)), gpu.up(np.ascontiguousarray(B.T).reshape(-1))
    full = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k)
    for ws in (full, full // 2, 0):
        say("weighed product", m, n, k, "workspace", ws, "plan", _plan(m, n, k, ws))
        c, scratch = gpu.up(np.full(m * n, np.nan, np.float32)), gpu.up(np.full(max(1, ws // 4), np.nan, np.float32))
        gpu.call("mnv_sgemm_nn", a.p, b.p, c.p, m, n, k, scratch.p, ctypes.c_size_t(ws))
        assert np.all(np.abs(gpu.down(c).reshape(n, m).T - exact) <= bound), ws


def _rounding(sums, k, ranges):
    """Relative rms error of sums of positive terms in `ranges` ranges of k, rounded at every eighth k, that are added four at a
    time: a rounding is evenly spread over a unit in the last place of the partial sum, whose size is its share of the whole."""
    shares = [np.arange(8, k / ranges, 8) / k] * ranges
    for first in range(0, ranges, 4):
        four = min(4, ranges - first)
        shares += [np.array([2, 2, 4] if four == 4 else range(2, four + 1)) / ranges]  # (0 + 1) + (2 + 3); what is left in order
        shares += [np.array([first + four] if first else []) / ranges]
    units = np.exp2(np.floor(np.log2(sums[:, None] * np.concatenate(shares))) - 23)
    return np.sqrt((units ** 2).sum(1).mean() / 12 / (sums ** 2).mean())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,ranges", [(379, 646, 3505, 14), (123, 2426, 3647, 13), (255, 1163, 3665, 12)])
def test_partial_results_are_added_four_at_a_time(m, n, k, ranges):
    """Both operands from a ReLU.  One after the other, the additions make the error 1.19 to 1.4 times the bound."""
    from gpu_util import Gpu, say
    gpu = Gpu()
    rng = np.random.default_rng(k)
    A, B = (np.maximum(rng.standard_normal(s, np.float32), np.float32(0)) for s in ((m, k), (k, n)))
    exact = A.astype(np.float64) @ B.astype(np.float64)
    ws = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k)
    say("partial results", m, n, k, "plan", _plan(m, n, k, ws))
    assert _plan(m, n, k, ws) == (128, ranges, 1)
    a, b = gpu.up(np.ascontiguousarray(A.T).reshape(-1)), gpu.up(np.ascontiguousarray(B.T).reshape(-1))
    c, scratch = gpu.empty(m * n), gpu.empty(ws // 4)
    gpu.call("mnv_sgemm_nn", a.p, b.p, c.p, m, n, k, scratch.p, ctypes.c_size_t(ws))
    error = np.linalg.norm(gpu.down(c).reshape(n, m).T.astype(np.float64) - exact) / np.linalg.norm(exact)
    assert error <= 1.04 * _rounding(exact.reshape(-1)[::97], k, ranges)
