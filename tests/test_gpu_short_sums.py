"""What sharing a reduction among wavefronts and summing it in runs of 32 leaves of the rounding errors of small
products and convolutions: their distance from float64 against what sums of that length can show."""
import ctypes
import math

import numpy as np
import pytest

from gpu_util import Gpu, say
from test_gpu_conv import Conv, _rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return Gpu()


def _bound(k, wavefronts):
    """Relative error (2-norm) of sums of k products of random signs.  Each rounding is off by at most 2^-24 of a partial
    sum, evenly spread: 2^-24 / sqrt(3) rms.  Partial sums of i products are sqrt(i) of one: the squares of those of a run of 32
    add up to 512, those of a wavefront's runs to (k / wavefronts)^2 / 64, those of the wavefronts to k (wavefronts + 1) / 2."""
    return 2.0 ** -24 / math.sqrt(3) * math.sqrt(16 + k / (64.0 * wavefronts) + (wavefronts + 1) / 2)


def _closer_bound(k, wavefronts, run):
    """The same for runs of `run` and the mean rounding: ulp / sqrt(12), which for values whose logarithms are evenly spread is
    0.4247 * 2^-24 of them; a twelfth on top."""
    return 1.08 * 0.4247 * 2.0 ** -24 * math.sqrt(run / 2 + k / (2.0 * run * wavefronts) + (wavefronts + 1) / 2)


def _error(got, want):
    return np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want)


# 16 x 16 and 32 x 32 tiles, four and eight wavefronts
@pytest.mark.parametrize("m,n,k,wavefronts", [(57, 3024, 2539, 8), (246, 1164, 1070, 4), (328, 53, 1276, 8), (1001, 250, 4099, 4)])
def test_small_products(gpu, m, n, k, wavefronts):
    say("error of a small product", m, n, k)
    rng = np.random.default_rng(k)
    A, B = rng.standard_normal((m, k), np.float32), rng.standard_normal((k, n), np.float32)
    a, b = gpu.up(np.ascontiguousarray(A.T).reshape(-1)), gpu.up(np.ascontiguousarray(B.T).reshape(-1))
    c = gpu.empty(m * n)
    gpu.call("mnv_sgemm_nn", a.p, b.p, c.p, m, n, k, None, ctypes.c_size_t(0))
    assert _error(gpu.down(c).reshape(n, m).T, A.astype(np.float64) @ B.astype(np.float64)) <= _bound(k, wavefronts)


def _convolution(gpu, p, passes):
    """Its error and the length of its longest sums."""
    import torch
    N, C, K, H, W, ph, pw, sv, sh, R, S = p
    say("error of a small convolution", p, passes)
    cv = Conv(gpu, *p)
    w = _rand(K * C * R * S, 1)
    flat = torch.from_numpy(w).double().view(K, C, R, S).flip(2, 3)  # a true convolution
    if passes == "fwd":
        x, bias = _rand(N * C * H * W, 2), np.zeros(K, np.float32)
        want = torch.nn.functional.conv2d(torch.from_numpy(x).double().view(N, C, H, W), flat, stride=(sv, sh), padding=(ph, pw))
        got, k = cv.fwd(x, w, bias), C * R * S
    else:
        dy = _rand(N * K * cv.Ho * cv.Wo, 3)
        rest = (H + 2 * ph - R) % sv, (W + 2 * pw - S) % sh
        want = torch.nn.functional.conv_transpose2d(torch.from_numpy(dy).double().view(N, K, cv.Ho, cv.Wo), flat, stride=(sv, sh),
                                                    padding=(ph, pw), output_padding=rest)
        got, k = cv.bwd_data(dy, w), K * -(-R // sv) * -(-S // sh)  # of the class with the most taps
    return _error(got, want.numpy().reshape(-1)), k


@pytest.mark.parametrize("p,passes", [  # no k ranges: each runs in the permuted filter or the filter in place
    ((15, 288, 32, 16, 32, 0, 0, 1, 1, 3, 3), "fwd"), ((2, 48, 160, 31, 49, 1, 1, 1, 1, 3, 3), "bwd_data"),
    ((60, 16, 280, 26, 14, 1, 1, 1, 1, 3, 3), "bwd_data"), ((32, 48, 80, 10, 32, 0, 0, 1, 1, 5, 5), "bwd_data"),
    ((59, 80, 32, 48, 20, 2, 2, 2, 2, 5, 5), "fwd"), ((21, 40, 288, 51, 9, 0, 0, 2, 2, 3, 3), "bwd_data"),
    ((34, 120, 120, 26, 11, 1, 1, 2, 2, 2, 2), "bwd_data"), ((47, 64, 64, 16, 27, 1, 1, 2, 2, 3, 3), "bwd_data"),
], ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else v)
def test_small_convolutions(gpu, p, passes):
    error, k = _convolution(gpu, p, passes)
    assert error <= _bound(k, 4)


@pytest.mark.parametrize("p,passes", [  # up to three slabs of 16 per wavefront, one of them a run
    ((23, 216, 72, 8, 11, 1, 1, 2, 2, 2, 2), "bwd_data"), ((3, 192, 72, 48, 8, 0, 0, 2, 2, 2, 2), "bwd_data"),
    ((45, 24, 96, 13, 37, 0, 0, 2, 2, 2, 2), "bwd_data"), ((27, 48, 16, 8, 34, 0, 0, 2, 2, 5, 5), "bwd_data"),
], ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else v)
def test_short_reductions_of_convolutions(gpu, p, passes):
    error, k = _convolution(gpu, p, passes)
    assert error <= _closer_bound(k, 4, 16)


@pytest.mark.parametrize("p", [(51, 112, 48, 33, 50, 1, 1, 2, 2, 3, 3), (80, 136, 64, 24, 12, 2, 2, 2, 2, 5, 5)], ids=lambda p: "-".join(map(str, p)))
def test_strided_data_gradients_in_parts(gpu, p):
    """One rounding of the full sum for 8 products: the partial sums' squares add up to k^2 / 16, and those of the smaller
    terms, at 2^-8 of them, do not count."""
    error, k = _convolution(gpu, p, "bwd_data")
    assert error <= 2.0 ** -24 / math.sqrt(3) * math.sqrt(k / 16 + 1)
