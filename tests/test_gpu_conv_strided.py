"""GPU parity of the data gradient of strided convolutions, whose positions are taken class by class
modulo the strides: against the CPU oracle on all tiles, with and without k ranges, and where classes
are empty, have no taps, or hold one position more or less than the others."""
import ctypes

import numpy as np
import pytest

from gpu_util import Gpu, TOL, normwise, say
from test_gpu_conv import Conv, _out, _rand
from oracle import mnv_oracle as ora

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return Gpu()


CASES = [  # N, C, K, H, W, ph, pw, sv, sh, R, S
    (2, 16, 16, 9, 9, 1, 1, 2, 2, 3, 3),
    (3, 40, 20, 11, 8, 0, 0, 2, 2, 3, 3),       # channels padded to 32
    (1, 33, 5, 13, 7, 2, 2, 2, 2, 5, 5),        # 5 channels to 16
    (2, 24, 48, 14, 15, 0, 0, 2, 2, 1, 1),      # three of four classes meet no tap
    (2, 17, 16, 12, 9, 1, 0, 2, 1, 3, 2),       # one direction only
    (2, 17, 16, 9, 12, 0, 1, 1, 3, 2, 4),
    (1, 20, 32, 23, 23, 0, 0, 4, 4, 11, 11),
    (2, 16, 16, 7, 6, 0, 0, 5, 4, 3, 3),        # filter below the stride: rows that meet nothing
    (1, 16, 16, 2, 2, 1, 1, 3, 3, 3, 3),        # planes below the stride: empty classes
    (2, 9, 16, 8, 7, 4, 3, 2, 3, 3, 2),         # padding beyond the filter
    (13, 24, 232, 49, 19, 0, 0, 2, 2, 3, 3),    # 128 x 32 tiles, k ranges
    (21, 184, 120, 31, 7, 0, 0, 2, 2, 3, 3),    # 64 x 64 tiles, k ranges
    (64, 144, 16, 20, 20, 1, 1, 2, 2, 3, 3),    # 128 x 128 / 96 tiles
    (40, 192, 96, 28, 28, 1, 1, 2, 2, 3, 3),    # bf16 parts, 96 columns
    (24, 256, 104, 15, 45, 2, 2, 2, 2, 5, 5),   # bf16 parts, 128 columns, channels padded
]


@pytest.mark.parametrize("p", CASES, ids=lambda p: "-".join(map(str, p)))
def test_strided_data_gradient_matches_the_oracle(gpu, p):
    N, C, K, H, W, ph, pw, sv, sh, R, S = p
    say("strided data gradient", p)
    cv = Conv(gpu, *p)
    dy, w = _rand(N * K * cv.Ho * cv.Wo, 5), _rand(K * C * R * S, 6)
    ref = ora.conv_bwd_data(dy, w, *p)
    for workspace in (True, False):  # without: the generic gathers
        assert normwise(cv.bwd_data(dy, w, workspace), ref) <= TOL


BEYOND = [  # strides beyond the plane in one direction or both: fewer classes than sv * sh
    (64, 64, 64, 2, 2, 1, 1, 20, 20, 3, 3),
    (17, 24, 344, 5, 3, 1, 0, 1, 6, 5, 2),
    (32, 16, 224, 5, 2, 0, 0, 1, 7, 5, 2),      # k ranges
    (9, 33, 40, 1, 37, 0, 1, 2, 2, 1, 3),       # one row
    (7, 20, 48, 3, 4, 2, 3, 5, 4, 4, 5),        # the other direction's stride is the plane's extent
    (700, 64, 128, 3, 2, 1, 2, 4, 8, 5, 5),
    (900, 96, 256, 3, 2, 1, 1, 4, 4, 3, 3),     # bf16 parts
]


@pytest.mark.parametrize("p", BEYOND, ids=lambda p: "-".join(map(str, p)))
def test_strides_beyond_the_plane_match_the_oracle(gpu, p):
    N, C, K, H, W, ph, pw, sv, sh, R, S = p
    say("strides beyond the plane", p)
    cv = Conv(gpu, *p)
    dy, w = _rand(N * K * cv.Ho * cv.Wo, 5), _rand(K * C * R * S, 6)
    ref = ora.conv_bwd_data(dy, w, *p)
    for workspace in (True, False):
        assert normwise(cv.bwd_data(dy, w, workspace), ref) <= TOL


@pytest.mark.parametrize("share", [0.0, 0.4, 0.999, 1.5])
def test_any_workspace_gives_the_gradient(gpu, share):
    """The queried bytes, fewer, which give fewer k ranges or the generic gathers where the
    permuted filter has no room, and more."""
    p = (13, 24, 232, 49, 19, 0, 0, 2, 2, 3, 3)
    N, C, K, H, W = p[:5]
    cv = Conv(gpu, *p)
    dy, w = _rand(N * K * cv.Ho * cv.Wo, 7), _rand(K * C * 9, 8)
    query = gpu.L.mnv_conv_bwd_data_workspace_bytes(*p)
    filter_bytes = 4 * C * 9 * 240
    assert query >= filter_bytes
    nbytes = int(share * query) if share else filter_bytes
    ddy, dw, out = gpu.up(dy), gpu.up(w), gpu.up(np.full(N * C * H * W, np.nan, np.float32))
    ws = gpu.empty(nbytes // 4 + 1)
    gpu.call("mnv_conv_bwd_data", ddy.p, dw.p, out.p, *p, ws.p, ctypes.c_size_t(nbytes))
    assert normwise(gpu.down(out), ora.conv_bwd_data(dy, w, *p)) <= TOL


def test_relu_gate_selects(gpu):
    p = (3, 40, 20, 11, 8, 1, 1, 2, 2, 3, 3)
    N, C, K, H, W = p[:5]
    cv = Conv(gpu, *p)
    dy, w, x = _rand(N * K * cv.Ho * cv.Wo, 9), _rand(K * C * 9, 10), _rand(N * C * H * W, 11)
    plain = cv.bwd_data(dy, w)
    ddy, dw, dx, out = gpu.up(dy), gpu.up(w), gpu.up(x), gpu.up(np.full(N * C * H * W, np.nan, np.float32))
    nbytes = gpu.L.mnv_conv_bwd_data_workspace_bytes(*p)
    ws = gpu.empty(nbytes // 4 + 1)
    gpu.call("mnv_conv_bwd_data_relu", ddy.p, dw.p, dx.p, out.p, *p, ws.p, ctypes.c_size_t(nbytes))
    np.testing.assert_array_equal(gpu.down(out), np.where(x > 0, plain, np.float32(0)))
