"""GPU parity of the data gradient of strided convolutions, whose positions are taken class by class
modulo the strides: against the CPU oracle on all tiles, with and without k ranges, and where classes
are empty, have no taps, or hold one position more or less than the others."""
import ctypes

import numpy as np
import pytest

from gpu_util import Gpu, TOL, normwise, say
from minerva_amd import capi
from test_gpu_conv import Conv, _out, _rand
from oracle import mnv_oracle as ora

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return Gpu()


def _plan(p, workspace=None):
    """Rows of the tile, k ranges, whether in bf16 parts, and classes (1: the generic gathers)."""
    L, v = capi.lib(), [ctypes.c_int() for _ in range(4)]
    ws = L.mnv_conv_bwd_data_workspace_bytes(*p) if workspace is None else workspace
    assert L.mnv_conv_bwd_data_plan(*p, ctypes.c_size_t(ws), *[ctypes.byref(x) for x in v]) == 0
    return tuple(x.value for x in v)


CASES = [  # N, C, K, H, W, ph, pw, sv, sh, R, S; the plan
    ((2, 16, 16, 9, 9, 1, 1, 2, 2, 3, 3), (32, 1, 0, 4)),
    ((3, 40, 20, 11, 8, 0, 0, 2, 2, 3, 3), (32, 1, 0, 4)),         # channels padded to 32
    ((1, 33, 5, 13, 7, 2, 2, 2, 2, 5, 5), (64, 1, 0, 1)),          # 5 channels: more padding than product
    ((2, 24, 48, 14, 15, 0, 0, 2, 2, 1, 1), (128, 1, 0, 1)),       # few short sums
    ((2, 17, 16, 12, 9, 1, 0, 2, 1, 3, 2), (32, 1, 0, 2)),         # one direction only
    ((2, 17, 16, 9, 12, 0, 1, 1, 3, 2, 4), (32, 1, 0, 3)),
    ((1, 20, 32, 23, 23, 0, 0, 4, 4, 11, 11), (32, 1, 0, 16)),
    ((2, 16, 16, 7, 6, 0, 0, 5, 4, 3, 3), (32, 1, 0, 20)),         # filter below the stride: rows that meet nothing
    ((1, 16, 16, 2, 2, 1, 1, 3, 3, 3, 3), (128, 1, 0, 1)),         # planes below the stride
    ((2, 9, 16, 8, 7, 4, 3, 2, 3, 3, 2), (32, 1, 0, 6)),           # padding beyond the filter
    ((13, 24, 232, 49, 19, 0, 0, 2, 2, 3, 3), (32, 1, 0, 4)),
    ((21, 184, 120, 31, 7, 0, 0, 2, 2, 3, 3), (32, 1, 0, 4)),
    ((1, 20, 168, 10, 6, 0, 0, 2, 2, 5, 5), (32, 8, 0, 4)),        # k ranges
    ((95, 51, 17, 28, 9, 0, 0, 4, 4, 2, 2), (64, 1, 0, 16)),       # 12 of 16 classes meet no tap
    ((40, 33, 210, 37, 22, 0, 0, 4, 4, 1, 1), (64, 2, 0, 16)),     # 15 of 16, with k ranges
    ((77, 11, 177, 29, 27, 0, 0, 4, 4, 1, 1), (128, 2, 0, 16)),
    ((121, 8, 24, 11, 50, 1, 1, 4, 4, 2, 2), (128, 1, 0, 16)),     # 128 x 32 tiles
    ((64, 144, 16, 20, 20, 1, 1, 2, 2, 3, 3), (128, 1, 0, 4)),     # 128 x 96
    ((40, 192, 96, 28, 28, 1, 1, 2, 2, 3, 3), (128, 1, 1, 4)),     # bf16 parts, 96 columns
    ((24, 256, 104, 15, 45, 2, 2, 2, 2, 5, 5), (128, 1, 1, 4)),    # bf16 parts, 128 columns, channels padded
    ((43, 104, 82, 10, 8, 0, 0, 2, 2, 7, 7), (128, 8, 1, 4)),      # bf16 parts with k ranges
    ((62, 96, 198, 9, 7, 0, 0, 3, 3, 7, 7), (128, 8, 1, 9)),
    ((81, 144, 16, 8, 43, 0, 0, 4, 4, 5, 5), (128, 1, 1, 16)),     # bf16 parts, classes of one tap
]


@pytest.mark.parametrize("p,plan", CASES, ids=lambda v: "-".join(map(str, v)))
def test_strided_data_gradient_matches_the_oracle(gpu, p, plan):
    N, C, K, H, W, ph, pw, sv, sh, R, S = p
    say("strided data gradient", p)
    assert _plan(p) == plan and _plan(p, 0)[3] == 1
    cv = Conv(gpu, *p)
    dy, w = _rand(N * K * cv.Ho * cv.Wo, 5), _rand(K * C * R * S, 6)
    ref = ora.conv_bwd_data(dy, w, *p)
    for workspace in (True, False):  # without: the generic gathers
        assert normwise(cv.bwd_data(dy, w, workspace), ref) <= TOL


BEYOND = [  # strides beyond the plane in one direction or both: fewer classes than sv * sh
    (64, 64, 64, 2, 2, 1, 1, 20, 20, 3, 3),
    (17, 24, 344, 5, 3, 1, 0, 1, 6, 5, 2),
    (32, 16, 224, 5, 2, 0, 0, 1, 7, 5, 2),      # k ranges, as the one above
    (9, 33, 40, 1, 37, 0, 1, 2, 2, 1, 3),       # one row
    (7, 20, 48, 3, 4, 2, 3, 5, 4, 4, 5),        # the other direction's stride is the plane's extent
    (700, 64, 128, 3, 2, 1, 2, 4, 8, 5, 5),
    (900, 96, 256, 3, 2, 1, 1, 4, 4, 3, 3),
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


@pytest.mark.parametrize("p", [
    (13, 24, 232, 49, 19, 0, 0, 2, 2, 3, 3),                                               # no k ranges
    (1, 20, 168, 10, 6, 0, 0, 2, 2, 5, 5), (40, 33, 210, 37, 22, 0, 0, 4, 4, 1, 1), (43, 104, 82, 10, 8, 0, 0, 2, 2, 7, 7),
], ids=lambda p: "-".join(map(str, p)))
@pytest.mark.parametrize("share", [0.0, 0.4, 0.999, 1.0, 1.5])
def test_any_workspace_gives_the_gradient(gpu, p, share):
    """The queried bytes, fewer, which give fewer k ranges or the generic gathers where the
    permuted filter has no room, and more; 0: the filter alone.  Nothing is written past them."""
    N, C, K, H, W = p[:5]
    cv = Conv(gpu, *p)
    dy, w = _rand(N * K * cv.Ho * cv.Wo, 7), _rand(K * C * p[9] * p[10], 8)
    query = gpu.L.mnv_conv_bwd_data_workspace_bytes(*p)
    filter_bytes = 4 * C * p[9] * p[10] * -(-K // 16) * 16
    ranges = _plan(p)[1]
    assert (query > filter_bytes) == (ranges > 1) and query >= filter_bytes
    nbytes = int(share * query) // 4 * 4 if share else filter_bytes
    if share < 1 and ranges > 1:
        assert _plan(p, nbytes) != _plan(p)
    ddy, dw, out = gpu.up(dy), gpu.up(w), gpu.up(np.full(N * C * H * W, np.nan, np.float32))
    ws = gpu.up(np.full(nbytes // 4 + 1024, 7.0, np.float32))
    gpu.call("mnv_conv_bwd_data", ddy.p, dw.p, out.p, *p, ws.p, ctypes.c_size_t(nbytes))
    assert normwise(gpu.down(out), ora.conv_bwd_data(dy, w, *p)) <= TOL
    assert np.all(gpu.down(ws)[nbytes // 4:] == 7.0)


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
