"""GPU parity of small convolutions on 32 x 32 tiles whose wavefronts share the reduction: the three passes
against the CPU oracle with and without k ranges, at ragged extents, with channels off the multiples
of 16, unit and larger strides, with and without padding, and in too small a workspace."""
import ctypes

import numpy as np
import pytest

from gpu_util import Gpu, TOL, normwise, say
from test_gpu_conv import Conv, _rand
from oracle import mnv_oracle as ora

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return Gpu()


CASES = [  # N, C, K, H, W, ph, pw, sv, sh, R, S; passes that are meant to run so
    ((19, 32, 32, 44, 12, 0, 0, 1, 1, 3, 3), "fwd"),                # no padding: the filter in place
    ((7, 48, 33, 14, 41, 1, 1, 1, 1, 3, 3), "fwd bwd_data"),        # a column past a tile
    ((4, 24, 56, 22, 47, 1, 1, 1, 1, 3, 3), "fwd bwd_filter"),      # 24 channels padded to 32
    ((1, 152, 368, 24, 16, 0, 0, 1, 1, 5, 5), "fwd bwd_filter"),    # k ranges; positions off the multiples of 16
    ((59, 80, 32, 48, 20, 2, 2, 2, 2, 5, 5), "fwd"),
    ((14, 240, 64, 16, 14, 1, 1, 2, 2, 3, 3), "bwd_data"),          # classes of positions
    ((2, 17, 40, 31, 29, 1, 1, 2, 1, 3, 2), "bwd_data"),
    ((2, 48, 352, 27, 36, 1, 1, 2, 2, 3, 3), "bwd_filter"),         # a table of taps
    ((3, 41, 50, 9, 7, 1, 0, 1, 1, 3, 1), ""),                      # ragged everywhere
    ((1, 256, 384, 13, 13, 1, 1, 1, 1, 3, 3), ""),
    ((1, 16, 16, 1, 1, 0, 0, 1, 1, 1, 1), ""),                      # one position
]


@pytest.mark.parametrize("p,passes", CASES, ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else v.replace(" ", "+"))
def test_small_convolutions_match_the_oracle(gpu, p, passes):
    N, C, K, H, W = p[:5]
    say("small convolution", p)
    cv = Conv(gpu, *p)
    x, w, b = _rand(N * C * H * W, 1), _rand(K * C * p[9] * p[10], 2), _rand(K, 3)
    dy = _rand(N * K * cv.Ho * cv.Wo, 4)
    x = np.maximum(x, 0)
    if "bwd_filter" in passes:
        plan = [ctypes.c_int() for _ in range(3)]
        nbytes = gpu.L.mnv_conv_bwd_filter_workspace_bytes(*p)
        assert gpu.L.mnv_conv_bwd_filter_plan(*p, ctypes.c_size_t(nbytes), *[ctypes.byref(v) for v in plan]) == 0
        assert plan[0].value == 32, "the case is meant to run on the small tiles"
    for workspace in (True, False):
        assert normwise(cv.fwd(x, w, b, workspace), ora.conv_fwd(x, w, b, *p)) <= TOL
        assert normwise(cv.bwd_data(dy, w, workspace), ora.conv_bwd_data(dy, w, *p)) <= TOL
        assert normwise(cv.bwd_filter(dy, x, workspace), ora.conv_bwd_filter(dy, x, *p)) <= TOL


@pytest.mark.parametrize("share", [0.3, 0.7, 0.999, 2.0])
def test_any_workspace_gives_the_results(gpu, share):
    """Less than the queried bytes: fewer k ranges or other kernels, and nothing is written past them."""
    p = (1, 256, 384, 13, 13, 1, 1, 1, 1, 3, 3)
    N, C, K, H, W = p[:5]
    x, w, b, dy = _rand(C * H * W, 1), _rand(K * C * 9, 2), _rand(K, 3), _rand(K * H * W, 4)
    dx, dw, db, ddy = gpu.up(x), gpu.up(w), gpu.up(b), gpu.up(dy)
    for name, args, size, ref in (
            ("fwd", (dx, dw, db), K * H * W, ora.conv_fwd(x, w, b, *p)),
            ("bwd_data", (ddy, dw), C * H * W, ora.conv_bwd_data(dy, w, *p)),
            ("bwd_filter", (dx, ddy), K * C * 9, ora.conv_bwd_filter(dy, x, *p))):
        nbytes = int(share * getattr(gpu.L, "mnv_conv_%s_workspace_bytes" % name)(*p)) // 4 * 4
        guard = np.full(nbytes // 4 + 1024, 7.0, np.float32)
        ws, out = gpu.up(guard), gpu.up(np.full(size, np.nan, np.float32))
        gpu.call("mnv_conv_" + name, *[a.p for a in args], out.p, *p, ws.p, ctypes.c_size_t(nbytes))
        assert normwise(gpu.down(out), ref) <= TOL, name
        assert np.all(gpu.down(ws)[nbytes // 4:] == 7.0), name
