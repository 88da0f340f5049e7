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


def _tile(gpu, name, p):
    """Rows of the tile, k ranges and, of a data gradient, classes of positions with the queried workspace."""
    v = [ctypes.c_int() for _ in range(4 if name == "bwd_data" else 3)]
    nbytes = getattr(gpu.L, "mnv_conv_%s_workspace_bytes" % name)(*p)
    assert getattr(gpu.L, "mnv_conv_%s_plan" % name)(*p, ctypes.c_size_t(nbytes), *[ctypes.byref(x) for x in v]) == 0
    return v[0].value, v[1].value, v[-1].value if name == "bwd_data" else 1


CASES = [  # N, C, K, H, W, ph, pw, sv, sh, R, S; passes that are meant to run so
    ((19, 32, 32, 44, 12, 0, 0, 1, 1, 3, 3), "fwd bwd_data"),       # no padding: the filter in place
    ((7, 48, 33, 14, 41, 1, 1, 1, 1, 3, 3), "fwd bwd_data"),        # a column past a tile
    ((4, 24, 56, 22, 47, 1, 1, 1, 1, 3, 3), "fwd bwd_filter"),      # 24 channels padded to 32
    ((1, 152, 368, 24, 16, 0, 0, 1, 1, 5, 5), "fwd bwd_filter"),    # k ranges; positions off the multiples of 16
    ((59, 80, 32, 48, 20, 2, 2, 2, 2, 5, 5), "fwd"),
    ((14, 240, 64, 16, 14, 1, 1, 2, 2, 3, 3), "bwd_data"),          # classes of positions
    ((2, 17, 40, 31, 29, 1, 1, 2, 1, 3, 2), "bwd_data"),
    ((2, 48, 352, 27, 36, 1, 1, 2, 2, 3, 3), "bwd_filter"),         # a table of taps
    ((3, 41, 50, 9, 7, 1, 0, 1, 1, 3, 1), "fwd bwd_data"),          # ragged everywhere
    ((1, 256, 384, 13, 13, 1, 1, 1, 1, 3, 3), "bwd_data"),
    ((1, 16, 16, 1, 1, 0, 0, 1, 1, 1, 1), "fwd bwd_data"),          # one position
]


@pytest.mark.parametrize("p,passes", CASES, ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else v.replace(" ", "+"))
def test_small_convolutions_match_the_oracle(gpu, p, passes):
    N, C, K, H, W = p[:5]
    say("small convolution", p)
    cv = Conv(gpu, *p)
    x, w, b = _rand(N * C * H * W, 1), _rand(K * C * p[9] * p[10], 2), _rand(K, 3)
    dy = _rand(N * K * cv.Ho * cv.Wo, 4)
    x = np.maximum(x, 0)
    for name in passes.split():
        assert _tile(gpu, name, p)[0] == 32, "the case is meant to run on the small tiles"
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


RANGES = [  # with k ranges, whose partial results are added by a second launch
    ("fwd", (1, 27, 17, 10, 6, 0, 0, 1, 1, 5, 5), 1),       # the filter in place
    ("fwd", (1, 152, 368, 24, 16, 0, 0, 1, 1, 5, 5), 1),
    ("fwd", (1, 88, 18, 6, 7, 1, 1, 1, 1, 3, 3), 1),        # channels padded
    ("fwd", (1, 80, 22, 5, 6, 1, 1, 2, 2, 3, 3), 1),
    ("bwd_data", (1, 20, 80, 6, 5, 1, 1, 1, 1, 3, 3), 1),
    ("bwd_data", (1, 16, 33, 5, 6, 0, 0, 1, 1, 5, 5), 1),   # channels padded
    ("bwd_data", (2, 16, 128, 6, 13, 2, 2, 2, 2, 5, 5), 4),  # classes of positions
    ("bwd_data", (2, 16, 291, 7, 9, 0, 0, 2, 2, 3, 3), 4),
]


@pytest.mark.parametrize("name,p,classes", RANGES, ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else str(v))
@pytest.mark.parametrize("share", [0.999, 1.0])
def test_small_tiles_with_k_ranges(gpu, name, p, classes, share):
    """The queried workspace, and a little less of it, which gives fewer ranges or other kernels."""
    N, C, K, H, W = p[:5]
    say("small convolution with k ranges", name, p, share)
    rows, ranges, n = _tile(gpu, name, p)
    assert rows == 32 and ranges > 1 and n == classes
    cv = Conv(gpu, *p)
    w, b, x, dy = _rand(K * C * p[9] * p[10], 2), _rand(K, 3), _rand(N * C * H * W, 1), _rand(N * K * cv.Ho * cv.Wo, 4)
    ref = ora.conv_fwd(x, w, b, *p) if name == "fwd" else ora.conv_bwd_data(dy, w, *p)
    nbytes = int(share * getattr(gpu.L, "mnv_conv_%s_workspace_bytes" % name)(*p)) // 4 * 4
    ws, out = gpu.up(np.full(nbytes // 4 + 1024, 7.0, np.float32)), gpu.up(np.full(ref.size, np.nan, np.float32))
    ins = [gpu.up(a) for a in ((x, w, b) if name == "fwd" else (dy, w))]
    gpu.call("mnv_conv_" + name, *[a.p for a in ins], out.p, *p, ws.p, ctypes.c_size_t(nbytes))
    assert normwise(gpu.down(out), ref) <= TOL
    assert np.all(gpu.down(ws)[nbytes // 4:] == 7.0)


@pytest.mark.parametrize("p", [(2, 24, 32, 9, 11, 1, 1, 1, 1, 3, 3), (3, 20, 40, 12, 7, 0, 0, 1, 1, 3, 3), (2, 40, 56, 13, 10, 1, 1, 2, 2, 3, 3)],
                         ids=lambda p: "-".join(map(str, p)))
def test_infinities_stay_where_they_are_summed(gpu, p):
    """What is past the channels, the rows or the reduction of a tile, or fetched ahead, is never multiplied into a result."""
    import torch
    N, C, K, H, W, ph, pw, sv, sh, R, S = p
    cv = Conv(gpu, *p)
    x, dy, w = _rand(N * C * H * W, 1), _rand(N * K * cv.Ho * cv.Wo, 2), _rand(K * C * R * S, 3)
    x4, dy4 = x.reshape(N, C, H, W), dy.reshape(N, K, cv.Ho, cv.Wo)
    x4[1, 0, 0, 0], x4[0, C - 1, H - 1, W - 1], x4[N - 1, C // 2, 3, W - 2] = np.inf, np.nan, -np.inf
    dy4[1, 0, 0, 0], dy4[0, K - 1, cv.Ho - 1, cv.Wo - 1], dy4[N - 1, K // 2, 1, 2] = np.nan, np.inf, -np.inf
    X, D = (torch.from_numpy(v).double() for v in (x4, dy4))
    F = torch.from_numpy(w).double().view(K, C, R, S).flip(2, 3)  # a true convolution
    rest = (H + 2 * ph - R) % sv, (W + 2 * pw - S) % sh
    cols = torch.nn.functional.unfold(X, (R, S), padding=(ph, pw), stride=(sv, sh))
    want = {"fwd": torch.nn.functional.conv2d(X, F, stride=(sv, sh), padding=(ph, pw)),
            "bwd_data": torch.nn.functional.conv_transpose2d(D, F, stride=(sv, sh), padding=(ph, pw), output_padding=rest),
            "bwd_filter": torch.matmul(D.flatten(2), cols.transpose(1, 2)).sum(0).view(K, C, R, S).flip(2, 3)}
    for name, got in (("fwd", cv.fwd(x, w, np.zeros(K, np.float32))), ("bwd_data", cv.bwd_data(dy, w)), ("bwd_filter", cv.bwd_filter(dy, x))):
        assert _tile(gpu, name, p)[0] == 32, name
        ref = want[name].numpy().reshape(-1)
        finite = np.isfinite(ref)
        assert 0 < finite.sum() < finite.size and np.array_equal(np.isfinite(got), finite), name
        assert normwise(got[finite], ref[finite]) <= TOL, name
