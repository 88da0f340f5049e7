"""Which data gradients and forward passes have their channels padded to the multiples of 16: host
arithmetic on the extents alone, seen from the workspace that holds the padded filter."""
import ctypes

import pytest

from minerva_amd import capi


def _query(direction, N, C, K, H, W, pad, R):
    return getattr(capi.lib(), "mnv_conv_%s_workspace_bytes" % direction)(N, C, K, H, W, pad, pad, 1, 1, R, R)


@pytest.mark.parametrize("dims,padded", [  # N, C, K, H, W, pad, R; the reduction runs over K
    ((1, 8, 8, 14, 14, 0, 1), False), ((4, 24, 24, 14, 14, 0, 1), False),     # one and two slabs: the permutation's launch
    ((64, 8, 12, 28, 28, 0, 1), False),                                       # costs more than they do
    ((50, 312, 24, 23, 14, 0, 1), True),                                      # or does not, over many tiles
    ((1, 24, 40, 14, 14, 0, 1), True), ((1, 40, 40, 14, 14, 0, 1), False),    # three slabs; 64 x 64 tiles
    ((16, 8, 8, 14, 14, 1, 3), False), ((64, 8, 8, 28, 28, 1, 3), True), ((1, 8, 12, 14, 14, 1, 3), True),
    ((4, 8, 8, 14, 14, 2, 5), True), ((16, 40, 8, 28, 28, 2, 5), False),      # twice the work,
    ((2, 40, 8, 28, 28, 2, 5), True),                                         # of few tiles
    ((16, 200, 10, 28, 28, 1, 3), True), ((32, 104, 10, 28, 28, 2, 5), True),  # 60% more work, in parts
    ((16, 40, 10, 28, 28, 2, 5), False), ((16, 256, 10, 14, 14, 2, 5), False), ((64, 200, 8, 28, 28, 1, 3), False),
    ((4, 40, 10, 14, 14, 1, 3), False),
    ((64, 24, 17, 28, 28, 1, 3), False), ((64, 24, 20, 28, 28, 1, 3), True),
])
def test_channels_of_small_data_gradients_are_padded_where_it_pays(dims, padded):
    N, C, K, H, W, pad, R = dims
    filter_bytes = 4 * C * R * R * ((K + 15) // 16 * 16)
    ws = _query("bwd_data", *dims)
    partial = 4 * N * H * W * C  # what k ranges ask for, in whole results
    if padded:
        assert ws >= filter_bytes and (ws - filter_bytes) % partial in (0, (256 - filter_bytes) % 256)
    else:
        assert ws % partial == 0


@pytest.mark.parametrize("C,padded", [(8, False), (9, False), (12, True), (24, True)])
def test_channels_of_forward_passes_are_padded_where_it_pays(C, padded):
    dims = (64, C, 88, 28, 28, 2, 5)
    assert (_query("fwd", *dims) >= 4 * 88 * 25 * ((C + 15) // 16 * 16)) == padded


@pytest.mark.parametrize("dims", [  # N, C, K, H, W, ph, pw, sv, sh, R, S
    (1, 32, 256, 2, 2, 1, 1, 65536, 65536, 3, 3), (1, 16, 16, 1, 1, 0, 0, 8192, 4096, 1, 1),
    (1, 1, 64, 8192, 4096, 0, 0, 8192, 4096, 1, 1), (1, 2, 16, 15000, 15000, 0, 0, 15000, 15000, 1, 1),
    (1, 32, 256, 2, 2, 1, 1, 2 ** 31 - 1, 2 ** 31 - 1, 3, 3),
])
def test_strides_of_millions_of_classes_have_a_workspace(dims):
    """A data gradient of strides sv x sh takes its positions in sv * sh classes, whose rows, each class
    filled up to whole tiles, may be more than an int holds."""
    N, C, K, H, W, ph, pw, sv, sh, R, S = dims
    ws = capi.lib().mnv_conv_bwd_data_workspace_bytes(*dims)
    # no more than the permuted filter and some partial results
    assert ws <= 4 * C * R * S * ((K + 15) // 16 * 16) + 256 + 64 * 4 * N * H * W * C


@pytest.mark.parametrize("dims,rows", [  # N, C, K, H, W, ph, pw, sv, sh, R, S; rows of the classes that hold a position
    ((2254, 64, 264, 3, 2, 1, 0, 8, 4, 2, 1), 0), ((929, 64, 240, 2, 4, 2, 2, 7, 5, 2, 1), 0), ((1057, 48, 200, 2, 4, 0, 2, 8, 1, 1, 1), 0),
    ((32, 16, 224, 5, 2, 0, 0, 1, 7, 5, 2), 2 * 160),
])
def test_classes_without_a_position_take_no_workspace(dims, rows):
    """Strides beyond the plane: of the sv * sh classes only min(sv, H) * min(sh, W) hold a position, and only
    those are rows of the product (0: no partial results, one range of each class)."""
    C, K, R, S = dims[1], dims[2], dims[9], dims[10]
    filter_bytes = 4 * C * R * S * ((K + 15) // 16 * 16)
    ws = capi.lib().mnv_conv_bwd_data_workspace_bytes(*dims)
    assert ws >= filter_bytes and filter_bytes % 256 == 0
    assert (ws == filter_bytes) if not rows else (ws > filter_bytes and (ws - filter_bytes) % (4 * rows * C) == 0)


def _data_plan(dims, workspace=None):
    """Rows of the tile, k ranges, whether in bf16 parts, classes of positions (1: the generic gathers of strides above 1)."""
    v = [ctypes.c_int() for _ in range(4)]
    ws = capi.lib().mnv_conv_bwd_data_workspace_bytes(*dims) if workspace is None else workspace
    assert capi.lib().mnv_conv_bwd_data_plan(*dims, ctypes.c_size_t(ws), *[ctypes.byref(x) for x in v]) == 0
    return tuple(x.value for x in v)


@pytest.mark.parametrize("dims,classes", [  # N, C, K, H, W, pad, R; stride 2
    ((52, 256, 32, 14, 12, 0, 1), 1), ((36, 272, 24, 32, 18, 0, 1), 1), ((81, 120, 24, 26, 18, 0, 1), 1), ((58, 96, 32, 26, 39, 0, 1), 1),
    ((35, 304, 56, 9, 32, 0, 1), 1), ((69, 224, 128, 32, 7, 0, 1), 1), ((10, 376, 120, 16, 37, 0, 1), 1), ((79, 136, 16, 8, 19, 1, 3), 1),
    ((93, 328, 32, 53, 22, 0, 1), 1), ((86, 176, 48, 34, 28, 0, 1), 1),
    ((39, 192, 72, 21, 54, 0, 1), 4), ((70, 128, 72, 52, 46, 0, 1), 4), ((26, 208, 128, 50, 45, 0, 1), 4), ((59, 72, 160, 13, 48, 0, 1), 4),
    ((27, 288, 16, 33, 39, 0, 3), 4), ((44, 304, 192, 15, 14, 0, 1), 4),
    ((4, 70, 70, 14, 14, 0, 1), 1), ((66, 24, 128, 46, 10, 0, 1), 4),    # few tiles
])
def test_strided_data_gradients_by_classes_where_it_pays(dims, classes):
    N, C, K, H, W, pad, R = dims
    assert _data_plan((N, C, K, H, W, pad, pad, 2, 2, R, R))[3] == classes


@pytest.mark.parametrize("dims,plan", [  # N, C, K, H, W, pad, R; stride 2
    ((34, 120, 120, 26, 11, 1, 2), (32, 0)), ((47, 64, 64, 16, 27, 1, 3), (32, 0)), ((120, 48, 24, 27, 30, 1, 3), (32, 0)),  # more k ranges
    ((108, 32, 56, 30, 21, 1, 3), (32, 0)),
    ((51, 112, 48, 33, 50, 1, 3), (128, 1)), ((113, 264, 248, 17, 16, 0, 1), (128, 1)), ((80, 136, 64, 24, 12, 2, 5), (128, 1)),  # a cut tail
    ((45, 120, 80, 56, 16, 0, 2), (128, 0)), ((116, 56, 80, 32, 36, 0, 1), (64, 0)),                      # as long sums either way
])
def test_strided_data_gradients_sum_no_longer_than_the_generic_gathers(dims, plan):
    """Rows of the tile and whether in bf16 parts: layers whose generic launch shortens its sums by k ranges or a cut tail go where
    sums are short as well."""
    N, C, K, H, W, pad, R = dims
    got = _data_plan((N, C, K, H, W, pad, pad, 2, 2, R, R))
    assert (got[0], got[2], got[3]) == plan + (4,)


@pytest.mark.parametrize("direction,dims,small", [  # N, C, K, H, W, pad, R, stride
    ("fwd", (15, 24, 96, 22, 43, 0, 1, 1), False), ("fwd", (78, 24, 32, 9, 56, 0, 1, 1), False), ("fwd", (23, 24, 96, 46, 46, 0, 1, 2), False),
    ("fwd", (67, 40, 64, 32, 8, 0, 1, 1), False), ("bwd_data", (10, 176, 56, 10, 45, 0, 1, 1), False),
    ("bwd_data", (16, 136, 56, 54, 9, 0, 1, 1), False),                                          # few slabs, many tiles
    ("fwd", (26, 64, 168, 9, 11, 0, 1, 1), True), ("bwd_data", (52, 24, 72, 18, 19, 0, 1, 1), True), ("fwd", (64, 88, 24, 49, 17, 0, 1, 2), True),
    ("fwd", (4, 200, 328, 10, 8, 0, 5, 2), False), ("fwd", (6, 264, 264, 19, 8, 2, 5, 2), False),   # a large filter to permute
    ("fwd", (35, 216, 24, 34, 8, 0, 5, 2), False), ("fwd", (97, 376, 24, 8, 47, 0, 5, 2), False),   # scattered positions
    ("fwd", (26, 160, 32, 28, 55, 0, 3, 2), False), ("fwd", (18, 32, 160, 9, 38, 0, 3, 2), True),
    ("fwd", (2, 104, 384, 11, 25, 2, 5, 2), False), ("fwd", (2, 136, 280, 11, 14, 1, 3, 2), True), ("fwd", (1, 120, 224, 25, 33, 1, 3, 2), True),
])
def test_layers_that_small_tiles_slow_down_stay_on_larger_ones(direction, dims, small):
    N, C, K, H, W, pad, R, stride = dims
    full = (N, C, K, H, W, pad, pad, stride, stride, R, R)
    v = [ctypes.c_int() for _ in range(4 if direction == "bwd_data" else 3)]
    ws = getattr(capi.lib(), "mnv_conv_%s_workspace_bytes" % direction)(*full)
    assert getattr(capi.lib(), "mnv_conv_%s_plan" % direction)(*full, ctypes.c_size_t(ws), *[ctypes.byref(x) for x in v]) == 0
    assert (v[0].value == 32) == small
