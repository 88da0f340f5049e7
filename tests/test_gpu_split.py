"""The matrix products that run in bf16 parts (csrc/gemm_split.h): at the edges of their tiles and
k steps, with each operand transposed, with every epilogue, against float64 element by element; and
with operands that have no such parts (infinities, NaN, values from 2^111 on) or hardly any
(denormals), where they must do what fp32 arithmetic does."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import Gpu, assert_bits_equal, normwise, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return Gpu()


def _plan(gpu, m, n, k, ws_bytes):
    v = [ctypes.c_int() for _ in range(3)]
    assert gpu.L.mnv_sgemm_nn_plan(m, n, k, ctypes.c_size_t(ws_bytes), *[ctypes.byref(x) for x in v]) == 0
    return tuple(x.value for x in v)


def _bound(A, B):
    """Element-wise: the sum of a1 b1 is rounded at every eight k, in two sets of accumulators and (k
    ranges) their sums, each time by at most one unit in the last place (the instruction cuts) of a partial sum of
    |a||b|; what the cut into parts leaves out is 3 x 2^-25 of every product."""
    k = A.shape[1]
    return (k / 8 + 24) * 2.0 ** -23 * (np.abs(B) @ np.abs(A).T)


def _products(gpu, A, B, workspace=True):
    """C{m,n} by the three entry points; A is {m,k}, B {n,k} here (float32)."""
    m, k = A.shape
    n = B.shape[0]
    a, at = gpu.up(np.ascontiguousarray(A.T).reshape(-1)), gpu.up(np.ascontiguousarray(A).reshape(-1))
    b, bt = gpu.up(np.ascontiguousarray(B).reshape(-1)), gpu.up(np.ascontiguousarray(B.T).reshape(-1))
    nb = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k) if workspace else 0
    ws = gpu.empty(nb // 4 + 1)
    out = {}
    for name, args in (("nn", (a, b)), ("tn", (at, b)), ("nt", (a, bt))):
        c = gpu.up(np.full(m * n + 4, np.float32(7.5), np.float32))
        extra = (None,) if name == "tn" else ()
        gpu.call("mnv_sgemm_" + name, args[0].p, args[1].p, *extra, c.p, m, n, k, ws.p if nb else None, ctypes.c_size_t(nb))
        got = gpu.down(c)
        assert (got[m * n:] == 7.5).all(), "wrote past C"
        out[name] = got[:m * n].reshape(n, m)
    return out


def _rand(shape, seed, relu=False):
    x = np.random.default_rng(seed).standard_normal(shape).astype(np.float32)
    return np.maximum(x, 0) if relu else x


SHAPES = [  # m, n, k: what the tile, the k step (32), the slab (16) and the planner divide them into
    (2048, 2048, 96),      # whole tiles, three steps, two workgroups per CU
    (2561, 2047, 97),      # one past and one short of a tile, one k in the last slab: an odd step
    (3841, 2177, 33), (3968, 1985, 31), (2500, 2500, 17),  # one slab and a bit, and less than a step
    (2303, 3073, 112),     # the second half of the last step is missing
    (1793, 2047, 1001),    # one workgroup per CU
    (200, 3000, 4001),     # k ranges
    (4095, 4096, 515), (4093, 4095, 514),  # 256 x 128 tiles
    (2307, 3549, 530),     # the tiles past two per CU cut into k ranges
]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("workspace", [True, False])
def test_products_in_parts_against_float64(gpu, m, n, k, workspace):
    ws = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k) if workspace else 0
    tile = _plan(gpu, m, n, k, ws)
    if workspace:
        assert tile[0] in (128, 256), "the case is meant to run in parts"
    A, B = _rand((m, k), m + k, relu=True), _rand((n, k), n)
    say("product in parts", m, n, k, "plan", tile)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    want, bound = B64 @ A64.T, _bound(A64, B64)
    got = _products(gpu, A, B, workspace)
    for name, c in got.items():
        bad = np.abs(c - want) > bound
        assert not bad.any(), "%s: %d elements, first %s" % (name, int(bad.sum()), np.argwhere(bad)[0])
    assert_bits_equal(got["tn"], got["nn"], "A given transposed")


@pytest.mark.parametrize("m,n,k", [(2561, 2047, 97), (1793, 2047, 1001), (200, 3000, 4001), (4095, 4096, 515)])
def test_products_in_parts_next_to_values_without_parts(gpu, m, n, k):
    """Infinities, NaN and finite values that a bf16 part or the scale in front of it cannot hold: the
    result is infinite, NaN or finite where float32 arithmetic has it so (inf times 1, which has
    two zero parts, is inf), and finite ones are as close as elsewhere."""
    rng = np.random.default_rng(k)
    A, B = _rand((m, k), 11), _rand((n, k), 12)
    B[:, 3] = 1.0  # meets the infinities of A: parts 1, 0, 0
    A[5, 3], A[m - 1, 3], A[m // 2, 3] = np.inf, -np.inf, np.nan
    A[7, k - 1] = np.float32(3.4e38)   # rounds to infinity in bf16; its products stay finite
    B[:, k - 1] = rng.uniform(0.25, 0.5, n).astype(np.float32)
    B[n - 1, 0], A[:, 0] = np.float32(2.0 ** 120), np.float32(2.0 ** -20) * rng.uniform(1, 2, m).astype(np.float32)
    B[2, 1], A[9, 1] = np.inf, 0.0     # inf times 0
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = B64 @ A64.T
        # the redone blocks add in the order of fp32 arithmetic: one rounding per k
        bound = (k + 8) * 2.0 ** -24 * (np.abs(B64) @ np.abs(A64).T)
    say("product in parts next to infinities", m, n, k)
    for name, c in _products(gpu, A, B).items():
        assert np.array_equal(np.isnan(c), np.isnan(want)), name
        inf = np.isinf(want)
        assert np.array_equal(np.isinf(c), inf) and np.array_equal(c[inf] > 0, want[inf] > 0), name
        fin = np.isfinite(want)
        assert (np.abs(c[fin] - want[fin]) <= bound[fin]).all(), name


@pytest.mark.parametrize("m,n,k", [(4093, 4099, 13), (4096, 4096, 16), (4099, 5003, 1)])
def test_products_of_one_slab_round_as_the_fp32_instruction(gpu, m, n, k):
    """Up to 16 k the large tiles stay with the fp32 instruction: one rounding per k."""
    A, B = _rand((m, k), 71), _rand((n, k), 72)
    assert _plan(gpu, m, n, k, 0) == (128, 1, 1)
    say("products of one slab", m, n, k)
    got = _products(gpu, A, B)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    want, bound = B64 @ A64.T, k * 2.0 ** -24 * (np.abs(B64) @ np.abs(A64).T)
    for name, c in got.items():
        assert (np.abs(c - want) <= bound).all(), name
        assert_bits_equal(c, got["nn"], name)
        if k == 1:
            assert_bits_equal(c, np.outer(B, A), name)


@pytest.mark.parametrize("m,n,k", [(2561, 2047, 97), (1793, 2047, 1002), (200, 3000, 4003), (257, 300, 145), (70, 90, 3)])
def test_rows_that_begin_with_infinities(gpu, m, n, k):
    """With k off the multiples of 4 the last vector of a row of A given transposed (a column of B) runs into
    the next row (column): what it brings from there must not reach the row's own results."""
    A, B = _rand((m, k), 61), _rand((n, k), 62)
    A[1::2, :3], B[1::2, :3] = np.inf, np.nan
    A64, B64 = A[::2].astype(np.float64), B[::2].astype(np.float64)
    want, bound = B64 @ A64.T, (k + 8) * 2.0 ** -24 * (np.abs(B64) @ np.abs(A64).T)
    say("rows that begin with infinities", m, n, k)
    for name, c in _products(gpu, A, B).items():
        assert (np.abs(c[::2, ::2] - want) <= bound).all(), name
        assert np.isnan(c[1::2]).all() and not np.isfinite(c[:, 1::2]).any(), name


def test_products_in_parts_of_denormals(gpu):
    """The smallest operands keep all their bits: denormals times values near 1, and normal values whose
    third part would be below the smallest bf16 number but for the scale."""
    m, n, k = 2048, 2048, 96
    rng = np.random.default_rng(3)
    A = (rng.integers(1, 1 << 23, (m, k)) * 2.0 ** -149).astype(np.float32)   # denormals
    A[m // 2:] = (_rand((m - m // 2, k), 5) * np.float32(2.0 ** -112)).astype(np.float32)
    B = (_rand((n, k), 6) * np.float32(2.0 ** 30)).astype(np.float32)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    want, bound = B64 @ A64.T, _bound(A64, B64)
    say("product in parts of denormals")
    for name, c in _products(gpu, A, B).items():
        assert (np.abs(c - want) <= bound).all(), name
        assert normwise(c[:, :m // 2], want[:, :m // 2]) <= 1e-6, name


def test_products_in_parts_are_no_less_exact_than_one_rounding_per_k(gpu):
    """2-norm of the error against float64, for a left operand from a ReLU (whose zeros a sum of one
    rounding per k gets for nothing): below what such a sum has, computed here in float32."""
    m, n, k = 2048, 2048, 576
    A, B = _rand((m, k), 21, relu=True), _rand((n, k), 22)
    want = B[:64].astype(np.float64) @ A.astype(np.float64).T
    acc = np.zeros((64, m), np.float32)
    for q in range(k):  # a fused multiply-add per k
        acc = (acc.astype(np.float64) + np.outer(B[:64, q].astype(np.float64), A[:, q].astype(np.float64))).astype(np.float32)
    ref = np.linalg.norm(acc - want)
    for name, c in _products(gpu, A, B).items():
        assert np.linalg.norm(c[:64] - want) <= 0.6 * ref, name


@pytest.mark.parametrize("m,n,k", [(2048, 2048, 96), (1793, 2047, 1001), (4095, 4096, 515)])
def test_sums_of_one_term(gpu, m, n, k):
    """A sum whose other terms are zero has no rounding of a running value to gain from.  What is left is
    that of the result, 2^-24, which the fp32 instruction has too, and the three products of parts that are
    left out: |second part| <= 2^-8, |third| <= 2^-17 of a value, 2 x 2^-25 and 2^-34 of the product
    (the sums of the small parts, at 2^-8, add less than 2^-28)."""
    rng = np.random.default_rng(k)
    hot, value, B = rng.integers(0, k, m), _rand(m, 43), _rand((n, k), 42)
    A = np.zeros((m, k), np.float32)
    A[np.arange(m), hot] = value
    want = B[:, hot].astype(np.float64) * value.astype(np.float64)
    say("sums of one term", m, n, k)
    for name, c in _products(gpu, A, B).items():
        assert (np.abs(c - want) <= (2.0 ** -23 + 2.0 ** -28) * np.abs(want)).all(), name
    A[np.arange(m), hot] = 1.0  # 1 = 1 + 0 + 0: times a value, its three parts and their sum
    for name, c in _products(gpu, A, B).items():
        assert_bits_equal(c, B[:, hot], name)


@pytest.mark.parametrize("m,n,k,rows", [(2562, 2047, 100, 128), (4094, 4095, 514, 256)])
def test_epilogues_of_products_in_parts(gpu, m, n, k, rows):
    """Bias, ReLU, gate and update on a product in parts have the bits of the separate operators."""
    A, B = _rand((m, k), 31), _rand((n, k), 32)
    rng = np.random.default_rng(33)
    bias, gate, w = (rng.standard_normal(s).astype(np.float32) for s in (m, m * n, m * n))
    nb = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k)
    assert _plan(gpu, m, n, k, nb)[0] == rows
    plain = _products(gpu, A, B)["nn"].reshape(-1)
    ws, c = gpu.empty(nb // 4 + 1), gpu.empty(m * n)
    a, b = gpu.up(np.ascontiguousarray(A.T).reshape(-1)), gpu.up(B.reshape(-1))
    at, bt = gpu.up(A.reshape(-1)), gpu.up(np.ascontiguousarray(B.T).reshape(-1))
    tail = (m, n, k)
    wsz = (ws.p, ctypes.c_size_t(nb))
    say("epilogues of products in parts")
    dbias, dgate, dw = gpu.up(bias), gpu.up(gate), gpu.up(w)
    gpu.call("mnv_sgemm_nn_bias", a.p, b.p, dbias.p, c.p, *tail, 1, *wsz)
    biased = (plain.reshape(n, m) + bias).reshape(-1)
    assert_bits_equal(gpu.down(c), np.where(biased > 0, biased, np.float32(0)), "bias and ReLU")
    gpu.call("mnv_sgemm_tn", at.p, b.p, dgate.p, c.p, *tail, *wsz)
    assert_bits_equal(gpu.down(c), np.where(gate > 0, plain, np.float32(0)), "gate")
    gpu.call("mnv_sgemm_nt_sgd", a.p, bt.p, dw.p, ctypes.c_float(0.25), c.p, *tail, *wsz)
    assert_bits_equal(gpu.down(c), w - np.float32(0.25) * plain, "update")


@pytest.mark.parametrize("C,K,tile", [(96, 136, 4), (64, 256, 5), (40, 130, 3)])
def test_filtering_passes_of_values_without_parts(gpu, C, K, tile):
    """The minimal-filtering passes multiply transformed tensors in parts: inputs scaled by 2^100 and more, whose
    transforms have none, give the scaled results of ordinary ones to the rounding of the sums."""
    N, H = 6, 13
    p = (N, C, K, H, H, 1, 1, 1, 1, 3, 3)
    if C % 16:
        p = (N, 48, K, H, H, 1, 1, 1, 1, 3, 3)
    C = p[1]
    rng = np.random.default_rng(C + K)
    x, w, b = (rng.standard_normal(s).astype(np.float32) for s in (N * C * H * H, K * C * 9, K))
    dy = rng.standard_normal(N * K * H * H).astype(np.float32)
    up, down = np.float32(2.0 ** 112), np.float32(2.0 ** -30)
    mode = gpu.L.mnv_conv_winograd_mode(tile)
    try:
        nb = max(gpu.L.mnv_conv_fwd_workspace_bytes(*p), gpu.L.mnv_conv_bwd_filter_workspace_bytes(*p))
        ws = gpu.empty(nb // 4 + 1)
        top, fd = gpu.empty(N * K * H * H), gpu.empty(K * C * 9)

        def passes(sx, sw, sd):
            say("filtering passes", p, "tile mode", tile, "scale", float(sx))
            dx, dw, db, ddy = (gpu.up(v) for v in (x * sx, w * sw, b * sx * sw, dy * sd))
            gpu.call("mnv_conv_fwd", dx.p, dw.p, db.p, top.p, *p, ws.p, ctypes.c_size_t(nb))
            gpu.call("mnv_conv_bwd_filter", dx.p, ddy.p, fd.p, *p, ws.p, ctypes.c_size_t(nb))
            return gpu.down(top).astype(np.float64) / (float(sx) * float(sw)), gpu.down(fd).astype(np.float64) / (float(sx) * float(sd))

        one = np.float32(1)
        ordinary, scaled = passes(one, one, one), passes(up, down, down)
    finally:
        gpu.L.mnv_conv_winograd_mode(mode)
    for got, want in zip(scaled, ordinary):
        assert np.isfinite(got).all() and normwise(got, want) <= 2e-5


DIRECT = [  # N, C, K, H, W, pad, stride, filter
    (10, 96, 256, 27, 27, 2, 1, 5),    # k ranges; 96 columns in the data gradient
    (3, 48, 130, 57, 55, 1, 1, 3),     # an odd number of slabs, two columns in the last tile
    (9, 16, 200, 41, 43, 0, 1, 3),     # one slab per tap, no padding
    (12, 3, 96, 131, 127, 0, 4, 11),   # the channels of an image, every k its own gather
    (6, 7, 70, 83, 85, 0, 1, 8),       # whole groups of four taps; 96-column tiles
    (5, 9, 130, 77, 80, 0, 2, 7),      # one tap short of them, an odd number of channels
    (8, 400, 136, 33, 33, 0, 1, 1),
    (8, 64, 192, 61, 59, 1, 2, 3),     # 96-column tiles
    (1, 256, 80, 70, 67, 1, 1, 3),     # one image, a tile that is not full
]


@pytest.mark.parametrize("case", DIRECT, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("infinite", [False, True])
def test_direct_convolutions_in_parts_against_float64(gpu, case, infinite):
    """The implicit products of the convolutions, forward, data and filter gradient, with all of the
    workspace, with what the permuted filter alone takes, and (forward) with none; once with an
    infinity among the inputs, which reaches the outputs that it reaches in exact arithmetic."""
    N, C, K, H, W, pad, st, R = case
    p = (N, C, K, H, W, pad, pad, st, st, R, R)
    Ho, Wo = (H + 2 * pad - R) // st + 1, (W + 2 * pad - R) // st + 1
    rng = np.random.default_rng(sum(case))
    x, w, b, dy = (rng.standard_normal(s).astype(np.float32) for s in ((N, C, H, W), (K, C, R, R), (K,), (N, K, Ho, Wo)))
    if infinite:
        x[N - 1, C // 2, H // 2, W // 2] = np.inf
        dy[0, K - 1, Ho // 3, Wo // 3] = -np.inf
    x64, w64, dy64 = (torch.from_numpy(v).double() for v in (x, w, dy))

    def passes(x, w, dy):
        xs, ws = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
        y = torch.nn.functional.conv2d(xs, ws.flip(2, 3), None, st, pad)
        dx, dw = torch.autograd.grad(y, (xs, ws), dy)
        return [v.detach().numpy() for v in (y, dx, dw)]

    # |sum| <= (roundings) 2^-23 sum |a||b|: one per eight k, those of the k ranges, and in fp32
    # arithmetic next to an infinity one of 2^-24 per k
    fin = [torch.nan_to_num(v, posinf=0.0, neginf=0.0) for v in (x64, dy64)]
    size = passes(fin[0].abs(), w64.abs(), fin[1].abs())
    want = passes(x64, w64, dy64) if not infinite else None
    if infinite:  # where the infinity goes, with its sign; torch's products would mix it with zeros
        base = passes(fin[0], w64, fin[1])
        mark_x, mark_dy = torch.isinf(x64).double() * torch.sign(x64), torch.isinf(dy64).double() * torch.sign(dy64)
        reach = [torch.nn.functional.conv2d(mark_x, w64.flip(2, 3), None, st, pad).numpy(),
                 passes(fin[0], w64, mark_dy)[1]]
        # every tap of the marked pixel and every pixel of the marked gradient meets one finite value
        dw_x, dw_dy = passes(mark_x, w64, fin[1])[2], passes(fin[0], w64, mark_dy)[2]
        reach.append(dw_x)
        both = (dw_x != 0) & (dw_dy != 0) & (np.sign(dw_x) != np.sign(dw_dy))
        reach[2] = np.where(dw_dy != 0, dw_dy, reach[2])
        want = []
        for v, r in zip(base, reach):
            v = v.copy()
            v[r != 0] = np.inf * np.sign(r[r != 0])
            want.append(v)
        want[2][both] = np.nan
    bias = np.broadcast_to(b.astype(np.float64)[None, :, None, None], want[0].shape)
    want[0] = want[0] + bias
    ks = (C * R * R, K * R * R, N * Ho * Wo)
    bound = [(k / 8 + 64 if not infinite else k + 64) * 2.0 ** -23 * v for k, v in zip(ks, size)]
    bound[0] = bound[0] + np.abs(bias) * 2.0 ** -20
    dx_, dw_, db_, ddy = (gpu.up(np.ascontiguousarray(v).reshape(-1)) for v in (x, w, b, dy))
    mode = gpu.L.mnv_conv_winograd_mode(0)
    try:
        jobs = [("fwd", want[0], bound[0], gpu.L.mnv_conv_fwd_workspace_bytes(*p), w.size * 4),
                ("bwd_data", want[1], bound[1], gpu.L.mnv_conv_bwd_data_workspace_bytes(*p), w.size * 4),
                ("bwd_filter", want[2], bound[2], gpu.L.mnv_conv_bwd_filter_workspace_bytes(*p), 0)]
        for name, ref, tol, full, small in jobs:
            ws, out = gpu.empty(full // 4 + 1), gpu.empty(ref.size)
            for nb in ((full, small, 0) if name == "fwd" else (full, small)):
                say("direct convolution", case, name, "workspace", nb, "infinite", infinite)
                args = {"fwd": (dx_.p, dw_.p, db_.p), "bwd_data": (ddy.p, dw_.p), "bwd_filter": (dx_.p, ddy.p)}[name]
                gpu.call("mnv_conv_" + name, *args, out.p, *p, ws.p if nb else None, ctypes.c_size_t(nb))
                got = gpu.down(out).reshape(ref.shape)
                assert np.array_equal(np.isnan(got), np.isnan(ref)), (name, nb)
                inf = np.isinf(ref)
                assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf] > 0, ref[inf] > 0), (name, nb)
                ok = np.isfinite(ref)
                assert (np.abs(got[ok] - ref[ok]) <= tol[ok]).all(), (name, nb, float(np.max(np.abs(got[ok] - ref[ok]) / tol[ok])))
    finally:
        gpu.L.mnv_conv_winograd_mode(mode)


CHANNELS = [  # N, C, K, H, W, pad, stride, filter: channels of the reduction 16 at a time, the last ones padded
    (2, 8, 9, 7, 7, 1, 1, 3),         # half of a slab; 128 x 32 tiles with k ranges
    (3, 17, 24, 12, 11, 1, 1, 3),     # one channel in the last slab
    (3, 15, 31, 9, 20, 1, 2, 3),      # one short of a slab; strided, the data gradient by the generic gathers
    (2, 40, 88, 33, 31, 2, 1, 5),     # 64 x 64 tiles
    (3, 72, 136, 57, 50, 1, 1, 3),    # in parts
    (3, 104, 200, 40, 41, 0, 1, 3),   # no padding: 96-column tiles in the data gradient
]


@pytest.mark.parametrize("case", CHANNELS, ids=lambda c: "x".join(map(str, c)))
def test_channels_off_the_multiples_of_16(gpu, case):
    """Forward and data gradient with all of the workspace, with just the permuted filter's, and with one
    byte less.  The last image is all infinities: it must not reach the images before it, whose
    missing channels lie where its first ones are."""
    N, C, K, H, W, pad, st, R = case
    p = (N, C, K, H, W, pad, pad, st, st, R, R)
    Ho, Wo = (H + 2 * pad - R) // st + 1, (W + 2 * pad - R) // st + 1
    rng = np.random.default_rng(sum(case))
    x, w, b, dy = (rng.standard_normal(s).astype(np.float32) for s in ((N, C, H, W), (K, C, R, R), (K,), (N, K, Ho, Wo)))
    x[N - 1], dy[N - 1] = np.inf, np.inf
    conv, m = torch.nn.functional, N - 1
    x64, w64, dy64 = (torch.from_numpy(v).double() for v in (x[:m], w.copy(), dy[:m]))

    def passes(x, w, dy):
        dx = conv.conv_transpose2d(dy, w.flip(2, 3), None, st, pad, ((H + 2 * pad - R) % st, (W + 2 * pad - R) % st))
        return conv.conv2d(x, w.flip(2, 3), None, st, pad).numpy(), dx.numpy()

    want, size = passes(x64, w64, dy64), passes(x64.abs(), w64.abs(), dy64.abs())
    want = want[0] + b.astype(np.float64)[None, :, None, None], want[1]
    assert want[0].shape == (m, K, Ho, Wo) and want[1].shape == (m, C, H, W)
    # one rounding per k at most, those of the k ranges, the bias
    bound = [(k * R * R + 64) * 2.0 ** -23 * v + 1e-6 for k, v in zip((C, K), size)]
    d = {n: gpu.up(np.ascontiguousarray(v).reshape(-1)) for n, v in (("x", x), ("w", w), ("b", b), ("dy", dy))}
    mode = gpu.L.mnv_conv_winograd_mode(0)
    try:
        for name, args, ref, tol, count, inner in (("fwd", ("x", "w", "b"), want[0], bound[0], K, C),
                                                   ("bwd_data", ("dy", "w"), want[1], bound[1], C, K)):
            full = getattr(gpu.L, "mnv_conv_%s_workspace_bytes" % name)(*p)
            permuted = count * R * R * ((inner + 15) // 16 * 16) * 4
            per_image = ref[0].size
            for nb in (full, permuted, permuted - 1):
                say("channels off 16", case, name, "workspace", nb)
                out, ws = gpu.up(np.full(N * per_image + 4, np.float32(7.5), np.float32)), gpu.empty(max(full, nb) // 4 + 1)
                gpu.call("mnv_conv_" + name, *[d[a].p for a in args], out.p, *p, ws.p, ctypes.c_size_t(nb))
                got = gpu.down(out)
                assert (got[N * per_image:] == 7.5).all(), "wrote past the result"
                got = got[:m * per_image].reshape(ref.shape)
                assert (np.abs(got - ref) <= tol).all(), (name, nb, float(np.nanmax(np.abs(got - ref) / tol)))
    finally:
        gpu.L.mnv_conv_winograd_mode(mode)
