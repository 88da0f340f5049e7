"""Products and operators whose extents or addresses are off the 16-byte grid: the paths that
fetch 16 bytes at a time there, at their edges."""
import ctypes

import numpy as np
import pytest

import test_gpu_winograd as tw
from gpu_util import Gpu, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return Gpu()


def _rand(n, seed):
    return np.random.default_rng(seed).standard_normal(n).astype(np.float32)


@pytest.mark.parametrize("m,n,k", [(65, 67, 1), (66, 33, 3), (129, 65, 18), (7, 130, 31), (131, 17, 46), (257, 66, 1027)])
@pytest.mark.parametrize("form", ["nn", "tn", "nt"])
def test_sgemm_vectors_past_an_edge_bring_nothing_in(gpu, m, n, k, form):
    """A vector that reaches past a row or column end meets the next one's values: an infinity and
    a NaN there reach their own row and column of the result only, and operands 4 bytes off the
    16-byte grid give the bits of aligned ones.  Sums of k products against float64: k + 1
    roundings of 2^-24 at most, relative to the sum of magnitudes."""
    say("sgemm", form, m, n, k)
    a, b = _rand(m * k, 1).reshape(k, m).T, _rand(k * n, 2).reshape(n, k).T  # A{m,k}, B{k,n}
    a, b = a.copy(), b.copy()
    a[0, :] = np.inf          # every vector that begins in row m - 1 ends in the next column's row 0
    b[0, n - 1] = np.nan      # a vector past K of column n - 2 meets it
    stored = {"nn": (a.T, b.T), "tn": (a, b.T), "nt": (a.T, b)}[form]
    got = []
    for shift in (0, 1):
        dev = [gpu.up(np.concatenate([np.zeros(shift, np.float32), np.ascontiguousarray(v).reshape(-1)])) for v in stored]
        dc = gpu.empty(m * n)
        ws_bytes = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k)
        ws = gpu.empty(ws_bytes // 4 + 1)
        args = [ctypes.c_void_p(ctypes.cast(d.p, ctypes.c_void_p).value + 4 * shift) for d in dev]
        if form == "tn":
            args.append(None)
        gpu.call("mnv_sgemm_" + form, *args, dc.p, m, n, k, ws.p, ctypes.c_size_t(ws_bytes))
        got.append(gpu.down(dc).reshape(n, m).T)
    assert got[0].tobytes() == got[1].tobytes()
    want = a[1:].astype(np.float64) @ b[:, :n - 1].astype(np.float64)
    bound = (k + 1) * 2.0 ** -24 * (np.abs(a[1:]).astype(np.float64) @ np.abs(b[:, :n - 1]))
    assert np.all(np.abs(got[0][1:, :n - 1] - want) <= bound)
    assert not np.isfinite(got[0][0]).any() and np.isnan(got[0][:, n - 1]).all()


# N, C, K, H, W, pad: groups of 256 tiles that begin and end inside a plane, planes whose size is
# no multiple of four (the last chunk of a plane reaches into the next one, or past the tensor),
# one tile per plane (every group spans many whole planes)
SPANS = [(2, 16, 32, 67, 61, 1), (1, 16, 16, 101, 99, 2), (3, 16, 32, 57, 55, 0), (70, 16, 16, 3, 5, 1)]


@pytest.mark.parametrize("q", SPANS, ids=lambda q: "x".join(map(str, q)))
@pytest.mark.parametrize("tile", [tw.F2, tw.F4, tw.F5], ids=["2x2", "4x4", "5x5"])
def test_transforms_of_tiles_that_cross_planes(gpu, ora, q, tile):
    """All three minimal-filtering passes against the oracle, with that path's own bounds."""
    tw._passes_against_oracle(gpu, ora, q + (q[5],), tile, 3, tw.BOUND[tile])


@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 9, 12])
@pytest.mark.parametrize("m,k", [(256, 4096), (257, 4098), (1003, 1047), (4099, 4101)])
def test_sgemm_of_few_columns(gpu, m, n, k):
    """Row blocks of 256 (64 for a transposed A), k ranges of four wavefronts, each width the
    columns are rounded up to.  k + 1 roundings against float64; the transposed forms and a fused
    bias have the bits of the plain product; so has a second call; a workspace for fewer k ranges and
    none at all stay within the bound."""
    say("sgemm, few columns", m, n, k)
    a, b, bias = _rand(m * k, 3), _rand(k * n, 4), _rand(m, 5)
    A, B = a.reshape(k, m).T, b.reshape(n, k).T
    ws_bytes = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k)
    ws, dc = gpu.empty(ws_bytes // 4 + 1), gpu.empty(m * n)
    at, bt = gpu.up(np.ascontiguousarray(A).reshape(-1)), gpu.up(np.ascontiguousarray(B).reshape(-1))
    da, db, dbias = gpu.up(a), gpu.up(b), gpu.up(bias)

    def run(name, *args, nbytes=ws_bytes):
        gpu.call("mnv_sgemm_" + name, *args, ws.p if nbytes else None, ctypes.c_size_t(nbytes))
        return gpu.down(dc).copy()

    got = run("nn", da.p, db.p, dc.p, m, n, k)
    want = A.astype(np.float64) @ B.astype(np.float64)
    bound = (k + 1) * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(B))
    assert np.all(np.abs(got.reshape(n, m).T - want) <= bound)
    for other in (run("nn", da.p, db.p, dc.p, m, n, k), run("tn", at.p, db.p, None, dc.p, m, n, k),
                  run("nt", da.p, bt.p, dc.p, m, n, k)):
        assert other.tobytes() == got.tobytes()
    assert run("nn_bias", da.p, db.p, dbias.p, dc.p, m, n, k, 1).tobytes() == \
        np.maximum(got.reshape(n, m) + bias, np.float32(0)).reshape(-1).tobytes()
    for nbytes in (ws_bytes // 3 // 4 * 4, 0):
        few = run("nn", da.p, db.p, dc.p, m, n, k, nbytes=nbytes)
        assert np.all(np.abs(few.reshape(n, m).T - want) <= bound)


# m, n, offset of the operands in floats: lines and columns that end in 1, 2 or 3 values, at every
# alignment, around the widths that the kernels change at (64 and 128 columns of a tile, 2048, 4096
# and 8192 values of a line)
ODD = [(1, 1, 0), (3, 5, 1), (63, 65, 2), (65, 63, 3), (130, 127, 0), (128, 128, 1), (1001, 257, 0), (1027, 1021, 2),
       (2049, 9, 0), (4093, 7, 3), (8191, 5, 1), (8192, 6, 2), (8197, 3, 0), (2047, 2051, 1)]


@pytest.mark.parametrize("m,n,off", ODD)
def test_matrix_operators_off_the_16_byte_grid(gpu, m, n, off):
    """Results against numpy, and the floats before and behind them untouched.  Data movement,
    single operations and maxima have no error.  A sum of L values: L roundings of 2^-24 relative
    to the sum of magnitudes.  Soft-max: an exponential, a sum of L and a quotient, L + 8 roundings."""
    say("matrix operators", m, n, off)
    x, y, row, col = _rand(m * n, 6), _rand(m * n, 7), _rand(m, 8), _rand(n, 9)
    lead = off + 4
    at = lambda d: ctypes.c_void_p(ctypes.cast(d.p, ctypes.c_void_p).value + 4 * lead)  # noqa: E731
    up = lambda v: gpu.up(np.concatenate([np.full(lead, 7, np.float32), v, np.full(5, 7, np.float32)]))  # noqa: E731
    dx, dy_, drow, dcol = up(x), up(y), gpu.up(row), gpu.up(col)

    def run(name, size, *args):
        out = up(np.full(size, 3, np.float32))
        gpu.call("mnv_" + name, *[at(out) if a == "out" else a for a in args])
        whole = gpu.down(out)
        assert np.all(whole[:lead] == 7) and np.all(whole[lead + size:] == 7), name
        return whole[lead:lead + size].copy()

    X, Y = x.reshape(n, m), y.reshape(n, m)  # X[column, row]
    assert np.array_equal(run("transpose", m * n, at(dx), "out", m, n).reshape(m, n), X.T)
    assert np.array_equal(run("norm_add_row", m * n, at(dx), drow.p, "out", m, n).reshape(n, m), X + row)
    assert np.array_equal(run("norm_mul_col", m * n, at(dx), dcol.p, "out", m, n).reshape(n, m), X * col[:, None])
    assert np.array_equal(run("reduce_max_col", n, at(dx), "out", m, n), X.max(1))
    assert np.array_equal(run("reduce_max_row", m, at(dx), "out", m, n), X.max(0))
    assert np.array_equal(run("maxindex_col", n, at(dx), "out", m, n), X.argmax(1))
    assert np.array_equal(run("maxindex_row", m, at(dx), "out", m, n), X.argmax(0))
    X64, Y64, u = X.astype(np.float64), Y.astype(np.float64), 2.0 ** -24
    for name, axis, length in (("reduce_sum_col", 1, m), ("reduce_sum_row", 0, n)):
        got = run(name, m * n // length, at(dx), "out", m, n)
        assert np.all(np.abs(got - X64.sum(axis)) <= length * u * np.abs(X64).sum(axis))
    e = np.exp(X64 - X64.max(1, keepdims=True))
    p = e / e.sum(1, keepdims=True)
    got = run("softmax_instance_fwd", m * n, at(dx), "out", n, m, 1, 1).reshape(n, m)
    # the hardware exponential's argument -- up to 10 here -- is rounded once, 10 u more
    assert np.all(np.abs(got - p) <= (m + 18) * u * p)
    dot = (X64 * Y64).sum(1, keepdims=True)
    got = run("softmax_instance_bwd", m * n, at(dy_), at(dx), "out", n, m, 1, 1).reshape(n, m)
    bound = np.abs(X64) * ((m + 2) * u * np.abs(X64 * Y64).sum(1, keepdims=True) + 3 * u * np.abs(Y64 - dot))
    assert np.all(np.abs(got - X64 * (Y64 - dot)) <= bound)


@pytest.mark.parametrize("N,K,H,W", [(256, 16, 3, 5), (300, 7, 2, 2), (37, 65, 9, 7), (5, 3, 1, 1)])
def test_bias_gradient_of_many_image_groups(gpu, N, K, H, W):
    """One to more than 64 group sums per channel, channels off the four of a workgroup: a sum of
    L values against float64, L roundings of 2^-24 relative to the sum of magnitudes."""
    say("bias gradient", N, K, H, W)
    dy = _rand(N * K * H * W, 10)
    nbytes = gpu.L.mnv_conv_bwd_bias_workspace_bytes(N, K)
    ws, db, ddy = gpu.empty(nbytes // 4 + 1), gpu.empty(K), gpu.up(dy)
    gpu.call("mnv_conv_bwd_bias", ddy.p, db.p, N, K, H, W, ws.p, ctypes.c_size_t(nbytes))
    t = dy.reshape(N, K, H * W).astype(np.float64)
    bound = N * H * W * 2.0 ** -24 * np.abs(t).sum((0, 2))
    assert np.all(np.abs(gpu.down(db) - t.sum((0, 2))) <= bound)
