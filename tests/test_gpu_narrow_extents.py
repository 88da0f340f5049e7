"""Products and matrix operators with one narrow extent: the kernel that each of them takes at the
sizes where the choice changes, and that none of them costs a multiple of the same work in a form
that reads its operands alike.  Times are medians of calls of both forms in turn; the bounds
leave a third and more to what the forms measured (both figures beside each bound)."""
import ctypes

import numpy as np
import pytest

from gpu_util import Gpu, assert_bits_equal, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return Gpu()


def _rand(n, seed):
    return np.random.default_rng(seed).standard_normal(n).astype(np.float32)


def _ratio(gpu, slow, fast, iters=20):
    """Median time of slow() over that of fast(), measured in turn."""
    t = [[gpu.dev.time_ms(f, iters=iters, warmup=2) for f in (slow, fast)] for _ in range(9)]
    a, b = (sorted(x)[4] for x in zip(*t))
    say("  %.2f us against %.2f us" % (a * 1e3, b * 1e3))
    return a / b


def _plan(gpu, m, n, k, ws_bytes):
    v = [ctypes.c_int() for _ in range(3)]
    assert gpu.L.mnv_sgemm_nn_plan(m, n, k, ctypes.c_size_t(ws_bytes), *[ctypes.byref(x) for x in v]) == 0
    return tuple(x.value for x in v)


def _bits(gpu, form, a, b, m, n, k, ws_bytes, *more):
    """The product through mnv_sgemm_<form>: a, b on the device as the form takes them."""
    ws, dc = gpu.empty(ws_bytes // 4 + 1), gpu.empty(m * n)
    gpu.call("mnv_sgemm_" + form, a.p, b.p, *more, dc.p, m, n, k, ws.p, ctypes.c_size_t(ws_bytes))
    return gpu.down(dc)


# 64 rows to a workgroup: one row, 63 and all of the last one's; k ranges that end in 1 to 4 values of
# a vector, in the first half of a run of 32 and in the second; at most 16 k per wavefront and more
@pytest.mark.parametrize("m,k,n", [(257, 16385, 1), (257, 16385, 5), (319, 16384, 4), (319, 16384, 8), (4160, 4110, 3),
                                   (4160, 4110, 12), (4097, 8207, 1), (4097, 8207, 11)])
def test_few_columns_of_a_transposed_operand_have_the_plain_forms_bits(gpu, m, k, n):
    """Values over the whole exponent range (products that underflow and that overflow among them), an
    infinity and a NaN in a row of A and in a column of B: the bits of mnv_sgemm_nn, and the other
    rows and columns finite where all their products are."""
    say("few columns, transposed", m, n, k)
    ws_bytes = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k)
    tile, _, groups = _plan(gpu, m, n, k, ws_bytes)
    assert (tile, groups) == (256, 4), "the case must run the few-column kernels"
    for wide in (False, True):
        a, b = _rand(m * k, 20).reshape(k, m), _rand(n * k, 21).reshape(n, k)
        if wide:
            a[::7] *= np.float32(1e-30)
            b[:, ::5] *= np.float32(1e-12)
        else:
            a[k - 1, m - 1], a[3, 7] = np.inf, np.nan
            b[n - 1, 5] = -np.inf
        da, dat = gpu.up(a.reshape(-1)), gpu.up(np.ascontiguousarray(a.T).reshape(-1))
        db = gpu.up(b.reshape(-1))
        want = _bits(gpu, "nn", da, db, m, n, k, ws_bytes)
        assert _bits(gpu, "tn", dat, db, m, n, k, ws_bytes, None).tobytes() == want.tobytes()
        if not wide:
            C = want.reshape(n, m)
            assert np.isfinite(np.delete(np.delete(C, n - 1, 0), (7, m - 1), 1)).all()
            assert not np.isfinite(C[n - 1]).any() and not np.isfinite(C[:, (7, m - 1)]).any()
        gate = _rand(m * n, 22)
        dgate = gpu.up(gate)
        got = _bits(gpu, "tn", dat, db, m, n, k, ws_bytes, dgate.p)
        assert got.tobytes() == np.where(gate > 0, want, np.float32(0)).tobytes()


@pytest.mark.parametrize("m,n,k", [(4096, 12, 4096), (9216, 2, 4096), (4096, 8, 9216)])
def test_few_columns_of_a_transposed_operand_cost_what_the_plain_form_does(gpu, m, n, k):
    """18.0 against 20.6 us, 35.3 / 26.5 and 33.2 / 30.4 (one lane per row of A: 92.8, 58.1 and 62.5)."""
    say("few columns, transposed, time", m, n, k)
    ws_bytes = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k)
    a, b, c, ws = gpu.empty(m * k), gpu.empty(n * k), gpu.empty(m * n), gpu.empty(ws_bytes // 4 + 1)
    for d, count in ((a, m * k), (b, n * k)):
        gpu.call("mnv_randn", d.p, ctypes.c_size_t(count), ctypes.c_uint64(5), ctypes.c_float(0), ctypes.c_float(1))
    tail = (c.p, m, n, k, ws.p, ctypes.c_size_t(ws_bytes), gpu.dev.stream)
    assert _ratio(gpu, lambda: gpu.L.mnv_sgemm_tn(a.p, b.p, None, *tail), lambda: gpu.L.mnv_sgemm_nn(a.p, b.p, *tail)) < 1.8


def _at(d, floats):
    return ctypes.c_void_p(d.ptr + 4 * floats)


def _guarded(v, lead):
    """v behind `lead` floats of 7 and in front of 5."""
    return np.concatenate([np.full(lead, 7, np.float32), v, np.full(5, 7, np.float32)])


# either extent within the small tile and past it, with and without 128 large tiles; three tile columns
# of the result and one value more (shifted runs), rows that end with every shift; a result whose last
# tile column is full with the shift (52 and 116 modulo 128)
@pytest.mark.parametrize("m,n", [(1, 20001), (20001, 1), (3, 16387), (16387, 3), (64, 8197), (65, 16389), (16389, 64),
                                 (16389, 65), (8191, 127), (8193, 129), (6145, 383), (6145, 384), (6145, 385), (6148, 388),
                                 (1000, 52), (4096, 116), (2052, 1012), (33, 401), (5, 500)])
@pytest.mark.parametrize("off", [0, 1, 3])
def test_transpose_of_narrow_matrices(gpu, m, n, off):
    """Bit for bit, and the floats around the result untouched."""
    say("transpose", m, n, off)
    x = _rand(m * n, 30)
    lead = off + 4
    src, dst = gpu.up(_guarded(x, lead)), gpu.up(_guarded(np.zeros(m * n, np.float32), lead))
    gpu.call("mnv_transpose", _at(src, lead), _at(dst, lead), m, n)
    assert gpu.down(dst).tobytes() == _guarded(x.reshape(n, m).T.reshape(-1), lead).tobytes()


@pytest.mark.parametrize("m,n", [(1714285, 7), (5, 2400001)])
def test_transpose_of_narrow_matrices_costs_a_few_copies(gpu, m, n):
    """Off the 16-byte grid: 35 and 46 us, copies of the same bytes 15 (large tiles: 104 and 102)."""
    say("transpose, time", m, n)
    a, c = gpu.empty(m * n), gpu.empty(m * n)
    gpu.call("mnv_fill", a.p, ctypes.c_size_t(m * n), ctypes.c_float(1))
    s = gpu.dev.stream
    assert _ratio(gpu, lambda: gpu.L.mnv_transpose(a.p, c.p, m, n, s), lambda: gpu.L.mnv_copy(a.p, c.p, m * n, s)) < 4.5


# rows: one per thread and four (16), a cut last vector of each length, one and several wavefronts and
# workgroups to a column, a last workgroup with a single row's vector (1025)
@pytest.mark.parametrize("m", [1, 3, 15, 16, 17, 18, 19, 255, 257, 1023, 1025, 1026, 1283, 2049])
@pytest.mark.parametrize("off", [0, 2])
def test_broadcast_over_few_rows(gpu, m, off):
    """Bit for bit into another matrix and in place, and the floats around the result untouched."""
    n = 41
    say("broadcast", m, n, off)
    x, row, col = _rand(m * n, 31), _rand(m, 32), _rand(n, 33)
    X, lead = x.reshape(n, m), off + 4
    drow, dcol = gpu.up(row), gpu.up(col)
    for name, vec, want in (("norm_sub_row", drow, X - row), ("norm_div_col", dcol, X / col[:, None])):
        src, dst = gpu.up(_guarded(x, lead)), gpu.up(_guarded(np.zeros(m * n, np.float32), lead))
        for to in (dst, src):
            gpu.call("mnv_" + name, _at(src, lead), vec.p, _at(to, lead), m, n)
            assert gpu.down(to).tobytes() == _guarded(want.reshape(-1), lead).tobytes(), name


@pytest.mark.parametrize("m,n", [(10, 2000000), (15, 1333333), (7, 2857143)])
def test_broadcast_over_few_rows_costs_a_few_streams(gpu, m, n):
    """86, 60 and 136 us, adding a constant to as many values 26 (four rows per thread and the last ones
    element by element: 316, 278 and 551)."""
    say("broadcast, time", m, n)
    a, c, v = gpu.empty(m * n), gpu.empty(m * n), gpu.empty(m)
    for d, count in ((a, m * n), (v, m)):
        gpu.call("mnv_fill", d.p, ctypes.c_size_t(count), ctypes.c_float(1))
    s = gpu.dev.stream
    assert _ratio(gpu, lambda: gpu.L.mnv_norm_add_row(a.p, v.p, c.p, m, n, s),
                  lambda: gpu.L.mnv_const_add(a.p, c.p, ctypes.c_float(2), m * n, s)) < 8


# rows: one per thread, four, and a cut last vector of each length behind a full workgroup and alone; columns
# at the sizes where the kernels change (4, 32, 48, 128 and 256), and enough for several trips of a thread
ROW_SHAPES = [(1, 300), (2, 5), (3, 260), (5, 4), (6, 5), (7, 31), (33, 33), (34, 47), (35, 48), (36, 127), (66, 130), (67, 255),
              (37, 256), (255, 513), (1001, 300), (4099, 6), (70001, 3)]


@pytest.mark.parametrize("m,n", ROW_SHAPES)
@pytest.mark.parametrize("off", [0, 1, 2])
def test_row_reductions_with_ties_nan_and_infinities(gpu, ora, m, n, off):
    """Maxima and arg-maxima bit for bit: many ties, zeros of both signs, NaN first in some rows and inside
    others, rows of -inf and of NaN.  Sums of the finite values against float64: n roundings of 2^-24
    relative to the sum of magnitudes.  The floats around the results untouched."""
    say("row reductions", m, n, off)
    rng = np.random.default_rng(40)
    x = rng.integers(-2, 3, m * n).astype(np.float32)
    x[x == 0] = np.where(rng.random(np.count_nonzero(x == 0)) < 0.5, 0.0, -0.0)
    finite = x.copy()
    x[rng.random(m * n) < 0.1] = np.nan
    X = x.reshape(n, m)  # X[column, row]
    X[0, ::3] = np.nan
    X[:, 1::7] = -np.inf
    X[:, 4::11] = np.nan
    lead = off + 4
    for name, v, want in (("reduce_max_row", x, ora.reduction(ora.MAX, x, [m, n], [1])),
                          ("maxindex_row", x, ora.maxindex(x, [m, n], 1)), ("reduce_sum_row", finite, None)):
        src, dst = gpu.up(_guarded(v, lead)), gpu.up(_guarded(np.zeros(m, np.float32), lead))
        gpu.call("mnv_" + name, _at(src, lead), _at(dst, lead), m, n)
        got = gpu.down(dst)
        assert np.all(got[:lead] == 7) and np.all(got[lead + m:] == 7), name
        if want is not None:
            assert_bits_equal(got[lead:lead + m], want, name)
        else:
            f = finite.reshape(n, m).astype(np.float64)
            assert np.all(np.abs(got[lead:lead + m] - f.sum(0)) <= n * 2.0 ** -24 * np.abs(f).sum(0))


@pytest.mark.parametrize("m,n", [(3000001, 1), (1000001, 3)])
def test_row_reductions_of_few_columns_cost_a_few_copies(gpu, m, n):
    """17.3 us for the first, a copy of its bytes 4.5 (64 column groups: 210)."""
    say("row maxima, time", m, n)
    a, c, r = gpu.empty(m * n), gpu.empty(m * n), gpu.empty(m)
    gpu.call("mnv_fill", a.p, ctypes.c_size_t(m * n), ctypes.c_float(1))
    s = gpu.dev.stream
    assert _ratio(gpu, lambda: gpu.L.mnv_reduce_max_row(a.p, r.p, m, n, s), lambda: gpu.L.mnv_copy(a.p, c.p, m * n, s)) < 12


# values per column: one per lane (up to 64, and two for some), vectors with a cut last one (from 96 on, from
# 2049 on by a whole workgroup), few lanes to merge
@pytest.mark.parametrize("m,n", [(1, 9), (2, 5), (3, 300), (5, 7), (33, 33), (63, 65), (65, 11), (95, 13), (96, 6), (97, 6), (98, 5),
                                 (255, 4), (2047, 3), (2050, 3), (8195, 2)])
@pytest.mark.parametrize("off", [0, 1, 3])
def test_column_reductions_with_ties_nan_and_infinities(gpu, ora, m, n, off):
    """As above, along the columns: NaN first in some, columns of -inf and of NaN."""
    say("column reductions", m, n, off)
    rng = np.random.default_rng(41)
    x = rng.integers(-2, 3, m * n).astype(np.float32)
    x[x == 0] = np.where(rng.random(np.count_nonzero(x == 0)) < 0.5, 0.0, -0.0)
    finite = x.copy()
    x[rng.random(m * n) < 0.1] = np.nan
    X = x.reshape(n, m)  # X[column, row]
    X[::3, 0] = np.nan
    X[1::7] = -np.inf
    X[4::11] = np.nan
    lead = off + 4
    for name, v, want in (("reduce_max_col", x, ora.reduction(ora.MAX, x, [m, n], [0])),
                          ("maxindex_col", x, ora.maxindex(x, [m, n], 0)), ("reduce_sum_col", finite, None)):
        src, dst = gpu.up(_guarded(v, lead)), gpu.up(_guarded(np.zeros(n, np.float32), lead))
        gpu.call("mnv_" + name, _at(src, lead), _at(dst, lead), m, n)
        got = gpu.down(dst)
        assert np.all(got[:lead] == 7) and np.all(got[lead + n:] == 7), name
        if want is not None:
            assert_bits_equal(got[lead:lead + n], want, name)
        else:
            f = finite.reshape(n, m).astype(np.float64)
            assert np.all(np.abs(got[lead:lead + n] - f.sum(1)) <= m * 2.0 ** -24 * np.abs(f).sum(1))


def test_short_columns_cost_what_aligned_ones_do(gpu):
    """Sums of 11 and of 12 values: 82 us each (vectors at any address: 117 for 11)."""
    n = 1000000
    a, r, s = gpu.empty(12 * n), gpu.empty(n), gpu.dev.stream
    gpu.call("mnv_fill", a.p, ctypes.c_size_t(12 * n), ctypes.c_float(1))
    assert _ratio(gpu, lambda: gpu.L.mnv_reduce_sum_col(a.p, r.p, 11, n, s), lambda: gpu.L.mnv_reduce_sum_col(a.p, r.p, 12, n, s)) < 1.25


def _softmax64(x):
    with np.errstate(invalid="ignore"):
        e = np.exp(x - x.max(1, keepdims=True))
        return e / e.sum(1, keepdims=True)


# lines of one value per lane, of a vector per lane and of several, around the lengths where that changes
# (40 forward, 128 backward, 256, 1024, 4096, 8192), and shorter than a vector
@pytest.mark.parametrize("length", [1, 2, 3, 4, 5, 10, 36, 39, 41, 126, 127, 129, 130, 131, 252, 255, 257, 259, 1022, 1027, 2050, 4097,
                                    8191, 8194])
@pytest.mark.parametrize("off", [0, 1, 2])
def test_softmax_lines_off_the_16_byte_grid(gpu, ora, length, off):
    """Against float64: the exponential's argument is rounded once (up to 10 u relative), a thread adds up to
    length / 64 values and the threads' sums meet in a tree, (length / 64 + 32) u in all, u = 2^-24.
    Backward: a dot product of that depth, relative to its sum of magnitudes, and three roundings.  Lines with
    an infinity, a NaN, or nothing but -inf: NaN and zero where the oracle has them.  Both in place as
    well, and the floats around the results untouched."""
    lines, u, lead = 11, 2.0 ** -24, off + 4
    say("softmax lines", length, lines, off)
    x, dy = _rand(lines * length, 50), _rand(lines * length, 51)
    X = x.reshape(lines, length)
    X[3, length // 2] = np.nan
    X[5, -1] = np.inf
    X[7] = -np.inf
    X[8, : length - 1] = -np.inf
    plain = [i for i in range(lines) if i not in (3, 5, 7, 8)]
    src, ddy, dst = gpu.up(_guarded(x, lead)), gpu.up(_guarded(dy, lead)), gpu.up(_guarded(np.zeros_like(x), lead))

    def floats(d):
        whole = gpu.down(d)
        assert np.all(whole[:lead] == 7) and np.all(whole[lead + x.size:] == 7)
        return whole[lead:lead + x.size].reshape(lines, length)

    gpu.call("mnv_softmax_instance_fwd", _at(src, lead), _at(dst, lead), lines, length, 1, 1)
    got = floats(dst)
    want = _softmax64(X.astype(np.float64))
    depth = length / 64 + 32
    assert np.all(np.abs(got - want)[plain] <= depth * u * want[plain])
    ref = ora.softmax_instance_fwd(x, lines, length, 1, 1).reshape(lines, length)
    for i in (3, 5, 7, 8):
        assert np.array_equal(np.isnan(got[i]), np.isnan(ref[i])) and np.array_equal(got[i] == 0, ref[i] == 0), i
    gpu.call("mnv_softmax_instance_fwd", _at(src, lead), _at(src, lead), lines, length, 1, 1)
    assert floats(src).tobytes() == got.tobytes()

    gpu.call("mnv_softmax_instance_bwd", _at(ddy, lead), _at(src, lead), _at(dst, lead), lines, length, 1, 1)
    back = floats(dst)
    y, d = got[plain].astype(np.float64), dy.reshape(lines, length)[plain].astype(np.float64)
    dot = (y * d).sum(1, keepdims=True)
    bound = y * (depth * u * np.abs(y * d).sum(1, keepdims=True) + 3 * u * np.abs(d - dot))
    assert np.all(np.abs(back[plain] - y * (d - dot)) <= bound)
    assert np.isnan(back[3]).all() and np.isnan(back[7]).all()
    gpu.call("mnv_softmax_instance_bwd", _at(ddy, lead), _at(src, lead), _at(ddy, lead), lines, length, 1, 1)
    assert floats(ddy).tobytes() == back.tobytes()


def test_short_softmax_lines_backward_cost_what_aligned_ones_do(gpu):
    """10 and 12 values to a line: 125 and 133 us (a vector per lane for 10: 212)."""
    n, s = 1000000, gpu.dev.stream
    dy, y, dx = gpu.empty(12 * n), gpu.empty(12 * n), gpu.empty(12 * n)
    for d in (dy, y):
        gpu.call("mnv_fill", d.p, ctypes.c_size_t(12 * n), ctypes.c_float(0.1))
    assert _ratio(gpu, lambda: gpu.L.mnv_softmax_instance_bwd(dy.p, y.p, dx.p, n, 10, 1, 1, s),
                  lambda: gpu.L.mnv_softmax_instance_bwd(dy.p, y.p, dx.p, n, 12, 1, 1, s)) < 1.5


def _few(gpu, m, n, k, ws_bytes):
    tile, ranges, groups = _plan(gpu, m, n, k, ws_bytes)
    assert (tile, groups) == (256, 4), "the case must run the few-column kernels"
    return ranges


# every width the columns are rounded up to, at odd and even extents of the three lines of the rule; k ranges that
# end in a step of 8, of 4 and in 1 to 3 values; m one row past a block
FEW = [(1, 257, 4111), (2, 1027, 1039), (3, 300, 5002), (4, 513, 1029), (5, 257, 4109), (6, 1501, 2503), (7, 1027, 4099), (8, 4097, 1021),
       (9, 4099, 4101), (10, 1025, 16391), (11, 9001, 1870), (12, 4097, 4098)]


@pytest.mark.parametrize("n,m,k", FEW)
def test_few_columns_off_the_16_byte_grid_next_to_infinities(gpu, n, m, k):
    """Operands at 1, 2 and 3 floats past a 16-byte boundary, every float around them a NaN; a row of A and a
    column of B that hold an infinity.  k + 1 roundings of 2^-24 against float64, and the fused forms
    (bias and ReLU, ReLU gate, weight update) bit for bit the separate steps on the same product."""
    say("few columns off the grid", n, m, k)
    ws_bytes = gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k)
    _few(gpu, m, n, k, ws_bytes)
    a, b = _rand(m * k, 60).reshape(k, m), _rand(n * k, 61).reshape(n, k)
    a[k - 1, 0], b[n - 1, k - 1] = np.inf, -np.inf
    ok = np.ix_(range(n - 1), range(1, m))  # rows and columns without an infinity
    want = (b[:-1].astype(np.float64) @ a[:, 1:].astype(np.float64))
    bound = (k + 1) * 2.0 ** -24 * (np.abs(b[:-1]).astype(np.float64) @ np.abs(a[:, 1:]).astype(np.float64))
    nan = np.full(4, np.nan, np.float32)
    ws, dc = gpu.empty(ws_bytes // 4 + 1), gpu.empty(m * n)

    def run(form, da, db, *extra, off, tail=()):
        gpu.call("mnv_sgemm_" + form, _at(da, off), _at(db, off), *extra, m, n, k, *tail, ws.p, ctypes.c_size_t(ws_bytes))
        return gpu.down(dc).reshape(n, m).copy()

    first = None
    for off in (1, 2, 3):
        wrap = lambda v: gpu.up(np.concatenate([nan[:off], np.ascontiguousarray(v).reshape(-1), nan]))  # noqa: E731
        da, db, dat, dbt = wrap(a), wrap(b), wrap(a.T), wrap(b.T)
        got = run("nn", da, db, dc.p, off=off)
        assert np.all(np.abs(got[ok] - want) <= bound)
        assert not np.isfinite(got[:, 0]).any() and not np.isfinite(got[n - 1]).any()
        first = got if first is None else first
        for other in (got, run("tn", dat, db, None, dc.p, off=off), run("nt", da, dbt, dc.p, off=off)):
            assert other.tobytes() == first.tobytes(), off
    bias, gate, w = _rand(m, 62), _rand(m * n, 63).reshape(n, m), _rand(m * n, 64).reshape(n, m)
    dbias, dgate, dw = gpu.up(bias), gpu.up(gate.reshape(-1)), gpu.up(w.reshape(-1))
    with np.errstate(invalid="ignore"):
        biased = first + bias
        assert run("nn_bias", da, db, dbias.p, dc.p, off=3, tail=(1,)).tobytes() == np.where(biased > 0, biased, np.float32(0)).tobytes()
        assert run("nn_relu_bwd", da, db, dgate.p, dc.p, off=3).tobytes() == np.where(gate > 0, first, np.float32(0)).tobytes()
        sgd = run("nt_sgd", da, dbt, dw.p, ctypes.c_float(0.125), dc.p, off=3)
        assert sgd.tobytes() == (w - np.float32(0.125) * first).tobytes()


@pytest.mark.parametrize("m,n,k", [(4096, 3, 5000), (2050, 2, 4100), (8200, 12, 2100)])
def test_few_columns_with_a_part_of_the_workspace(gpu, m, n, k):
    """Fewer k ranges, down to the least that the rule accepts: within k + 1 roundings of float64 each."""
    say("few columns, part of the workspace", m, n, k)
    full = _few(gpu, m, n, k, gpu.L.mnv_sgemm_nn_workspace_bytes(m, n, k))
    least = -(-128 // -(-m // 256))
    a, b = _rand(m * k, 65), _rand(n * k, 66)
    A, B = a.reshape(k, m).astype(np.float64), b.reshape(n, k).astype(np.float64)
    want, bound = B @ A, (k + 1) * 2.0 ** -24 * (np.abs(B) @ np.abs(A))
    da, db = gpu.up(a), gpu.up(b)
    assert least < full
    for have in sorted({least, least + 1, (least + full) // 2, full}):
        assert _few(gpu, m, n, k, 4 * m * n * have) <= have
        got = _bits(gpu, "nn", da, db, m, n, k, 4 * m * n * have).reshape(n, m)
        assert np.all(np.abs(got - want) <= bound), have


@pytest.mark.parametrize("m,n,k", [(32769, 2, 64), (33001, 1, 127), (40003, 3, 100), (66001, 4, 1000)])
def test_few_columns_in_one_range(gpu, m, n, k):
    """128 row blocks and more, or few k: one range, stored by the kernel itself, without a workspace."""
    say("few columns, one range", m, n, k)
    assert _few(gpu, m, n, k, 0) == 1
    a, b = _rand(m * k, 67), _rand(n * k, 68)
    A, B = a.reshape(k, m).astype(np.float64), b.reshape(n, k).astype(np.float64)
    bound = (k + 1) * 2.0 ** -24 * (np.abs(B) @ np.abs(A))
    da, db, dat = gpu.up(a), gpu.up(b), gpu.up(np.ascontiguousarray(a.reshape(k, m).T).reshape(-1))
    got = _bits(gpu, "nn", da, db, m, n, k, 0)
    assert np.all(np.abs(got.reshape(n, m) - B @ A) <= bound)
    assert _bits(gpu, "tn", dat, db, m, n, k, 0, None).tobytes() == got.tobytes()


def test_few_columns_of_an_operand_past_32_bit_offsets(gpu):
    """A of 2^29 elements and more: two k panels, the second accumulated into C, both by the few-column
    kernel.  Sampled rows against float64, k + 2 roundings."""
    m, n, k = 70001, 3, 8192
    assert m * k >= 1 << 29
    first = ((1 << 29) - 1 - m) // m + 1
    first -= first % 16
    assert 64 <= k - first and _few(gpu, m, n, first, 0) == 1 and _few(gpu, m, n, k - first, 0) == 1
    say("few columns, two panels", m, n, k)
    da, db, dc = gpu.empty(m * k), gpu.up(_rand(n * k, 69)), gpu.up(np.full(m * n, np.nan, np.float32))
    gpu.call("mnv_randn", da.p, ctypes.c_size_t(m * k), ctypes.c_uint64(70), ctypes.c_float(0), ctypes.c_float(1))
    gpu.call("mnv_sgemm_nn", da.p, db.p, dc.p, m, n, k, None, ctypes.c_size_t(0))
    rows = np.unique(np.concatenate([[0, 255, 256, m - 1], np.random.default_rng(71).integers(0, m, 60)]))
    A = gpu.down(da).reshape(k, m)[:, rows].astype(np.float64)
    B, got = gpu.down(db).reshape(n, k).astype(np.float64), gpu.down(dc).reshape(n, m)[:, rows]
    assert np.all(np.abs(got - B @ A) <= (k + 2) * 2.0 ** -24 * (np.abs(B) @ np.abs(A)))


@pytest.mark.parametrize("N,K,H,W", [(8192, 1, 1, 3), (4000, 3, 2, 1), (1500, 5, 1, 1)])
def test_bias_gradient_of_several_hundred_image_groups(gpu, N, K, H, W):
    """Up to 2048 group sums per channel, 32 to a lane: N H W roundings of 2^-24 against float64."""
    say("bias gradient", N, K, H, W)
    nbytes = gpu.L.mnv_conv_bwd_bias_workspace_bytes(N, K)
    assert nbytes // (4 * K) >= 375
    dy = _rand(N * K * H * W, 72)
    ws, db, ddy = gpu.empty(nbytes // 4 + 1), gpu.empty(K), gpu.up(dy)
    gpu.call("mnv_conv_bwd_bias", ddy.p, db.p, N, K, H, W, ws.p, ctypes.c_size_t(nbytes))
    t = dy.reshape(N, K, H * W).astype(np.float64)
    assert np.all(np.abs(gpu.down(db) - t.sum((0, 2))) <= N * H * W * 2.0 ** -24 * np.abs(t).sum((0, 2)))
