"""Which kernel a product takes, those of at most 12 columns above all: host arithmetic on the extents
and the workspace alone, so checked without a GPU."""
import ctypes
import os
import random
import re
import struct
import subprocess
import time

import pytest

from minerva_amd import capi


def _query(m, n, k):
    return capi.lib().mnv_sgemm_nn_workspace_bytes(m, n, k)


def _plan(m, n, k, ws_bytes):
    v = [ctypes.c_int() for _ in range(3)]
    assert capi.lib().mnv_sgemm_nn_plan(m, n, k, ctypes.c_size_t(ws_bytes), *[ctypes.byref(x) for x in v]) == 0
    return tuple(x.value for x in v)


def _few(plan):
    return plan[0] == 256 and plan[2] == 4


@pytest.mark.parametrize("m", [256, 512, 513, 1000])
def test_ranges_do_not_depend_on_how_k_ends(m):
    """16 k per wavefront up to 65 ranges and 32 beyond, whatever k is modulo 64, with the workspace
    that the query asks for and with more."""
    for k in range(2048, 8321):
        ws = _query(m, 1, k)
        plan = _plan(m, 1, k, ws)
        assert _few(plan), k
        assert plan[1] == -(-k // (64 if k <= 4160 else 128)), k
        assert ws == plan[1] * m * 4 and _plan(m, 1, k, 1 << 40) == plan, k


@pytest.mark.parametrize("n,least", [(1, 1 << 19), (4, 1 << 19), (5, 7 << 19), (8, 7 << 19), (9, 1 << 24), (12, 1 << 24)])
def test_elements_of_the_left_operand_from_which_few_columns_have_their_kernel(n, least):
    for m in (1024, 2048):
        k = least // m
        assert _few(_plan(m, n, k, 1 << 40)) and not _few(_plan(m, n, k - 1, 1 << 40)), (m, k)
    assert not _few(_plan(4096, 13, 4096, 1 << 40)) and not _few(_plan(255, n, 1 << 20, 1 << 40))


def test_few_columns_over_few_or_many_k():
    assert _few(_plan(256, 8, 4096, 1 << 40)) and not _few(_plan(257, 8, 4095, 1 << 40))   # from 4096 k on, 2^20 elements
    assert not _few(_plan(40000, 8, 100, 1 << 40)) and _few(_plan(100000, 8, 64, 1 << 40))  # below 256 k, 6 x 2^20
    assert _few(_plan(40000, 4, 100, 1 << 40)) and not _few(_plan(40000, 4, 63, 1 << 40))


def test_few_columns_with_less_workspace():
    """A quarter of the 512 workgroups at least, or the tiles; the ranges never need more than there is."""
    m, n, k = 4096, 3, 5000
    full = _plan(m, n, k, _query(m, n, k))
    assert full == (256, 27, 4)
    for have in range(full[1] + 1):
        plan = _plan(m, n, k, have * m * n * 4)
        assert _few(plan) == (have >= 8), have
        assert not _few(plan) or plan[1] <= have
    for m, few in ((127 * 256, False), (127 * 256 + 1, True)):  # 128 row blocks: one range, no workspace
        assert _few(_plan(m, 1, 1000, 0)) == few and _plan(m, 1, 1000, 0)[1] == 1


def _extents(count):
    rng = random.Random(6)
    span = lambda low, high: int(low * (high / low) ** rng.random())
    return [(span(16, 4097), span(16, 4097), span(32, 4097)) for _ in range(count)]


NAMED = [  # planned with k ranges on the large tiles by one of the two instructions and without by the other
    (3530, 2630, 3872), (2921, 3395, 3933), (3372, 3896, 3982), (1500, 1500, 1501), (978, 1316, 3098), (9216, 256, 4096),
]


def test_the_queried_workspace_gives_the_plan_of_an_unlimited_one():
    """A caller that lends what the query asks for gets the plan that the query was made for, and the
    query asks for the partial results of that plan and no more."""
    for m, n, k in NAMED + _extents(6000):
        ws, most = _query(m, n, k), _plan(m, n, k, 1 << 40)
        assert _plan(m, n, k, ws) == most, (m, n, k, ws)
        slabs = -(-k // 16)
        if most[1] > 1 and not _few(most):  # the launch rounds the planned ranges to equal ones
            planned = ws // (4 * m * n)
            assert ws == planned * 4 * m * n and -(-slabs // -(-slabs // planned)) == most[1], (m, n, k, ws)


def test_a_plan_without_k_ranges_needs_no_workspace():
    for m, n, k in NAMED + _extents(6000):
        most = _plan(m, n, k, 1 << 40)
        if most[1] == 1:
            assert _plan(m, n, k, 0) == most, (m, n, k)


@pytest.mark.parametrize("m,n,k", [(307, 270, 143), (78, 382, 127), (2271, 261, 215), (3059, 183, 194), (329, 1452, 164)])
def test_short_products_stay_on_small_tiles_without_k_ranges(m, n, k):
    """A few slabs of k: the 64 x 64 tiles without ranges beat those with ranges, which the tiles in parts
    are weighed against first, and the tiles in parts."""
    for ws in (0, _query(m, n, k), 1 << 40):
        assert _plan(m, n, k, ws) == (64, 1, 1)


@pytest.mark.parametrize("m,n,k,rows", [
    (2871, 1047, 42, 64), (603, 3437, 70, 64), (1519, 1490, 36, 64),     # one workgroup per CU, nothing to overlap
    (3189, 2290, 49, 128), (2882, 2636, 172, 128), (2015, 1742, 107, 128),
])
def test_products_of_few_steps(m, n, k, rows):
    assert _plan(m, n, k, 0) == (rows, 1, 1)


@pytest.mark.parametrize("m,n,k,cut", [
    (3909, 1954, 260, False), (2716, 2401, 242, False),  # two tiles per CU, short k: all at once
    (2307, 3549, 528, True), (3530, 2630, 3872, True),   # a few tiles more than that
    (1298, 4851, 1634, False), (4096, 4096, 256, False), # many parts of long ranges; nothing left over
])
def test_products_in_parts_cut_their_tail_where_the_partial_tiles_cost_less(m, n, k, cut):
    assert _plan(m, n, k, 1 << 40) == (128, 1, 1)
    assert (_query(m, n, k) > 0) == cut


def test_weighing_many_launches_costs_little_host_time():
    """Every call plans its product.  One whose k ranges are weighed for both instructions takes at most
    twice and a half the time of one that has no choice; asking the runtime for the device in every
    estimate made it four times."""
    def fastest(m, n, k):
        best = float("inf")
        for _ in range(15):
            t = time.perf_counter()
            for _ in range(500):
                _query(m, n, k)
            best = min(best, time.perf_counter() - t)
        return best
    assert min(fastest(256, 256, 784) / fastest(10, 256, 256) for _ in range(3)) <= 2.5


@pytest.mark.parametrize("m,n,k,tile,wavefronts", [
    (16, 16, 32, 16, 8), (100, 7, 257, 16, 8), (257, 255, 783, 16, 8), (5, 300, 1023, 16, 8),
    (513, 511, 509, 16, 4), (784, 256, 255, 32, 8), (57, 3024, 2539, 32, 8),
    (1421, 284, 487, 32, 4), (1001, 250, 4099, 32, 4), (1770, 721, 430, 32, 4), (450, 1796, 288, 32, 4),
    (555, 2773, 156, 0, 0), (2411, 630, 201, 0, 0), (433, 3053, 133, 0, 0), (3921, 332, 232, 0, 0),  # more tiles than the CUs hold
    (509, 513, 1935, 0, 0), (597, 428, 1999, 0, 0), (600, 447, 1819, 0, 0), (2468, 102, 1441, 32, 4),  # a fifth 16 x 16 tile on a CU, long k
    (143, 1592, 2779, 32, 8), (1586, 158, 2770, 32, 8), (2138, 704, 499, 32, 4),  # weighed against k ranges in parts
    (509, 513, 1020, 16, 4), (365, 680, 1890, 16, 4),                     # shorter k; four of them
    (864, 1196, 89, 32, 4), (1752, 632, 126, 32, 4), (536, 2220, 117, 32, 4),  # more than four of them to a CU, short k
    (1, 1, 1, 0, 0), (15, 17, 3, 0, 0),                                   # one slab: the 64 x 64 tile
    (200, 1000, 4099, 0, 0), (500, 500, 3000, 0, 0), (4096, 3, 5000, 0, 0),  # k ranges: only with a workspace
    (4096, 4096, 4096, 0, 0),
])
def test_tiles_of_small_products(m, n, k, tile, wavefronts):
    """Which products run on 16 x 16 and 32 x 32 tiles, and how many wavefronts share their k.  They ask for no workspace."""
    assert not tile or _query(m, n, k) == 0
    for ws in (_query(m, n, k), 1 << 40):
        v = [ctypes.c_int() for _ in range(2)]
        assert capi.lib().mnv_sgemm_nn_small_plan(m, n, k, ctypes.c_size_t(ws), *[ctypes.byref(x) for x in v]) == 0
        assert (v[0].value, v[1].value) == (tile, wavefronts), ws
        assert not tile or _plan(m, n, k, ws) == (64, 1, 1)


def _device_code(path):
    """The code objects in a library's bundles."""
    data, magic, at = open(path, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        pos = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, pos - 8)[0]):
            offset, size, chars = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + chars]
            pos += 24 + chars
            if b"gfx950" in name:
                yield data[at + offset:at + offset + size]
        at += len(magic)


READELF = "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_products_in_parts_keep_their_loop_in_registers(tmp_path):
    """Two workgroups per CU leave 128 registers.  The few that do not fit are those of the result's
    addresses, outside the loop; with a fetch of four loads per vector, which a transposed A of a k off
    the multiples of 4 once took, there were 17 and the loop waited for them."""
    found = 0
    for i, image in enumerate(_device_code(capi.LIB_PATH)):
        if b"mnv_gemm_split_kernel" not in image or b"SgemmNN" not in image:
            continue
        co = tmp_path / ("%d.co" % i)
        co.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(co)], capture_output=True, text=True, check=True).stdout
        for kernel in notes.split(".agpr_count")[1:]:
            name = re.search(r"\.name: +(\S+)", kernel).group(1)
            if "mnv_gemm_split_kernel" in name and "SgemmNN" in name:
                found += 1
                assert int(re.search(r"\.vgpr_spill_count: +(\d+)", kernel).group(1)) <= 8, name
    assert found == 18  # three tiles, six forms of the operands
