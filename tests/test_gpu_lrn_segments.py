"""GPU parity of normalisations of few positions, whose channels are cut into segments of a window's reach:
against the CPU oracle at channel counts around one and several segments and on small and re-cut planes."""
import ctypes

import numpy as np
import pytest

from gpu_util import Gpu, TOL, normwise, say
from oracle import mnv_oracle as ora

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return Gpu()


@pytest.mark.parametrize("size", [3, 5, 7])
@pytest.mark.parametrize("N,C,H,W", [(1, 1, 3, 3), (2, 3, 4, 5), (1, 4, 1, 1), (3, 5, 7, 7), (1, 6, 9, 2), (2, 13, 23, 23), (5, 29, 33, 16),
                                     (2, 64, 25, 31), (40, 24, 17, 19), (130, 37, 12, 28)])
def test_short_segments_match_the_oracle(gpu, size, N, C, H, W):
    say("lrn", size, N, C, H, W)
    rng = np.random.default_rng(size * C + H)
    x = np.maximum(rng.standard_normal(N * C * H * W) * 2, 0).astype(np.float32)
    dy = rng.standard_normal(N * C * H * W).astype(np.float32)
    a, b = ctypes.c_float(1e-2), ctypes.c_float(0.75)
    dx, ddy = gpu.up(x), gpu.up(dy)
    nan = np.full(x.size, np.nan, np.float32)
    scale, top, out = gpu.up(nan), gpu.up(nan), gpu.up(nan)
    gpu.call("mnv_lrn_fwd", dx.p, scale.p, top.p, size, a, b, N, C, H, W)
    want_top, want_scale = ora.lrn_fwd(x, size, 1e-2, 0.75, N, C, H, W)
    assert normwise(gpu.down(scale), want_scale) <= TOL and normwise(gpu.down(top), want_top) <= TOL
    gpu.call("mnv_lrn_bwd", dx.p, top.p, scale.p, ddy.p, out.p, size, a, b, N, C, H, W)
    assert normwise(gpu.down(out), ora.lrn_bwd(x, want_top, want_scale, dy, size, 1e-2, 0.75, N, C, H, W)) <= TOL
