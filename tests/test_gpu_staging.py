"""Host tensors through the pinned staging area, whose small copies stay in flight: the caller's buffer may change
as soon as a call returns, the area's halves are reused only when their copies have left, and small, large
and read-back copies share it."""
import numpy as np
import pytest

from gpu_util import say
from minerva_amd import hostapi

pytestmark = pytest.mark.gpu

HALF = (8 << 20) // 4  # floats of half a staging area


@pytest.mark.parametrize("dataflow", [False, True])
@pytest.mark.parametrize("sizes", [[1], [HALF], [HALF + 1, 5, HALF - 64], [700001] * 9, [HALF // 2, HALF // 2, 3, 2 * HALF + 7, 100, HALF]],
                         ids=["one value", "a half", "large, small", "several rounds", "mixed"])
def test_buffers_may_change_after_the_call(sizes, dataflow):
    say("staged uploads", sizes, dataflow)
    rt = hostapi.Runtime(0, sync_each_op=False, dataflow=dataflow)
    want, tensors = [], []
    for i, n in enumerate(sizes):
        a = (np.arange(n, dtype=np.int64) * 7919 + i).astype(np.float32)
        want.append(a.copy())
        tensors.append(rt.tensor(a, [n]))
        a[:] = np.nan
        if i % 4 == 2:  # a result between uploads
            np.testing.assert_array_equal(tensors[i - 1].read(), want[i - 1])
    for t, w in zip(tensors, want):
        np.testing.assert_array_equal(t.read(), w)
    for t in tensors:
        t.free()
    rt.close()
