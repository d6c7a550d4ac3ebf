"""Environment maps of more than 2^24 columns or rows, whose texel index floor(k / n * n) in FP32 can come to
n: the projection reads no texel past the map. The map is all ones and the memory behind it, in the same
allocation, 1e30, which one such read would bring into the sum."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide", [True, False])
def test_no_read_past_the_map(ctx, wide):
    from banshee_amd import hip
    n, guard = (1 << 24) + 4, 64
    k = np.float32(n - 1)
    assert np.floor(k / np.float32(n) * np.float32(n)) == n   # the last column's index in FP32
    buf = np.ones((n + guard, 3), np.float32)
    buf[n:] = 1e30
    dev, out = ctx.to_device(buf), ctx.alloc((1, 3), np.float32)
    w, h = (n, 1) if wide else (1, n)
    r = hip.lib().bsh_sh_project_env(ctx.h, dev.ptr, ctypes.c_int(w), ctypes.c_int(h), ctypes.c_int(0), out.ptr,
                                     ctypes.c_void_p(None))
    assert r == 0, hip.lib().bsh_last_error()
    ctx.sync()
    # Y_00 times the cells' solid angles: one row has sin(theta) = 1 and steps pi and 2 pi / n; one column
    # sums sin(theta) pi / n over theta, 2, times 2 pi. Additions in a row: 32 + 3 in a block, 1025 + 6 over the
    # 65,537 blocks, so at most 1066 2^-24 = 6.4e-5 relative; the angles' own rounding averages out
    want = 0.28209479177387814 * (np.pi * 2 * np.pi if wide else 2 * 2 * np.pi)
    np.testing.assert_allclose(out.numpy(), want, rtol=1e-4)
