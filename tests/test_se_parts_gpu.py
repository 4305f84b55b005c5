"""Global average pool and channel scale at the edges of their pixel pairs: planes of one pixel, odd planes
(a pair in two planes), counts off a lane group and off a block, ragged channels, every lane count.

The mean is an fp32 sum of HW fp16 values, rounded once to fp16: within 2^-11 of the float64 mean plus
HW * 2^-24 of the mean magnitude. The scaled pixel is one correctly rounded fp16 product: exact.
"""
import numpy as np
import pytest

import vknn_amd as V
from tests.gpu_helpers import check, from_device_nc4, round_half, to_device_nc4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C,H,W", [(1, 1, 1, 1), (3, 5, 1, 1), (2, 9, 1, 2), (5, 7, 7, 7), (3, 20, 9, 8), (2, 12, 15, 17), (1, 6, 23, 23), (1, 8, 61, 67),
                                     (9, 672, 14, 14), (1, 4, 1, 1023), (1, 4, 32, 33)])
def test_pool_and_scale(gpu, N, C, H, W):
    lib, r = V.vkhip(), np.random.default_rng(N + C + H * W)
    x, g = round_half(r.standard_normal((N, C, H, W))), round_half(r.standard_normal((N, C, 1, 1)))
    dx, dg = to_device_nc4(x), to_device_nc4(g)
    da, dy = V.DeviceBuffer(V.nc4_elems(N, C, 1, 1) * 2), V.DeviceBuffer(V.nc4_elems(N, C, H, W) * 2)
    check(lib.vkhip_global_avg_pool(dx.ptr, da.ptr, N, C, H, W, None))
    check(lib.vkhip_channel_scale(dx.ptr, dg.ptr, dy.ptr, N, C, H * W, None))
    check(lib.vkhip_stream_sync(None))
    mean, got = x.astype(np.float64).mean((2, 3), keepdims=True), from_device_nc4(da, (N, C, 1, 1))
    bound = np.abs(mean) * 2.0 ** -11 + H * W * 2.0 ** -24 * np.abs(x).mean((2, 3), keepdims=True) + 2.0 ** -25
    assert (np.abs(got - mean) <= bound * 1.01).all()
    assert np.array_equal(from_device_nc4(dy, (N, C, H, W)), (x.astype(np.float16) * g.astype(np.float16)).astype(np.float32))
