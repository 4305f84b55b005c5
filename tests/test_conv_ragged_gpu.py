"""The halo tiles for any channel count (50-53) against the CPU oracle: channel counts around a
16-channel K stage and around a 4-channel block, even and odd widths, both strides, split-K, several
images. The tiles they share their kernels with keep refusing such counts. Bar as for every conv
kernel: max|d|/max|ref| <= 2e-2, cosine >= 0.9999."""
import ctypes

import numpy as np
import pytest

import vknn_amd as V
from tests.gpu_helpers import conv_desc, gpu_conv, round_half
from tests.oracle_lib import oracle_conv, parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [50, 51, 52, 53])
@pytest.mark.parametrize("cin,cout,h,w,s,ks", [(1, 3, 7, 7, 1, 0), (15, 33, 9, 12, 1, 0), (16, 16, 8, 8, 2, 0), (17, 70, 13, 11, 2, 0), (30, 40, 5, 30, 1, 2),
                                               (67, 20, 12, 14, 1, 3), (130, 65, 7, 9, 2, 0)])
def test_halo_any_channel_count(gpu, tile, cin, cout, h, w, s, ks):
    r = np.random.default_rng(cin * 3 + cout + s)
    x = round_half(r.standard_normal((3, cin, h, w)))
    wt = round_half(r.standard_normal((cout, cin, 3, 3)) * np.sqrt(2.0 / (9 * cin)))
    b = (r.standard_normal(cout) * 0.1).astype(np.float32)
    algo = V.CONV_SPLITK if ks else V.CONV_GEMM
    got, plan, _ = gpu_conv(x, wt, b, (s, s), (1, 1, 1, 1), act=1, algo=algo, tile=tile, ksplit=ks)
    assert plan.tile == tile
    rel, cos = parity(got, oracle_conv(x, wt, b, (s, s), (1, 1, 1, 1), act=1))
    assert rel <= 2e-2 and cos >= 0.9999, (rel, cos)
    if cin % 16:
        d, _ = conv_desc(x.shape, wt.shape, (s, s), (1, 1, 1, 1))
        base = {50: 18, 51: 26, 52: 32, 53: 33}[tile]
        assert V.vkhip().vkhip_conv_plan_make(ctypes.byref(d), V.CONV_GEMM, base, 0, ctypes.byref(V.ConvPlan())) != 0
