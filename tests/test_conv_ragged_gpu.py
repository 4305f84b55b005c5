"""The halo tiles for any channel count (50-53) against the CPU oracle: channel counts around a
16-channel K stage and around a 4-channel block, even and odd widths, both strides, split-K, several
images. The tiles whose geometry they have keep refusing such counts. Bar as for every conv
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


@pytest.mark.parametrize("tile", [50, 51, 52, 53])
@pytest.mark.parametrize("cin,w,s", [(17, 8, 1), (30, 9, 1), (5, 8, 2), (41, 11, 2)])
def test_halo_fills_the_last_stage_with_zeros(gpu, tile, cin, w, s):
    """The channel slots past the last block come after the image in memory, where the next one begins:
    what that one holds (infinities here, which a zero weight would turn into NaN) reaches no output of
    this one, to the bit."""
    r = np.random.default_rng(cin)
    x = round_half(r.standard_normal((2, cin, 8, w)))
    wt = round_half(r.standard_normal((40, cin, 3, 3)) * 0.2)
    b = (r.standard_normal(40) * 0.1).astype(np.float32)
    ref = gpu_conv(x, wt, b, (s, s), (1, 1, 1, 1), algo=V.CONV_GEMM, tile=tile)[0]
    x[1] = np.inf
    got = gpu_conv(x, wt, b, (s, s), (1, 1, 1, 1), algo=V.CONV_GEMM, tile=tile)[0]
    assert np.isfinite(ref).all() and not np.isfinite(got[1]).all()
    np.testing.assert_array_equal(got[0], ref[0])
