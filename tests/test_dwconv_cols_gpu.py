"""The matrix-core depthwise kernel (dwconv_cols_kernel, plan tile 0) against the CPU oracle at the
edges of its column split: planes narrower than a window, one column left over, row bands, odd
widths, odd output rows at stride 2, pads above and beside K/2, ragged channels, every activation,
residual and pool sums; and infinities, which may only reach the outputs whose window holds them.

The kernel sums the same fp16 x fp16 products in fp32 as the oracle, in another order, and rounds
once to fp16: bar max|d|/max|ref| <= 2e-2 and cosine >= 0.9999, as for every conv kernel here.
"""
import ctypes

import numpy as np
import pytest

import vknn_amd as V
from tests.gpu_helpers import check, conv_desc, from_device_nc4, gpu_conv, round_half, to_device_nc4
from tests.oracle_lib import oracle_conv, parity

pytestmark = pytest.mark.gpu


def case(shape, k, s, pads, act, res):
    r = np.random.default_rng(shape[1] * 7 + shape[2] + k + s)
    x = round_half(r.standard_normal(shape))
    w = round_half(r.standard_normal((shape[1], 1, k, k)) * 0.3)
    b = (r.standard_normal(shape[1]) * 0.1).astype(np.float32)
    d, ys = conv_desc(shape, w.shape, (s, s), pads, group=shape[1], act=act, has_res=int(res))
    return x, w, b, d, ys, round_half(r.standard_normal(ys)) if res else None


@pytest.mark.parametrize("k,s", [(3, 1), (3, 2), (5, 1), (5, 2)])
@pytest.mark.parametrize("shape,act,res", [((1, 4, 1, 1), 0, False), ((1, 6, 2, 3), 1, True), ((3, 20, 7, 7), 4, False), ((2, 5, 15, 33), 5, True),
                                           ((17, 8, 9, 14), 2, False), ((1, 16, 112, 112), 3, False), ((128, 12, 14, 14), 4, True)])
def test_cols_against_oracle(gpu, shape, act, res, k, s):
    p = k // 2
    x, w, b, d, ys, rr = case(shape, k, s, (p,) * 4, act, res)
    lo, hi = (-0.5, 0.7) if act == 3 else (0.0, 0.0)
    got, plan, _ = gpu_conv(x, w, b, (s, s), (p,) * 4, group=shape[1], act=act, lo=lo, hi=hi, res=rr)
    assert plan.algo == V.CONV_DEPTHWISE and plan.tile == 0
    ref = oracle_conv(x, w, b, (s, s), (p,) * 4, group=shape[1], res=rr, act=act, lo=lo, hi=hi)
    rel, cos = parity(got, ref)
    assert rel <= 2e-2 and cos >= 0.9999, (rel, cos)


@pytest.mark.parametrize("shape,k,s,tile", [((2, 6, 9, 14), 3, 1, 0), ((1, 8, 6, 300), 5, 1, 0), ((2, 5, 15, 33), 5, 2, 0), ((2, 6, 9, 14), 3, 1, 4),
                                            ((2, 8, 28, 28), 5, 1, 207), ((9, 12, 7, 7), 3, 1, 907), ((1, 8, 6, 300), 7, 1, 0)])
@pytest.mark.parametrize("res", [False, True])
def test_hard_sigmoid(gpu, shape, k, s, tile, res):
    """clamp(lo v + hi, 0, 1) on every depthwise kernel (columns, also on rows wider than a strip;
    strips, pipelined and persistent ones; any shape): the oracle's plain sums, then the formula,
    which the kernel applies to its own fp32 sums before the rounding to fp16."""
    p = k // 2
    x, w, b, d, ys, rr = case(shape, k, s, (p,) * 4, 6, res)
    lo, hi = 0.2, 0.5
    got, plan, _ = gpu_conv(x, w, b, (s, s), (p,) * 4, group=shape[1], act=6, lo=lo, hi=hi, res=rr, algo=V.CONV_DEPTHWISE, tile=tile)
    ref = np.clip(lo * oracle_conv(x, w, b, (s, s), (p,) * 4, group=shape[1], res=rr) + hi, 0, 1)
    assert ref.min() == 0 and ref.max() == 1
    rel, cos = parity(got, ref)
    assert rel <= 2e-2 and cos >= 0.9999, (rel, cos)


# pads (top, left, bottom, right); 5x5 stride 1 with an odd left pad does not fit the window: strip kernel
@pytest.mark.parametrize("k,s,pads", [(3, 1, (0, 0, 0, 0)), (3, 2, (0, 0, 1, 1)), (3, 1, (2, 2, 2, 2)), (5, 2, (1, 1, 2, 2)), (5, 1, (1, 1, 1, 1)),
                                      (5, 1, (0, 0, 4, 4)), (5, 1, (4, 4, 0, 0)), (3, 2, (3, 3, 3, 3))])
def test_cols_pads(gpu, k, s, pads):
    x, w, b, d, ys, _ = case((2, 10, 13, 18), k, s, pads, 0, False)
    got, _, _ = gpu_conv(x, w, b, (s, s), pads, group=10)
    rel, cos = parity(got, oracle_conv(x, w, b, (s, s), pads, group=10))
    assert rel <= 2e-2 and cos >= 0.9999, (rel, cos)


@pytest.mark.parametrize("k,s,p", [(3, 1, 7), (3, 1, 8), (5, 1, 10), (3, 2, 10), (5, 2, 12)])
def test_cols_bands_in_the_top_padding(gpu, k, s, p):
    """A plane split into 4-row bands whose first band lies wholly above the image: its outputs see
    padding only, in every plane (a row of the plane before is no row of this one)."""
    x, w, b, d, ys, _ = case((1, 16, 20, 20), k, s, (p,) * 4, 0, False)
    got, plan, _ = gpu_conv(x, w, b, (s, s), (p,) * 4, group=16)
    assert plan.tile == 0
    ref = oracle_conv(x, w, b, (s, s), (p,) * 4, group=16)
    assert np.array_equal(got[:, :, :1], np.broadcast_to(b.astype(np.float16).astype(np.float32)[None, :, None, None], got[:, :, :1].shape))
    rel, cos = parity(got, ref)
    assert rel <= 2e-2 and cos >= 0.9999, (rel, cos)


@pytest.mark.parametrize("k,s", [(3, 1), (3, 2), (5, 1), (5, 2)])
def test_cols_infinities_stay_in_their_window(gpu, k, s):
    p = k // 2
    x, w, b, d, ys, _ = case((2, 8, 17, 22), k, s, (p,) * 4, 0, False)
    x[0, 2, 5, 7], x[1, 6, 0, 21], x[1, 1, 16, 0] = np.inf, -np.inf, np.nan
    got, _, _ = gpu_conv(x, w, b, (s, s), (p,) * 4, group=8)
    ref = oracle_conv(x, w, b, (s, s), (p,) * 4, group=8)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    inf, fin = np.isinf(ref), np.isfinite(ref)
    assert inf.any() and np.array_equal(got[inf], ref[inf])
    rel, cos = parity(got[fin], ref[fin])
    assert rel <= 2e-2 and cos >= 0.9999, (rel, cos)


@pytest.mark.parametrize("k,s", [(3, 1), (3, 2), (5, 1), (5, 2)])
@pytest.mark.parametrize("pooled", [False, True])
def test_cols_residual_in_place_beside_infinities(gpu, k, s, pooled):
    """A residual that is the output's own memory gives the bits of one that is not, also in windows
    whose outputs are computed again tap by tap."""
    lib, p = V.vkhip(), k // 2
    x, w, b, d, ys, rr = case((2, 8, 17, 22), k, s, (p,) * 4, 0, True)
    x[0, 2, 5, 7], x[1, 6, 0, 21], x[1, 1, 16, 0] = np.inf, -np.inf, np.nan
    ref, plan, _ = gpu_conv(x, w, b, (s, s), (p,) * 4, group=8, res=rr)
    assert not np.isfinite(ref).all()
    blob = np.zeros(plan.weight_bytes, np.uint8)
    check(lib.vkhip_conv_pack_weights(ctypes.byref(d), ctypes.byref(plan), w.ctypes.data, b.ctypes.data, blob.ctypes.data))
    dx, db, dy = to_device_nc4(x), V.DeviceBuffer.from_array(blob), to_device_nc4(rr)
    if pooled:
        dp = V.DeviceBuffer(2 * 2 * lib.vkhip_conv_pool_parts(ctypes.byref(d), ctypes.byref(plan)) * 16)
        check(lib.vkhip_conv_forward_pooled(ctypes.byref(d), ctypes.byref(plan), dx.ptr, db.ptr, dy.ptr, dy.ptr, dp.ptr, None))
    else:
        check(lib.vkhip_conv_forward(ctypes.byref(d), ctypes.byref(plan), dx.ptr, db.ptr, dy.ptr, dy.ptr, None, None))
    check(lib.vkhip_stream_sync(None))
    np.testing.assert_array_equal(from_device_nc4(dy, ys), ref)


@pytest.mark.parametrize("shape,k,s", [((3, 22, 14, 14), 3, 1), ((4, 960, 7, 7), 5, 1), ((2, 12, 29, 31), 5, 2), ((1, 8, 40, 9), 3, 2),
                                       ((2, 8, 20, 112), 3, 1), ((1, 5, 140, 77), 3, 1), ((1, 4, 37, 300), 5, 2)])
def test_cols_pool_sums(gpu, shape, k, s):
    """The parts of a plane add up to the sum of the stored fp16 outputs: fp32 sums of at most
    H * W values each, so their relative error is below H * W * 2^-24 < 1e-4."""
    lib, p = V.vkhip(), k // 2
    x, w, b, d, ys, _ = case(shape, k, s, (p,) * 4, 4, False)
    ref, plan, dref = gpu_conv(x, w, b, (s, s), (p,) * 4, group=shape[1], act=4)
    blob = np.zeros(plan.weight_bytes, np.uint8)
    check(lib.vkhip_conv_pack_weights(ctypes.byref(d), ctypes.byref(plan), w.ctypes.data, b.ctypes.data, blob.ctypes.data))
    parts = lib.vkhip_conv_pool_parts(ctypes.byref(d), ctypes.byref(plan))
    cb = (shape[1] + 3) // 4
    dx, db = to_device_nc4(x), V.DeviceBuffer.from_array(blob)
    dy, dp = V.DeviceBuffer(V.nc4_elems(*ys) * 2), V.DeviceBuffer(shape[0] * cb * parts * 16)
    check(lib.vkhip_conv_forward_pooled(ctypes.byref(d), ctypes.byref(plan), dx.ptr, db.ptr, None, dy.ptr, dp.ptr, None))
    check(lib.vkhip_stream_sync(None))
    assert np.array_equal(from_device_nc4(dy, ys), ref)
    got = dp.download(np.float32, shape[0] * cb * parts * 4).reshape(shape[0], cb, parts, 4).astype(np.float64).sum(2)
    want = ref.astype(np.float64).sum((2, 3))
    np.testing.assert_allclose(got.reshape(shape[0], -1)[:, :shape[1]], want, atol=1e-4 * np.abs(ref).sum((2, 3)).max())
