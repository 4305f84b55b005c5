"""The matrix-core depthwise + projection kernel (dwpw_cols_kernel) against the CPU oracle at the edges
of its split: planes narrower than a window, one column left over, row bands, pads beside K/2, channel
counts off the chunk of 32 and the block of 4, one and two output fragments, every depthwise
activation; and infinities, which may only reach the outputs whose window holds them.

The kernel and the oracle round the depthwise result to fp16 and sum fp16 x fp16 products in fp32, in
another order: bar max|d|/max|ref| <= 2e-2 and cosine >= 0.9999, as for every conv kernel here.
"""
import ctypes

import numpy as np
import pytest

import vknn_amd as V
from tests.gpu_helpers import check, conv_desc, from_device_nc4, round_half, to_device_nc4
from tests.oracle_lib import oracle_dwpw, parity

pytestmark = pytest.mark.gpu


def run(shape, k, s, pads, cout, dw_act, act, res, spoil=None):
    lib, E = V.vkhip(), shape[1]
    r = np.random.default_rng(E + cout + shape[2] + k + s)
    x = round_half(r.standard_normal(shape))
    if spoil:
        spoil(x)
    w1 = round_half(r.standard_normal((E, 1, k, k)) * 0.3)
    b1, b2 = (r.standard_normal(E) * 0.1).astype(np.float32), (r.standard_normal(cout) * 0.1).astype(np.float32)
    w2 = round_half(r.standard_normal((cout, E)) * E ** -0.5)
    dwd, ys = conv_desc(shape, w1.shape, (s, s), pads, group=E, act=dw_act)
    ys = (shape[0], cout) + tuple(ys[2:])
    rr = round_half(r.standard_normal(ys)) if res else None
    lo, hi = (-0.5, 0.7) if act == 3 else (0.0, 0.0)
    d = V.DwPwDesc(dw=dwd, Cout=cout, act=act, act_lo=lo, act_hi=hi, has_res=int(res))
    blob = np.zeros(lib.vkhip_dwpw_weight_bytes(ctypes.byref(d)), np.uint8)
    check(lib.vkhip_dwpw_pack_weights(ctypes.byref(d), w1.ctypes.data, b1.ctypes.data, w2.ctypes.data, b2.ctypes.data, blob.ctypes.data))
    dx, db, dr = to_device_nc4(x), V.DeviceBuffer.from_array(blob), to_device_nc4(rr) if res else None
    dy = V.DeviceBuffer(V.nc4_elems(*ys) * 2)
    check(lib.vkhip_dwpw_forward(ctypes.byref(d), dx.ptr, db.ptr, dr.ptr if res else None, dy.ptr, None))
    check(lib.vkhip_stream_sync(None))
    return from_device_nc4(dy, ys), oracle_dwpw(x, w1, b1, w2, b2, (s, s), pads, dw_act=dw_act, res=rr, act=act, lo=lo, hi=hi)


@pytest.mark.parametrize("k,s", [(3, 1), (3, 2), (5, 1), (5, 2)])
@pytest.mark.parametrize("shape,cout,dw_act,act,res", [((1, 4, 1, 2), 1, 0, 0, False), ((3, 33, 5, 8), 33, 1, 1, True), ((2, 62, 17, 34), 64, 2, 3, True),
                                                       ((17, 96, 9, 14), 32, 2, 0, False), ((40, 8, 14, 14), 7, 0, 4, True), ((2, 1024, 7, 8), 40, 2, 0, False)])
def test_cols_against_oracle(gpu, shape, cout, dw_act, act, res, k, s):
    got, ref = run(shape, k, s, (k // 2,) * 4, cout, dw_act, act, res)
    rel, cos = parity(got, ref)
    assert rel <= 2e-2 and cos >= 0.9999, (rel, cos)


# pads (top, left, bottom, right); 5x5 stride 1 with an odd left pad does not fit the window: ring kernel
@pytest.mark.parametrize("k,s,pads", [(3, 1, (0, 0, 0, 0)), (3, 2, (0, 0, 1, 1)), (3, 1, (2, 2, 2, 2)), (5, 2, (1, 1, 2, 2)), (5, 1, (1, 1, 1, 1)),
                                      (5, 1, (0, 0, 4, 4)), (5, 1, (4, 4, 0, 0)), (3, 2, (3, 3, 3, 3))])
def test_cols_pads(gpu, k, s, pads):
    got, ref = run((2, 42, 13, 18), k, s, pads, 20, 2, 0, False)
    rel, cos = parity(got, ref)
    assert rel <= 2e-2 and cos >= 0.9999, (rel, cos)


# one or two projection fragments x strips of 4, 2 and 1 rows per thread; ragged channels, one chunk
# and many, a strip of several row groups and one cut off by the last row
@pytest.mark.parametrize("shape,pads,cout,dw_act,act,res", [((2, 72, 12, 16), (2, 1, 2, 3), 40, 2, 0, True), ((1, 144, 14, 14), (2, 3, 2, 1), 24, 1, 3, False),
                                                            ((3, 20, 4, 64), (1, 1, 1, 3), 24, 0, 1, False), ((3, 20, 4, 64), (1, 1, 1, 3), 33, 2, 0, True),
                                                            ((2, 33, 3, 38), (1, 3, 1, 1), 7, 2, 0, False), ((2, 33, 3, 38), (1, 3, 1, 1), 64, 2, 4, False),
                                                            ((1, 1024, 6, 8), (2, 1, 2, 3), 64, 2, 0, False), ((2, 4, 9, 100), (2, 1, 2, 3), 16, 2, 0, True)])
def test_ring_kernel_on_odd_left_pads(gpu, shape, pads, cout, dw_act, act, res):
    """5x5 stride 1 with an odd left pad, the one case that stays on the ring kernel."""
    got, ref = run(shape, 5, 1, pads, cout, dw_act, act, res)
    rel, cos = parity(got, ref)
    assert rel <= 2e-2 and cos >= 0.9999, (rel, cos)


@pytest.mark.parametrize("k,s", [(3, 1), (3, 2), (5, 1), (5, 2)])
@pytest.mark.parametrize("dw_act", [0, 2])
def test_cols_infinities_stay_in_their_window(gpu, k, s, dw_act):
    def spoil(x):
        x[0, 2, 5, 7], x[1, 30, 0, 21], x[1, 34, 16, 0] = np.inf, -np.inf, np.inf

    got, ref = run((2, 38, 17, 22), k, s, (k // 2,) * 4, 12, dw_act, 0, False, spoil)
    fin = np.isfinite(ref)
    assert np.array_equal(np.isfinite(got), fin) and (dw_act or not fin.all())
    rel, cos = parity(got[fin], ref[fin])
    assert rel <= 2e-2 and cos >= 0.9999, (rel, cos)
