"""What AUTO picks for dense convolutions, host only: every pick is a plan that its own explicit
request gives again (algorithm, tile, splits, sizes), needs no more workspace than the
allocation-free entry point holds, and shapes that none of the modelled kernels takes keep a gather
plan. The picks' results are compared with the oracle in test_conv_sweep_gpu.py."""
import ctypes
import random

import pytest

import vknn_amd as V

SCRATCH = 64 << 20


def plan_of(algo, tile, ks, **kw):
    d = V.ConvDesc(**{**dict(SH=1, SW=1, PT=0, PL=0, DH=1, DW=1, group=1, act=1, act_lo=0.0, act_hi=0.0, has_res=0), **kw})
    p = V.ConvPlan()
    return V.vkhip().vkhip_conv_plan_make(ctypes.byref(d), algo, tile, ks, ctypes.byref(p)), p


@pytest.mark.parametrize("k,s", [(1, 1), (1, 2), (3, 1), (3, 2)])
def test_auto_picks_are_plans_of_their_own(k, s):
    r = random.Random(k * 10 + s)
    for n, cin, cout, h, w in [(1, 1, 1, 1, 1), (1, 16, 4, 7, 7), (128, 2048, 2048, 7, 7), (1, 2048, 2048, 2, 2), (3, 5, 33, 1, 640)] + [
            (r.randint(1, 64), r.randint(1, 700), r.randint(1, 700), r.randint(1, 60), r.randint(1, 60)) for _ in range(60)]:
        for res in (0, 1, 2):
            c = dict(N=n, Cin=cin, H=h, W=w, Cout=cout, OH=(h - 1) // s + 1, OW=(w - 1) // s + 1, KH=k, KW=k, SH=s, SW=s, PT=k // 2, PL=k // 2, has_res=res)
            rc, p = plan_of(V.CONV_AUTO, -1, 0, **c)
            assert rc == 0, c
            rc, q = plan_of(p.algo, p.tile, p.ksplit, **c)
            assert rc == 0 and bytes(p) == bytes(q), (c, p.algo, p.tile, p.ksplit)
            assert p.workspace_bytes <= SCRATCH, c


@pytest.mark.parametrize("kw", [dict(KH=5, KW=5, PT=2, PL=2, OH=20, OW=20), dict(KH=3, KW=3, PT=0, PL=0, OH=18, OW=18), dict(KH=1, KW=3, PT=0, PL=1, OH=20, OW=20),
                                dict(KH=3, KW=3, PT=2, PL=2, DH=2, DW=2, OH=20, OW=20), dict(KH=1, KW=1, SH=3, SW=3, OH=7, OW=7),
                                dict(KH=1, KW=1, PT=1, PL=1, OH=22, OW=22)])
def test_auto_keeps_gather_plans_elsewhere(kw):
    rc, p = plan_of(V.CONV_AUTO, -1, 0, N=2, Cin=40, H=20, W=20, Cout=72, **kw)
    assert rc == 0 and p.tile < 8


def test_auto_with_a_given_tile_or_split_keeps_it():
    c = dict(N=8, Cin=64, H=14, W=14, Cout=64, OH=14, OW=14, KH=1, KW=1)
    for t in (0, 3, 24):
        rc, p = plan_of(V.CONV_AUTO, t, 0, **c)
        assert rc == 0 and p.tile == t
