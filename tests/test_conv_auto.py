"""What AUTO picks for dense convolutions, host only: every pick is a plan that its own explicit
request gives again (algorithm, tile, splits, sizes), needs no more workspace than the
allocation-free entry point holds, and shapes that none of the modelled kernels takes keep a gather
plan. The picks' results are compared with the oracle in test_conv_sweep_gpu.py."""
import ctypes
import random
import time

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


def band_copies(d, bn, slots, waves):
    """The 1 KB copies per channel slot of a halo tile's largest band, by walking every tile."""
    ohw, p, rows = d.OH * d.OW, d.N * d.OH * d.OW, 0
    for p0 in range(0, p, bn):
        p1 = min(p, p0 + bn) - 1
        rows = max(rows, (p1 // ohw - p0 // ohw) * (d.H + 2) + d.SH * (p1 % ohw // d.OW - p0 % ohw // d.OW) + 3)
    n = -(-rows * (((d.W + 3) & ~1) // 2) // 64)
    while slots * n % waves:
        n += 1
    return n


# tile -> (pixels, channel slots, waves of a workgroup); most copies its kernels are built for
HALO = {18: (256, 4, 4, 15), 26: (128, 4, 4, 8), 19: (256, 4, 4, 10), 50: (256, 4, 4, 15), 53: (128, 4, 4, 8)}


def test_halo_band_matches_the_walk_over_all_tiles():
    """A halo plan's band, found without walking the layer's tiles, over random layers: tiles that
    divide an image or not, one image or many, rows shorter and longer than a tile."""
    r, made = random.Random(5), 0
    for _ in range(1500):
        s, big = r.choice((1, 2)), r.random()
        h, w = (r.randint(1, 90 if big < 0.2 else 24) for _ in range(2))
        tile = r.choice(list(HALO))
        bn, slots, waves, most = HALO[tile]
        c = dict(N=r.randint(1, 40 if big < 0.2 else 140), Cin=32, H=h, W=w, Cout=32, OH=(h - 1) // s + 1, OW=(w - 1) // s + 1, KH=3, KW=3, SH=s, SW=s, PT=1, PL=1)
        rc, p = plan_of(V.CONV_GEMM, tile, 0, **c)
        want = band_copies(V.ConvDesc(**c), bn, slots, waves)
        assert (rc == 0) == (want <= most), (tile, c, want)
        if rc == 0:
            made += 1
            assert p.reserved == want, (tile, c, want)
    assert made > 300


def test_plans_of_large_maps_cost_no_walk():
    """Host time of a plan does not grow with the number of tiles (12800 here, which took 29 us per call
    to walk): best of several, against the same layer on one image."""
    best = {}
    for n in (1, 128):
        c = dict(N=n, Cin=16, H=80, W=80, Cout=16, OH=80, OW=80, KH=3, KW=3, SH=1, SW=1, PT=1, PL=1)
        best[n] = 1e9
        for _ in range(30):
            t = time.perf_counter()
            for _ in range(20):
                assert plan_of(V.CONV_GEMM, 33, 0, **c)[0] == 0
            best[n] = min(best[n], (time.perf_counter() - t) / 20)
    assert best[128] < best[1] + 10e-6, best


@pytest.mark.parametrize("c,h,w,k,s", [(64, 112, 112, 3, 1), (96, 112, 112, 3, 2), (32, 224, 224, 3, 1), (72, 56, 56, 5, 2), (960, 7, 7, 5, 1)])
def test_pool_parts_do_not_grow_with_the_row_bands(c, h, w, k, s):
    """The FC after a depthwise conv adds its parts up one by one: at most 4 bands of a plane (8 past
    128 rows), each with the 16-window groups that its row can lie in, also for one image, where the
    conv without pool sums splits into many more."""
    d = V.ConvDesc(N=1, Cin=c, H=h, W=w, Cout=c, OH=(h - 1) // s + 1, OW=(w - 1) // s + 1, KH=k, KW=k, SH=s, SW=s, PT=k // 2, PL=k // 2, DH=1, DW=1, group=c, act=1)
    p = V.ConvPlan()
    assert V.vkhip().vkhip_conv_plan_make(ctypes.byref(d), V.CONV_DEPTHWISE, -1, 0, ctypes.byref(p)) == 0
    windows = -(-d.OW // (4 if s == 1 else 2))
    parts = V.vkhip().vkhip_conv_pool_parts(ctypes.byref(d), ctypes.byref(p))
    assert 0 < parts <= (8 if d.OH > 128 else 4) * ((windows + 14) // 16 + 1)


@pytest.mark.parametrize("tile,kernel,c", [
    (-1, "dwconv_cols_kernel", dict(KH=3, KW=3)), (-1, "dwconv_cols_kernel", dict(KH=5, KW=5, PT=2, PL=2)),
    (7, "dwconv_lds_kernel", dict(KH=3, KW=3)), (907, "dwconv_lds_kernel", dict(KH=3, KW=3, H=7, W=7, OH=7, OW=7)),
    (-1, "dwconv_lds_kernel", dict(KH=5, KW=5, OH=16, OW=16)),  # left pad 1: the taps leave the window
    (-1, "dwconv_lds_kernel", dict(N=128, Cin=64, Cout=64, group=64, H=112, W=112, OH=56, OW=56, KH=3, KW=3, SH=2, SW=2)),  # 257 MB
    (-1, "dwconv_kernel", dict(KH=7, KW=7, PT=3, PL=3)), (7, "dwconv_kernel", dict(KH=7, KW=7, PT=3, PL=3)),
    (-1, "dwconv_kernel", dict(KH=3, KW=3, DH=2, DW=2, PT=2, PL=2)), (4, "dwconv_kernel", dict(H=6, W=300, OH=6, OW=300, KH=3, KW=3))])
def test_depthwise_plans_name_the_kernel_they_run(tile, kernel, c):
    """Reports and profiles take a layer's kernel from its plan, which knows what its tile comes to."""
    d = V.ConvDesc(**{**dict(N=2, Cin=8, H=18, W=18, Cout=8, OH=18, OW=18, SH=1, SW=1, PT=1, PL=1, DH=1, DW=1, group=8, act=1), **c})
    p = V.ConvPlan()
    assert V.vkhip().vkhip_conv_plan_make(ctypes.byref(d), V.CONV_DEPTHWISE, tile, 0, ctypes.byref(p)) == 0
    assert V.vkhip().vkhip_conv_plan_kernel(ctypes.byref(p)).decode() == kernel
