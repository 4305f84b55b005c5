// Fused depthwise 3x3 / 5x5 + 1x1 projection with both stages on the matrix cores.
#include "conv_kernels.h"
#include "dwpw.h"

namespace vkhip {

    // The depthwise stage is dwconv_cols_kernel's (dwconv_cols.hip): an 8-pixel x 4-channel row window
    // times the taps as a banded matrix gives 16 outputs of 16 windows per v_mfma_f32_16x16x32_f16, its
    // operands straight from global memory. A workgroup of 8 waves owns 16 windows (image, band of BR = 4
    // output rows, window in the row) over all channels and walks them in chunks of 32: wave w computes
    // channel block w of the chunk, applies the depthwise activation and writes fp16 vectors into an LDS
    // chunk [channel block pair][pixel], which is the B operand of the projection's
    // v_mfma_f32_32x32x16_f16; after one barrier each wave adds the chunk's 32 channels into the
    // projection of its 32 pixels (two LDS chunks, so that the next one is written meanwhile). The next
    // chunk's rows and taps are loaded before the activation and the projection.
    //
    // Bound by the chunk's instructions and its wait for the rows (about 1 us per chunk and workgroup,
    // two workgroups per CU), so every load of a chunk is one instruction on offsets computed once, the
    // activation is two packed fp16 operations, and nothing in the chunk waits for loads of the next
    // one; loading two chunks ahead measured no faster (registers). The ring kernel does the depthwise
    // sums on the vector units from LDS. Ring -> this kernel, us, 3x3 unless noted, ReLU6:
    //   N 32 144 -> 24 at 56x56  28.9 -> 14.8     N 128 144 -> 24 at 56x56     68.0 -> 50.4
    //   N 1  144 -> 24 at 56x56  22.7 -> 8.7      N 32 96 -> 24 at 112x112 s2  25.9 -> 22.1
    //   N 32 384 -> 64 at 14x14  50.5 -> 18.1     N 32 240 -> 40 at 28x28 5x5  46.7 -> 15.9
    //   N 2  1024 -> 64 at 8x8   44.3 -> 37.8     N 32 72 -> 40 at 56x56 5x5 s2 18.7 -> 8.7
    // and 1.1 - 3.3x on 24 more shapes, none slower.
    //
    // Windows with an infinity or NaN are recomputed tap by tap, as in dwconv_cols_kernel.
    template <int K, int S, int MF>
    __global__ __launch_bounds__(512, K == 3 && S == 1 && MF == 1 ? 4 : 2) void dwpw_cols_kernel(DwPwArgs a, DwPwCols t) {
        constexpr int BR = 4, F = S == 1 ? K : K + 2, DX = S == 1 ? 4 : 2;
        constexpr int RIN = BR * S + K - S;       // input rows of a band
        constexpr int PX = 16 * DX * BR;          // pixels of a workgroup
        constexpr int NA = S == 1 ? BR : BR / 2;  // depthwise accumulators: output rows, or row pairs
        constexpr int MW = S == 1 ? MF : 1;       // projection fragments per wave (stride 2: half as many pixels)
        constexpr unsigned kInvalid = 0x80000000u;
        __shared__ __attribute__((aligned(16))) u32x2 bch[2][4][PX][2]; // pixel slots swizzled by swz()
        __shared__ u32x4 ach[2][4][MF * 32];
        auto swz = [](int px) { return px ^ ((px >> 4) & 3); };
        using std::integral_constant;
        const int lane = threadIdx.x & 63, n16 = lane & 15, g = lane >> 4;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int grp  = xcd_remap(blockIdx.x, gridDim.x);
        const int H = a.H, W = a.W, OH = a.OH, OW = a.OW, HW8 = H * W * 8;

        // this lane's window: image, band, position; and its pixel pair of every input row
        const int  q    = grp * 16 + n16;
        const bool live = q < t.Q;
        const int  xbq  = (live ? q : 0) % t.XB, nbq = (live ? q : 0) / t.XB;
        const int  img  = nbq / t.NB, y0 = (nbq % t.NB) * BR, iy0 = y0 * S - a.PT;
        const int  x0   = xbq * 4 - (t.off + a.PL) + 2 * g;
        const bool ok0  = live && x0 >= 0 && x0 < W; // x0 and W are even
        // Byte offset in channel block 0 of each input row, past every range where the row or the window
        // is outside the image (reads zero); and of the two taps (8 bytes each, after one tap of slack in
        // front) of A row (d, c) in each of the F tap rows, with the mask that keeps channel c of the taps
        // that exist. Computed once, so that a chunk costs one instruction per load.
        unsigned roff[RIN], woff[F];
#pragma unroll
        for (int r = 0; r < RIN; ++r)
            roff[r] = ok0 & ((unsigned) (iy0 + r) < (unsigned) H) ? (unsigned) ((img * a.Eb * H + iy0 + r) * W + x0) * 8u : kInvalid;
        const int c4 = n16 & 3, d4 = n16 >> 2, dy4 = S == 1 ? 0 : d4 >> 1, dx4 = S == 1 ? d4 : d4 & 1;
        const int kx0 = 2 * g - t.off - dx4 * S; // first of the two taps
#pragma unroll
        for (int f = 0; f < F; ++f) {
            const int ky = f - 2 * dy4;
            woff[f]      = ((unsigned) ky < (unsigned) K) & (kx0 >= -1) & (kx0 < K) ? (unsigned) (ky * K + kx0 + 1) * 8u : kInvalid;
        }
        const unsigned keep = 0xFFFFu << (16 * (c4 & 1));
        const bool     t0   = (unsigned) kx0 < (unsigned) K, t1 = (unsigned) (kx0 + 1) < (unsigned) K;
        const u32x4    wmask = u32x4_make(t0 && c4 < 2 ? keep : 0u, t0 && c4 >= 2 ? keep : 0u, t1 && c4 < 2 ? keep : 0u, t1 && c4 >= 2 ? keep : 0u);
        const int      xbytes = a.N * a.Eb * HW8;
        const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc((void *) a.pw_w, (short) 0, a.m_frags * 32 * a.Kp * 2, 0x00020000);
        u32x4   buf[RIN], wt[F];
        float4v b0;
        auto    fetch = [&](int ch) __attribute__((always_inline)) {
            const int     cb = ch * 8 + wave;
            const bool    in = cb < a.Eb; // wave-uniform; past the last block everything reads zero
            const __amdgpu_buffer_rsrc_t xrs =
                __builtin_amdgcn_make_buffer_rsrc((char *) a.x + (in ? (long long) cb * HW8 : 0), (short) 0, in ? xbytes - cb * HW8 : 0, 0x00020000);
            const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
                (char *) a.dw_h + (in ? cb * K * K * 8 : 0) - 8, (short) 0, in ? K * K * 8 + 16 : 0, 0x00020000); // the blob goes on at both ends
            const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc((char *) a.dw_b + (in ? cb * 16 : 0), (short) 0, in ? 16 : 0, 0x00020000);
#pragma unroll
            for (int r = 0; r < RIN; ++r) buf[r] = __builtin_amdgcn_raw_buffer_load_b128(xrs, roff[r], 0, 0);
#pragma unroll
            for (int f = 0; f < F; ++f) wt[f] = __builtin_amdgcn_raw_buffer_load_b128(wrs, woff[f], 0, 0);
            b0 = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(brs, 0, 0, 0));
        };

        // this wave's share of the projection: pixel fragment and first output-channel fragment
        const int fr = S == 1 ? wave : wave & 3, m0 = S == 1 ? 0 : wave >> 2;
        float16v  pacc[MW];
#pragma unroll
        for (int m = 0; m < MW; ++m)
#pragma unroll
            for (int r = 0; r < 16; ++r) pacc[m][r] = 0.f;

        // projection weights of a chunk: lane row l % 32, halves ch * 32 + ks * 16 + (l / 32) * 8 ..
        // The chunk's 64 bytes of every projection row are staged by all threads, MF * 4 bytes each. Issued
        // before the rows of the same chunk, so that the wait for those covers them.
        constexpr int LPR = 16 / MF; // threads per row
        typedef std::conditional_t<MF == 1, unsigned, u32x2> stage_t;
        const int      arow = threadIdx.x / LPR, apc = threadIdx.x % LPR;
        const unsigned poff = (unsigned) (arow * a.Kp * 2 + apc * (MF * 4));
        char          *adst = (char *) &ach[0][apc * MF / 4][arow] + apc * MF % 4 * 4;
        stage_t        pw;
        auto           fetch_pw = [&](int ch) __attribute__((always_inline)) {
            if constexpr (MF == 1) pw = __builtin_amdgcn_raw_buffer_load_b32(prs, poff, ch * 64, 0);
            else pw = __builtin_amdgcn_raw_buffer_load_b64(prs, poff, ch * 64, 0);
        };

        const half_t dl = (half_t) (a.dw_act == VKHIP_ACT_NONE ? -__builtin_inff() : 0.f), dh = (half_t) (a.dw_act == VKHIP_ACT_RELU6 ? 6.f : __builtin_inff());
        const half4  dlo = {dl, dl, dl, dl}, dhi = {dh, dh, dh, dh};
        auto         chunk = [&](int ch, auto more) __attribute__((always_inline)) {
            half8 fa[F];
#pragma unroll
            for (int f = 0; f < F; ++f) fa[f] = __builtin_bit_cast(half8, wt[f] & wmask);
            float4v       acc[NA];
            // input row r is tap row r - y of output row y (stride 2: tap row r - 4 i of the row pair i)
            static_for<0, RIN>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                const half8   fb = __builtin_bit_cast(half8, buf[r]);
                static_for<0, NA>([&](auto ic) {
                    constexpr int i = decltype(ic)::value, f = S == 1 ? r - i : r - 4 * i;
                    if constexpr (f == 0) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[0], fb, b0, 0, 0, 0);
                    else if constexpr (f > 0 && f < F) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[f], fb, acc[i], 0, 0, 0);
                });
            });
            *reinterpret_cast<stage_t *>(adst + (ch & 1) * (int) sizeof(ach[0])) = pw;
            if constexpr (decltype(more)::value) {
                fetch_pw(ch + 1);
                fetch(ch + 1);
            }
            float nf = 0.f; // NaN once a sum of this lane was not finite
#pragma unroll
            for (int i = 0; i < NA; ++i) nf = __builtin_fmaf((acc[i].x + acc[i].y) + (acc[i].z + acc[i].w), 0.f, nf);
            // fp16 outputs into the chunk: pixel 64 y + 4 n + g (stride 2: 64 i + 32 dy + 2 n + dx). Zero, six
            // and the infinities are fp16 values, so finite sums are clamped after the conversion, in pairs.
            const int px  = S == 1 ? 4 * n16 + g : (g >> 1) * 32 + 2 * n16 + (g & 1);
            u32x2    *dst = &bch[ch & 1][wave >> 1][swz(px)][wave & 1];
            if (!__any(nf != nf)) {
#pragma unroll
                for (int i = 0; i < NA; ++i)
                    dst[i * 64 * 2] = __builtin_bit_cast(u32x2, __builtin_elementwise_min(__builtin_elementwise_max(f4_to_h4(acc[i]), dlo), dhi));
            } else {
                const int cb = ch * 8 + wave, ox = xbq * DX + (S == 1 ? g : g & 1);
#pragma unroll
                for (int i = 0; i < NA; ++i) {
                    float4v v = acc[i];
                    if (nf != nf) {
                        const int oy = y0 + (S == 1 ? i : 2 * i + (g >> 1));
                        v            = *reinterpret_cast<const float4v *>(a.dw_b + cb * 4);
#pragma unroll 1
                        for (int k = 0; k < K * K; ++k) {
                            const int iy = oy * S - a.PT + k / K, ix = ox * S - a.PL + k % K;
                            if ((unsigned) iy >= (unsigned) H || (unsigned) ix >= (unsigned) W) continue;
                            const half4 xv = u2_as_h4(a.x[((long long) (img * a.Eb + cb) * H + iy) * W + ix]);
                            const half4 wv = *reinterpret_cast<const half4 *>(a.dw_h + ((long long) cb * K * K + k) * 4);
                            v.x = __builtin_fmaf((float) xv.x, (float) wv.x, v.x);
                            v.y = __builtin_fmaf((float) xv.y, (float) wv.y, v.y);
                            v.z = __builtin_fmaf((float) xv.z, (float) wv.z, v.z);
                            v.w = __builtin_fmaf((float) xv.w, (float) wv.w, v.w);
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = apply_act(v[e], a.dw_act, 0.f, 6.f);
                    dst[i * 64 * 2] = __builtin_bit_cast(u32x2, f4_to_h4(v));
                }
            }
            // the chunk is in LDS; the next rows stay in flight
            __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (m0 < MF) {
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    const half8 bf = *reinterpret_cast<const half8 *>(&bch[ch & 1][ks * 2 + (lane >> 5)][swz(fr * 32 + (lane & 31))][0]);
#pragma unroll
                    for (int m = 0; m < MW; ++m) {
                        const half8 af = __builtin_bit_cast(half8, ach[ch & 1][ks * 2 + (lane >> 5)][(m0 + m) * 32 + (lane & 31)]);
                        pacc[m]        = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, bf, pacc[m], 0, 0, 0);
                    }
                }
            }
        };
        // the last chunk loads nothing ahead: a branch around the loads would make the compiler wait for
        // them at the next use of any earlier load
        fetch_pw(0);
        fetch(0);
        int ch = 0;
        for (; ch + 1 < t.chunks; ++ch) chunk(ch, std::true_type {});
        chunk(ch, std::false_type {});

        // epilogue: bias (+ residual) + activation, fp16 NC4HW4 store
        if (m0 >= MF) return;
        const int px = fr * 32 + (lane & 31), lk = lane >> 5;
        const int n  = S == 1 ? (px & 63) >> 2 : (px & 31) >> 1;
        const int yr = S == 1 ? px >> 6 : (px >> 6) * 2 + ((px >> 5) & 1);
        const int qo = grp * 16 + n;
        if (qo >= t.Q) return;
        const int xo = qo % t.XB, no = qo / t.XB, oy = (no % t.NB) * BR + yr, ox = xo * DX + (S == 1 ? px & 3 : px & 1);
        if (oy >= OH || ox >= OW) return;
        const long long base = ((long long) (no / t.NB) * a.Coutb * OH + oy) * OW + ox;
        auto            finish = [&](auto act_c) __attribute__((always_inline)) {
            constexpr int ACT = decltype(act_c)::value;
#pragma unroll
            for (int m = 0; m < MW; ++m)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int oc = (m0 + m) * 32 + k * 8 + lk * 4, ocb = oc >> 2;
                    if (ocb >= a.Coutb) continue;
                    float4v v = {pacc[m][k * 4 + 0], pacc[m][k * 4 + 1], pacc[m][k * 4 + 2], pacc[m][k * 4 + 3]};
                    v += *reinterpret_cast<const float4v *>(a.pw_b + oc);
                    const long long yi = base + (long long) ocb * OH * OW;
                    if (a.has_res) v += h4_to_f4(u2_as_h4(a.res[yi]));
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e] = apply_act(v[e], ACT < 0 ? a.act : ACT, a.lo, a.hi);
                        if (oc + e >= a.Cout) v[e] = 0.f;
                    }
                    a.y[yi] = h4_as_u2(f4_to_h4(v));
                }
        };
        if (a.act == VKHIP_ACT_NONE) finish(integral_constant<int, VKHIP_ACT_NONE> {});
        else if (a.act == VKHIP_ACT_RELU) finish(integral_constant<int, VKHIP_ACT_RELU> {});
        else finish(integral_constant<int, -1> {});
    }

    // The column split of a shape that dwpw_ring_fits accepts (square 3x3 / 5x5, stride 1 or 2, no
    // dilation, even width, at most 64 output channels, 31-bit buffer offsets), or false where the taps
    // of a window's outputs reach past its 8 pixels (5x5 stride 1 with an odd left pad).
    bool dwpw_cols_plan(const vkhip_dwpw_desc *d, DwPwCols &t) {
        const vkhip_conv_desc &c = d->dw;
        const int     DX = c.SH == 1 ? 4 : 2;
        const int64_t Eb = ceil_div(c.Cin, 4);
        t.off = ((c.PL + 1) & ~1) - c.PL;
        if ((DX - 1) * c.SW + c.KW - 1 + t.off > 7) return false;
        t.XB     = (int) ceil_div(c.OW, DX);
        t.NB     = (int) ceil_div(c.OH, 4);
        t.chunks = (int) ceil_div(Eb, 8);
        const int64_t Q = (int64_t) c.N * t.NB * t.XB;
        if (Q >= (1LL << 30)) return false;
        t.Q = (int) Q;
        return true;
    }

    int dwpw_cols_launch(const DwPwArgs &a, const DwPwCols &t, hipStream_t st) {
        const dim3 grid((unsigned) ceil_div(t.Q, 16));
        using std::integral_constant;
        auto go = [&](auto k, auto s) {
            constexpr int K = decltype(k)::value, S = decltype(s)::value;
            if (a.m_frags == 1) dwpw_cols_kernel<K, S, 1><<<grid, 512, 0, st>>>(a, t);
            else dwpw_cols_kernel<K, S, 2><<<grid, 512, 0, st>>>(a, t);
        };
        if (a.KH == 3 && a.SH == 1) go(integral_constant<int, 3> {}, integral_constant<int, 1> {});
        else if (a.KH == 3) go(integral_constant<int, 3> {}, integral_constant<int, 2> {});
        else if (a.SH == 1) go(integral_constant<int, 5> {}, integral_constant<int, 1> {});
        else go(integral_constant<int, 5> {}, integral_constant<int, 2> {});
        return check_launch("dwpw_cols");
    }

} // namespace vkhip
