// Depthwise 3x3 / 5x5 convolution (stride 1 or 2) on the matrix cores, straight from global memory.
#include "conv_kernels.h"

namespace vkhip {

    // One v_mfma_f32_16x16x32_f16 takes an input row window of 8 pixels x 4 channels (one channel
    // block, K = 32) to 16 outputs x 16 windows. The A operand is the row's taps as a banded matrix:
    // its row (d, c) holds channel c's taps at the pixels that output d of the window sees, zero
    // elsewhere. Stride 1: the outputs are 4 neighbouring pixels, and an input row updates the K
    // output rows it is a tap row of (K products, K live accumulators). Stride 2: 2 pixels of 2
    // output rows, so K + 2 input rows make a row pair. The 16 columns of B are 16 windows of the
    // same channel block: (image, row band, window) in that order, flattened, so that 7-wide planes
    // fill the tile as well as 112-wide ones. A lane's B registers are 16 contiguous bytes of a row
    // (2 pixels x 4 channels) and its result is one NC4HW4 vector: nothing passes through LDS.
    //
    // Bound: memory, then the epilogue's VALU work. The LDS strip kernel (dwconv_lds_kernel) is VALU
    // bound: for a 5x5 tap row and one output pixel of 4 channels it issues 12 dot products and mixed
    // fmas plus the packing of their operands, where here 256 outputs cost one product of 16 cycles.
    // Measured at batch 128, hard-swish, from memory (strip kernel's best plan -> this): 672 channels
    // at 14x14 5x5 27.7 -> 16.3 us (4.1 TB/s) and 3x3 20.8 -> 14.8, 960 at 7x7 5x5 14.8 -> 11.4,
    // 72 at 56x56 5x5 stride 2 20.7 -> 12.7, 672 at 14x14 5x5 stride 2 16.7 -> 10.2; one image:
    // 672 at 14x14 5.8 -> 4.5. 108 VGPRs, four waves per SIMD; held to five or six it spills (27.6 and
    // 58.9 us on the first shape). Storing through a lane permutation (contiguous runs instead of 8-byte
    // vectors 32 bytes apart) was 5% slower; the order of the items and shorter bands made no
    // difference.
    //
    // A zero entry of the banded matrix times an infinity or NaN is NaN, so a window with one would
    // spoil its 16 outputs: such a window leaves every one of its sums non-finite, and the lanes that
    // saw one recompute their outputs tap by tap at the end.

    template <int K, int S>
    struct DwColsShape {
        static constexpr int F  = S == 1 ? K : K + 2;         // A fragments: tap rows (stride 2: of a row pair)
        static constexpr int U  = S == 1 ? (K == 3 ? 6 : 5) : 8; // rows in flight; a multiple of the accumulator period
        static constexpr int DX = S == 1 ? 4 : 2;             // output pixels of a window
    };

    // POOL: also leave the pool sums (without them the kernel holds fewer registers: 15.4 -> 15.0 us on the
    // first shape above). RES: with a residual (as a run-time branch of each row 15.3 us, as a variant
    // 14.2; both without a residual).
    template <int K, int S, int ACT, bool ODD, bool POOL, bool RES>
    __global__ __launch_bounds__(256, 4) void dwconv_cols_kernel(DwArgs a, DwCols t) {
        using Sh = DwColsShape<K, S>;
        constexpr int      F = Sh::F, U = Sh::U, DX = Sh::DX;
        constexpr unsigned kInvalid = 0x80000000u;
        const int lane = threadIdx.x & 63, n16 = lane & 15, g = lane >> 4;
        // channel block fastest: neighbouring waves read neighbouring planes
        const int item = __builtin_amdgcn_readfirstlane(xcd_remap(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6));
        if (item >= t.groups * a.Cb) return;
        const int cb = item % a.Cb, grp = item / a.Cb;

        // A fragments: lane holds row (d, c) = (n16 / 4, n16 % 4), window pixels 2g and 2g + 1
        half8 fa[F];
        {
            const int c = n16 & 3, d = n16 >> 2;
            const int dy = S == 1 ? 0 : d >> 1, dx = S == 1 ? d : d & 1;
            const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc((void *) (a.w + (long long) cb * K * K), (short) 0, K * K * 8, 0x00020000);
            unsigned short               wt[F][2]; // all loads first, out-of-window taps read zeros: one latency
#pragma unroll
            for (int f = 0; f < F; ++f)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int  kx = 2 * g + e - t.off - dx * S, ky = f - 2 * dy;
                    const bool ok = (unsigned) kx < (unsigned) K && (unsigned) ky < (unsigned) K;
                    wt[f][e]      = __builtin_amdgcn_raw_buffer_load_b16(wrs, ok ? (unsigned) (((ky * K + kx) * 4 + c) * 2) : kInvalid, 0, 0);
                }
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const unsigned s0 = (unsigned) wt[f][0] << (16 * (c & 1)), s1 = (unsigned) wt[f][1] << (16 * (c & 1));
                fa[f] = __builtin_bit_cast(half8, u32x4_make(c & 2 ? 0u : s0, c & 2 ? s0 : 0u, c & 2 ? 0u : s1, c & 2 ? s1 : 0u));
            }
        }
        const float4v b0 = *reinterpret_cast<const float4v *>(a.bias + cb * 4);

        // this lane's column: image, band, window
        const int  H = a.H, W = a.W, OH = a.OH, OW = a.OW;
        const int  q    = grp * 16 + n16;
        const bool live = q < t.Q;
        const int  xbq  = (live ? q : 0) % t.XB, nbq = (live ? q : 0) / t.XB;
        const int  band = nbq % t.NB, img = nbq / t.NB;
        const int  plane = img * a.Cb + cb;
        const int  y0    = band * t.BR;          // first output row
        const int  iy0   = y0 * S - a.PT;        // first input row
        const int  x0    = xbq * 4 - (t.off + a.PL) + 2 * g; // this lane's pixel pair (even)
        const bool ok0   = live && x0 >= 0 && x0 < W, ok1 = live && x0 >= 0 && x0 + 1 < W;
        const int  W8    = W * 8;
        const unsigned xb = (unsigned) ((plane * H + iy0) * W + x0) * 8u; // wraps for rows above the image: used only where valid
        const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc((void *) a.x, (short) 0, a.N * a.Cb * H * W * 8, 0x00020000);
        const __amdgpu_buffer_rsrc_t yrs = __builtin_amdgcn_make_buffer_rsrc((void *) a.y, (short) 0, a.N * a.Cb * OH * OW * 8, 0x00020000);
        const __amdgpu_buffer_rsrc_t rrs =
            __builtin_amdgcn_make_buffer_rsrc((void *) (RES ? a.res : a.y), (short) 0, RES ? a.N * a.Cb * OH * OW * 8 : 0, 0x00020000);
        // rows of the band inside the image; the others read zeros
        const int R    = t.BR * S + K - S; // input rows of a band
        const int ylast = max(0, min(H, iy0 + R)); // 0: the whole band lies in the top padding
        auto load = [&](int r) __attribute__((always_inline)) {
            const bool     row = (unsigned) (iy0 + r) < (unsigned) ylast;
            const unsigned o   = xb + (unsigned) (r * W8);
            if constexpr (ODD) {
                const u32x2 p = __builtin_amdgcn_raw_buffer_load_b64(xrs, row & ok0 ? o : kInvalid, 0, 0);
                const u32x2 s = __builtin_amdgcn_raw_buffer_load_b64(xrs, row & ok1 ? o + 8u : kInvalid, 0, 0);
                return u32x4_make(p.x, p.y, s.x, s.y);
            } else {
                return __builtin_amdgcn_raw_buffer_load_b128(xrs, row & ok0 ? o : kInvalid, 0, 0);
            }
        };

        // output: lane (n16, g) holds the 4 channels of one pixel of its window
        const int      ox   = xbq * DX + (S == 1 ? g : g & 1);
        const int      dyl  = S == 1 ? 0 : g >> 1;
        const int      ylim = min(t.BR, OH - y0); // output rows of this band
        const bool     xok  = live && ox < OW;
        const unsigned yb   = (unsigned) ((plane * OH + y0) * OW + ox) * 8u;
        const bool     rag  = (a.C & 3) != 0;
        float4v        psum = {0.f, 0.f, 0.f, 0.f};
        float          nf   = 0.f; // NaN once a sum of this lane was not finite
        int            kept = 0;   // RES: the rows stored until then
        auto finish = [&](float4v v, int y, bool ok, auto first_c) __attribute__((always_inline)) {
            // The residual may be the output's own memory: its rows from the first non-finite sum on are
            // left as they are for the recomputation (without one they are stored twice).
            if constexpr (RES && decltype(first_c)::value) {
                ok = ok && nf == nf;
                kept += nf == nf;
            }
            const unsigned o = ok ? yb + (unsigned) (y * OW) * 8u : kInvalid;
            if constexpr (RES) v += h4_to_f4(__builtin_bit_cast(half4, __builtin_amdgcn_raw_buffer_load_b64(rrs, o, 0, kStreamLoad)));
            v.x = apply_act(v.x, ACT, a.lo, a.hi);
            v.y = apply_act(v.y, ACT, a.lo, a.hi);
            v.z = apply_act(v.z, ACT, a.lo, a.hi);
            v.w = apply_act(v.w, ACT, a.lo, a.hi);
            if (rag) {
                if (cb * 4 + 0 >= a.C) v.x = 0.f;
                if (cb * 4 + 1 >= a.C) v.y = 0.f;
                if (cb * 4 + 2 >= a.C) v.z = 0.f;
                if (cb * 4 + 3 >= a.C) v.w = 0.f;
            }
            const half4 h = f4_to_h4(v);
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, h), yrs, o, 0, kStreamStore);
            if constexpr (POOL) {
                // the sum of the fp16 values just stored (one mixed fma each, the same single rounding
                // as converting and adding)
                const u32x2 hb = __builtin_bit_cast(u32x2, h);
                const half4 hs = __builtin_bit_cast(half4, u32x2 {ok ? hb.x : 0u, ok ? hb.y : 0u});
                psum.x = __builtin_fmaf((float) hs.x, 1.f, psum.x);
                psum.y = __builtin_fmaf((float) hs.y, 1.f, psum.y);
                psum.z = __builtin_fmaf((float) hs.z, 1.f, psum.z);
                psum.w = __builtin_fmaf((float) hs.w, 1.f, psum.w);
            }
        };
        auto emit = [&](const float4v &v, int y) __attribute__((always_inline)) {
            nf = __builtin_fmaf(v.x, 0.f, nf);
            finish(v, y + dyl, xok && y + dyl < ylim, std::true_type {});
        };

        u32x4 buf[U];
#pragma unroll
        for (int u = 0; u < U; ++u) buf[u] = load(u);
        float4v acc[S == 1 ? K : 2];
        // row r = r0 + u: its products, the load of row r + U, and the output rows it completes
        auto step = [&](int r, auto uc, auto first_c, auto more_c) __attribute__((always_inline)) {
            constexpr int  u     = decltype(uc)::value;
            constexpr bool first = decltype(first_c)::value; // the first U rows of the band
            const half8    fb    = __builtin_bit_cast(half8, buf[u]);
            if constexpr (decltype(more_c)::value) buf[u] = load(r + U);
            if constexpr (S == 1) {
                // output row r starts from the bias; r - K + 1 is complete
                acc[u % K] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[0], fb, b0, 0, 0, 0);
                static_for<1, K>([&](auto kc) {
                    constexpr int ky = decltype(kc)::value, i = (u - ky + 2 * K) % K;
                    if constexpr (!first || ky <= u) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[ky], fb, acc[i], 0, 0, 0);
                });
                if constexpr (!first || u >= K - 1) emit(acc[(u + 1) % K], r - (K - 1));
            } else {
                // pair r / 4 gets tap row r % 4 (the first one on top of the bias), the pair before it tap row r % 4 + 4
                constexpr int cur = (u / 4) & 1, tr = u % 4;
                if constexpr (tr == 0) acc[cur] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[tr], fb, b0, 0, 0, 0);
                else acc[cur] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[tr], fb, acc[cur], 0, 0, 0);
                if constexpr (tr + 4 < F && (!first || u >= 4)) {
                    acc[cur ^ 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[tr + 4], fb, acc[cur ^ 1], 0, 0, 0);
                    if constexpr (tr + 4 == F - 1) emit(acc[cur ^ 1], (r / 4 - 1) * 2);
                }
            }
        };
        // Whole blocks of U rows run without a branch between the loads, so that each wait counts the
        // loads after it; with an exit inside the block the compiler waits for every load in flight at
        // its top (18.2 us instead of 14.7 at 672 channels of 14x14 5x5, batch 128).
        using std::false_type;
        using std::true_type;
        int r0 = 0;
        if (R >= U) {
            static_for<0, U>([&](auto uc) { step(decltype(uc)::value, uc, true_type {}, true_type {}); });
            for (r0 = U; r0 + U <= R; r0 += U)
                static_for<0, U>([&](auto uc) { step(r0 + decltype(uc)::value, uc, false_type {}, true_type {}); });
            static_for<0, U - 1>([&](auto uc) {
                if (r0 + decltype(uc)::value < R) step(r0 + decltype(uc)::value, uc, false_type {}, false_type {});
            });
        } else {
            static_for<0, U - 1>([&](auto uc) {
                if (decltype(uc)::value < R) step(decltype(uc)::value, uc, true_type {}, false_type {});
            });
        }
        if (__any(nf != nf)) {
            if (nf != nf && xok) {
                if constexpr (!RES) psum = float4v {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                for (int y = dyl + kept * S; y < ylim; y += S) {
                    float4v v = b0;
#pragma unroll 1
                    for (int k = 0; k < K * K; ++k) {
                        const int iy = (y0 + y) * S - a.PT + k / K, ix = ox * S - a.PL + k % K;
                        if ((unsigned) iy >= (unsigned) H || (unsigned) ix >= (unsigned) W) continue;
                        const half4 xv = u2_as_h4(a.x[((long long) plane * H + iy) * W + ix]), wv = a.w[(long long) cb * K * K + k];
                        v.x = __builtin_fmaf((float) xv.x, (float) wv.x, v.x);
                        v.y = __builtin_fmaf((float) xv.y, (float) wv.y, v.y);
                        v.z = __builtin_fmaf((float) xv.z, (float) wv.z, v.z);
                        v.w = __builtin_fmaf((float) xv.w, (float) wv.w, v.w);
                    }
                    finish(v, y, true, std::false_type {});
                }
            }
        }
        if constexpr (POOL) {
            // A window's pixels are lanes n16, n16 + 16, + 32 and + 48; then the windows of one (plane,
            // band) that this group holds add up into the first of them, in a fixed order.
            auto from = [&](float4v v, int src) __attribute__((always_inline)) { return float4v {__shfl(v.x, src), __shfl(v.y, src), __shfl(v.z, src), __shfl(v.w, src)}; };
            psum += from(psum, lane ^ 16);
            psum += from(psum, lane ^ 32);
            for (int o = 1; o < 16 && o < t.XB; o <<= 1) {
                const float4v v = from(psum, lane + o);
                if (n16 + o < 16 && xbq + o < t.XB && q + o < t.Q) psum += v;
            }
            const int g0 = (q - xbq) >> 4, part = grp - g0; // the groups of this (plane, band): g0 ..
            if (live && g == 0 && (n16 == 0 || xbq == 0)) {
                float4v *p = a.pool + (((long long) plane * t.NB + band) * t.parts);
                p[part]    = psum;
                if (grp == (q - xbq + t.XB - 1) >> 4)
                    for (int k = part + 1; k < t.parts; ++k) p[k] = float4v {0.f, 0.f, 0.f, 0.f};
            }
        }
    }

    // The column split of a depthwise conv, or false where the kernel does not apply: unit dilation,
    // square 3x3 / 5x5, stride 1 or 2, and taps that stay inside the 8-pixel window.
    // Bands: whole planes while that makes enough waves (2048, two per SIMD), else down to 4 rows
    // (the K - 1 extra input rows of a band are read again by its neighbour).
    // With pool sums every band adds t.parts of them to what each FC tile after it sums up, 0.15 us each,
    // where a row less per band saves 0.2 us: 4 bands, 8 past 128 rows. Conv and squeeze-excite of one
    // image, bands as without the sums (by the wave count) -> 4 or 8: 64 channels 112x112 3x3 27.8 -> 17.0
    // us, 96 at 112 / 2 3x3 21.5 -> 14.2, 72 at 56 3x3 16.4 -> 14.1, 32 at 224 3x3 63.2 -> 23.3.
    // A 3x3 stride-2 conv whose tensors exceed the last-level cache stays with the strip kernel, which
    // reads them in longer runs: 64 channels 112 -> 56 at batch 128 (257 MB) 49.3 us against 59.1,
    // 56 -> 28 at batch 512 49.8 against 55.3; below (77 MB) 17.3 against 15.3, and the other kernel
    // sizes and strides are level or faster here on both sides (3x3 stride 1, 321 MB: 72.8 / 73.0;
    // 5x5 stride 2, 201 MB: 51.2 / 45.2).
    bool dw_cols_plan(const vkhip_conv_desc *d, bool pooled, DwCols &t) {
        const int K = d->KH, S = d->SH;
        if (d->DH != 1 || d->DW != 1 || d->KW != K || d->SW != S || (K != 3 && K != 5) || (S != 1 && S != 2)) return false;
        const int DX = S == 1 ? 4 : 2;
        t.off = ((d->PL + 1) & ~1) - d->PL;
        if ((DX - 1) * S + K - 1 + t.off > 7) return false;
        const int64_t Cb = ceil_div(d->Cin, 4);
        if (K == 3 && S == 2 && d->OW > 14 && d->N * Cb * ((int64_t) d->H * d->W + (int64_t) d->OH * d->OW) * 8 > ((int64_t) 160 << 20)) return false;
        t.XB = (int) ceil_div(d->OW, DX);
        t.NB = 1;
        auto rows = [&](int nb) { return (int) round_up(ceil_div(d->OH, nb), S); };
        const int most = !pooled ? d->OH : d->OH > 128 ? 8 : 4;
        while (t.NB < most && Cb * ceil_div((int64_t) d->N * t.XB * t.NB, 16) < 2048 && rows(t.NB) > 4) ++t.NB;
        t.BR = rows(t.NB);
        t.NB = (int) ceil_div(d->OH, t.BR);
        const int64_t Q = (int64_t) d->N * t.XB * t.NB;
        if (Q * Cb >= (1LL << 31)) return false;
        t.Q      = (int) Q;
        t.parts  = t.XB <= 16 && 16 % t.XB == 0 ? 1 : (t.XB + 14) / 16 + 1;
        t.groups = (int) ceil_div(Q, 16);
        return true;
    }

    template <int K, int S>
    static void launch_cols(const DwArgs &a, const DwCols &t, hipStream_t st) {
        const dim3 grid((unsigned) ceil_div((int64_t) t.groups * a.Cb, 4));
        auto       go = [&](auto act_c) {
            constexpr int ACT = decltype(act_c)::value;
            auto          with = [&](auto odd_c, auto pool_c) {
                constexpr bool ODD = decltype(odd_c)::value, POOL = decltype(pool_c)::value;
                if (a.has_res) dwconv_cols_kernel<K, S, ACT, ODD, POOL, true><<<grid, 256, 0, st>>>(a, t);
                else dwconv_cols_kernel<K, S, ACT, ODD, POOL, false><<<grid, 256, 0, st>>>(a, t);
            };
            using std::false_type;
            using std::true_type;
            if (a.W % 2) a.pool ? with(true_type {}, true_type {}) : with(true_type {}, false_type {});
            else a.pool ? with(false_type {}, true_type {}) : with(false_type {}, false_type {});
        };
        using std::integral_constant;
        switch (a.act) {
            case VKHIP_ACT_RELU: go(integral_constant<int, VKHIP_ACT_RELU> {}); break;
            case VKHIP_ACT_RELU6: go(integral_constant<int, VKHIP_ACT_RELU6> {}); break;
            case VKHIP_ACT_CLIP: go(integral_constant<int, VKHIP_ACT_CLIP> {}); break;
            case VKHIP_ACT_HARDSWISH: go(integral_constant<int, VKHIP_ACT_HARDSWISH> {}); break;
            case VKHIP_ACT_SILU: go(integral_constant<int, VKHIP_ACT_SILU> {}); break;
            case VKHIP_ACT_HARDSIGMOID: go(integral_constant<int, VKHIP_ACT_HARDSIGMOID> {}); break;
            default: go(integral_constant<int, VKHIP_ACT_NONE> {}); break;
        }
    }

    int dw_cols_launch(const DwArgs &a, const DwCols &t, hipStream_t st) {
        if (a.KH == 3 && a.SH == 1) launch_cols<3, 1>(a, t, st);
        else if (a.KH == 3) launch_cols<3, 2>(a, t, st);
        else if (a.SH == 1) launch_cols<5, 1>(a, t, st);
        else launch_cols<5, 2>(a, t, st);
        return check_launch("dwconv_cols");
    }

} // namespace vkhip
