// Arguments shared by the fused depthwise + projection kernels (dwpw.hip, dwpw_cols.hip).
#pragma once
#include "common.h"

namespace vkhip {

    struct DwPwArgs {
        const uint2  *x;
        const float  *dw_b;  // [Eb*4]
        const float  *dw_w;  // [Eb][KH][KW][4]
        const float  *pw_b;  // [Coutp]
        const half_t *pw_w;  // [Coutp][Kp]
        const uint2  *res;
        uint2        *y;
        int           N, E, Eb, Ebp, H, W, OH, OW, KH, KW, SH, SW, PT, PL, DH, DW;
        int           dw_act;
        int           Cout, Coutb, m_frags, Kp, P;
        int           act;
        float         lo, hi;
        int           has_res;
        const half_t *dw_h;  // [Eb][KH][KW][4], the depthwise weights in fp16
    };

    // Column split of dwpw_cols_kernel (dwpw_cols.hip): windows per row, row bands per plane, window
    // pixel of tap 0 of output 0, columns, chunks of 8 channel blocks.
    struct DwPwCols {
        int XB, NB, off, Q, chunks;
    };
    bool dwpw_cols_plan(const vkhip_dwpw_desc *d, DwPwCols &t);
    int  dwpw_cols_launch(const DwPwArgs &a, const DwPwCols &t, hipStream_t st);

} // namespace vkhip
