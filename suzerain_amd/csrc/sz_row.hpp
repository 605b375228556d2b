// Multiply-adds with a factor broadcast from a lane of the 16-lane row (gfx950).
#pragma once
#include <hip/hip_runtime.h>

namespace sz {

// a_i -= l[lane L0 + i] u for i < N (N = 1 or 4), l read from lanes L0 .. of
// the same 16-lane row: the two nested multiply-adds of sz::cfnms.  Written
// as instructions because the compiler does not fold a 64-bit row broadcast
// into the multiply-add; the leading s_nop covers the two wait states a DPP
// operand needs after the instruction that wrote it.  The accumulators are
// written before the other operands' last reads ("+&v"): without that an
// operand that starts with an accumulator's value may share its register.
template <int L0, typename R>
__device__ __forceinline__ void fnms_row1(R &ax, R &ay, R lx, R ly, R ux, R uy)
{
    if constexpr (sizeof(R) == 8)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, -%2, %4 row_newbcast:%c6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, -%2, %5 row_newbcast:%c6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %0, %3, %5 row_newbcast:%c6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, -%3, %4 row_newbcast:%c6 row_mask:0xf bank_mask:0xf"
            : "+&v"(ax), "+&v"(ay) : "v"(lx), "v"(ly), "v"(ux), "v"(uy), "n"(L0));
    else
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %0, -%2, %4 row_newbcast:%c6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %1, -%2, %5 row_newbcast:%c6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %0, %3, %5 row_newbcast:%c6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %1, -%3, %4 row_newbcast:%c6 row_mask:0xf bank_mask:0xf"
            : "+&v"(ax), "+&v"(ay) : "v"(lx), "v"(ly), "v"(ux), "v"(uy), "n"(L0));
}
#define PN_LINE(OP, A, L, U, C) OP " %" #A ", " L ", %" #U " row_newbcast:%c" #C         \
                                " row_mask:0xf bank_mask:0xf\n\t"
#define PN_FOUR(OP)                                                             \
    "s_nop 1\n\t"                                                               \
    PN_LINE(OP, 0, "-%8", 10, 12) PN_LINE(OP, 1, "-%8", 11, 12)                   \
    PN_LINE(OP, 2, "-%8", 10, 13) PN_LINE(OP, 3, "-%8", 11, 13)                   \
    PN_LINE(OP, 4, "-%8", 10, 14) PN_LINE(OP, 5, "-%8", 11, 14)                   \
    PN_LINE(OP, 6, "-%8", 10, 15) PN_LINE(OP, 7, "-%8", 11, 15)                   \
    PN_LINE(OP, 0, "%9", 11, 12) PN_LINE(OP, 1, "-%9", 10, 12)                    \
    PN_LINE(OP, 2, "%9", 11, 13) PN_LINE(OP, 3, "-%9", 10, 13)                    \
    PN_LINE(OP, 4, "%9", 11, 14) PN_LINE(OP, 5, "-%9", 10, 14)                    \
    PN_LINE(OP, 6, "%9", 11, 15) PN_LINE(OP, 7, "-%9", 10, 15)
template <int L0, typename R>
__device__ __forceinline__ void fnms_row4(R &ax0, R &ay0, R &ax1, R &ay1, R &ax2, R &ay2,
                                          R &ax3, R &ay3, R lx, R ly, R ux, R uy)
{
    if constexpr (sizeof(R) == 8)
        asm(PN_FOUR("v_fmac_f64_dpp")
            : "+&v"(ax0), "+&v"(ay0), "+&v"(ax1), "+&v"(ay1), "+&v"(ax2), "+&v"(ay2),
              "+&v"(ax3), "+&v"(ay3)
            : "v"(lx), "v"(ly), "v"(ux), "v"(uy), "n"(L0), "n"(L0 + 1), "n"(L0 + 2),
              "n"(L0 + 3));
    else
        asm(PN_FOUR("v_fmac_f32_dpp")
            : "+&v"(ax0), "+&v"(ay0), "+&v"(ax1), "+&v"(ay1), "+&v"(ax2), "+&v"(ay2),
              "+&v"(ax3), "+&v"(ay3)
            : "v"(lx), "v"(ly), "v"(ux), "v"(uy), "n"(L0), "n"(L0 + 1), "n"(L0 + 2),
              "n"(L0 + 3));
}
#undef PN_FOUR
#undef PN_LINE

}  // namespace sz
