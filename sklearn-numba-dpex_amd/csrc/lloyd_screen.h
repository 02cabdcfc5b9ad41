// What the kernels that screen labels on the fp16 matrix cores share (lloyd_mfma_screen.hip says how the screen
// works): the constants of its error bound, the scale, the split into two fp16 parts, and the fixed-point terms of the
// sums.
#pragma once

#include "kmx_common.h"

namespace {

// Error bound of one approximate score, in scaled units:
//   (SCR_ERR_SPLIT + r) ||x|| C + r H + SCR_ERR_ABS sqrt(d) (||x|| + C),
// r = SCR_ERR_ROUND * 51 * (K steps of 16 features): one ulp per addition of the accumulation
constexpr float SCR_ERR_SPLIT = 7.2e-7f;  // 3.01 * 2^-22, rounded up
// fp64 inputs reach the split through one rounding to fp32 (2^-24 relative, for x and for c): what
// the two fp16 parts leave out is then at most 1.25 * 2^-22 of a value instead of 2^-22, and the
// half norms in the scores are those of the rounded centroids (2^-23 relative)
constexpr float SCR_ERR_SPLIT_F64 = 9.6e-7f;  // 4.01 * 2^-22, rounded up
constexpr float SCR_ERR_HNEG_F64 = 1.2e-7f;   // 2^-23, rounded up
constexpr float SCR_ERR_ROUND = 1.2e-7f;  // 2^-23, rounded up
constexpr float SCR_ERR_ABS = 6.2e-5f;    // 2^-14, rounded up
// Scaled data lie in [2^(SCR_SCALE_EXP - 1), 2^SCR_SCALE_EXP): low enough for -0.5||c||^2 / SCR_HK_X1
// to stay inside fp16 for every d <= 31 (0.5 * 31 * 2^26 / 2^15 < 2^15), high enough for the
// absolute term of the bound to stay a few percent of the relative one.
constexpr int SCR_SCALE_EXP = 13;

// 1.5 * 2^(52 - q): adding it to |v| < 2^(51 - q) leaves round-to-nearest(v * 2^q) in the low
// mantissa bits, so the product x * w needs no separate scaling by 2^q.  The low word is zero.
__device__ __forceinline__ double fix_magic(int q) {
    return __hiloint2double((int)(0x43380000u - ((unsigned int)q << 20)), 0);
}
__device__ __forceinline__ unsigned long long to_fixed_q(double v_plus_magic, double magic) {
    // only the high words differ (asm: the optimiser would rebuild a 64-bit subtraction)
    unsigned int hi;
    asm("v_sub_u32 %0, %1, %2" : "=v"(hi) : "v"(__double2hiint(v_plus_magic)), "v"(__double2hiint(magic)));
    return ((unsigned long long)hi << 32) | (unsigned int)__double2loint(v_plus_magic);
}

// 2^-a with max|x| * 2^-a in [2^(SCR_SCALE_EXP - 1), 2^SCR_SCALE_EXP) (1 for all-zero or non-finite data)
__device__ __forceinline__ float screen_scale(const float xmax) {
    return (xmax > 0.0f && xmax < kmx_inf<float>()) ? ldexpf(1.0f, SCR_SCALE_EXP - 1 - ilogbf(xmax)) : 1.0f;
}

// The fp16 pair of eight scaled values, as operand registers: hi = fp16(x * 2^-a) and
// lo = fp16(x * 2^-a - hi), each one mixed-precision fused multiply-add with a single rounding
// (the product with a power of two and the difference are exact); value i goes to half i % 2 of
// register i / 2.  `scale` is a scalar operand.
// Sixteen instructions in ONE statement: between separate statements the compiler pads every
// dependency on an assembly result with a wait state (it must assume a partial register
// write).  The real rule - a 16-bit write needs one instruction between it and a read of that
// register - is kept by the order: the four registers are written in rotation.  The closing
// s_nop gives a vector-ALU result the two wait states it needs before a matrix instruction may
// read it.
__device__ __forceinline__ void split_eight(const float v0, const float v1, const float v2, const float v3,
                                            const float v4, const float v5, const float v6, const float v7,
                                            const float scale, unsigned int (&hw)[4], unsigned int (&lw)[4]) {
    asm("v_fma_mixlo_f16 %0, %8, %16, 0\n\t"
        "v_fma_mixlo_f16 %1, %10, %16, 0\n\t"
        "v_fma_mixlo_f16 %2, %12, %16, 0\n\t"
        "v_fma_mixlo_f16 %3, %14, %16, 0\n\t"
        "v_fma_mixhi_f16 %0, %9, %16, 0\n\t"
        "v_fma_mixhi_f16 %1, %11, %16, 0\n\t"
        "v_fma_mixhi_f16 %2, %13, %16, 0\n\t"
        "v_fma_mixhi_f16 %3, %15, %16, 0\n\t"
        "v_fma_mixlo_f16 %4, %8, %16, -%0 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %5, %10, %16, -%1 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %6, %12, %16, -%2 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %7, %14, %16, -%3 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %4, %9, %16, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %5, %11, %16, -%1 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %6, %13, %16, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %7, %15, %16, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "s_nop 1"
        : "=&v"(hw[0]), "=&v"(hw[1]), "=&v"(hw[2]), "=&v"(hw[3]), "=&v"(lw[0]), "=&v"(lw[1]), "=&v"(lw[2]),
          "=&v"(lw[3])
        : "v"(v0), "v"(v1), "v"(v2), "v"(v3), "v"(v4), "v"(v5), "v"(v6), "v"(v7), "s"(scale));
}

}  // namespace
