// fp32 products on the f16 matrix cores of gfx950 by a two-way split.
//
// A float row is scaled by a power of two so that its largest magnitude lies
// in [2^14, 2^15), and each scaled value v is held as two halves, hi = f16(v)
// and lo = f16(v - hi): 22 significand bits and lo's sign, about 23 in all,
// for every value within 2^-18 of the row's largest.  Smaller ones keep an
// absolute error of 2^-40 of it, which shows where the large values of a row
// meet zeros or small values: a row's code counts them, and what they may have
// spoilt is recomputed in floats (gemm_split_kernel).  A product of two such
// rows is
//     sum hi.hi + hi.lo + lo.hi      (lo.lo, below 2^-22 of hi.hi, dropped)
// accumulated in f32 by v_mfma_f32_16x16x32_f16: three instructions of 16
// cycles for 32 k-values against eight v_mfma_f32_16x16x4_f32 of 32 cycles.
// Against float64 the result is closer than the fp32 matrix instructions' for
// K >= 64 or so, because the products are summed 32 to a rounding instead
// of 4 (see launch_gemm_split for the measured errors).
//
// Storage, "split rows": row r, k-slice s (32 values) is 128 bytes at
// (r * K / 32 + s) * 128: hi of the 32 values, then lo.  The bytes are those
// of the f32 row, so a buffer of rows * K floats holds either form.  K is
// padded with zeros to a multiple of 32.
#pragma once

#include "common.h"
#include "kernels.h"

namespace vh {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// v_mfma_f32_16x16x32_f16.  Lane l supplies A row l % 16 and B column l % 16
// at k = 8 * (l / 16) .. + 7; D[4 * (l / 16) + r][l % 16] lands in register r.
__device__ __forceinline__ f32x4 mfma16x16x32_f16(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// hi and lo of a scaled value.
__device__ __forceinline__ void split_f16(float v, _Float16 &hi, _Float16 &lo) {
    hi = (_Float16)v;
    lo = (_Float16)(v - (float)hi);
}

// e with |x| * 2^-e in [2^14, 2^15) for the row maximum's bits (0: e = 0).
__device__ __forceinline__ int split_exponent(uint32_t maxbits) {
    if (maxbits >= 0x7f800000u) return kSplitNonFinite;
    if (maxbits == 0) return 0;
    // frexp exponent, subnormals included: |x| = f * 2^ex, f in [1/2, 1).
    return __builtin_amdgcn_frexp_expf(__uint_as_float(maxbits)) - 15;
}

// Largest of the 64 lanes, in each of them (the steps of wave_sum).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_umax(uint32_t v) {
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
    v = dpp_umax<0x140>(dpp_umax<0x141>(dpp_umax<0x4e>(dpp_umax<0xb1>(v))));
    v = max(v, (uint32_t)__shfl_xor((int)v, 16, kWave));
    return max(v, (uint32_t)__shfl_xor((int)v, 32, kWave));
}

// Small values of a split row (nonzero, below 2^-3 once scaled): those whose
// key, the magnitude's bits less one so that zero sorts above every number, is
// below the limit of the row's exponent.
__device__ __forceinline__ uint32_t small_key(float v) { return (__float_as_uint(v) & 0x7fffffffu) - 1u; }
__device__ __forceinline__ uint32_t small_limit(int e) {
    return max(__float_as_uint(__builtin_ldexpf(0.125f, e)), 1u) - 1u;
}
__device__ __forceinline__ int small_count4(f32x4 v, uint32_t limit) {
    int n = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) n += small_key(v[r]) < limit;
    return n;
}

// Running maximum of magnitudes as bit patterns (a NaN sorts above every number).
__device__ __forceinline__ uint32_t absmax4(uint32_t mx, f32x4 v) {
#pragma unroll
    for (int r = 0; r < 4; r++) mx = max(mx, __float_as_uint(v[r]) & 0x7fffffffu);
    return mx;
}

// One asynchronous copy of 16 bytes per lane, global base + voff to LDS
// lds + 16 * lane (global_load_lds_dwordx4; lds is wave-uniform).  In asm,
// because the compiler orders LDS reads behind every builtin copy in flight
// (s_waitcnt vmcnt(0) before the first read), which would empty the pipeline;
// split_wait states the wait instead.  It has no output registers.  s_nop: a
// scalar write of m0 needs one wait state before an LDS copy reads it.  (m0
// cannot be named as clobbered; a kernel that copies this way must hold no
// other use of it, such as the builtin copy.)
__device__ __forceinline__ void copy16_to_lds(const void *base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds), "v"(voff), "s"(base)
                 : "memory");
}

// Every copy but the last N of this wave landed, and its LDS reads returned.
template <int N>
__device__ __forceinline__ void split_wait() {
    static_assert(N >= 0 && N < 64, "vmcnt counts to 63");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

}  // namespace vh
