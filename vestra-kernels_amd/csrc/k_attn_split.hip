// Online-softmax attention on the f16 matrix cores, on split rows
// (split_gemm.h): head_dim 64, any scale.
//
// Q, K and V are split rows [bh][tokens] of 256 bytes (two slices of 32
// dims, hi then lo), each tensor with one exponent per head or one for all.
// A workgroup of eight waves owns 64 queries of one head; QG = 2 groups of
// waves each take 32 of the queries and KS = 4 key streams share the keys: of
// every step's 128 keys stream s takes PK = 32.  K and V
// panels are copied straight into LDS, one step ahead of their use.  Per
// panel a wave computes
//     S^T[key][query] = K . Q^T
// so that a lane holds its own query's scores, keys 16 t + 4 lh + r of tile
// t, which is the B operand of
//     O^T[d][query] += V^T[d][key] . P^T[key][query]
// if the 32 keys of a product are taken in the order (4 lh .. 4 lh + 3 of
// tile 2 g, then of tile 2 g + 1); V^T comes from the row-major panel by
// transposing LDS reads (ds_read_b64_tr_b16) of the same rows.  The output
// stays with the lane of its query, so a correction is a plain multiply.
//
// P is split like everything else.  It is held as 2^5 p, so that its halves
// are exact to 2^-23 for p above 2^-8 of the largest and to 2^-30 below (the
// offset also puts the usual exponents near zero, where their rounding is
// least); the running maximum is only raised when a score passes it by 2^8
// (still inside the half's range), so most panels need no correction.
//
// The output is floats, split rows (the next projection's input), or Q8_0 rows
// (the Q8_0 block's: two streams finish a block of 32 dims and exchange their
// largest magnitudes), which saves the launch that quantised the floats
// (4.8 us at 865 tokens).
//
// Where the halves may not hold what the floats do, a workgroup forms its
// queries again from the floats, on the fp32 matrix instructions (float_pass;
// 12 x 865 in 66 us, the split pass included): heads with an
// infinity or NaN, heads whose small values (split_gemm.h) may show in the scores
// (kScoreBound), and queries whose output is small against the head's largest
// V (kRowFloor, kDimFloor: the probabilities that matter were below P's
// range, or the values below V's).
//
// Error against float64 at 12 x 865 x 64, N(0, 1): 2.5e-7, against 4.3e-7 of the
// fp32 matrix instructions.  Time on split rows (kernel trace): 12 x 865 18 us
// against 28 (fp32 matrix instructions), 48 x 865 53 against 100, 12 x 3457
// 157 against 343.  Products alone would take a third of that: the softmax's
// VALU work and the products share the SIMD's issue (a product holds it
// for 8 of its 16 cycles, measured), and taking out the copies, the LDS reads or
// the exponentials one at a time saves 14%, 4% and 6% at 12 x 3457.  Single K and
// V buffers with two workgroups per CU (174, 210 with the registers for it
// spilled) and the copies spread between the products (167) were slower.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "split_gemm.h"

namespace vh {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kPBits = 5.0f;    // P is held as 2^kPBits p
constexpr float kMaxSlack = 8.0f; // scores may pass the running maximum by this (base 2)

constexpr int QG = 2, KS = 8 / QG;          // query groups and key streams of a workgroup
constexpr int PK = 128 / KS, KT = PK / 16;  // keys of a stream and step, and their tiles of 16

// Codes per head and tensor, one from each workgroup that split its rows: the
// exponent, and whether that workgroup has seen a small value.
constexpr int kCodes = 4;

struct AttnArgs {
    const char *q, *k, *v;        // split rows [bh][T][256 bytes]
    const int *ex;                // [3][bh][kCodes] codes of q, k, v, or null:
    int eq, ek, ev;               // these exponents for every head
    const float *qf, *kf, *vf;    // the float rows [bh][T][hd]
    int T, heads, bh, qtiles, hd;
    float scale_log2;             // softmax scale times log2(e)
    float *out;                   // f32: token-major [img][T][heads*hd] or [bh][T][hd]
    int token_major;
    char *out_split;              // split rows [img*T][heads*64] with exponent ev
    int8_t *q8_qs;                // Q8: blocks [heads*2][img*T][32] of the token-major
    uint16_t *q8_d;               // output and their scales (hd = 64)
};

enum class AOut : int { F32, Split, Q8 };

// quantize_row_q8_0's value (src/q8_0_dot.rs:38-44): half away from zero, NaN to 0.
__device__ __forceinline__ int q8_value(float v, float inv) {
    const float q = roundf(mul_rn(v, inv));
    return isnan(q) ? 0 : (int)fminf(fmaxf(q, -127.0f), 127.0f);
}

// Two floats to two halves (one v_cvt_pk_f16_f32; the empty asm keeps the
// compiler from converting each again where a half is used), and what the
// halves leave of them (v_fma_mix_f32, which the opaque minus one keeps from
// becoming a conversion and a subtraction).  No instruction is written out in
// asm here: the compiler keeps the wait states of a transcendental's result
// only towards instructions that it knows.
__device__ __forceinline__ f16x2 cvt_pk_f16(float a, float b) {
    f16x2 h;
    h[0] = (_Float16)a;
    h[1] = (_Float16)b;
    uint32_t u = __builtin_bit_cast(uint32_t, h);
    asm("" : "+v"(u));
    return __builtin_bit_cast(f16x2, u);
}
__device__ __forceinline__ f16x2 residual_pk_f16(f16x2 h, float a, float b) {
    float minus = -1.0f;
    asm("" : "+s"(minus));
    return cvt_pk_f16(__builtin_fmaf((float)h[0], minus, a), __builtin_fmaf((float)h[1], minus, b));
}

// max / sum with the lanes 16 and 32 away, on the VALU: a permlane swap of
// two copies of v leaves v in one and the partner's v in the other, in either
// order.
__device__ __forceinline__ void swap16(float &a, float &b) {
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void swap32(float &a, float &b) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ float max_groups(float v) {
    float a = v, b = v;
    swap16(a, b);
    a = b = fmaxf(a, b);
    swap32(a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float sum_groups(float v) {
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    return v;
}

// Four halves of column li of a 4 x 16 tile of halves in LDS, whose row r is
// in the lanes 4 r .. 4 r + 3 of each 16-lane group (lane i gives the address
// of row i / 4, columns 4 (i % 4) .. + 3, and receives column i).
__device__ __forceinline__ f16x4 read_tr(const char *p) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                         (__attribute__((address_space(3))) s16x4 *)p));
}

// A score's halves are off by at most 2 * 64 * 2^15 * 2^-25 in their own scale where
// Q or K holds small values: 2^-33 of (largest |q|) (largest |k|) scale, so 2^-21
// of the weight while that product is at most 2^12 (N(0, 1): about 3).
constexpr float kScoreBound = 0x1p12f;
// V, scaled to below 2^15, is off by 2^-25 where it is small, and P by 2^-31 of the
// largest weight: an output row whose largest |o| is at least kRowFloor, and a
// dim whose largest |o| over the queries is at least kDimFloor, hold that to
// 2^-25 of themselves (V; 2^-17 where a wave has fewer than four queries to tell
// by), or to 2^-33 times the number of keys at the worst (P).  N(0, 1) gives |o| of
// 2^8 at 865 tokens, 2^2 at ten million.
constexpr float kRowFloor = 4.0f, kDimFloor = 1.0f;

// max over the 16 lanes of a row (lane & 15), in every lane of it.
__device__ __forceinline__ float max_row16(float v) {
    v = fmaxf(v, dpp_f32<0xb1>(v));
    v = fmaxf(v, dpp_f32<0x4e>(v));
    v = fmaxf(v, dpp_f32<0x141>(v));
    return fmaxf(v, dpp_f32<0x140>(v));
}

// The wave's 32 queries against its stream's keys, from the floats: what the
// split pass leaves in o, m and l, without its exponents.  S^T = K . Q^T and
// O^T += V^T . P^T as there, 4 dims or keys to an instruction: lane (li, lh)
// holds dims 16 c + 4 lh + e of its row, and the key 4 lh + r of instruction
// r of P . V.
__device__ __forceinline__ void float_pass(const AttnArgs &fa, size_t off, int qw, int stream, int lane,
                                           f32x4 (&o)[4][2], float (&m)[2], float (&l)[2]) {
    const int li = lane & 15, lh = lane >> 4, T = fa.T, hd = fa.hd;
    const bool vec = (hd & 3) == 0;
    auto four = [&](const float *row, int d) {
        f32x4 v{0.0f, 0.0f, 0.0f, 0.0f};
        if (vec) {
            if (d < hd) v = *reinterpret_cast<const f32x4 *>(row + d);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (d + e < hd) v[e] = row[d + e];
        }
        return v;
    };
    f32x4 qv[2][4];
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int c = 0; c < 4; c++)
            qv[u][c] = four(fa.qf + off + (size_t)min(qw + 16 * u + li, T - 1) * hd, 16 * c + 4 * lh);
#pragma unroll
    for (int u = 0; u < 2; u++) {
        m[u] = -INFINITY;
        l[u] = 0.0f;
#pragma unroll
        for (int df = 0; df < 4; df++) o[df][u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (int k0 = stream * PK; k0 < T; k0 += 128) {
        f32x4 kv[2][4], s[2][2];
        float vv[2][4][4];  // [key tile][r][df]: V[k0 + 16 t + 4 lh + r][16 df + li]
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                kv[t][c] = four(fa.kf + off + (size_t)min(k0 + 16 * t + li, T - 1) * hd, 16 * c + 4 * lh);
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int df = 0; df < 4; df++) {
                    const int key = k0 + 16 * t + 4 * lh + r, d = 16 * df + li;
                    vv[t][r][df] = key < T && d < hd ? fa.vf[off + (size_t)key * hd + d] : 0.0f;
                }
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                s[t][u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int c = 0; c < 4; c++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        s[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[t][c][e], qv[u][c][e], s[t][u], 0, 0, 0);
            }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            float mx = -INFINITY;
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    s[t][u][r] = k0 + 16 * t + 4 * lh + r < T ? s[t][u][r] * fa.scale_log2 : -INFINITY;
                    mx = fmaxf(mx, s[t][u][r]);
                }
            const float mn = fmaxf(m[u], max_groups(mx)), ref = mn == -INFINITY ? 0.0f : mn;
            const float corr = __builtin_amdgcn_exp2f(m[u] - ref);
            m[u] = mn;
            l[u] *= corr;
#pragma unroll
            for (int df = 0; df < 4; df++) o[df][u] *= corr;
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float p = __builtin_amdgcn_exp2f(s[t][u][r] - ref);
                    l[u] += p;
#pragma unroll
                    for (int df = 0; df < 4; df++)
                        o[df][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[t][r][df], p, o[df][u], 0, 0, 0);
                }
        }
    }
}

template <AOut OUT>
__global__ __launch_bounds__(512, 2) void attn_split_kernel(AttnArgs fa) {
    constexpr int HALF = 128 * 256;  // bytes of a step's K (or V) panels
    extern __shared__ __attribute__((aligned(16))) char smem_c[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lh = lane >> 4;
    const int qg = wave % QG, stream = wave / QG;
    const int T = fa.T;

    // Workgroups go round-robin over the 8 XCDs; a head's query tiles are
    // kept on one XCD, whose L2 then holds its K and V.
    const int total = fa.bh * fa.qtiles, per = (total + 7) / 8;
    const int item = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (item >= total || (int)(blockIdx.x / 8) >= per) return;
    const int bh = item / fa.qtiles, q0 = (item % fa.qtiles) * (QG * 32);
    const int img = bh / fa.heads, head = bh - img * fa.heads;
    const size_t off = (size_t)bh * T * fa.hd;  // of the head's float rows
    int cq = 0, ck = 0, cv = 0;  // the head's codes
    if constexpr (OUT != AOut::Split) {
#pragma unroll
        for (int i = 0; i < kCodes; i++) {
            cq |= fa.ex[bh * kCodes + i];
            ck |= fa.ex[(fa.bh + bh) * kCodes + i];
            cv |= fa.ex[(2 * fa.bh + bh) * kCodes + i];
        }
    }
    bool floats = false;  // the head goes to float_pass

    const char *Qh = fa.q + (size_t)bh * T * 256;
    const char *Kh = fa.k + (size_t)bh * T * 256;
    const char *Vh = fa.v + (size_t)bh * T * 256;
    f32x4 o[4][2];  // o[df][t][r] = O[query tile t, li][16 df + 4 lh + r]
    float m[2], l[2];
    auto split_pass = [&] {
        // Q fragments: query tile t, slice c.
        f16x8 qh[2][2], ql[2][2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const char *row = Qh + (size_t)min(q0 + qg * 32 + 16 * t + li, T - 1) * 256 + lh * 16;
#pragma unroll
            for (int c = 0; c < 2; c++) {
                qh[t][c] = *reinterpret_cast<const f16x8 *>(row + c * 128);
                ql[t][c] = *reinterpret_cast<const f16x8 *>(row + c * 128 + 64);
            }
        }

        // One copy moves four rows of 256 bytes; this wave copies rows 32 i + 4
        // wave .. + 3 of a step's 128 K and 128 V rows (keys past T: the last).
        // K's granules are XOR-swizzled by the row (fragment reads take one
        // granule of 16 rows), V's pairs of granules by the row (transposing
        // reads take a pair of eight rows per 32 lanes).
        const int crow = 4 * wave + (lane >> 4), cg = lane & 15;
        const uint32_t kgr = (uint32_t)((cg ^ (crow & 15)) << 4), vgr = (uint32_t)((cg ^ (2 * (crow & 7))) << 4);
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem_c;
        auto copy_panels = [&](const char *base, int step, uint32_t gr, uint32_t dst0) {
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + dst0 + wave * 1024);
            if ((step + 1) * 128 <= T) {
                const char *panel = base + (size_t)step * 32768;
#pragma unroll
                for (int i = 0; i < 4; i++) copy16_to_lds(panel + i * 8192, crow * 256 + gr, dst + i * 8192);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    copy16_to_lds(base, (uint32_t)min(step * 128 + 32 * i + crow, T - 1) * 256 + gr, dst + i * 8192);
            }
        };

#pragma unroll
        for (int df = 0; df < 4; df++)
#pragma unroll
            for (int t = 0; t < 2; t++) o[df][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        m[0] = m[1] = -INFINITY;
        l[0] = l[1] = 0.0f;

        // LDS offsets of this lane in its stream's panels.
        const char *ks = smem_c + (stream * PK + li) * 256;
        const char *vs = smem_c + 2 * HALF + (stream * PK + 4 * lh + (li >> 2)) * 256 + (li & 1) * 8;
        const int vx = 2 * ((4 * lh + (li >> 2)) & 7), vg0 = (li & 3) >> 1;

        // K fragments of key tile t, slice c of the stream's panel.
        f16x8 kh[KT][2], kl[KT][2];
        auto read_k = [&](int buf) {
#pragma unroll
            for (int t = 0; t < KT; t++)
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    kl[t][c] = *reinterpret_cast<const f16x8 *>(ks + buf * HALF + t * 4096 + (((8 * c + 4 + lh) ^ li) << 4));
                    kh[t][c] = *reinterpret_cast<const f16x8 *>(ks + buf * HALF + t * 4096 + (((8 * c + lh) ^ li) << 4));
                }
        };
        // S^T = K . Q^T in six rounds of independent products, the small ones
        // first: only the last two additions round at the size of the score.
        auto score_round = [&](auto ic, f32x4(&s)[KT][2]) {
            constexpr int i = decltype(ic)::value;
#pragma unroll
            for (int t = 0; t < KT; t++)
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    if constexpr (i == 0) s[t][u] = mfma16x16x32_f16(kl[t][0], qh[u][0], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
                    if constexpr (i == 1) s[t][u] = mfma16x16x32_f16(kh[t][0], ql[u][0], s[t][u]);
                    if constexpr (i == 2) s[t][u] = mfma16x16x32_f16(kl[t][1], qh[u][1], s[t][u]);
                    if constexpr (i == 3) s[t][u] = mfma16x16x32_f16(kh[t][1], ql[u][1], s[t][u]);
                    if constexpr (i == 4) s[t][u] = mfma16x16x32_f16(kh[t][0], qh[u][0], s[t][u]);
                    if constexpr (i == 5) s[t][u] = mfma16x16x32_f16(kh[t][1], qh[u][1], s[t][u]);
                }
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        using I4 = std::integral_constant<int, 4>;
        using I5 = std::integral_constant<int, 5>;

        // Step t: the scores of step t + 1 are formed while step t's become P (the
        // matrix cores and the VALU work side by side in one wave; without this
        // the waves of a CU pass through the same phase together), then P . V.
        // Nothing waits for LDS: V's fragments are read while the softmax runs,
        // and K's, for the scores of the next step, behind P . V.  So K is copied
        // three steps ahead of its use as P and V one.
        const int steps = (T + 127) / 128;
        copy_panels(Kh, 0, kgr, 0);
        copy_panels(Kh, min(1, steps - 1), kgr, HALF);
        copy_panels(Vh, 0, vgr, 2 * HALF);
        split_wait<8>();
        __builtin_amdgcn_s_barrier();
        // The codes are looked at here, so that nothing above waits for them.
        int e_score = fa.eq + fa.ek;
        if constexpr (OUT != AOut::Split) {
            e_score = split_code_exponent(cq) + split_code_exponent(ck);
            floats = cq == kSplitNonFinite || ck == kSplitNonFinite || cv == kSplitNonFinite ||
                     ((split_code_small(cq) || split_code_small(ck)) &&
                      __builtin_ldexpf(fa.scale_log2, e_score + 30) > kScoreBound);
            if (floats) {
                split_wait<0>();
                return;
            }
        }
        // Kept off zero and infinity: a masked score (-inf) stays -inf.
        const float scale = fminf(fmaxf(__builtin_ldexpf(fa.scale_log2, e_score), 0x1p-126f), 0x1p127f);
        f32x4 s0[KT][2], s1[KT][2];
        read_k(0);
        score_round(I0{}, s0);
        score_round(I1{}, s0);
        score_round(I2{}, s0);
        score_round(I3{}, s0);
        score_round(I4{}, s0);
        score_round(I5{}, s0);
        split_wait<4>();  // K of step 1
        __builtin_amdgcn_s_barrier();
        if (steps > 2) copy_panels(Kh, 2, kgr, 0);
        read_k(1);
        auto one_step = [&](int step, auto bufc, f32x4(&s)[KT][2], f32x4(&sn)[KT][2]) {
            constexpr int buf = decltype(bufc)::value;
            const int k0 = step * 128 + stream * PK;
            split_wait<0>();  // K of step + 2 and V of this step
            __builtin_amdgcn_s_barrier();
            if (step + 3 < steps) copy_panels(Kh, step + 3, kgr, (buf ^ 1) * HALF);
            if (step + 1 < steps) copy_panels(Vh, step + 1, vgr, (3 - buf) * HALF);
            // Rows 4 lh .. + 3 and 16 below, columns 16 df .. + 15.
            f16x8 vh[4], vl[4];
#pragma unroll
            for (int df = 0; df < 4; df++) {
                const char *p0 = vs + buf * HALF;
                const int gh = ((8 * (df / 2) + 2 * (df % 2) + vg0) ^ vx) << 4;
                const int gl = ((8 * (df / 2) + 4 + 2 * (df % 2) + vg0) ^ vx) << 4;
                const f16x4 h0 = read_tr(p0 + gh), h1 = read_tr(p0 + 4096 + gh);
                const f16x4 l0 = read_tr(p0 + gl), l1 = read_tr(p0 + 4096 + gl);
                vh[df] = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
                vl[df] = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
            }
            if (k0 + PK > T) {
#pragma unroll
                for (int t = 0; t < KT; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (k0 + 16 * t + 4 * lh + r >= T) s[t][0][r] = s[t][1][r] = -INFINITY;
            }
            // The exponents; raise the maximum where one passes the slack (a lane
            // checks its own keys; only then is it reduced over the query's four
            // lanes).
            f32x4 e[KT][2];
            float mx[2];
            auto exponents = [&](int u) {
                const float off = kPBits - (m[u] == -INFINITY ? 0.0f : m[u]);
#pragma unroll
                for (int t = 0; t < KT; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) e[t][u][r] = __builtin_fmaf(s[t][u][r], scale, off);
                float a = fmaxf(fmaxf(e[0][u][0], e[0][u][1]), e[0][u][2]);
                a = fmaxf(fmaxf(a, e[0][u][3]), e[1][u][0]);
                a = fmaxf(fmaxf(a, e[1][u][1]), e[1][u][2]);
                mx[u] = fmaxf(a, e[1][u][3]);
            };
            exponents(0);
            exponents(1);
            // (Before any key was seen the maximum is -inf and always raised.)
            if (__any(fmaxf(mx[0], mx[1]) > kPBits + kMaxSlack || m[0] == -INFINITY)) {
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const float base = m[u] == -INFINITY ? 0.0f : m[u];
                    const float mn = fmaxf(m[u], max_groups(mx[u]) - kPBits + base);
                    // -inf only while no key was seen: then nothing to correct.
                    const float corr = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m[u] - mn);
                    m[u] = mn;
                    l[u] *= corr;
#pragma unroll
                    for (int df = 0; df < 4; df++) o[df][u] *= corr;
                    exponents(u);
                }
            }
            f16x8 ph[2], pl[2];
            float sum[2];
            auto softmax_part = [&](int u, int t) {
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; r++) p[r] = __builtin_amdgcn_exp2f(e[t][u][r]);
                const float four = (p[0] + p[1]) + (p[2] + p[3]);
                sum[u] = t == 0 ? four : sum[u] + four;
#pragma unroll
                for (int r = 0; r < 4; r += 2) {
                    const f16x2 hi = cvt_pk_f16(p[r], p[r + 1]), lo = residual_pk_f16(hi, p[r], p[r + 1]);
                    ph[u][4 * t + r] = hi[0];
                    ph[u][4 * t + r + 1] = hi[1];
                    pl[u][4 * t + r] = lo[0];
                    pl[u][4 * t + r + 1] = lo[1];
                }
            };
            // A round of four products with a quarter of the softmax between them.
            auto mixed = [&] {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x402, 5, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            __builtin_amdgcn_sched_barrier(0);
            score_round(I0{}, sn);
            softmax_part(0, 0);
            mixed();
            score_round(I1{}, sn);
            softmax_part(0, 1);
            mixed();
            score_round(I2{}, sn);
            softmax_part(1, 0);
            mixed();
            score_round(I3{}, sn);
            softmax_part(1, 1);
            mixed();
            score_round(I4{}, sn);
            score_round(I5{}, sn);
            l[0] += sum[0];
            l[1] += sum[1];
            __builtin_amdgcn_sched_barrier(0);
            read_k(buf);  // of step + 2; past the last step: not used
            auto each = [&](auto f) {
#pragma unroll
                for (int df = 0; df < 4; df++)
#pragma unroll
                    for (int u = 0; u < 2; u++) o[df][u] = f(df, u, o[df][u]);
            };
            each([&](int df, int u, f32x4 c) { return mfma16x16x32_f16(vl[df], ph[u], c); });
            each([&](int df, int u, f32x4 c) { return mfma16x16x32_f16(vh[df], pl[u], c); });
            each([&](int df, int u, f32x4 c) { return mfma16x16x32_f16(vh[df], ph[u], c); });
        };
        for (int step = 0; step < steps; step += 2) {
            one_step(step, I0{}, s0, s1);
            if (step + 1 < steps) one_step(step + 1, I1{}, s1, s0);
        }

        split_wait<0>();
    };

    // The key streams of a query group are merged through LDS in stream
    // order; stream s finishes the output dims of fragments [s * 4 / KS, ...).
    constexpr int DF = 4 / KS;
    f32x4 *xo = reinterpret_cast<f32x4 *>(smem_c);                   // [wave][8][64]
    float4 *xm = reinterpret_cast<float4 *>(smem_c + 8 * 8 * 64 * 16);  // [wave][64]
    // Q8: a block of 32 dims is finished by two streams (16 dims each); their
    // largest magnitudes meet in LDS.
    static_assert(OUT != AOut::Q8 || DF == 1, "two streams per Q8_0 block");
    float *xq = reinterpret_cast<float *>(smem_c + 8 * 8 * 64 * 16 + 8 * 64 * 16);  // [wave][2][16]
    int *xlow = reinterpret_cast<int *>(xq + 8 * 2 * 16);  // set: outputs too small
    f32x4 out[2][DF];
    auto merge = [&] {
        l[0] = sum_groups(l[0]);
        l[1] = sum_groups(l[1]);
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int df = 0; df < 4; df++)
#pragma unroll
            for (int u = 0; u < 2; u++) xo[(wave * 8 + df * 2 + u) * 64 + lane] = o[df][u];
        xm[wave * 64 + lane] = make_float4(m[0], m[1], l[0], l[1]);
        if (tid == 0) *xlow = 0;
        __syncthreads();
        float ms[KS][2], ls[KS][2];
#pragma unroll
        for (int z = 0; z < KS; z++) {
            const float4 t = xm[(z * QG + qg) * 64 + lane];
            ms[z][0] = t.x;
            ms[z][1] = t.y;
            ls[z][0] = t.z;
            ls[z][1] = t.w;
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            float mm = ms[0][u];
#pragma unroll
            for (int z = 1; z < KS; z++) mm = fmaxf(mm, ms[z][u]);
            float w[KS], lsum = 0.0f;
#pragma unroll
            for (int z = 0; z < KS; z++) {
                w[z] = __builtin_amdgcn_exp2f(ms[z][u] - mm);  // 0 for a stream without keys
                lsum += w[z] * ls[z][u];
            }
            const float inv = 1.0f / lsum;
#pragma unroll
            for (int i = 0; i < DF; i++) {
                const int df = stream * DF + i;
                f32x4 r = w[0] * xo[(qg * 8 + df * 2 + u) * 64 + lane];
#pragma unroll
                for (int z = 1; z < KS; z++) r += w[z] * xo[((z * QG + qg) * 8 + df * 2 + u) * 64 + lane];
                out[u][i] = r * inv;
            }
        }
    };
    // Marks in LDS if a query's or a dim's outputs are too small for the halves,
    // each stream looking at the dims it finishes (a query, if at least four
    // of them are real, at the first stream's anyway).
    auto mark_small = [&] {
        // Nearly always every lane's own values settle it (12 x 865 from floats 26.9
        // -> 26.3 us with this, the Q8_0 block at 865 tokens 99.1 -> 98.6).
        bool low = false;
#pragma unroll
        for (int i = 0; i < DF; i++) {
            const f32x4 v0 = out[0][i], v1 = out[1][i];
#pragma unroll
            for (int e = 0; e < 4; e++) low |= !(fmaxf(fabsf(v0[e]), fabsf(v1[e])) >= kDimFloor);
            low |= !(fmaxf(fmaxf(fabsf(v0[0]), fabsf(v0[1])), fmaxf(fabsf(v0[2]), fabsf(v0[3]))) >= kRowFloor);
            low |= !(fmaxf(fmaxf(fabsf(v1[0]), fabsf(v1[1])), fmaxf(fabsf(v1[2]), fabsf(v1[3]))) >= kRowFloor);
        }
        if (!__any(low)) return;
        low = false;
#pragma unroll
        for (int i = 0; i < DF; i++) {
            const int d0 = 16 * (stream * DF + i), queries = T - (q0 + qg * 32);
            const float dim_floor = queries >= 4 ? kDimFloor : kDimFloor * 0x1p-8f;
            f32x4 dim{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const bool real = q0 + qg * 32 + 16 * u + li < T;
                const f32x4 v = out[u][i];
                // (Dims past hd are zeros.)
                const float row = max_groups(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
                low |= real && (d0 + 4 <= fa.hd || d0 == 0) && row < kRowFloor;
#pragma unroll
                for (int e = 0; e < 4; e++) dim[e] = fmaxf(dim[e], real ? fabsf(v[e]) : 0.0f);
            }
            if (split_code_small(cv) && queries > 0)
#pragma unroll
                for (int e = 0; e < 4; e++) low |= d0 + 4 * lh + e < fa.hd && max_row16(dim[e]) < dim_floor;
        }
        if (low) *xlow = 1;
    };
    int ev = OUT == AOut::Split ? fa.ev : split_code_exponent(cv);
    auto store = [&] {
        f32x4 q8v[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int query = q0 + qg * 32 + 16 * u + li;
            if constexpr (OUT == AOut::Split) {
                if (query >= T) continue;
#pragma unroll
                for (int i = 0; i < DF; i++) {
                    const int df = stream * DF + i;
                    const f32x4 r = out[u][i];
                    const f16x2 h0 = cvt_pk_f16(r[0], r[1]), h1 = cvt_pk_f16(r[2], r[3]);
                    const f16x2 l0 = residual_pk_f16(h0, r[0], r[1]), l1 = residual_pk_f16(h1, r[2], r[3]);
                    char *dst = fa.out_split + (((size_t)img * T + query) * fa.heads + head) * 256 + (df / 2) * 128 +
                                (df % 2) * 32 + lh * 8;
                    *reinterpret_cast<f16x4 *>(dst) = __builtin_shufflevector(h0, h1, 0, 1, 2, 3);
                    *reinterpret_cast<f16x4 *>(dst + 64) = __builtin_shufflevector(l0, l1, 0, 1, 2, 3);
                }
            } else if constexpr (OUT == AOut::Q8) {
                float amax = 0.0f;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    q8v[u][e] = __builtin_ldexpf(out[u][0][e], ev);
                    amax = q8_absmax(amax, q8v[u][e]);
                }
                amax = q8_absmax(amax, __shfl_xor(amax, 16, kWave));
                amax = q8_absmax(amax, __shfl_xor(amax, 32, kWave));
                if (lh == 0) xq[(wave * 2 + u) * 16 + li] = amax;
            } else {
                if (query >= T) continue;
#pragma unroll
                for (int i = 0; i < DF; i++) {
                    const int d = 16 * (stream * DF + i) + 4 * lh;
                    float *dst = fa.token_major
                                     ? fa.out + (((size_t)img * T + query) * fa.heads + head) * fa.hd + d
                                     : fa.out + off + (size_t)query * fa.hd + d;
                    f32x4 v;
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = __builtin_ldexpf(out[u][i][e], ev);
                    if ((fa.hd & 3) == 0) {
                        if (d < fa.hd) *reinterpret_cast<f32x4 *>(dst) = v;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (d + e < fa.hd) dst[e] = v[e];
                    }
                }
            }
        }
        if constexpr (OUT == AOut::Q8) {
            __syncthreads();
            const size_t rows = (size_t)(fa.bh / fa.heads) * T;
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int query = q0 + qg * 32 + 16 * u + li;
                const int other = (stream ^ 1) * QG + qg;
                float d, inv;
                q8_scale(fmaxf(xq[(wave * 2 + u) * 16 + li], xq[(other * 2 + u) * 16 + li]), d, inv);
                if (query >= T) continue;
                uint32_t w = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) w |= (uint32_t)(q8_value(q8v[u][e], inv) & 0xff) << (8 * e);
                const size_t slot = (size_t)(head * 2 + stream / 2) * rows + (size_t)img * T + query;
                *reinterpret_cast<uint32_t *>(fa.q8_qs + slot * 32 + (stream & 1) * 16 + 4 * lh) = w;
                if (lh == 0 && (stream & 1) == 0) fa.q8_d[slot] = __builtin_bit_cast(uint16_t, (_Float16)d);
            }
        }
    };
    split_pass();
    if (!floats) {
        merge();
        if constexpr (OUT != AOut::Split) {
            // The mark is read behind a barrier, for Q8_0 rows their own.  (Floats
            // are stored after it: they may go where the queries are.)
            mark_small();
            if constexpr (OUT == AOut::Q8) store();
            else __syncthreads();
            floats = *xlow != 0;
        }
    }
    if constexpr (OUT != AOut::Split) {
        if (floats) {
            float_pass(fa, off, q0 + qg * 32, stream, lane, o, m, l);
            merge();
            ev = 0;
            if constexpr (OUT == AOut::Q8) store();
        }
    }
    if constexpr (OUT != AOut::Q8) store();
}

// Largest magnitude (as bits) of n floats, over a workgroup of NT threads
// (valid in every thread), and the least key (split_gemm.h): of all of them, or
// of share 0 .. 3 where the other workgroups of a head take the other shares.
// Four 16-byte loads per thread in flight where the run is 16-byte aligned.
struct Range {
    uint32_t most, least;
};
template <int NT>
__device__ __forceinline__ Range block_range(const float *__restrict__ src, size_t n, int share) {
    Range a{0u, ~0u};
    auto least4 = [&](f32x4 v) {
#pragma unroll
        for (int r = 0; r < 4; r++) a.least = min(a.least, small_key(v[r]));
    };
    size_t i = threadIdx.x;
    if ((reinterpret_cast<uintptr_t>(src) & 15) == 0) {
        const f32x4 *s4 = reinterpret_cast<const f32x4 *>(src);
        const size_t n4 = n / 4;
        for (; i + 3 * NT < n4; i += 4 * NT) {
            const f32x4 v[4] = {s4[i], s4[i + NT], s4[i + 2 * NT], s4[i + 3 * NT]};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                a.most = absmax4(a.most, v[j]);
                if (share < 0 || share == j) least4(v[j]);
            }
        }
        for (; i < n4; i += NT) {
            const f32x4 v = s4[i];
            a.most = absmax4(a.most, v);
            least4(v);
        }
        i = 4 * n4 + threadIdx.x;
    }
    for (; i < n; i += NT) {
        a.most = max(a.most, __float_as_uint(src[i]) & 0x7fffffffu);
        a.least = min(a.least, small_key(src[i]));
    }
    a.most = wave_umax(a.most);
    a.least = ~wave_umax(~a.least);
    __shared__ Range red[NT / 64];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NT / 64; w++) {
        a.most = max(a.most, red[w].most);
        a.least = min(a.least, red[w].least);
    }
    return a;
}

// The range of each chunk of a head's floats: grid (chunks, bh, 3), part
// [3][bh][chunks].
__global__ __launch_bounds__(256) void attn_range_kernel(const float *__restrict__ q, const float *__restrict__ k,
                                                         const float *__restrict__ v, Range *__restrict__ part,
                                                         size_t head_floats) {
    const float *src = (blockIdx.z == 0 ? q : (blockIdx.z == 1 ? k : v)) + (size_t)blockIdx.y * head_floats;
    const size_t per = ((head_floats + gridDim.x - 1) / gridDim.x + 3) & ~(size_t)3;
    const size_t lo = min(blockIdx.x * per, head_floats), hi = min(lo + per, head_floats);
    const Range a = block_range<256>(src + lo, hi - lo, -1);
    if (threadIdx.x == 0) part[((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = a;
}

// Split rows of Q, K and V with one exponent per head, rows of hd floats
// widened to 64 with zeros, and the head's codes: grid (workgroups, bh, 3), 16
// lanes per row.  The head's range comes from attn_range_kernel's chunks, or,
// with part == nullptr, each of at most kCodes workgroups takes the largest
// magnitude over the whole head itself, looks for small values in its share
// (or, if there are fewer, everywhere) and stores its own codes.
template <int NT>
__global__ __launch_bounds__(NT) void attn_split_rows_kernel(const float *__restrict__ q,
                                                             const float *__restrict__ k,
                                                             const float *__restrict__ v,
                                                             const Range *__restrict__ part, int chunks,
                                                             char *__restrict__ out, int *__restrict__ ex, int T,
                                                             int hd) {
    const int bh = blockIdx.y, BH = gridDim.y, z = blockIdx.z;
    const float *src = (z == 0 ? q : (z == 1 ? k : v)) + (size_t)bh * T * hd;
    Range a{0u, ~0u};
    if (part)
        for (int c = 0; c < chunks; c++) {
            const Range b = part[((size_t)z * BH + bh) * chunks + c];
            a = Range{max(a.most, b.most), min(a.least, b.least)};
        }
    else
        a = block_range<NT>(src, (size_t)T * hd, gridDim.x == 4 ? (int)blockIdx.x : -1);
    const int e = split_exponent(a.most);
    static_assert(kCodes == 4, "as many as shares");
    const int code = e == kSplitNonFinite ? e : split_code(e, a.least < small_limit(e));
    if (threadIdx.x == 0)
        for (int i = blockIdx.x; i < kCodes; i += part ? 1 : gridDim.x) ex[(z * BH + bh) * kCodes + i] = code;
    if (e == kSplitNonFinite) return;
    char *dst = out + ((size_t)z * BH + bh) * T * 256;
    const int d = 4 * (threadIdx.x & 15);
    const bool vec = (hd & 3) == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0;
    for (int row = blockIdx.x * (NT / 16) + (threadIdx.x >> 4); row < T; row += gridDim.x * (NT / 16)) {
        f32x4 x{0.0f, 0.0f, 0.0f, 0.0f};
        if (vec) {
            if (d < hd) x = *reinterpret_cast<const f32x4 *>(src + (size_t)row * hd + d);
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (d + r < hd) x[r] = src[(size_t)row * hd + d + r];
        }
        f32x4 y;
#pragma unroll
        for (int r = 0; r < 4; r++) y[r] = __builtin_ldexpf(x[r], -e);
        const f16x2 h0 = cvt_pk_f16(y[0], y[1]), h1 = cvt_pk_f16(y[2], y[3]);
        const f16x2 l0 = residual_pk_f16(h0, y[0], y[1]), l1 = residual_pk_f16(h1, y[2], y[3]);
        char *p = dst + (size_t)row * 256 + (d / 32) * 128 + (d % 32) * 2;
        *reinterpret_cast<f16x4 *>(p) = __builtin_shufflevector(h0, h1, 0, 1, 2, 3);
        *reinterpret_cast<f16x4 *>(p + 64) = __builtin_shufflevector(l0, l1, 0, 1, 2, 3);
    }
}

template <AOut OUT>
hipError_t run_attn(hipStream_t s, AttnArgs fa) {
    constexpr size_t lds = 4 * 128 * 256;  // two steps of K and of V panels
    static_assert(lds >= 8 * 8 * 64 * 16 + 8 * 64 * 16 + 8 * 2 * 16 * 4 + 4, "the merge fits the panels' LDS");
    auto kernel = attn_split_kernel<OUT>;
    static std::atomic<uint64_t> configured{0};
    if (hipError_t e = ensure_dynamic_lds(kernel, lds, configured); e != hipSuccess) return e;
    fa.qtiles = (fa.T + QG * 32 - 1) / (QG * 32);
    const int total = fa.bh * fa.qtiles;
    kernel<<<(unsigned)((total + 7) / 8 * 8), 512, lds, s>>>(fa);
    return hipGetLastError();
}

constexpr int kRangeChunks = 16;

}  // namespace

bool attn_split_fits(size_t bh, size_t tokens) {
    // 32-bit row offsets of a head, and the grid of 64-query tiles.
    return bh > 0 && bh <= 65535 && tokens > 0 && tokens <= ((size_t)1 << 23) - 256 &&
           bh * ((tokens + 63) / 64) <= (size_t)INT32_MAX / 1024;
}

// From floats the split costs a launch of its own (10 us at 12 x 865), so it needs
// enough keys to earn that, and enough workgroups that the fp32 kernels' key
// splits no longer fill the idle CUs.  Both forms at head_dim 64 on MI355X (us a
// call, fp32 and split): 12 x 193 9 and 14, 12 x 384 12 and 17, 12 x 505 18 and
// 20, 24 x 384 19 and 20, 48 x 350 34 and 39, 1 x 3457 42 and 55; 12 x 600 23 and
// 22, 12 x 865 33 and 27, 24 x 420 28 and 25, 8 x 700 22 and 23, 48 x 560 63 and
// 52, 12 x 3457 332 and 159.  Three or five tiles of 64 keys the fp32 kernels do
// not split evenly: 12 x 150 14 and 14, 12 x 300 20 and 16, but 48 x 150 18 and
// 21.  Narrower heads have padding launches on that side (8 x 500 x 40 23 and 17,
// 2 x 64 x 16 21 and 11).
bool attn_split_pays(size_t bh, size_t tokens, size_t hd) {
    if (hd < 64) return true;
    const double rows = (double)bh * (double)tokens;
    const size_t tiles = (tokens + 63) / 64;
    if ((tiles == 3 || tiles == 5) && bh * tiles <= 128) return true;
    if (tokens <= 512 && bh * tiles > 256) return false;
    return rows >= 4800.0 && rows * (double)tokens >= 3.5e6;
}

size_t attn_split_bytes(size_t bh, size_t tokens) {
    return 3 * bh * tokens * 256 + 3 * bh * (kRangeChunks * sizeof(Range) + kCodes * sizeof(int));
}

hipError_t launch_attn_split_f32(hipStream_t s, const float *q, const float *k, const float *v, float *out,
                                 size_t bh, size_t tokens, size_t heads, size_t hd, bool token_major,
                                 float softmax_scale, void *ws, int8_t *q8_qs, uint16_t *q8_d) {
    if (bh == 0 || tokens == 0) return hipSuccess;
    if (!attn_split_fits(bh, tokens) || hd == 0 || hd > 64) return hipErrorInvalidValue;
    if (q8_qs && (hd != 64 || !q8_d || heads == 0 || bh % heads != 0)) return hipErrorInvalidValue;
    char *planes = static_cast<char *>(ws);
    const size_t each = bh * tokens * 256;
    int *ex = reinterpret_cast<int *>(planes + 3 * each);
    Range *part = reinterpret_cast<Range *>(ex + 3 * bh * kCodes);
    const size_t head_floats = tokens * hd;
    // Heads of up to 64 K floats (1024 tokens): one launch whose workgroups
    // each read the whole head for its largest magnitude, from the cache past
    // the first (12 x 865 x 64: 10 us; two launches 13.4).  Longer heads take
    // it in a launch of its own.
    if (head_floats <= 65536) {
        const unsigned wgs = (unsigned)std::min<size_t>((tokens + 63) / 64, kCodes);
        attn_split_rows_kernel<1024><<<dim3(wgs, (unsigned)bh, 3), 1024, 0, s>>>(q, k, v, nullptr, 0, planes, ex,
                                                                                (int)tokens, (int)hd);
    } else {
        attn_range_kernel<<<dim3(kRangeChunks, (unsigned)bh, 3), 256, 0, s>>>(q, k, v, part, head_floats);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        const unsigned wgs = (unsigned)std::min<size_t>((tokens + 31) / 32, 64);
        attn_split_rows_kernel<256><<<dim3(wgs, (unsigned)bh, 3), 256, 0, s>>>(
            q, k, v, part, kRangeChunks, planes, ex, (int)tokens, (int)hd);
    }
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    AttnArgs fa{};
    fa.q = planes;
    fa.k = planes + each;
    fa.v = planes + 2 * each;
    fa.ex = ex;
    fa.qf = q;
    fa.kf = k;
    fa.vf = v;
    fa.T = (int)tokens;
    fa.heads = (int)heads;
    fa.bh = (int)bh;
    fa.hd = (int)hd;
    fa.scale_log2 = softmax_scale * kLog2e;
    fa.out = out;
    fa.token_major = token_major ? 1 : 0;
    fa.q8_qs = q8_qs;
    fa.q8_d = q8_d;
    return q8_qs ? run_attn<AOut::Q8>(s, fa) : run_attn<AOut::F32>(s, fa);
}

hipError_t launch_attn_split(hipStream_t s, const SplitQkv &p, void *out_split, size_t bh, size_t tokens,
                             size_t heads) {
    if (bh == 0 || tokens == 0) return hipSuccess;
    if (!attn_split_fits(bh, tokens)) return hipErrorInvalidValue;
    AttnArgs fa{};
    fa.q = static_cast<const char *>(p.q);
    fa.k = static_cast<const char *>(p.k);
    fa.v = static_cast<const char *>(p.v);
    fa.eq = p.eq;
    fa.ek = p.ek;
    fa.ev = p.ev;
    fa.T = (int)tokens;
    fa.heads = (int)heads;
    fa.bh = (int)bh;
    fa.hd = 64;
    fa.scale_log2 = 0.125f * kLog2e;
    fa.out_split = static_cast<char *>(out_split);
    return run_attn<AOut::Split>(s, fa);
}

}  // namespace vh
