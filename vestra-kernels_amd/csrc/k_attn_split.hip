// Online-softmax attention on the f16 matrix cores, on split rows
// (split_gemm.h): head_dim 64, any scale.
//
// Q, K and V are split rows [bh][tokens] of 256 bytes (two slices of 32
// dims, hi then lo), each tensor with one exponent per head or one for all.
// A workgroup of eight waves owns QG * 32 queries of one head; QG groups of
// waves each take 32 of the queries and KS = 8 / QG key streams share the
// keys: of every step's 128 keys stream s takes PK = 128 / KS.  K and V
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
// Error against float64 at 12 x 865 x 64, N(0, 1): 2.5e-7, against 4.3e-7 of the
// fp32 matrix instructions.  Time on split rows (kernel trace): 12 x 865 18 us
// against 28 (fp32 matrix instructions), 48 x 865 54 against 100, 12 x 3457
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

struct AttnArgs {
    const char *q, *k, *v;        // split rows [bh][T][256 bytes]
    const int *ex;                // [3][bh] exponents of q, k, v, or null:
    int eq, ek, ev;               // these for every head
    const float *qf, *kf, *vf;    // the float rows [bh][T][hd] (non-finite heads)
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

// A head with an infinity or NaN, in floats, one query per wave at a time:
// rare, so plain.  64 keys per step, one per lane; output dim `lane` (< hd).
__device__ __attribute__((noinline)) float attention_floats(const float *q, const float *k, const float *v, int T,
                                                            int hd, float scale_log2, int query, int lane) {
    float m = -INFINITY, l = 0.0f, o = 0.0f;
    for (int k0 = 0; k0 < T; k0 += 64) {
        const int key = k0 + lane;
        float s = -INFINITY;
        if (key < T) {
            s = 0.0f;
            for (int d = 0; d < hd; d++) s = fmaf(q[(size_t)query * hd + d], k[(size_t)key * hd + d], s);
            s *= scale_log2;
        }
        const float mn = fmaxf(m, wave_max(s)), ref = mn == -INFINITY ? 0.0f : mn;
        const float corr = __builtin_amdgcn_exp2f(m - ref), p = __builtin_amdgcn_exp2f(s - ref);
        l = l * corr + wave_sum(p);
        o *= corr;
        m = mn;
        for (int j = 0; j < min(64, T - k0); j++) {
            const float pj = __shfl(p, j, 64);
            if (lane < hd) o = fmaf(pj, v[(size_t)(k0 + j) * hd + lane], o);
        }
    }
    return o / l;
}

template <int QG, AOut OUT>
__global__ __launch_bounds__(512, 2) void attn_split_kernel(AttnArgs fa) {
    constexpr int KS = 8 / QG, PK = 128 / KS, KT = PK / 16;
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
    const int eq = fa.ex ? fa.ex[bh] : fa.eq, ek = fa.ex ? fa.ex[fa.bh + bh] : fa.ek;
    const int ev = fa.ex ? fa.ex[2 * fa.bh + bh] : fa.ev;
    const int img = bh / fa.heads, head = bh - img * fa.heads;

    if constexpr (OUT != AOut::Split) {
        if (eq == kSplitNonFinite || ek == kSplitNonFinite || ev == kSplitNonFinite) {
            const size_t off = (size_t)bh * T * fa.hd;
            for (int i = wave; i < QG * 32 && q0 + i < T; i += 8) {
                const float o =
                    attention_floats(fa.qf + off, fa.kf + off, fa.vf + off, T, fa.hd, fa.scale_log2, q0 + i, lane);
                if constexpr (OUT == AOut::Q8) {
                    float amax = q8_absmax(0.0f, o), d, inv;
#pragma unroll
                    for (int x = 1; x < 32; x *= 2) amax = q8_absmax(amax, __shfl_xor(amax, x, kWave));
                    q8_scale(amax, d, inv);
                    const size_t rows = (size_t)(fa.bh / fa.heads) * T;
                    const size_t slot = (size_t)(head * 2 + lane / 32) * rows + (size_t)img * T + q0 + i;
                    fa.q8_qs[slot * 32 + lane % 32] = (int8_t)q8_value(o, inv);
                    if (lane % 32 == 0) fa.q8_d[slot] = __builtin_bit_cast(uint16_t, (_Float16)d);
                } else {
                    float *orow = fa.token_major
                                      ? fa.out + (((size_t)img * T + q0 + i) * fa.heads + head) * fa.hd
                                      : fa.out + off + (size_t)(q0 + i) * fa.hd;
                    if (lane < fa.hd) orow[lane] = o;
                }
            }
            return;
        }
    }

    const char *Qh = fa.q + (size_t)bh * T * 256;
    const char *Kh = fa.k + (size_t)bh * T * 256;
    const char *Vh = fa.v + (size_t)bh * T * 256;
    // Kept off zero and infinity: a masked score (-inf) stays -inf.
    const float scale = fminf(fmaxf(__builtin_ldexpf(fa.scale_log2, eq + ek), 0x1p-126f), 0x1p127f);

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

    f32x4 o[4][2];  // o[df][t][r] = O[query tile t, li][16 df + 4 lh + r]
#pragma unroll
    for (int df = 0; df < 4; df++)
#pragma unroll
        for (int t = 0; t < 2; t++) o[df][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.0f, 0.0f};

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
    static_assert(KT == 2, "32 keys per stream and step");
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

    // The key streams of a query group are merged through LDS in stream
    // order; stream s finishes the output dims of fragments [s * 4 / KS, ...).
    l[0] = sum_groups(l[0]);
    l[1] = sum_groups(l[1]);
    split_wait<0>();
    __builtin_amdgcn_s_barrier();
    f32x4 *xo = reinterpret_cast<f32x4 *>(smem_c);                   // [wave][8][64]
    float4 *xm = reinterpret_cast<float4 *>(smem_c + 8 * 8 * 64 * 16);  // [wave][64]
#pragma unroll
    for (int df = 0; df < 4; df++)
#pragma unroll
        for (int u = 0; u < 2; u++) xo[(wave * 8 + df * 2 + u) * 64 + lane] = o[df][u];
    xm[wave * 64 + lane] = make_float4(m[0], m[1], l[0], l[1]);
    __syncthreads();
    constexpr int DF = 4 / KS;
    // Q8: a block of 32 dims is finished by two streams (16 dims each); their
    // largest magnitudes meet in LDS.
    static_assert(OUT != AOut::Q8 || DF == 1, "two streams per Q8_0 block");
    float *xq = reinterpret_cast<float *>(smem_c + 8 * 8 * 64 * 16 + 8 * 64 * 16);  // [wave][2][16]
    f32x4 q8v[2];
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
        const int query = q0 + qg * 32 + 16 * u + li;
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
        f32x4 r[DF];
#pragma unroll
        for (int i = 0; i < DF; i++) {
            const int df = stream * DF + i;
            r[i] = w[0] * xo[(qg * 8 + df * 2 + u) * 64 + lane];
#pragma unroll
            for (int z = 1; z < KS; z++) r[i] += w[z] * xo[((z * QG + qg) * 8 + df * 2 + u) * 64 + lane];
            r[i] *= inv;
        }
        if constexpr (OUT == AOut::Split) {
            if (query >= T) continue;
#pragma unroll
            for (int i = 0; i < DF; i++) {
                const int df = stream * DF + i;
                const f16x2 h0 = cvt_pk_f16(r[i][0], r[i][1]), h1 = cvt_pk_f16(r[i][2], r[i][3]);
                const f16x2 l0 = residual_pk_f16(h0, r[i][0], r[i][1]), l1 = residual_pk_f16(h1, r[i][2], r[i][3]);
                char *dst = fa.out_split + (((size_t)img * T + query) * fa.heads + head) * 256 + (df / 2) * 128 +
                            (df % 2) * 32 + lh * 8;
                *reinterpret_cast<f16x4 *>(dst) = __builtin_shufflevector(h0, h1, 0, 1, 2, 3);
                *reinterpret_cast<f16x4 *>(dst + 64) = __builtin_shufflevector(l0, l1, 0, 1, 2, 3);
            }
        } else if constexpr (OUT == AOut::Q8) {
            float amax = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                q8v[u][e] = __builtin_ldexpf(r[0][e], ev);
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
                                 : fa.out + ((size_t)bh * T + query) * fa.hd + d;
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = __builtin_ldexpf(r[i][e], ev);
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
}

// Largest magnitude (as bits) of n floats, over a workgroup of NT threads
// (valid in every thread); four 16-byte loads per thread in flight where the
// run is 16-byte aligned.
template <int NT>
__device__ __forceinline__ uint32_t block_absmax(const float *__restrict__ src, size_t n) {
    uint32_t mx = 0;
    size_t i = threadIdx.x;
    if ((reinterpret_cast<uintptr_t>(src) & 15) == 0) {
        const f32x4 *s4 = reinterpret_cast<const f32x4 *>(src);
        const size_t n4 = n / 4;
        for (; i + 3 * NT < n4; i += 4 * NT) {
            const f32x4 a = s4[i], b = s4[i + NT], c = s4[i + 2 * NT], d = s4[i + 3 * NT];
            mx = absmax4(absmax4(absmax4(absmax4(mx, a), b), c), d);
        }
        for (; i < n4; i += NT) mx = absmax4(mx, s4[i]);
        i = 4 * n4 + threadIdx.x;
    }
    for (; i < n; i += NT) mx = max(mx, __float_as_uint(src[i]) & 0x7fffffffu);
    mx = wave_umax(mx);
    __shared__ uint32_t red[NT / 64];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) mx = max(mx, red[w]);
    return mx;
}

// Largest magnitude of each chunk of a head's floats: grid (chunks, bh, 3),
// part [3][bh][chunks].
__global__ __launch_bounds__(256) void attn_absmax_kernel(const float *__restrict__ q, const float *__restrict__ k,
                                                          const float *__restrict__ v, uint32_t *__restrict__ part,
                                                          size_t head_floats) {
    const float *src = (blockIdx.z == 0 ? q : (blockIdx.z == 1 ? k : v)) + (size_t)blockIdx.y * head_floats;
    const size_t per = ((head_floats + gridDim.x - 1) / gridDim.x + 3) & ~(size_t)3;
    const size_t lo = min(blockIdx.x * per, head_floats), hi = min(lo + per, head_floats);
    const uint32_t mx = block_absmax<256>(src + lo, hi - lo);
    if (threadIdx.x == 0) part[((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = mx;
}

// Split rows of Q, K and V with one exponent per head, rows of hd floats
// widened to 64 with zeros: grid (workgroups, bh, 3), 16 lanes per row.  The
// head's largest magnitude comes from attn_absmax_kernel's chunks, or, with
// part == nullptr, every workgroup takes it over the whole head itself.
template <int NT>
__global__ __launch_bounds__(NT) void attn_split_rows_kernel(const float *__restrict__ q,
                                                             const float *__restrict__ k,
                                                             const float *__restrict__ v,
                                                             const uint32_t *__restrict__ part, int chunks,
                                                             char *__restrict__ out, int *__restrict__ ex, int T,
                                                             int hd) {
    const int bh = blockIdx.y, BH = gridDim.y, z = blockIdx.z;
    const float *src = (z == 0 ? q : (z == 1 ? k : v)) + (size_t)bh * T * hd;
    uint32_t mx = 0;
    if (part)
        for (int c = 0; c < chunks; c++) mx = max(mx, part[((size_t)z * BH + bh) * chunks + c]);
    else
        mx = block_absmax<NT>(src, (size_t)T * hd);
    const int e = split_exponent(mx);
    if (blockIdx.x == 0 && threadIdx.x == 0) ex[z * BH + bh] = e;
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

template <int QG, AOut OUT>
hipError_t run_attn(hipStream_t s, AttnArgs fa) {
    constexpr size_t lds = 4 * 128 * 256;  // two steps of K and of V panels
    static_assert(lds >= 8 * 8 * 64 * 16 + 8 * 64 * 16 + 8 * 2 * 16 * 4, "the merge fits the panels' LDS");
    auto kernel = attn_split_kernel<QG, OUT>;
    static std::atomic<uint64_t> configured{0};
    if (hipError_t e = ensure_dynamic_lds(kernel, lds, configured); e != hipSuccess) return e;
    fa.qtiles = (fa.T + QG * 32 - 1) / (QG * 32);
    const int total = fa.bh * fa.qtiles;
    kernel<<<(unsigned)((total + 7) / 8 * 8), 512, lds, s>>>(fa);
    return hipGetLastError();
}

template <AOut OUT>
hipError_t dispatch_attn(hipStream_t s, const AttnArgs &fa) {
    return run_attn<2, OUT>(s, fa);
}

constexpr int kAbsmaxChunks = 16;

}  // namespace

bool attn_split_fits(size_t bh, size_t tokens) {
    // 32-bit row offsets of a head, and the grid of 64-query tiles.
    return bh > 0 && bh <= 65535 && tokens > 0 && tokens <= ((size_t)1 << 23) - 256 &&
           bh * ((tokens + 63) / 64) <= (size_t)INT32_MAX / 1024;
}

size_t attn_split_bytes(size_t bh, size_t tokens) {
    return 3 * bh * tokens * 256 + 3 * bh * (kAbsmaxChunks + 1) * sizeof(int);
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
    uint32_t *part = reinterpret_cast<uint32_t *>(ex + 3 * bh);
    const size_t head_floats = tokens * hd;
    // Heads of up to 64 K floats (1024 tokens): one launch whose workgroups
    // each read the whole head for its largest magnitude, from the cache past
    // the first (12 x 865 x 64: 10 us; two launches 13.4).  Longer heads take
    // it in a launch of its own.
    if (head_floats <= 65536) {
        const unsigned wgs = (unsigned)std::min<size_t>((tokens + 63) / 64, 4);
        attn_split_rows_kernel<1024><<<dim3(wgs, (unsigned)bh, 3), 1024, 0, s>>>(q, k, v, nullptr, 0, planes, ex,
                                                                                (int)tokens, (int)hd);
    } else {
        attn_absmax_kernel<<<dim3(kAbsmaxChunks, (unsigned)bh, 3), 256, 0, s>>>(q, k, v, part, head_floats);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        const unsigned wgs = (unsigned)std::min<size_t>((tokens + 31) / 32, 64);
        attn_split_rows_kernel<256><<<dim3(wgs, (unsigned)bh, 3), 256, 0, s>>>(
            q, k, v, part, kAbsmaxChunks, planes, ex, (int)tokens, (int)hd);
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
    return q8_qs ? dispatch_attn<AOut::Q8>(s, fa) : dispatch_attn<AOut::F32>(s, fa);
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
    return dispatch_attn<AOut::Split>(s, fa);
}

}  // namespace vh
