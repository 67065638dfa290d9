// Projection GEMMs on split rows (split_gemm.h): C[m][n] = sum_k X[m][k] W[n][k],
// X the activation rows, W the weight rows, both k-contiguous.
//
// A workgroup owns a BM x BN tile; KG groups of WM x WN waves take every
// KG-th k-slice of 32 and sum their tiles in group order through LDS.  A
// slice (128 bytes per row) is copied straight into LDS (no registers, no
// LDS stores) through a ring of three stages: while the products of slice t
// run from registers, the fragments of slice t + 1 are read from LDS and
// slices t + 2 and t + 3 are in flight from L2 (t + 2 alone on the largest
// tile, whose ring is two stages).  One barrier per slice.  The granules of a
// row are XOR-swizzled by the row on the way in, so that a fragment read (16
// rows x 4 granules) touches every bank once per 256 bytes.  W is the A
// operand of the matrix instruction, so that a lane ends with four
// consecutive columns of one row and stores 16 bytes.
//
// What bounds it: at 3460 x 2304 x 768 the f16 matrix cores, whose clock
// drops to 1.7-1.9 GHz under this load (40.4 us, 910 TFLOP/s of f16 products; a
// register-only loop of the same instruction reaches 1.9 PFLOP/s on random
// data and 2.4 on zeros, an 8192^3 library product in f16 1.13 PFLOP/s); at 865
// rows the one round of tiles and its start and end (13.6 us for N = 2304
// against 28 on the fp32 matrix instructions, which are bound at 19.5).
//
// Error against float64 (2-norm, N(0, 1) rows times N(0, 0.02^2) weights):
// 1.5e-7 to 2.0e-7 at K = 768 and 2.6e-7 to 3.6e-7 at K = 3072 (3.2e-7 and
// 6.2e-7 on the 128 x 256 tile), against 2.5e-7 to 5.0e-7 and 5.8e-7 to
// 9.9e-7 of the fp32 matrix instructions.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "split_gemm.h"

namespace vh {
namespace {

struct SplitArgs {
    const char *x, *w;      // split rows of X [M][Kp] and W [N][Kp]
    const int *ex, *ew;     // row codes (ex null: exponent ex_c for every row)
    int ex_c;
    int M, N, slices;       // slices = Kp / 32
    // K pieces: a tile's slices are shared out over `pieces` workgroups, whose
    // tiles (in `partial`, [tile][piece][value][thread]) the last to finish
    // sums in piece order; piece_cnt counts a tile's arrivals, zero between
    // launches.
    int pieces;
    float *partial;  // null: whole tiles only
    unsigned *piece_cnt;
    const float *xf, *wf;   // the f32 rows [M][K], [N][K], or null
    int K, wf_n;            // wf_n: 0, or wf is [K][wf_n]
    float *c;
    const float *bias, *gamma;
    float *q, *k, *v;
    float qkv_scale[3];     // Qkv: 0 for floats, or split rows of the values times this
    int tokens, heads;
    const float *rot;
    // Conv: X is a zero-padded channel-last image of split rows, one per
    // pixel of its grid of width conv_wp, with the one exponent ex[0]; the
    // slices of W walk the taps (ky, kx), conv_cs channel slices each, and
    // row m of the product reads image row m + ky * conv_wp + kx.  C^T goes to
    // c[n][y][x] for x < conv_ow (m = y * conv_wp + x), conv_plane floats a
    // channel.  xf is the CHW image [conv_cs * 32][conv_ih][conv_iw] and wf
    // [N][taps][channels], and conv_small [M] the small values of each
    // output's window.
    const int *conv_small;
    int conv_cs, conv_kw, conv_wp, conv_ow, conv_ih, conv_iw, conv_pad, conv_relu;
    size_t conv_plane;
    char *out_split;        // GeluSplit: split rows [M][N] of the output times out_scale
    float out_scale;
};

constexpr int kSplitMaxPieces = 4;

enum class SEpi : int { Store, Gelu, Residual, Qkv, GeluSplit, Chw, Conv };

// ---- outputs recomputed in floats -------------------------------------------------
// The halves of a value below 2^-3 of the scaled row (a "small" one, at most 2^-17
// of the row's largest) are off by up to 2^-25, so n_x of them in a row of X and
// n_w in a row of W leave an error of at most (n_x + n_w) 2^-25 2^15 in a
// scaled product of the rows.  Where the product is at least 2^22 times
// that, it is right to the halves' own 2^-22; where it is less (the large
// values cancelled, or met zeros), it is formed again from the floats.
// Rows of ordinary data hold a small value once in a hundred (N(0, 1), K =
// 768), and then one product in 10^5 or so is that small.
constexpr float kSmallBound = 0x1p12f;
// Up to this many outputs of a wave's tile one at a time (2 us each), else the
// tile on the fp32 matrix instructions, at about their rate in the fp32 GEMM.
constexpr int kFewOutputs = 12;

// Convolution: the floats (tap, channel) k and on, N of one tap, of output m's
// window; 0 outside the image.
template <int N>
__device__ __forceinline__ void conv_values(const SplitArgs &ar, int m, int k, float (&v)[N]) {
    const int cin = ar.conv_cs * 32, t = k / cin, c = k - t * cin, y = m / ar.conv_wp;
    const int yy = y + t / ar.conv_kw - ar.conv_pad, xx = m - y * ar.conv_wp + t % ar.conv_kw - ar.conv_pad;
    const bool in = yy >= 0 && yy < ar.conv_ih && xx >= 0 && xx < ar.conv_iw;
#pragma unroll
    for (int e = 0; e < N; e++) {
        v[e] = in ? ar.xf[((size_t)(c + e) * ar.conv_ih + yy) * ar.conv_iw + xx] : 0.0f;
        if (ar.conv_relu) v[e] = fmaxf(v[e], 0.0f);
    }
}

// Output (m, n) by a whole wave (the same m and n in every lane).  A
// convolution's taps and channels are walked in steps of 64 channels of one tap,
// whose place is the same in every lane, instead of dividing every lane's k by
// the channels and the width (a DPT level at 24 x 36, mean of ten inputs, 133.7
// -> 133.0 us).
template <bool CONV>
__device__ __forceinline__ float float_dot(const SplitArgs &ar, int m, int n, int lane) {
    const float *w = ar.wf + (ar.wf_n ? (size_t)n : (size_t)n * ar.K);
    float s = 0.0f;
    if constexpr (CONV) {
        const int cin = ar.conv_cs * 32, steps = (ar.K / cin) * ((cin + 63) / 64);
        const int y = m / ar.conv_wp - ar.conv_pad, x = m % ar.conv_wp - ar.conv_pad;
        int c0 = 0, ky = 0, kx = 0;
#pragma unroll 8
        for (int i = 0; i < steps; i++) {
            const int c = min(c0 + lane, cin - 1), yy = y + ky, xx = x + kx;
            const bool in = yy >= 0 && yy < ar.conv_ih && xx >= 0 && xx < ar.conv_iw;
            float v = ar.xf[((size_t)c * ar.conv_ih + (in ? yy : 0)) * ar.conv_iw + (in ? xx : 0)];
            if (ar.conv_relu) v = fmaxf(v, 0.0f);
            const float wv = w[c];
            s = in && c0 + lane < cin ? fmaf(v, wv, s) : s;
            c0 += 64;
            if (c0 >= cin) {
                c0 = 0;
                w += cin;
                if (++kx == ar.conv_kw) {
                    kx = 0;
                    ky++;
                }
            }
        }
    } else {
        const size_t step = ar.wf_n ? (size_t)ar.wf_n : 1;
#pragma unroll 8
        for (int k = lane; k < ar.K; k += 64) s = fmaf(ar.xf[(size_t)m * ar.K + k], w[k * step], s);
    }
    return wave_sum(s);
}

// A wave's tile, FO x FN fragments of 16 x 16 in the layout of the split
// products: rows m = mb + 16 i (mb with the lane's row), columns from nb on.
// The 16 values of a step go to the lanes as k = k0 + 4 (lane / 16) + 0 .. 3.
template <int FO, int FN, bool CONV>
__device__ __forceinline__ void float_tile(const SplitArgs &ar, int mb, int nb, int lane, f32x4 (&out)[FO][FN]) {
    const int li = lane & 15, lh = lane >> 4;
    constexpr int D = 12 / (FO + FN) < 1 ? 1 : 12 / (FO + FN);  // steps loaded at once
    const bool vec = (ar.K & 3) == 0, xvec = vec && !CONV, wvec = vec && !ar.wf_n;
    auto four = [&](const float *p, size_t step, bool v16, int k) {
        f32x4 v{0.0f, 0.0f, 0.0f, 0.0f};
        if (v16) {
            if (k < ar.K) v = *reinterpret_cast<const f32x4 *>(p + k);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (k + e < ar.K) v[e] = p[(size_t)(k + e) * step];
        }
        return v;
    };
#pragma unroll
    for (int i = 0; i < FO; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) out[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int k0 = 0; k0 < ar.K; k0 += 16 * D) {
        f32x4 xv[D][FO], wv[D][FN];
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int k = k0 + 16 * d + 4 * lh;
#pragma unroll
            for (int i = 0; i < FO; i++) {
                const int m = min(mb + 16 * i, ar.M - 1);
                if constexpr (CONV) {
                    float v[4]{};
                    if (k < ar.K) conv_values(ar, m, k, v);
                    xv[d][i] = f32x4{v[0], v[1], v[2], v[3]};
                } else {
                    xv[d][i] = four(ar.xf + (size_t)m * ar.K, 1, xvec, k);
                }
            }
#pragma unroll
            for (int j = 0; j < FN; j++) {
                const size_t n = min(nb + 16 * j + li, ar.N - 1);
                wv[d][j] = four(ar.wf + (ar.wf_n ? n : n * ar.K), ar.wf_n ? ar.wf_n : 1, wvec, k);
            }
        }
#pragma unroll
        for (int d = 0; d < D; d++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int i = 0; i < FO; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++)
                        out[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[d][j][e], xv[d][i][e], out[i][j], 0, 0, 0);
    }
}

template <int BM, int BN, int WM, int WN, int KG, int ST, SEpi EPI, bool PIECES>
__global__ __launch_bounds__(WM *WN *KG * 64) void gemm_split_kernel(SplitArgs ar) {
    constexpr int NW = WM * WN, GT = NW * 64;
    constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;
    constexpr int ROWS = BM + BN;
    constexpr int CP = ROWS / 8;               // copies of 8 rows in a stage
    constexpr int LD = (CP + NW - 1) / NW;     // per wave; past CP the last one again
    constexpr int STAGE = ROWS * 128;
    static_assert(BM % 8 == 0 && BN % 8 == 0, "whole copies");
    static_assert(TM % 16 == 0 && TN % 16 == 0 && FM % KG == 0, "fragments");
    static_assert(ST == 2 || ST == 3, "a stage being filled besides the one being read");
    constexpr int FO = FM / KG;  // fragment rows (of 16 m) a K group finishes
    static_assert(EPI != SEpi::Qkv || TN % 32 == 0, "whole 32-wide RoPE halves per wave");
    extern __shared__ __attribute__((aligned(16))) char smem_c[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = KG == 1 ? 0 : wave / NW, gw = wave % NW;
    const int wm = gw / WN, wn = gw % WN;
    const int li = lane & 15, lh = lane >> 4;

    // Workgroups go round-robin over the 8 XCDs; renumbered so that an XCD's
    // share is a run of tiles that walks 8 row tiles column by column.
    const int nx = (ar.N + BN - 1) / BN, ny = (ar.M + BM - 1) / BM;
    int tm, tn, piece = 0, tile;
    {
        const int total = nx * ny * (PIECES ? ar.pieces : 1), bid = blockIdx.x;
        const int q = total / 8, r = total % 8, xcd = bid % 8;
        int t = xcd * q + min(xcd, r) + bid / 8;
        if constexpr (PIECES) {
            piece = t % ar.pieces;
            t /= ar.pieces;
        }
        tile = t;
        const int gm = min(8, ny), group = t / (gm * nx), first = group * gm;
        const int rows = min(ny - first, gm), local = t - group * gm * nx;
        tm = first + local % rows;
        tn = local / rows;
    }
    const int m0 = tm * BM, n0 = tn * BN;
    const size_t pitch = (size_t)ar.slices * 128;
    const size_t xpitch = EPI == SEpi::Conv ? (size_t)ar.conv_cs * 128 : pitch;
    const char *xb = ar.x + (size_t)m0 * xpitch, *wb = ar.w + (size_t)n0 * pitch;

    const int mb = m0 + wm * TM + kg * FO * 16 + li;  // this lane's first row of the epilogue

    // Copy i of this wave moves rows 8 b .. 8 b + 7 (b = i * NW + gw) of the
    // stage; LDS granule p of a row holds global granule p ^ (row % 8), so
    // that the 16 rows of a fragment read spread over all banks.
    uint32_t voff[LD];
#pragma unroll
    for (int i = 0; i < LD; i++) {
        const int b = min(i * NW + gw, CP - 1), row = b * 8 + lane / 8;
        const int r = row < BM ? min(row, ar.M - 1 - m0) : min(row - BM, ar.N - 1 - n0);
        voff[i] = (uint32_t)(r * (int)(row < BM ? xpitch : pitch) + (((lane & 7) ^ (lane >> 3)) << 4));
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem_c + kg * ST * STAGE;
    int conv_at = 0, conv_kin = 0, conv_kx = 0;  // Conv: the slice last copied and its place
    size_t conv_off = 0;
    auto copy_stage = [&](int slice, int buf) {
        const size_t ko = (size_t)slice * 128;
        size_t xo = ko;
        if constexpr (EPI == SEpi::Conv) {
            // Stages are copied in slice order: step to this one.
            while (conv_at < slice) {
                conv_at++;
                conv_off += 128;
                if (++conv_kin == ar.conv_cs) {
                    // conv_off now holds the next pixel: the next tap of the row.
                    conv_kin = 0;
                    if (++conv_kx == ar.conv_kw) {
                        conv_kx = 0;
                        conv_off += (size_t)(ar.conv_wp - ar.conv_kw) * xpitch;
                    }
                }
            }
            xo = conv_off;
        }
#pragma unroll
        for (int i = 0; i < LD; i++) {
            const int b = min(i * NW + gw, CP - 1);
            const char *base = b * 8 < BM ? xb + xo : wb + ko;
            copy16_to_lds(base, voff[i], __builtin_amdgcn_readfirstlane(lds0 + buf * STAGE + b * 1024));
        }
    };

    // The cross products hi.lo and lo.hi sum apart from hi.hi where there are
    // registers for it: their sum is 2^-11 of the other's, so only a third
    // of the additions round at full size (64 x 64 tiles,
    // error against float64 at K = 768: 2.4e-7 -> 1.5e-7).
    constexpr bool SEP = FM * FN <= 8;
    f32x4 acc[FM][FN], cross[SEP ? FM : 1][SEP ? FN : 1];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) {
            acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (SEP) cross[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    auto low = [&](int i, int j) -> f32x4 & {
        if constexpr (SEP) return cross[i][j];
        else return acc[i][j];
    };

    // Fragment i of X: row wm*TM + 16 i + li, hi granule lh, lo granule 4 + lh.
    const char *gs = smem_c + kg * ST * STAGE;
    const int ohi = (lh ^ (li & 7)) << 4, olo = ((4 + lh) ^ (li & 7)) << 4;
    f16x8 xh[2][FM], xl[2][FM], wh[2][FN], wl[2][FN];
    auto fetch = [&](int set, int buf) {
        const char *xs = gs + buf * STAGE + (wm * TM + li) * 128;
        const char *ws = gs + buf * STAGE + (BM + wn * TN + li) * 128;
#pragma unroll
        for (int i = 0; i < FM; i++) xh[set][i] = *reinterpret_cast<const f16x8 *>(xs + i * 2048 + ohi);
#pragma unroll
        for (int j = 0; j < FN; j++) wh[set][j] = *reinterpret_cast<const f16x8 *>(ws + j * 2048 + ohi);
#pragma unroll
        for (int j = 0; j < FN; j++) wl[set][j] = *reinterpret_cast<const f16x8 *>(ws + j * 2048 + olo);
#pragma unroll
        for (int i = 0; i < FM; i++) xl[set][i] = *reinterpret_cast<const f16x8 *>(xs + i * 2048 + olo);
    };
    // W is the A operand: a lane ends with four consecutive n of one m.
    auto products = [&](int set) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) acc[i][j] = mfma16x16x32_f16(wh[set][j], xh[set][i], acc[i][j]);
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) low(i, j) = mfma16x16x32_f16(wl[set][j], xh[set][i], low(i, j));
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) low(i, j) = mfma16x16x32_f16(wh[set][j], xl[set][i], low(i, j));
    };

    // Of the piece's slices [beg, beg + S) group kg takes every KG-th; every
    // group runs the same number of steps (barriers are workgroup-wide).
    int beg = 0, S = ar.slices;
    if constexpr (PIECES) {
        const int each = (ar.slices + ar.pieces - 1) / ar.pieces;
        beg = piece * each;
        S = min(each, ar.slices - beg);
    }
    const int steps = (S + KG - 1) / KG;
    auto slice_of = [&](int t) { return beg + min(kg + t * KG, S - 1); };
    copy_stage(slice_of(0), 0);
    copy_stage(slice_of(1), 1);
    if constexpr (ST == 3) copy_stage(slice_of(2), 2);
    split_wait<(ST - 1) * LD>();
    __builtin_amdgcn_s_barrier();
    fetch(0, 0);
    int window_small[EPI == SEpi::Conv ? FO : 1];  // landed by the time the loop ends
    if constexpr (EPI == SEpi::Conv)
#pragma unroll
        for (int i = 0; i < FO; i++) window_small[i] = ar.conv_small[min(mb + 16 * i, ar.M - 1)];
    // Step t: products of slice t (fragments in registers) while the
    // fragments of slice t + 1 are read; the buffer of slice t, whose reads
    // ended before this step's barrier, takes slice t + ST.  Copies past the
    // last slice reload it into a buffer that is not read again, so that
    // every step is the same basic block.
    auto step = [&](int t, auto setc, int buf) {
        constexpr int set = decltype(setc)::value;
        split_wait<(ST - 2) * LD>();  // slice t + 1 landed; of three, t + 2 may be in flight
        __builtin_amdgcn_s_barrier();
        copy_stage(slice_of(t + ST), buf);
        fetch(set ^ 1, buf == ST - 1 ? 0 : buf + 1);
        products(set);
        // Issue order: a fragment read behind each of the first products.
        constexpr int NR = 2 * (FM + FN), NM = 3 * FM * FN, PER = NM / NR < 1 ? 1 : (NM / NR > 2 ? 2 : NM / NR);
#pragma unroll
        for (int r = 0; r < NR; r++) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, NM, 0);
    };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    // A group without a slice for the last step (S % KG) leaves it out.
    const int mine = (S - kg + KG - 1) / KG;
    int buf = 0, t = 0;
    for (; t + 1 < mine; t += 2) {
        step(t, P0{}, buf);
        buf = buf == ST - 1 ? 0 : buf + 1;
        step(t + 1, P1{}, buf);
        buf = buf == ST - 1 ? 0 : buf + 1;
    }
    if (t < mine) {
        step(t, P0{}, buf);
        t++;
    }
    if (t < steps) __builtin_amdgcn_s_barrier();
    split_wait<0>();
    if constexpr (SEP) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) acc[i][j] += cross[i][j];
    }

    // The K groups' partial tiles are summed in group order through LDS:
    // group g finishes fragment rows [g * FO, (g + 1) * FO), in accs[0 .. FO).
    f32x4 fin[FO][FN];
    if constexpr (KG > 1) {
        __builtin_amdgcn_s_barrier();
        f32x4 *xch = reinterpret_cast<f32x4 *>(smem_c);
        const int gt = tid % GT;
        // [source group][fragment][thread]; a group leaves out its own rows.
#pragma unroll
        for (int i = 0; i < FM; i++)
            if (i / FO != kg)
#pragma unroll
                for (int j = 0; j < FN; j++) xch[((kg * FM + i) * FN + j) * GT + gt] = acc[i][j];
        __syncthreads();
#pragma unroll
        for (int o = 0; o < KG; o++) {
            if (o != kg) continue;
#pragma unroll
            for (int i = 0; i < FO; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    const int row = o * FO + i;
                    f32x4 sum = o == 0 ? acc[row][j] : xch[(row * FN + j) * GT + gt];
#pragma unroll
                    for (int g = 1; g < KG; g++) sum += g == o ? acc[row][j] : xch[((g * FM + row) * FN + j) * GT + gt];
                    fin[i][j] = sum;
                }
        }
    } else {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) fin[i][j] = acc[i][j];
    }

    if constexpr (PIECES) {
        // Publish, count in, and go on only as the last of the tile.  The
        // partials are agent-scope atomic stores, which write through the
        // XCD's L2 to where every XCD reads; each thread waits for its own to
        // be acknowledged (vmcnt counts stores; the asm's memory clobber keeps
        // them before it), the barrier orders those waits before thread 0's
        // increment, and the last piece reads with agent-scope atomic loads
        // after it.  No piece waits for another, so the grid drains at any
        // residency.
        constexpr int NT = NW * KG * 64, PER = FO * FN * 4;
        __shared__ int last_piece;
        float *base = ar.partial + (size_t)tile * ar.pieces * PER * NT + tid;
        float *mine = base + (size_t)piece * PER * NT;
#pragma unroll
        for (int i = 0; i < FO; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    __hip_atomic_store(mine + ((i * FN + j) * 4 + r) * NT, fin[i][j][r], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0)
            last_piece = __hip_atomic_fetch_add(ar.piece_cnt + tile, 1u, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(ar.pieces - 1);
        __syncthreads();
        if (!last_piece) return;
        if (tid == 0) __hip_atomic_store(ar.piece_cnt + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // Every load before the first sum, under a uniform branch per piece.
        float pv[kSplitMaxPieces][PER];
#pragma unroll
        for (int p = 0; p < kSplitMaxPieces; p++)
#pragma unroll
            for (int e = 0; e < PER; e++)
                pv[p][e] = p < ar.pieces ? __hip_atomic_load(base + ((size_t)p * PER + e) * NT, __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_AGENT)
                                         : 0.0f;
#pragma unroll
        for (int i = 0; i < FO; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int e = (i * FN + j) * 4 + r;
                    float v = pv[0][e];
#pragma unroll
                    for (int p = 1; p < kSplitMaxPieces; p++)
                        if (p < ar.pieces) v += pv[p][e];
                    fin[i][j][r] = v;
                }
    }

    // Epilogue: lane (li, lh) holds C[m][n .. n + 3], m = mb + 16 i, n = nb + 16 j.
    const int nb = n0 + wn * TN + 4 * lh;
    if (n0 + wn * TN >= ar.N) return;
    const bool vec = (ar.N & 3) == 0;
    int xcode[FO], wcode[FN][4];
    float bias[FN][4], gamma[FN][4];
#pragma unroll
    for (int i = 0; i < FO; i++)
        if constexpr (EPI == SEpi::Conv) xcode[i] = ar.ex[0] + split_code(-512, window_small[i]);
        else xcode[i] = ar.ex ? ar.ex[min(mb + 16 * i, ar.M - 1)] : split_code(ar.ex_c, 0);
#pragma unroll
    for (int j = 0; j < FN; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int cn = min(nb + 16 * j + r, ar.N - 1);
            wcode[j][r] = ar.ew[cn];
            bias[j][r] = load_or(ar.bias, reinterpret_cast<const float *>(ar.ew), cn, 0.0f);
            gamma[j][r] = load_or(ar.gamma, reinterpret_cast<const float *>(ar.ew), cn, 1.0f);
        }
    f32x4 old[EPI == SEpi::Residual ? FO : 1][FN];
    auto load_old = [&] {
        if constexpr (EPI == SEpi::Residual) {
            if (vec) {
#pragma unroll
                for (int i = 0; i < FO; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++)
                        old[i][j] = *reinterpret_cast<const f32x4 *>(
                            ar.c + (size_t)min(mb + 16 * i, ar.M - 1) * ar.N + min(nb + 16 * j, ar.N - 4));
            }
        }
    };
    // Early, behind what follows; on the largest tile its registers are needed.
    constexpr bool EARLY = FO * FN < 16;
    if constexpr (EARLY) load_old();
    // Qkv: the wave's columns lie in one head of one of Q, K, V.
    const int colw = n0 + wn * TN;
    float *head_dst = nullptr;
    float head_scale = 0.0f;
    bool rope = false;
    if constexpr (EPI == SEpi::Qkv) {
        const int per = ar.heads * 64, group = colw / per;
        head_dst = group == 0 ? ar.q : (group == 1 ? ar.k : ar.v);
        head_scale = group == 0 ? ar.qkv_scale[0] : (group == 1 ? ar.qkv_scale[1] : ar.qkv_scale[2]);
        rope = ar.rot != nullptr && group < 2;
    }
    // The products in their own scale, and from the floats where small values
    // may show (kSmallBound) or a value is not finite.  First the lane's least
    // product against its largest counts (a product of finite rows is no NaN; a
    // convolution's may be), then each of them.
    bool spoilt = false;
    float xs[FO], ws[FN][4];
#pragma unroll
    for (int i = 0; i < FO; i++)
        xs[i] = mb + 16 * i < ar.M ? (float)split_code_small(xcode[i]) * kSmallBound : -INFINITY;
#pragma unroll
    for (int j = 0; j < FN; j++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            ws[j][r] = nb + 16 * j + r < ar.N ? (float)split_code_small(wcode[j][r]) * kSmallBound : -INFINITY;
    if (ar.xf && ar.wf) {
        float least = INFINITY, nx = 0.0f, nw = 0.0f;
#pragma unroll
        for (int i = 0; i < FO; i++) nx = fmaxf(nx, xs[i]);
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                nw = fmaxf(nw, ws[j][r]);
#pragma unroll
                for (int i = 0; i < FO; i++) {
                    const float p = __builtin_fabsf(fin[i][j][r]);
                    if constexpr (EPI == SEpi::Conv) spoilt |= p != p;
                    least = fminf(least, p);
                }
            }
        spoilt |= least < nx + nw;
    }
    uint64_t bad = 0;  // of this lane, bit (i * FN + j) * 4 + r
    static_assert(FO * FN * 4 <= 64, "one bit per output");
    spoilt = __any(spoilt);
    // (The code of this and of what follows is seldom in the instruction cache,
    // so it is kept short: which outputs exist is only asked of the marked ones.
    // A DPT level at 24 x 36 133.0 -> 129.5 us, 128.8 without the checks.)
    if (spoilt) {
#pragma unroll
        for (int e = 0; e < FO * FN * 4; e++) {
            const int i = e / (4 * FN), j = e / 4 % FN, r = e % 4;
            if (!(__builtin_fabsf(fin[i][j][r]) >= xs[i] + ws[j][r])) bad |= (uint64_t)1 << e;
        }
    }
#pragma unroll
    for (int j = 0; j < FN; j++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int i = 0; i < FO; i++)
                fin[i][j][r] = __builtin_ldexpf(fin[i][j][r], split_code_exponent(xcode[i]) + split_code_exponent(wcode[j][r]));
    if (spoilt) {
        // The arguments are read again here, so that the loop above need not
        // hold those of this rare path, nor the registers of `old`.
        const auto *again = (const __attribute__((address_space(4))) SplitArgs *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(again));
        SplitArgs late;
        __builtin_memcpy(&late, (const void *)again, sizeof(late));
        if (wave_sum((float)__popcll(bad)) > (float)kFewOutputs) {
            float_tile<FO, FN, EPI == SEpi::Conv>(late, mb, nb - 4 * lh, lane, fin);
        } else {
            for (uint64_t lanes; (lanes = __ballot(bad != 0));) {
                const int src = (int)__ffsll((unsigned long long)lanes) - 1;
                const int bit = __builtin_amdgcn_readlane((int)__ffsll((unsigned long long)bad) - 1, src);
                const int m = __builtin_amdgcn_readlane(mb, src) + 16 * (bit / (4 * FN));
                const int n = __builtin_amdgcn_readlane(nb, src) + 16 * (bit / 4 % FN) + bit % 4;
                if (lane == src) bad &= bad - 1;
                if (m >= late.M || n >= late.N) continue;
                if constexpr (EPI == SEpi::Conv)
                    if (m % late.conv_wp >= late.conv_ow) continue;
                const float s = float_dot<EPI == SEpi::Conv>(late, m, n, lane);
                if (lane == src) {
#pragma unroll
                    for (int e = 0; e < FO * FN * 4; e++)
                        if (e == bit) fin[e / (4 * FN)][e / 4 % FN][e % 4] = s;
                }
            }
        }
        if constexpr (EARLY) load_old();
    }
    if constexpr (!EARLY) load_old();
#pragma unroll
    for (int i = 0; i < FO; i++) {
        const int m = mb + 16 * i;
        if (m >= ar.M) continue;
        float v[FN][4];
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float t = fin[i][j][r];
                if (ar.bias) t = add_rn(t, bias[j][r]);
                if constexpr (EPI == SEpi::Store || EPI == SEpi::Residual || EPI == SEpi::Chw)
                    if (ar.gamma) t = mul_rn(t, gamma[j][r]);
                if constexpr (EPI == SEpi::Gelu || EPI == SEpi::GeluSplit) t = gelu_fast_form(t);
                v[j][r] = t;
            }
        if constexpr (EPI == SEpi::Qkv) {
            const int img = m / ar.tokens, tok = m - img * ar.tokens;
#pragma unroll
            for (int jp = 0; jp < FN; jp += 2) {
                const int col = colw + jp * 16;       // a 32-wide half of a head
                const int head = (col % (ar.heads * 64)) / 64, d0 = col % 64;
                if (col >= ar.N) continue;
                if (rope) {
                    // rope::rotate_half (src/rope.rs:84-93): dims (d, d + 16) of
                    // the half are fragments (jp, jp + 1) of this lane.
                    const float *rp = ar.rot + (((size_t)tok * 2 + d0 / 32) * 16 + 4 * lh) * 2;
                    const f32x4 r0 = *reinterpret_cast<const f32x4 *>(rp);
                    const f32x4 r1 = *reinterpret_cast<const f32x4 *>(rp + 4);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float sn = r < 2 ? r0[2 * r] : r1[2 * r - 4], cs = r < 2 ? r0[2 * r + 1] : r1[2 * r - 3];
                        const float a = v[jp][r], b = v[jp + 1][r];
                        v[jp][r] = sub_rn(mul_rn(a, cs), mul_rn(b, sn));
                        v[jp + 1][r] = add_rn(mul_rn(b, cs), mul_rn(a, sn));
                    }
                }
                float *row = head_dst + (((size_t)img * ar.heads + head) * ar.tokens + tok) * 64;
                if (head_scale != 0.0f) {
                    // Split row of 256 bytes: slice d0 / 32, hi then lo.
                    char *sd = reinterpret_cast<char *>(row) + d0 * 4 + lh * 8;
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        f16x4 hi, lo;
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            _Float16 a, b;
                            split_f16(v[jp + h][r] * head_scale, a, b);
                            hi[r] = a;
                            lo[r] = b;
                        }
                        *reinterpret_cast<f16x4 *>(sd + 32 * h) = hi;
                        *reinterpret_cast<f16x4 *>(sd + 32 * h + 64) = lo;
                    }
                    continue;
                }
                float *dst = row + d0 + 4 * lh;
                *reinterpret_cast<f32x4 *>(dst) = f32x4{v[jp][0], v[jp][1], v[jp][2], v[jp][3]};
                *reinterpret_cast<f32x4 *>(dst + 16) =
                    f32x4{v[jp + 1][0], v[jp + 1][1], v[jp + 1][2], v[jp + 1][3]};
            }
        } else if constexpr (EPI == SEpi::GeluSplit) {
            // Split rows of the output, N % 32 == 0: one exponent for all.
#pragma unroll
            for (int j = 0; j < FN; j++) {
                const int n = nb + 16 * j;
                if (n >= ar.N) continue;
                f16x4 hi, lo;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    _Float16 h, l;
                    split_f16(v[j][r] * ar.out_scale, h, l);
                    hi[r] = h;
                    lo[r] = l;
                }
                char *dst = ar.out_split + ((size_t)m * (ar.N / 32) + n / 32) * 128 + (n % 32) * 2;
                *reinterpret_cast<f16x4 *>(dst) = hi;
                *reinterpret_cast<f16x4 *>(dst + 64) = lo;
            }
        } else {
#pragma unroll
            for (int j = 0; j < FN; j++) {
                const int n = nb + 16 * j;
                if (n >= ar.N) continue;
                if constexpr (EPI == SEpi::Conv) {
                    const int y = m / ar.conv_wp, x = m - y * ar.conv_wp;
                    if (x >= ar.conv_ow) continue;
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (n + r < ar.N)
                            ar.c[(size_t)(n + r) * ar.conv_plane + (size_t)y * ar.conv_ow + x] = v[j][r];
                } else if constexpr (EPI == SEpi::Chw) {
                    // C^T: 16 lanes store 16 consecutive rows of one channel.
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (n + r < ar.N) ar.c[(size_t)(n + r) * ar.M + m] = v[j][r];
                } else {
                    float *dst = ar.c + (size_t)m * ar.N + n;
                    if (vec) {
                        f32x4 o{v[j][0], v[j][1], v[j][2], v[j][3]};
                        if constexpr (EPI == SEpi::Residual)
#pragma unroll
                            for (int r = 0; r < 4; r++) o[r] = add_rn(old[i][j][r], v[j][r]);
                        *reinterpret_cast<f32x4 *>(dst) = o;
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            if (n + r < ar.N) dst[r] = EPI == SEpi::Residual ? add_rn(dst[r], v[j][r]) : v[j][r];
                    }
                }
            }
        }
    }
}

// Split rows of 32-bit float rows, one wave per row.  The row maximum is
// taken on the bit patterns (magnitude order, and a NaN sorts above every
// number), then each value is scaled by its exact power of two and split.
// Rows of up to 1024 values stay in registers between the two passes (the
// row is read once: 865 x 768 in 2.4 us); longer rows are read again, from
// the cache.
__device__ __forceinline__ void store_split4(char *row, int k, f32x4 v, int e) {
    f16x4 hi, lo;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        _Float16 h, l;
        split_f16(__builtin_ldexpf(v[r], -e), h, l);
        hi[r] = h;
        lo[r] = l;
    }
    char *p = row + (k / 32) * 128 + (k % 32) * 2;
    *reinterpret_cast<f16x4 *>(p) = hi;
    *reinterpret_cast<f16x4 *>(p + 64) = lo;
}

// The code of a row of exponent e of which each lane of a wave has found n
// small values.
__device__ __forceinline__ int wave_split_code(int e, int n) {
    if (e == kSplitNonFinite) return kSplitNonFinite;
    return split_code(e, __any(n) ? (int)wave_sum((float)n) : 0);
}

// One row of K floats to its split row, by one wave.
__device__ __forceinline__ void split_row(const float *__restrict__ src, char *__restrict__ dst, int *__restrict__ ex,
                                          int K, int slices, int lane) {
    const int Kp = slices * 32;
    uint32_t mx = 0, limit;
    int e, small = 0;
    const f32x4 zero{0.0f, 0.0f, 0.0f, 0.0f};
    if ((K & 3) == 0) {
        const f32x4 *src4 = reinterpret_cast<const f32x4 *>(src);
        const int n4 = K >> 2, np4 = Kp >> 2;
        if (K <= 1024) {
            f32x4 r[4];
#pragma unroll
            for (int j = 0; j < 4; j++) r[j] = lane + j * 64 < n4 ? src4[lane + j * 64] : zero;
#pragma unroll
            for (int j = 0; j < 4; j++) mx = absmax4(mx, r[j]);
            e = split_exponent(wave_umax(mx));
            limit = small_limit(e);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (lane + j * 64 < np4) store_split4(dst, 4 * (lane + j * 64), e == kSplitNonFinite ? zero : r[j], e);
                small += small_count4(r[j], limit);
            }
        } else {
            int c = lane;
            for (; c + 192 < n4; c += 256)
                mx = absmax4(absmax4(absmax4(absmax4(mx, src4[c]), src4[c + 64]), src4[c + 128]), src4[c + 192]);
            for (; c < n4; c += 64) mx = absmax4(mx, src4[c]);
            e = split_exponent(wave_umax(mx));
            limit = small_limit(e);
#pragma unroll 4
            for (c = lane; c < np4; c += 64) {
                const f32x4 v = c < n4 && e != kSplitNonFinite ? src4[c] : zero;
                small += small_count4(v, limit);
                store_split4(dst, 4 * c, v, e);
            }
        }
    } else {
        // Rows that are not 16-byte aligned: lane-consecutive floats, sixteen
        // loads in flight, in registers when the row has at most 1024.
        auto store1 = [&](int k, float v) {
            _Float16 h, l;
            split_f16(__builtin_ldexpf(v, -e), h, l);
            _Float16 *p = reinterpret_cast<_Float16 *>(dst + (k / 32) * 128) + k % 32;
            p[0] = h;
            p[32] = l;
        };
        float r[16];
        for (int k0 = 0; k0 < K; k0 += 1024) {
#pragma unroll
            for (int j = 0; j < 16; j++) r[j] = k0 + lane + 64 * j < K ? src[k0 + lane + 64 * j] : 0.0f;
#pragma unroll
            for (int j = 0; j < 16; j++) mx = max(mx, __float_as_uint(r[j]) & 0x7fffffffu);
        }
        e = split_exponent(wave_umax(mx));
        limit = small_limit(e);
        for (int k0 = 0; k0 < Kp; k0 += 1024) {
            if (K > 1024) {
#pragma unroll
                for (int j = 0; j < 16; j++) r[j] = k0 + lane + 64 * j < K ? src[k0 + lane + 64 * j] : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < 16; j++) {
                if (k0 + lane + 64 * j < Kp) store1(k0 + lane + 64 * j, e == kSplitNonFinite ? 0.0f : r[j]);
                small += small_key(r[j]) < limit;
            }
        }
    }
    const int code = wave_split_code(e, small);
    if (lane == 0) *ex = code;
}

__global__ __launch_bounds__(256) void split_rows_kernel(const float *__restrict__ in, char *__restrict__ out,
                                                         int *__restrict__ ex, size_t rows, int K, int slices) {
    const size_t row = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (row >= rows) return;
    split_row(in + row * K, out + row * slices * 128, ex + row, K, slices, threadIdx.x & 63);
}

// LayerNorm of each row straight into split rows (launch_layernorm's bits,
// then split): cols % 32 == 0, cols <= 1024, one wave per row.  A row whose
// normalised values hold a NaN (an infinity cannot arise without one in
// the statistics) is stored as NaN with exponent 0.  Small values are not
// counted: its products take no float rows.
__global__ __launch_bounds__(256) void layernorm_split_kernel(const float *__restrict__ in,
                                                              const float *__restrict__ gamma,
                                                              const float *__restrict__ beta,
                                                              char *__restrict__ out, int *__restrict__ ex,
                                                              size_t rows, int cols, float eps) {
    const int lane = threadIdx.x & 63;
    const size_t row = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (row >= rows) return;
    const f32x4 *x4 = reinterpret_cast<const f32x4 *>(in + row * cols);
    const int n4 = cols >> 2;
    f32x4 r[4], g[4], b[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int idx = lane + j * 64, ci = idx < n4 ? idx : 0;
        r[j] = idx < n4 ? x4[idx] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        g[j] = reinterpret_cast<const f32x4 *>(gamma)[ci];
        b[j] = reinterpret_cast<const f32x4 *>(beta)[ci];
    }
    float mean, inv;
    ln_row_stats(r, lane, n4, cols, eps, mean, inv);
    uint32_t mx = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (lane + j * 64 >= n4) continue;
        r[j] = ln_apply(r[j], mean, inv, g[j], b[j]);
        mx = absmax4(mx, r[j]);
    }
    mx = wave_umax(mx);
    int e = split_exponent(mx);
    if (e == kSplitNonFinite) {
        e = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) r[j] = r[j] * __builtin_nanf("");
    }
    char *dst = out + row * (cols / 32) * 128;
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (lane + j * 64 < n4) store_split4(dst, 4 * (lane + j * 64), r[j], e);
    if (lane == 0) ex[row] = split_code(e, 0);
}

// One wave per weight row; the sums in doubles, which hold the squares of every
// float.
__global__ __launch_bounds__(256) void weight_range_kernel(const float *__restrict__ w, const float *__restrict__ t,
                                                           const float *__restrict__ u, WeightRange *__restrict__ out,
                                                           int N, int K) {
    const int lane = threadIdx.x & 63;
    const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (n >= N) return;
    double wt = 0.0, wu = 0.0, wa = 0.0, w2 = 0.0;
    float most = 0.0f;
    for (int k = lane; k < K; k += 64) {
        const float v = w[(size_t)n * K + k];
        const double a = (double)v * t[k], b = u ? (double)v * u[k] : 0.0;
        wt += a * a;
        wu += b;
        wa += fabs(b);
        w2 += (double)v * v;
        most = fmaxf(most, fabsf(v));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        wt += __shfl_xor(wt, o, kWave);
        wu += __shfl_xor(wu, o, kWave);
        wa += __shfl_xor(wa, o, kWave);
        w2 += __shfl_xor(w2, o, kWave);
    }
    most = wave_max(most);
    if (lane == 0)
        out[n] = WeightRange{(float)__builtin_sqrt(wt), (float)wu, (float)wa, (float)__builtin_sqrt(w2), most};
}

// Both operands of a row-major product a [M][K] . b [K][N] in one launch:
// workgroups [0, col_wgs) split 16 columns of b each, the rest 16 rows of a
// each, one per wave.  A column strip is read twice, the second time from
// the cache (strips of at most 1024 rows stay in registers): for the largest
// magnitudes, then 256 rows at a time through LDS, so that a column's slice
// is stored from consecutive lanes (1153 x 1003 x 771: both operands 12.4 us, against 28 in
// two launches with 64 rows at a time).
__global__ __launch_bounds__(1024) void split_operands_kernel(const float *__restrict__ a, char *__restrict__ as,
                                                              int *__restrict__ ea, int M, const float *__restrict__ b,
                                                              char *__restrict__ bs, int *__restrict__ eb, int K,
                                                              int N, int slices, int col_wgs) {
    if ((int)blockIdx.x >= col_wgs) {
        const size_t row = (size_t)(blockIdx.x - col_wgs) * 16 + (threadIdx.x >> 6);
        if (row < (size_t)M)
            split_row(a + row * K, as + row * slices * 128, ea + row, K, slices, threadIdx.x & 63);
        return;
    }
    const int c = threadIdx.x & 15, kr = threadIdx.x >> 4;  // column, row of the pass
    const int n0 = blockIdx.x * 16, nc = min(n0 + c, N - 1);
    __shared__ uint32_t red[16][17];
    __shared__ float tile[256][17];
    // Sixteen loads in flight: 1024 rows of the strip, which stay in registers
    // when there are no more.
    float r[16];
    auto load = [&](int k0) {
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int kk = k0 + kr + 64 * j;
            r[j] = kk < K ? b[(size_t)kk * N + nc] : 0.0f;
        }
    };
    uint32_t mx = 0;
    for (int k0 = 0; k0 < K; k0 += 1024) {
        load(k0);
#pragma unroll
        for (int j = 0; j < 16; j++) mx = max(mx, __float_as_uint(r[j]) & 0x7fffffffu);
    }
    mx = max(mx, (uint32_t)__shfl_xor((int)mx, 16, 64));
    mx = max(mx, (uint32_t)__shfl_xor((int)mx, 32, 64));
    if ((threadIdx.x & 63) < 16) red[threadIdx.x >> 6][c] = mx;
    __syncthreads();
    // Store role: column sc of the strip, rows 4 sk .. 4 sk + 3 of a tile.
    const int sc = threadIdx.x >> 6, sk = threadIdx.x & 63;
    uint32_t m = 0;
#pragma unroll
    for (int w = 0; w < 16; w++) m = max(m, red[w][sc]);
    const int e = split_exponent(m), sn = n0 + sc;
    const uint32_t limit = small_limit(e);
    int small = 0;
    for (int k0 = 0; k0 < slices * 32; k0 += 1024) {
        if (K > 1024) load(k0);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (k0 + 256 * q >= slices * 32) break;
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 4; j++) tile[kr + 64 * j][c] = r[4 * q + j];
            __syncthreads();
            const int ks = k0 + 256 * q + 4 * sk;
            if (sn < N && ks < slices * 32) {
                f32x4 v;
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = e == kSplitNonFinite ? 0.0f : tile[4 * sk + j][sc];
                small += small_count4(v, limit);
                store_split4(bs + (size_t)sn * slices * 128, ks, v, e);
            }
        }
    }
    const int code = wave_split_code(e, small);  // a column's tiles are stored by one wave
    if (sk == 0 && sn < N) eb[sn] = code;
}

// Largest finite magnitude (as bits) of each chunk of n floats, with ReLU
// applied first when relu: kConvChunks workgroups, part [kConvChunks].  Also
// clears the `outs` counters that conv_split_image_kernel adds to.
constexpr int kConvChunks = 256;
__global__ __launch_bounds__(256) void conv_absmax_kernel(const float *__restrict__ in, uint32_t *__restrict__ part,
                                                          size_t n, int relu, int *__restrict__ small, int outs) {
    for (int o = blockIdx.x * 256 + threadIdx.x; o < outs; o += gridDim.x * 256) small[o] = 0;
    uint32_t mx = 0;
    auto take = [&](float v) {
        if (relu) v = fmaxf(v, 0.0f);
        const uint32_t b = __float_as_uint(v) & 0x7fffffffu;
        mx = b < 0x7f800000u ? max(mx, b) : mx;
    };
    const f32x4 *in4 = reinterpret_cast<const f32x4 *>(in);
    const size_t n4 = n / 4, stride = (size_t)gridDim.x * 256;
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    for (; i + 3 * stride < n4; i += 4 * stride) {
        const f32x4 a = in4[i], b = in4[i + stride], c = in4[i + 2 * stride], d = in4[i + 3 * stride];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            take(a[e]);
            take(b[e]);
            take(c[e]);
            take(d[e]);
        }
    }
    for (; i < n4; i += stride) {
        const f32x4 a = in4[i];
#pragma unroll
        for (int e = 0; e < 4; e++) take(a[e]);
    }
    if (blockIdx.x == 0 && threadIdx.x < n - 4 * n4) take(in[4 * n4 + threadIdx.x]);
    mx = wave_umax(mx);
    __shared__ uint32_t red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = max(max(red[0], red[1]), max(red[2], red[3]));
}

// The CHW image [cs * 32][ih][iw] as split rows, one per pixel of the grid
// padded by `pad` (zeros; also the rows past the grid), with one exponent:
// grid (positions / 64, cs), a workgroup moving 64 positions of 32 channels
// through LDS (64 consecutive pixels per load, 8 bytes per store).  A pixel's
// small values (about one in 60000 of N(0, 1)) are counted in at the outputs
// whose taps read it, so that the product needs one count per output.
__global__ __launch_bounds__(256) void conv_split_image_kernel(const float *__restrict__ in,
                                                               const uint32_t *__restrict__ part,
                                                               char *__restrict__ out, int *__restrict__ ex, int cs,
                                                               int ih, int iw, int pad, int rows, int relu,
                                                               int *__restrict__ small, int outs, int kh, int kw) {
    __shared__ uint32_t red[4];
    __shared__ float tile[32][65];
    const uint32_t chunk = part[threadIdx.x];
    static_assert(kConvChunks == 256, "one chunk per thread");
    const int wp = iw + 2 * pad, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane, y = p / wp - pad, x = p % wp - pad;
    const bool inside = p < rows && y >= 0 && y < ih && x >= 0 && x < iw;
    const float *src = in + ((size_t)(blockIdx.y * 32 + wv * 8) * ih + (inside ? y : 0)) * iw + (inside ? x : 0);
    const size_t plane = (size_t)ih * iw;
    float v[8];
#pragma unroll
    for (int c = 0; c < 8; c++) v[c] = src[c * plane];
    const uint32_t mx = wave_umax(chunk);  // while the image's loads are in flight
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        if (relu) v[c] = fmaxf(v[c], 0.0f);
        tile[wv * 8 + c][lane] = inside ? v[c] : 0.0f;
    }
    __syncthreads();
    const int e = split_exponent(max(max(red[0], red[1]), max(red[2], red[3])));
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) ex[0] = split_code(e, 0);
    const int q0 = blockIdx.x * 64 + (threadIdx.x >> 3), c4 = 4 * (threadIdx.x & 7);
    const uint32_t limit = small_limit(e);
    int n[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int pos = i * 32 + (threadIdx.x >> 3), q = q0 + i * 32;
        if (q >= rows) continue;
        f16x4 hi, lo;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            _Float16 h, l;
            const float t = __builtin_ldexpf(tile[c4 + r][pos], -e);
            split_f16(t, h, l);
            hi[r] = h;
            lo[r] = __builtin_isfinite(t) ? l : (_Float16)0.0f;
            n[i] += small_key(tile[c4 + r][pos]) < limit;
        }
        char *dst = out + ((size_t)q * cs + blockIdx.y) * 128 + c4 * 2;
        *reinterpret_cast<f16x4 *>(dst) = hi;
        *reinterpret_cast<f16x4 *>(dst + 64) = lo;
    }
    if (n[0] + n[1] == 0) return;
    for (int i = 0; i < 2; i++)
        for (int ky = 0; ky < kh; ky++)
            for (int kx = 0; kx < kw; kx++)
                if (const int o = q0 + 32 * i - ky * wp - kx; n[i] && o >= 0 && o < outs) atomicAdd(small + o, n[i]);
}

// The tiles, and what a k-slice of one costs a CU in microseconds when the
// tile has it alone (slope between K = 768 and K = 3072 at 865 rows on
// MI355X) with the cost of a launch that does not depend on K.
struct SplitTile {
    int bm, bn;
    float slice_us, fixed_us;
    bool qkv;    // waves a whole number of 32-wide RoPE halves across
    bool alone;  // takes more than half the LDS
    bool pieces;
};
constexpr SplitTile kSplitTiles[] = {
    {128, 256, 0.858f, 5.0f, true, true, false},   // 2 x 4 waves
    {128, 192, 0.646f, 6.0f, false, true, false},  // 2 x 4 waves
    {128, 128, 0.480f, 5.9f, true, true, false},   // 2 x 4 waves
    {128, 96, 0.378f, 5.0f, false, true, false},   // 4 x 2 waves
    {64, 128, 0.286f, 3.9f, true, false, false},   // 2 x 4 waves, two workgroups per CU
    {64, 64, 0.211f, 3.0f, true, true, true},      // 2 x 2 waves, two K groups
    {64, 32, 0.125f, 3.7f, true, false, true},     // 2 x 1 waves, two K groups, two workgroups per CU
};

struct SplitPlan {
    int tile, pieces;
    float us;
};

// The tile with the lowest predicted time: every CU runs ceil(tiles / 256)
// tiles of slices * slice_us, and a tile that has the CU alone (more than
// half the LDS) adds about 2 us of prologue and epilogue per further round.
// Grids of at most half the CUs may share a tile's K out over 2 to 4
// workgroups of at least 8 slices: the partials, which go past the L2 both
// ways, take 1.5 us and 1.8 TB/s.  So it pays for few rows only (97 x 768 x
// 3072 10.0 us in 4 pieces, 14.9 whole; 865 x 768 x 3072 22.2 in 3 pieces of 64 x
// 128, 22.0 whole on 64 x 64).  The prediction names the fastest or comes
// within 3% of it on the shapes swept on MI355X (865 x 3072 x 768: 18.1 us
// here, 20.5 for 64 x 128, 23.9 for 64 x 64; 3460 x 2304 x 768: 40.4 for 128 x
// 256, 45.9 for 64 x 128; 3460 x 3072 x 768: 57.2 for 128 x 192, 63.9 for 128 x
// 128 and 65.2 for 128 x 256; 97 x 2304 x 768: 6.2 for 64 x 32, 10.3 for 64 x
// 128).
SplitPlan plan_split(size_t m, size_t n, int slices, bool qkv, bool pieces_ok) {
    SplitPlan best{0, 1, INFINITY};
    for (int i = 0; i < (int)(sizeof(kSplitTiles) / sizeof(kSplitTiles[0])); i++) {
        const SplitTile &t = kSplitTiles[i];
        if (qkv && !t.qkv) continue;
        const size_t tiles = ((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn);
        const float rounds = (float)((tiles + 255) / 256);
        const float whole = t.fixed_us + rounds * slices * t.slice_us + (t.alone ? 2.0f * (rounds - 1.0f) : 0.0f);
        if (whole < best.us) best = SplitPlan{i, 1, whole};
        for (int p = 2; pieces_ok && t.pieces && p <= kSplitMaxPieces; p++) {
            const int each = (slices + p - 1) / p;
            if (tiles * p > 256 || each < 8 || each * (p - 1) >= slices) continue;
            const float us = t.fixed_us + each * t.slice_us + 1.5f + (float)m * (float)n * (float)(8 * p) / 1.8e6f;
            if (us < best.us) best = SplitPlan{i, p, us};
        }
    }
    return best;
}

template <int BM, int BN, int WM, int WN, int KG, SEpi EPI, bool PIECES = false>
hipError_t launch_split_tile(hipStream_t s, const SplitArgs &ar) {
    // The largest tile's step is long enough for one stage in flight (40.4 us
    // against 42.5 for three stages at 3460 x 2304 x 768).
    constexpr int ST = BM * BN >= 128 * 256 ? 2 : 3;
    constexpr size_t stage = (size_t)KG * ST * (BM + BN) * 128;
    constexpr size_t xch = KG > 1 ? (size_t)KG * BM * BN * 4 : 0;
    constexpr size_t lds = stage > xch ? stage : xch;
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    auto kernel = gemm_split_kernel<BM, BN, WM, WN, KG, ST, EPI, PIECES>;
    static std::atomic<uint64_t> configured{0};
    if (hipError_t e = ensure_dynamic_lds(kernel, lds, configured); e != hipSuccess) return e;
    const size_t tiles = (size_t)((ar.M + BM - 1) / BM) * (size_t)((ar.N + BN - 1) / BN) * (size_t)ar.pieces;
    if (tiles > (size_t)INT32_MAX / (WM * WN * KG * 64)) return hipErrorInvalidValue;
    kernel<<<(unsigned)tiles, WM * WN * KG * 64, lds, s>>>(ar);
    return hipGetLastError();
}

template <SEpi EPI>
hipError_t launch_split_epi(hipStream_t s, SplitArgs ar) {
    const SplitPlan p = plan_split(ar.M, ar.N, ar.slices, EPI == SEpi::Qkv, ar.partial != nullptr);
    ar.pieces = p.pieces;
    constexpr bool Q = EPI == SEpi::Qkv;
    switch (p.tile) {
        case 0: return launch_split_tile<128, 256, 2, 4, 1, EPI>(s, ar);
        case 1:
            if constexpr (!Q) return launch_split_tile<128, 192, 2, 4, 1, EPI>(s, ar);
            return hipErrorInvalidValue;
        case 2: return launch_split_tile<128, 128, 2, 4, 1, EPI>(s, ar);
        case 3:
            if constexpr (!Q) return launch_split_tile<128, 96, 4, 2, 1, EPI>(s, ar);
            return hipErrorInvalidValue;
        case 4: return launch_split_tile<64, 128, 2, 4, 1, EPI>(s, ar);
        case 5:
            return p.pieces > 1 ? launch_split_tile<64, 64, 2, 2, 2, EPI, true>(s, ar)
                                : launch_split_tile<64, 64, 2, 2, 2, EPI>(s, ar);
        default:
            return p.pieces > 1 ? launch_split_tile<64, 32, 2, 1, 2, EPI, true>(s, ar)
                                : launch_split_tile<64, 32, 2, 1, 2, EPI>(s, ar);
    }
}

}  // namespace

bool split_gemm_fits(size_t m, size_t n, size_t k) {
    // A wave splits a row of either operand, both in one launch: fewer than
    // 2^32 threads.
    constexpr size_t kMaxRows = ((size_t)1 << 25) - 64;
    if (m > kMaxRows || n > kMaxRows) return false;
    // Row offsets inside a 256-row tile stay below 2^31 bytes, and the
    // chosen tile's grid (with or without Qkv's choice) below the launch limit.
    if (k == 0 || k > ((size_t)1 << 21) - 32) return false;
    if (m == 0 || n == 0) return true;
    for (bool qkv : {false, true}) {
        const SplitTile &t = kSplitTiles[plan_split(m, n, (int)((k + 31) / 32), qkv, false).tile];
        if ((m + t.bm - 1) / t.bm > (size_t)INT32_MAX / 512 / ((n + t.bn - 1) / t.bn)) return false;
    }
    return true;
}

// Splitting reads and writes four bytes per value at about 3 TB/s, in a launch
// of 2.5 us.  The fp32 GEMM runs 64 x 64 tiles at 0.55 us per k-slice of 32,
// the K of a grid below half the CUs in two parts at once (a long K, below a
// quarter, in more: a third of a round), a partial last round as K pieces (0.3
// of a round), and takes twice as long where K is no multiple of 32 (its masked
// loads).  Both forms of 240 linears on MI355X, K = 96 to 3072, N = 96 to 3072,
// 16 to 3460 rows (us a call, fp32 and split): 865 x 768 x 768 14.2 and 14.4,
// 500 x 768 x 768 13.3 and 11.6, 865 x 768 x 3072 40.8 and 22.7, 865 x 1536 x 384
// 23.4 and 18.1; the fp32 GEMM keeps K below 128 (865 x 96 x 3072 9.5 and 12.6,
// 3460 x 96 x 3072 27.3 and 30.7: the output's bytes bound both), 865 x 1536 x 96
// (12.1 and 15.0) and 500 x 1536 x 384 (13.9 and 17.2).  Where the rule takes
// the split form it is at most 2 us behind (500 x 1536 x 96 11.8 and 14.0).
// whole_tiles: the fp32 route is the channel-major one, which splits no K (865 x
// 768 x 96 19.3 and 11).
bool split_gemm_pays(size_t m, size_t n, size_t k, size_t split_values, bool whole_tiles) {
    if (k < 128 && k % 32 == 0) return false;
    const int slices = (int)((k + 31) / 32);
    const float gemm_us = plan_split(m, n, slices, false, true).us;
    const float split_us = 2.5f + (float)split_values * 8.0f / 3e6f + gemm_us;
    const float tiles = (float)((m + 63) / 64) * (float)((n + 63) / 64);
    float rounds = tiles > 256.0f ? tiles / 256.0f + 0.3f : (tiles > 128.0f ? tiles / 256.0f : 0.5f);
    if (tiles <= 64.0f && k > 1024) rounds = 0.33f;
    if (whole_tiles) rounds = ceilf(tiles / 256.0f);
    const float fp32_us = (4.0f + rounds * slices * 0.55f) * (k % 32 == 0 ? 1.0f : 2.0f);
    return split_us < fp32_us;
}

hipError_t launch_split_rows(hipStream_t s, const float *in, void *out, int *ex, size_t rows, size_t k) {
    if (rows == 0) return hipSuccess;
    const size_t wpb = rows <= 2048 ? 1 : 4;
    split_rows_kernel<<<(unsigned)((rows + wpb - 1) / wpb), (unsigned)(64 * wpb), 0, s>>>(
        in, static_cast<char *>(out), ex, rows, (int)k, (int)((k + 31) / 32));
    return hipGetLastError();
}

hipError_t launch_split_operands(hipStream_t s, const float *a, void *as, int *ea, size_t m, const float *b, void *bs,
                                 int *eb, size_t k, size_t n) {
    if (m == 0 || n == 0) return hipSuccess;
    const size_t cols = (n + 15) / 16, rows = (m + 15) / 16;
    split_operands_kernel<<<(unsigned)(cols + rows), 1024, 0, s>>>(a, static_cast<char *>(as), ea, (int)m, b,
                                                                   static_cast<char *>(bs), eb, (int)k, (int)n,
                                                                   (int)((k + 31) / 32), (int)cols);
    return hipGetLastError();
}

hipError_t launch_layernorm_split(hipStream_t s, const float *in, const float *gamma, const float *beta, void *out,
                                  int *ex, size_t rows, size_t cols, float eps) {
    if (rows == 0) return hipSuccess;
    if (cols % 32 != 0 || cols == 0 || cols > 1024) return hipErrorInvalidValue;
    const size_t wpb = rows <= 2048 ? 1 : 4;
    layernorm_split_kernel<<<(unsigned)((rows + wpb - 1) / wpb), (unsigned)(64 * wpb), 0, s>>>(
        in, gamma, beta, static_cast<char *>(out), ex, rows, (int)cols, eps);
    return hipGetLastError();
}

hipError_t launch_weight_ranges(hipStream_t s, const float *w, const float *t, const float *u, WeightRange *out,
                                size_t n, size_t k) {
    if (n == 0) return hipSuccess;
    weight_range_kernel<<<(unsigned)((n + 3) / 4), 256, 0, s>>>(w, t, u, out, (int)n, (int)k);
    return hipGetLastError();
}

size_t conv_split_bytes(const SplitConv &c) {
    const size_t wp = c.iw + 2 * c.pad, rows = (c.ih + 2 * c.pad) * wp + c.kw - 1;
    const size_t outs = (c.ih + 2 * c.pad - c.kh + 1) * wp;
    return rows * c.in_c * 4 + (kConvChunks + 1 + outs) * sizeof(int);
}

bool conv_split_fits(const SplitConv &c) {
    if (c.in_c % 32 != 0 || c.in_c == 0) return false;
    const size_t wp = c.iw + 2 * c.pad, hp = c.ih + 2 * c.pad, K = c.kh * c.kw * c.in_c;
    const size_t oh = hp - c.kh + 1, ow = wp - c.kw + 1;
    if (K < 256 || hp * wp + c.kw > (size_t)INT32_MAX / 512 || c.in_c / 32 > 65535 ||
        !split_gemm_fits(oh * wp, c.out_c, K))
        return false;
    // Below half the CUs in 64 x 64 tiles the fp32 kernel splits K over the idle
    // ones, and the staging launches here are no gain (384 -> 128 on 24 x 36: 18
    // us against about 25).
    const size_t tiles = ((c.out_c + 63) / 64) * ((oh * ow + 63) / 64);
    if (tiles < 128) return false;
    // Otherwise by the time of two staging launches at 1.5 TB/s of image and the
    // product, against 0.75 us per tile and k-slice of the fp32 kernel, a
    // partial last round as K pieces.  Per call on MI355X, split and fp32 (us):
    // 128 -> 128 on 96 x 144 30.7 and 53.6, 64 -> 32 on 384 x 576 89 and 171,
    // 32 -> 128 on 96 x 144 15.3 and 18.1, 1 x 1 256 -> 256 there 25.8 and
    // 27.9; the fp32 form keeps 32 -> 64 on 97 x 91 (12.1 and 10.8) and 1 x 1
    // with few outputs (256 -> 33 on 96 x 144 19.1 and 10.0).
    const int slices = (int)(K / 32);
    const float split_us =
        7.0f + (float)(c.in_c * c.ih * c.iw) * 4.0f / 1.5e6f + plan_split(oh * wp, c.out_c, slices, false, false).us;
    const float rounds = tiles > 256 ? (float)tiles / 256.0f + 0.3f : 1.0f;
    return split_us < 5.0f + rounds * (float)slices * 0.75f;
}

hipError_t launch_conv_split(hipStream_t s, const SplitConv &c, void *ws) {
    const int cs = (int)(c.in_c / 32), wp = (int)(c.iw + 2 * c.pad), hp = (int)(c.ih + 2 * c.pad);
    const int rows = hp * wp + (int)c.kw - 1, oh = hp - (int)c.kh + 1, ow = wp - (int)c.kw + 1;
    char *img = static_cast<char *>(ws);
    uint32_t *part = reinterpret_cast<uint32_t *>(img + (size_t)rows * c.in_c * 4);
    int *ex = reinterpret_cast<int *>(part + kConvChunks), *small = ex + 1;
    conv_absmax_kernel<<<kConvChunks, 256, 0, s>>>(c.in, part, c.in_c * c.ih * c.iw, c.relu ? 1 : 0, small, oh * wp);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    conv_split_image_kernel<<<dim3((rows + 63) / 64, cs), 256, 0, s>>>(
        c.in, part, img, ex, cs, (int)c.ih, (int)c.iw, (int)c.pad, rows, c.relu ? 1 : 0, small, oh * wp, (int)c.kh,
        (int)c.kw);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    SplitArgs ar{};
    ar.x = img;
    ar.w = static_cast<const char *>(c.w);
    ar.ex = ex;
    ar.ew = c.ew;
    ar.M = oh * wp;
    ar.N = (int)c.out_c;
    ar.K = (int)(c.kh * c.kw * c.in_c);
    ar.slices = ar.K / 32;
    ar.xf = c.in;
    ar.wf = c.wf;
    ar.c = c.out;
    ar.bias = c.bias;
    ar.conv_small = small;
    ar.conv_cs = cs;
    ar.conv_kw = (int)c.kw;
    ar.conv_wp = wp;
    ar.conv_ow = ow;
    ar.conv_ih = (int)c.ih;
    ar.conv_iw = (int)c.iw;
    ar.conv_pad = (int)c.pad;
    ar.conv_relu = c.relu ? 1 : 0;
    ar.conv_plane = (size_t)oh * ow;
    return launch_split_epi<SEpi::Conv>(s, ar);
}

hipError_t launch_gemm_split(hipStream_t s, const SplitGemm &g) {
    if (g.m == 0 || g.n == 0) return hipSuccess;
    if (!split_gemm_fits(g.m, g.n, g.k)) return hipErrorInvalidValue;
    SplitArgs ar{};
    ar.x = static_cast<const char *>(g.x);
    ar.w = static_cast<const char *>(g.w);
    ar.ex = g.ex;
    ar.ex_c = g.ex_c;
    ar.ew = g.ew;
    ar.M = (int)g.m;
    ar.N = (int)g.n;
    ar.K = (int)g.k;
    ar.slices = (int)((g.k + 31) / 32);
    ar.xf = g.xf;
    ar.wf = g.wf;
    ar.wf_n = g.wf_columns ? (int)g.n : 0;
    ar.c = g.c;
    ar.bias = g.bias;
    ar.gamma = g.gamma;
    ar.q = g.q;
    ar.k = g.k_out;
    ar.v = g.v;
    ar.tokens = (int)g.tokens;
    ar.heads = (int)g.heads;
    ar.rot = g.rot;
    for (int i = 0; i < 3; i++)
        ar.qkv_scale[i] = g.qkv_split[i] ? __builtin_ldexpf(1.0f, -g.qkv_ex[i]) : 0.0f;
    if (g.piece_cnt && g.piece_cnt_n >= 256 && g.partial_floats >= kSplitPieceFloats) {
        ar.partial = g.partial;
        ar.piece_cnt = g.piece_cnt;
    }
    ar.out_split = static_cast<char *>(g.out_split);
    ar.out_scale = g.out_split ? __builtin_ldexpf(1.0f, -g.out_ex) : 0.0f;
    if (g.out_split) {
        if (g.epi != Epi::Gelu || g.n % 32 != 0 || g.out_ex > 100 || g.out_ex < -100) return hipErrorInvalidValue;
        return launch_split_epi<SEpi::GeluSplit>(s, ar);
    }
    if (g.chw) return g.epi == Epi::Store ? launch_split_epi<SEpi::Chw>(s, ar) : hipErrorInvalidValue;
    switch (g.epi) {
        case Epi::Store: return launch_split_epi<SEpi::Store>(s, ar);
        case Epi::Gelu: return launch_split_epi<SEpi::Gelu>(s, ar);
        case Epi::Residual: return launch_split_epi<SEpi::Residual>(s, ar);
        case Epi::Qkv: return g.n == 3 * g.heads * 64 ? launch_split_epi<SEpi::Qkv>(s, ar) : hipErrorInvalidValue;
    }
    return hipErrorInvalidValue;
}

}  // namespace vh
