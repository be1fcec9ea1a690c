// Row-streaming projections of 1 .. 16 tokens (bf16): the decode steps' matrix products, each with its consumer's elementwise work as an epilogue.
//
// An epilogue E is called once per output, e(value, token, row, problem) (E::WAVES: by whole waves, e(value, token, row, in range)).  E::SUMSQ: it returns the square of what it stored and offers `sums`, which
// receives per token and workgroup the sum of those squares -- partial sums for an RMS norm whose 1 / rms the CONSUMER of the stored rows applies to its
// results (RowsIn::sq): W (r x) = r (W x), so no launch of its own stands between the two.
#pragma once
#include "elem.h"
#include <algorithm>
#include <type_traits>

namespace ad {

__device__ __forceinline__ u32x4 ldw16(const bf16_t* p) { return ld16_once(p); }   // a weight stream is read once
// acc[r] += W[row r] . x, a wave over two weight rows: four 16-byte chunks per row and lane requested before the first use, the token's row comes from the
// L1 / L2
__device__ __forceinline__ void two_rows(float (&acc)[2], const bf16_t* w0, const bf16_t* w1, const bf16_t* x, int K, int l) {
    const int nch = K >> 3;
    for (int c0 = l; c0 < nch; c0 += 256) {
        u32x4 a[2][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = min(c0 + 64 * u, nch - 1);
            a[0][u] = ldw16(w0 + c * 8);
            a[1][u] = ldw16(w1 + c * 8);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            u32x4 v = ld16(x + min(c0 + 64 * u, nch - 1) * 8);
            const bool in = c0 + 64 * u < nch;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t xv = in ? v[q] : 0u;
                acc[0] = dot2bf(a[0][u][q], xv, acc[0]);
                acc[1] = dot2bf(a[1][u][q], xv, acc[1]);
            }
        }
    }
    acc[0] = wave_sum_bcast(acc[0]);
    acc[1] = wave_sum_bcast(acc[1]);
}

struct RowsIn {
    const bf16_t* W;    // [N, K]
    const bf16_t* W2;   // second matrix of a gated pair
    const bf16_t* X;    // [T, ldx]
    long long ldx;
    int K, N;
    const float* sq = nullptr;   // [T, sq_n] partial sums of squares: results are multiplied by 1 / sqrt(sum inv_n + eps)
    int sq_n = 0;
    float inv_n = 0.f, eps = 0.f;
};
struct RowsPair {   // up to two problems of one launch (blockIdx.z): equal N and tokens
    RowsIn in[2];
};

namespace {
// one token: a wave per two weight rows (PAIR: per output, gate row and up row)
template <class E, bool PAIR>
__global__ __launch_bounds__(256) void row_kernel(RowsPair rp, E e) {
    ARIA_SMEM_STATIC float red[8];
    const RowsIn& in = rp.in[blockIdx.z];
    const int t = threadIdx.x, l = t & 63, w = t >> 6, N = in.N;
    const int row0 = PAIR ? blockIdx.x * 4 + w : (blockIdx.x * 4 + w) * 2;
    const int r0 = min(row0, N - 1), r1 = PAIR ? r0 : min(row0 + 1, N - 1);
    float ss = 0.f;
    if (in.sq) {
        for (int i = t; i < in.sq_n; i += 256) ss += in.sq[i];
    }
    float acc[2] = {0.f, 0.f};
    two_rows(acc, in.W + (long long)r0 * in.K, (PAIR ? in.W2 : in.W) + (long long)r1 * in.K, in.X, in.K, l);
    float v0 = acc[0], v1 = acc[1];
    if (in.sq) {
        ss = wave_sum_bcast(ss);
        if (l == 0) red[w] = ss;
        sync();
        const float r = 1.f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) * in.inv_n + in.eps);
        v0 *= r;
        v1 *= r;
    }
    float s = 0.f;
    if (PAIR) {
        if (l == 0 && row0 < N) e(v0, v1, 0, row0);
    } else if (l < 2 && row0 + l < N) {
        s = e(l ? v1 : v0, 0, row0 + l, int(blockIdx.z));
    }
    if (E::SUMSQ) {
        s += shfl_xor(s, 1);
        if (l == 0) red[4 + w] = s;
        sync();
        if (t == 0) e.sums[blockIdx.x] = (red[4] + red[5]) + (red[6] + red[7]);
    }
}
// Several tokens: a workgroup of NW waves runs through the groups [g0, g1) of 16 weight rows with MT x 16 tokens.  Tokens are the rows of A, weight rows
// the columns of B: both k-contiguous in memory, so fragments come straight from global memory, and the matrix pipe takes the multiply-adds of sixteen tokens
// at the price of one.  Wave w owns the KS 32-column steps of the reduction that start at column 32 KS w: its part of the tokens is loaded ONCE and stays
// in registers, and a weight fragment's register is refilled with the next group's as soon as it is used, so up to 16 kilobytes a wave are in flight
// without a break between the groups.  The NW partial results meet in LDS (two images in turn: one barrier a group), where whole waves sum them and call
// out(value, token, column of the group, group).  wrow(g, r): row r of group g, xrow(i): this lane's token row of tile i; both from column 0.
//
// A load takes eight rows' whole cache lines (64 columns), the next one the other eight rows'; the two fragments of 16 rows and 32 columns are these with their halves
// exchanged between the lanes of a row (whole_lines).  So the weights, which are read once, can be non-temporal: a fragment loaded as it is wanted touches half a line of 16 rows,
// and the hint then fetches every line twice.  Reading 500 MB: half lines 87 us, non-temporal 104, whole lines 86, non-temporal 77 (6.8 TB/s); 34 MB 8.3, 10.4, 7.9, 7.4.
// A step left over (KS odd) is a half line that another wave shares: a plain load.  !ONCE: half lines, plain (rows_once, experts_once).
template <int NW, int MT>
struct RowsRed {
    float v[2][NW][16 * MT][17];
};
template <int NW, int KS, int MT, bool ONCE, class WRow, class XRow, class Out>
__device__ __forceinline__ void stream_rows(int K, const WRow& wrow, const XRow& xrow, int g0, int g1, RowsRed<NW, MT>& red, const Out& out) {
    constexpr int P = KS / 2;                                          // ONCE: pairs of steps, and a left-over one where KS is odd
    constexpr int SLOTS = ONCE ? KS <= 16 ? P : 6 : 1;   // pairs in flight: pair p in slot p % SLOTS (seven of 26 steps: an expert pair's registers spill)
    constexpr int DEPTH = ONCE ? 1 : KS <= 16 ? KS : KS / 2;           // else: fragments in flight
    static_assert(KS % DEPTH == 0, "a step keeps its register");
    const int t = threadIdx.x, l = t & 63, w = t >> 6, q4 = l >> 4, c16 = l & 15;
    // the last waves' windows are moved down into the row, the columns that another wave owns zeroed in the tokens: every address is base + constant
    const int own = w * KS * 32, start = min(own, K - KS * 32);
    // the column of x[][u]: in order, but the left-over step last, which is the window's first where that begins in the middle of a line
    const int odd = ONCE && KS % 2 ? first_lane(start >> 5 & 1) : 0;
    auto column = [&](int u) __attribute__((always_inline)) { return start + 32 * (ONCE && KS % 2 && u == KS - 1 ? odd ? 0 : KS - 1 : u + odd); };
    const int row = c16 & 7, line = column(0) + (q4 + 4 * (c16 >> 3)) * 8;
    u32x4 x[MT][KS], a[SLOTS], b[SLOTS], f[DEPTH];   // f[0] of ONCE: the left-over step
    const bf16_t *wa = wrow(g0, ONCE ? row : c16), *wb = ONCE ? wrow(g0, row + 8) : wa, *wf = wrow(g0, c16);
    if constexpr (ONCE) {
#pragma unroll
        for (int p = 0; p < SLOTS; ++p) a[p] = ldw16(wa + line + 64 * p), b[p] = ldw16(wb + line + 64 * p);
        if (KS % 2) f[0] = ld16(wf + column(KS - 1) + q4 * 8);
    } else {
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) f[u] = ld16(wf + column(u) + q4 * 8);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const bf16_t* xp = xrow(i) + q4 * 8;
#pragma unroll
        for (int u = 0; u < KS; ++u) x[i][u] = ld16(xp + column(u));
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int u = 0; u < KS; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) x[i][u][q] = column(u) + q4 * 8 >= own ? x[i][u][q] : 0u;
    for (int g = g0; g < g1; ++g) {
        const int ph = (g - g0) & 1;
        f32x4 acc[MT];   // (one chain a tile whatever MT is: a token's sums do not depend on how many tokens there are)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto step = [&](int u, const s16x8& v) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i] = mfma16(__builtin_bit_cast(s16x8, x[i][u]), v, acc[i]);
        };
        // the group's steps; its registers are refilled with its own later steps and (`on`) the next group's
        auto steps = [&](auto on_, const bf16_t* na, const bf16_t* nb, const bf16_t* nf) __attribute__((always_inline)) {
            constexpr bool on = decltype(on_)::value;
            if constexpr (ONCE) {   // (the steps in the row's order in either form: the same bits)
                if (KS % 2 && odd) step(KS - 1, __builtin_bit_cast(s16x8, f[0]));
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    const int s = p % SLOTS;
                    u32x4 lo, hi;
                    whole_lines(a[s], b[s], lo, hi);
                    step(2 * p, __builtin_bit_cast(s16x8, lo));
                    step(2 * p + 1, __builtin_bit_cast(s16x8, hi));
                    if (p + SLOTS < P)
                        a[s] = ldw16(wa + line + 64 * (p + SLOTS)), b[s] = ldw16(wb + line + 64 * (p + SLOTS));
                    else if (on)
                        a[s] = ldw16(na + line + 64 * s), b[s] = ldw16(nb + line + 64 * s);
                }
                if (KS % 2 && !odd) step(KS - 1, __builtin_bit_cast(s16x8, f[0]));
                if (KS % 2 && on) f[0] = ld16(nf + column(KS - 1) + q4 * 8);
            } else {
#pragma unroll
                for (int u = 0; u < KS; ++u) {
                    step(u, __builtin_bit_cast(s16x8, f[u % DEPTH]));
                    if (u + DEPTH < KS)
                        f[u % DEPTH] = ld16(wf + column(u + DEPTH) + q4 * 8);
                    else if (on)
                        f[u % DEPTH] = ld16(nf + column(u + DEPTH - KS) + q4 * 8);
                }
            }
        };
        if (g + 1 < g1) {
            const bf16_t *na = wrow(g + 1, ONCE ? row : c16), *nb = ONCE ? wrow(g + 1, row + 8) : na, *nf = wrow(g + 1, c16);
            steps(std::true_type{}, na, nb, nf);
            wa = na, wb = nb, wf = nf;
        } else {
            steps(std::false_type{}, wa, wb, wf);
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) red.v[ph][w][16 * i + 4 * q4 + r][c16] = acc[i][r];
        sync();
        // (whole waves; one tile of sums: the halves of the workgroup in turn)
        for (int i = MT == 1 ? ((t >> 8) == ((g - g0) & (NW / 4 - 1)) ? t & 255 : 256) : t; i < 256 * MT; i += NW * 64) {
            const int tok = i >> 4, n = i & 15;
            float v = 0.f;
#pragma unroll
            for (int ww = 0; ww < NW; ++ww) v += red.v[ph][ww][tok][n];
            out(v, tok, n, g);
        }
    }
}
// 1 / rms of sixteen tokens from their partial sums of squares, a wave per token
__device__ __forceinline__ void token_rms(float* rms, const RowsIn& in, int t0, int n_tok, int waves) {
    const int l = threadIdx.x & 63;
    for (int i = threadIdx.x >> 6; i < 16 && t0 + i < n_tok; i += waves) {
        float s = 0.f;
        for (int j = l; j < in.sq_n; j += 64) s += in.sq[(long long)(t0 + i) * in.sq_n + j];
        s = wave_sum_bcast(s);
        if (l == 0) rms[i] = 1.f / sqrtf(s * in.inv_n + in.eps);
    }
}
// PAIR: a group is 8 gate rows and the 8 up rows of the same outputs
template <int NW, int KS, int MT, class E, bool PAIR, bool ONCE>
__global__ __launch_bounds__(NW * 64) void rows_kernel(RowsPair rp, int n_tok, int per, E e) {
    ARIA_SMEM_STATIC RowsRed<NW, MT> red;
    ARIA_SMEM_STATIC float rms[16];
    constexpr int OUT = PAIR ? 8 : 16;
    const RowsIn& in = rp.in[blockIdx.z];
    const int c16 = threadIdx.x & 15, t0 = blockIdx.y * 16 * MT, groups = (in.N + OUT - 1) / OUT, g0 = blockIdx.x * per;
    if (g0 >= groups) return;
    if (MT == 1 && in.sq) token_rms(rms, in, t0, n_tok, NW);   // (published by the first group's barrier)
    stream_rows<NW, KS, MT, ONCE>(
        in.K, [&](int g, int r) { return (PAIR && r >= 8 ? in.W2 : in.W) + (long long)min(g * OUT + (PAIR ? r & 7 : r), in.N - 1) * in.K; },
        [&](int i) { return in.X + (long long)min(t0 + 16 * i + c16, n_tok - 1) * in.ldx; }, g0, min(groups, g0 + per), red,
        [&](float v, int tok, int n, int g) {
            const float u = PAIR ? shfl_xor(v, 8) : 0.f;
            const int row = g * OUT + n;
            const bool in_range = t0 + tok < n_tok && row < in.N && n < OUT;
            const float r = MT == 1 && in.sq && in_range ? rms[tok] : 1.f;
            float s = 0.f;
            if constexpr (PAIR) {
                if (in_range) e(v * r, u * r, t0 + tok, row);
            } else if constexpr (E::WAVES) {   // (all lanes: the epilogue exchanges values)
                e(v, t0 + tok, row, in_range);
            } else if (in_range) {
                s = e(v * r, t0 + tok, row, int(blockIdx.z));
            }
            if constexpr (E::SUMSQ) {   // sixteen lanes hold a token's outputs
                s = group_sum<16>(s);
                if (n == 0 && t0 + tok < n_tok) e.sums[(long long)(t0 + tok) * groups + g] = s;
            }
        });
}
// any reduction (below a wave's window of stream_rows or beyond what it holds in registers): the 8 waves on interleaved 128-column blocks of it, a workgroup per 16 rows
template <class E, bool PAIR>
__global__ __launch_bounds__(512) void rows_long_kernel(RowsPair rp, int n_tok, E e) {
    constexpr int NW = 8, RG = PAIR ? 2 : 1;
    ARIA_SMEM_STATIC float red[NW][16][16 * RG + 1];
    ARIA_SMEM_STATIC float rms[16];
    const RowsIn& in = rp.in[blockIdx.z];
    const int t = threadIdx.x, l = t & 63, w = t >> 6, q4 = l >> 4, c16 = l & 15, K = in.K, N = in.N;
    const int n0 = blockIdx.x * 16, t0 = blockIdx.y * 16;
    const bf16_t* wp[RG];
#pragma unroll
    for (int g = 0; g < RG; ++g) wp[g] = (g ? in.W2 : in.W) + (long long)min(n0 + c16, N - 1) * K;
    const bf16_t* xp = in.X + (long long)min(t0 + c16, n_tok - 1) * in.ldx;
    f32x4 acc[RG][2];
#pragma unroll
    for (int g = 0; g < RG; ++g) acc[g][0] = acc[g][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = w * 128; k0 < K; k0 += 2 * NW * 128) {   // two blocks in flight: every weight fragment before the first use
        u32x4 a[8], b[RG][8];
#pragma unroll
        for (int g = 0; g < RG; ++g)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int k = k0 + (u >> 2) * NW * 128 + (u & 3) * 32 + q4 * 8;
                b[g][u] = ld16(wp[g] + (k < K ? k : 0));
            }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int k = k0 + (u >> 2) * NW * 128 + (u & 3) * 32 + q4 * 8;
            a[u] = ld16(xp + (k < K ? k : 0));
#pragma unroll
            for (int q = 0; q < 4; ++q) a[u][q] = k < K ? a[u][q] : 0u;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int g = 0; g < RG; ++g) acc[g][u & 1] = mfma16(__builtin_bit_cast(s16x8, a[u]), __builtin_bit_cast(s16x8, b[g][u]), acc[g][u & 1]);
    }
    if (in.sq) token_rms(rms, in, t0, n_tok, NW);
#pragma unroll
    for (int g = 0; g < RG; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[w][4 * q4 + r][16 * g + c16] = acc[g][0][r] + acc[g][1][r];
    sync();
    if (t >= 256) return;
    const int tok = t >> 4, n = t & 15;
    const bool in_range = t0 + tok < n_tok && n0 + n < N;
    float v = 0.f, u = 0.f, s = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) {
        v += red[ww][tok][n];
        if (PAIR) u += red[ww][tok][16 * (RG - 1) + n];
    }
    if (in_range) {
        if (in.sq) {
            v *= rms[tok];
            u *= rms[tok];
        }
        if constexpr (PAIR)
            e(v, u, t0 + tok, n0 + n);
        else
            s = e(v, t0 + tok, n0 + n, int(blockIdx.z));
    }
    if constexpr (E::SUMSQ) {
        s = group_sum<16>(s);
        if (n == 0 && t0 + tok < n_tok) e.sums[(long long)(t0 + tok) * gridDim.x + blockIdx.x] = s;
    }
}

// workgroups of one problem, i.e. the partial sums per token that an epilogue with SUMSQ leaves
inline int rows_parts(int64_t T, int64_t N) { return int(T == 1 ? (N + 7) / 8 : (N + 15) / 16); }

// Whether weights [N, K] that `passes` rows of workgroups go through come by whole lines, non-temporal (stream_rows): read once, lines that do not straddle rows, and enough of them.
// Us, half lines / whole: 100352 x 2560 at 2, 16, 64 tokens 93 / 82, 103 / 85, 123 / 117; 32000 x 1024 14.0 / 12.9 (2 tokens); 2560 x 2560 5.7 / 5.5; gate and up of 3328 x 2560 at 40 tokens
// 15.8 / 14.9.  In several passes (found in the L2): 7680 x 2560, 280 tokens, 37.4 / 38.8.  1024 x 1024, 64 x 2560: 3.15 / 3.26, 4.8 / 4.9; 1000 x 1000 2.7 / 3.4.
inline bool rows_once(int64_t passes, int64_t N, int64_t K) { return passes == 1 && K % 64 == 0 && N * K >= (3 << 20); }

// Whether weights by expert, E times [N, K] in all, come so: lines that do not straddle rows, and at least `least` Mi weights.  Fewer are still in the Infinity Cache from the use before, which the
// hint passes by: 32 for a step's few rows, 16 for sorted ones.  A model's steps, 16 experts of 768 x 1024 (pairs 25 M, down 12.6 M), half lines / whole: 4, 8, 16 tokens 151 / 153, 161 / 164, 176 / 179 us; 32 of 1024 x 1536: 238 / 219, 278 /
// 254, 308 / 276.  Sorted rows, launches in turn, rows an expert: 16 of 768 x 1024, down: 12 9.7 / 10.2, 26 10.4 / 11.5, a quarter of the experts with 100 and the rest with one 15.9 / 17.1, but
// pairs, whose two tensors are twice as many: 4 11.6 / 11.8, 12 15.2 / 13.5, 26 17.3 / 15.5, 19.9 / 19.8.  An expert of several tiles of rows fetches its weights anew for each, and is ahead or
// level with it even so: 64 of 1664 x 2560, a quarter of the experts with 80 rows and the rest with 8: pairs 276 / 237, down 146 / 144, with 100 and one 281 / 239, 150 / 143; 32 of 1024 x 1536: 61 /
// 53, 32.2 / 32.3, 62 / 55, 33.7 / 33.5.  Not where one expert has all rows (26 times 64): 85 / 85, 48.5 / 54.
inline bool experts_once(int64_t E, int64_t N, int64_t K, int64_t least) { return K % 64 == 0 && E * N * K >= least << 20; }

// Row groups per workgroup: one round of the 256 CUs.  More workgroups read the tokens more often (7680 x 2560, 16 tokens: 240 workgroups 10.4 us, 480
// 13.1), fewer leave CUs idle (4448 rows: two groups each on 139 workgroups 9.5 us, one each on 278 -- a second, nearly empty round -- 12.1).
inline int rows_per_workgroup(int64_t groups, int64_t problems) { return int(std::max<int64_t>(1, (groups * problems + 255) / 256)); }

// stream_rows' shape for a reduction of K columns: CALL(waves, steps per wave).  The steps of a wave are registers (4 a step for the tokens, as many for
// up to 16 fragments in flight), rounded up to a few values; OTHER runs beyond 6656 columns, and below 128 (a wave's window).
// One launch, 16 tokens, this form (by whole lines) against rows_long_kernel: 100352 x 2560 87 us (5.9 TB/s) against 147, 7680 x 2560 10.7 against 15.8, 2560 x 2560 7.4
// against 8.9, 6656 x 2560 10.2 against 15.6; at 2 tokens 76 (6.7 TB/s) against 117, 9.6 against 10.6, 6.1 against 6.3, 9.1 against 10.4.  What is left beside the
// 6.8 TB/s of a plain non-temporal read is the launch itself (about 4 us until the first results) and the tokens' rows from the L2, once per workgroup.
// Six steps from 1025 columns on, for the seven of up to 1792, a window of which a sixth lay over another wave's there.  us, seven / six: 4608 x 1536 at 48, 200 tokens 11.4 / 10.2, 17.7 / 15.7,
// 8192 x 1536 11.8 / 10.8, 23.4 / 20.9, 64000 x 1536 at 2, 16 32.8 / 31.7, 38.9 / 34.5, 32000 x 1536 at 16, 48 20.1 / 19.1, 27.8 / 25.9, 4096 x 1280 at 200 15.6 / 13.8, 5120 x 1088 17.6 / 15.6.
// Duguzen's steps, 1536 wide, three layers, 2, 4, 8, 16 tokens: 190 / 186, 230 / 222, 265 / 258, 292 / 281.  The waves' sums are other ones with it; a product's error against 64 bits, seven / six
// steps: 1088 9.1e-8 / 8.7e-8, 1280 9.3e-8 / 9.0e-8, 1536 9.5e-8 / 9.2e-8.
#define ARIA_ROWS_SHAPE(K, CALL, OTHER) \
    if ((K) < 128)                      \
        OTHER                           \
    else if ((K) <= 1024)               \
        CALL(8, 4)                      \
    else if ((K) <= 1536)               \
        CALL(8, 6)                      \
    else if ((K) <= 1792)               \
        CALL(8, 7)                      \
    else if ((K) <= 2560)               \
        CALL(8, 10)                     \
    else if ((K) <= 3328)               \
        CALL(8, 13)                     \
    else if ((K) <= 4096)               \
        CALL(8, 16)                     \
    else if ((K) <= 6656)               \
        CALL(8, 26)                     \
    else                                \
        OTHER

// The same for up to a few hundred tokens: 16, 32 or 64 at a time past the weights, as many as the registers hold beside a wave's window of the
// reduction.  K < 128 or > 4096: not served.
inline int rows_tiles(int64_t K, int64_t T) {
    const int most = K <= 2560 ? 4 : 2, need = int((T + 15) / 16);
    return need <= 1 ? 1 : need <= 2 ? 2 : most;
}
// Whether M tokens times N rows of K columns go by rows where the tiles would take them too: every pass over the weights costs about as much as the first, from
// the L2 / MALL (100352 x 2560: 16 tokens 100 us, tiles 110; 64: 120, 119; 320: 405, 212; 13312 x 2560: 192 tokens 45, 44; 256: 51, 46; 7680 x 4096: 96 tokens 35, 36;
// 128: 44, 37).
inline bool rows_ahead(int64_t M, int64_t N, int64_t K) {
    return M <= 16 || (K <= 2560 ? N * ((M + 63) / 64) <= 52000 : N * ((M + 31) / 32) <= 26000);
}
template <bool PAIR, class E>
int launch_rows_wide(const RowsIn& in, int64_t T, const E& e, void* stream) {
    const RowsPair rp{{in, in}};
    const int mt = rows_tiles(in.K, T);
    const int64_t groups = (in.N + (PAIR ? 7 : 15)) / (PAIR ? 8 : 16), ty = (T + 16 * mt - 1) / (16 * mt);
    // one round of the 256 CUs; eight workgroups on that go through the same weight rows for the next tokens, so that they are on the same XCD and find them in
    // its L2 (16384 x 2560, 160 tokens: 86 us with the others elsewhere, 49; 8192 x 1536, 320 tokens: 56, 34)
    const int64_t most = ty == 1 ? 256 : std::max<int64_t>(256 / ty / 8 * 8, 8);
    const int per = int((groups + most - 1) / most);
    const int64_t tx = (groups + per - 1) / per;
    const dim3 grid(unsigned(ty == 1 ? tx : (tx + 7) / 8 * 8), unsigned(ty));
#define ARIA_WIDE(KS, MT)                                                                                            \
    if (once)                                                                                                        \
        ARIA_LAUNCH((rows_kernel<8, KS, MT, E, PAIR, true>), grid, dim3(512), 0, stream, rp, int(T), per, e);        \
    else                                                                                                             \
        ARIA_LAUNCH((rows_kernel<8, KS, MT, E, PAIR, false>), grid, dim3(512), 0, stream, rp, int(T), per, e)
#define ARIA_WIDE_TILES(KS)  \
    if (mt == 1) {           \
        ARIA_WIDE(KS, 1);    \
    } else if (mt == 2) {    \
        ARIA_WIDE(KS, 2);    \
    } else {                 \
        ARIA_WIDE(KS, 4);    \
    }
    if (in.K < 128 || in.K > 4096) return ARIA_ERR_UNSUPPORTED;
    const bool once = rows_once(ty, in.N * (PAIR ? 2 : 1), in.K);
    if (in.K <= 1024) {
        ARIA_WIDE_TILES(4);
    } else if (in.K <= 1536) {
        ARIA_WIDE_TILES(6);
    } else if (in.K <= 1792) {
        ARIA_WIDE_TILES(7);
    } else if (in.K <= 2560) {
        ARIA_WIDE_TILES(10);
    } else if (in.K <= 3328) {
        if (mt == 1) {
            ARIA_WIDE(13, 1);
        } else {
            ARIA_WIDE(13, 2);
        }
    } else if (mt == 1) {
        ARIA_WIDE(16, 1);
    } else {
        ARIA_WIDE(16, 2);
    }
#undef ARIA_WIDE
#undef ARIA_WIDE_TILES
    return aria_check_launch();
}

template <bool PAIR, class E>
int launch_rows_of(const RowsPair& rp, int problems, int64_t T, const E& e, void* stream) {
    const int64_t groups = (rp.in[0].N + (PAIR ? 7 : 15)) / (PAIR ? 8 : 16), long_groups = (rp.in[0].N + 15) / 16;
    const int per = rows_per_workgroup(groups, problems), other = rp.in[problems - 1].K;
    const int K = std::max(rp.in[0].K, other), least = std::min(rp.in[0].K, other);
    const dim3 grid(unsigned((groups + per - 1) / per), unsigned((T + 15) / 16), unsigned(problems));
    const bool once = rows_once(grid.y, rp.in[0].N * problems, rp.in[0].K) && other % 64 == 0;   // (a pair's 2816 x 1024 at 2, 8 tokens, half lines / whole: 5.1 / 5.5, 5.8 / 6.0)
#define ARIA_ROWS_LONG ARIA_LAUNCH((rows_long_kernel<E, PAIR>), dim3(unsigned(long_groups), grid.y, grid.z), dim3(512), 0, stream, rp, int(T), e);
#define ARIA_ROWS(NW, KS)                                                                                                     \
    {                                                                                                                         \
        if (least < KS * 32) /* (a wave's window would end beyond the shorter reduction) */                                   \
            ARIA_ROWS_LONG                                                                                                    \
        else if (once)                                                                                                        \
            ARIA_LAUNCH((rows_kernel<NW, KS, 1, E, PAIR, true>), grid, dim3(NW * 64), 0, stream, rp, int(T), per, e);         \
        else                                                                                                                  \
            ARIA_LAUNCH((rows_kernel<NW, KS, 1, E, PAIR, false>), grid, dim3(NW * 64), 0, stream, rp, int(T), per, e);        \
    }
    ARIA_ROWS_SHAPE(K, ARIA_ROWS, ARIA_ROWS_LONG)
#undef ARIA_ROWS
#undef ARIA_ROWS_LONG
    return aria_check_launch();
}

template <class E>
int launch_rows(const RowsPair& rp, int problems, int64_t T, const E& e, void* stream) {
    if (T > 1) return launch_rows_of<false>(rp, problems, T, e, stream);
    ARIA_LAUNCH((row_kernel<E, false>), dim3(unsigned((rp.in[0].N + 7) / 8), 1, unsigned(problems)), dim3(256), 0, stream, rp, e);
    return aria_check_launch();
}
// gated pair: outputs e(gate, up, token, row)
template <class E>
int launch_row_pairs(const RowsIn& in, int64_t T, const E& e, void* stream) {
    const RowsPair rp{{in, in}};
    if (T > 1) return launch_rows_of<true>(rp, 1, T, e, stream);
    ARIA_LAUNCH((row_kernel<E, true>), dim3(unsigned((in.N + 3) / 4)), dim3(256), 0, stream, rp, e);
    return aria_check_launch();
}

}  // namespace
}  // namespace ad
