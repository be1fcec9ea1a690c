// C = A W^T in true 32-bit (v_mfma_f32_16x16x4_f32: 32-bit products, 32-bit sums, 128 multiply-adds a cycle and CU -- twice the vector pipe's unpacked rate).
//
// Both operands are k-contiguous: a lane loads 16 bytes of a row, four multiply steps whose reduction indices are whatever the four lanes of a row hold -- the same for
// both operands.
//
// Few outputs (gemm_f32_kernel): fragments straight from global memory.  A workgroup computes a tile of 16 MT x 16 NT outputs, its NW waves on interleaved 16-column
// steps of the reduction, DEPTH steps in flight; the partial tiles meet in LDS once.  Splitting the REDUCTION over the waves is what fills the chip where a
// serving step has a few rows only (1 .. 16 rows of a 1024-wide layer are 16 tiles of 64 columns: 100 us a launch as one 64 x 64 tile per workgroup with its
// waves side by side), and costs one pass over the tile in LDS.  16 x 16 x 8 waves up to 16 rows, where the weights' stream bounds it; 32 x 32 x 4 and 64 x 32 x 4 up to a round of tiles.
//
// More (gemm_f32_tiles_kernel): stages in the LDS.  Read from global memory, the half lines of a 16-column step are fetched from the L2 twice, which bound those tiles.
// M x N x K, us with the reduction over the waves (64 x 32 a workgroup) / by stages: 883 x 2112 x 1024 61 / 44, 883 x 2816 x 1024 77 / 53, 883 x 1024 x 2816 74 / 59,
// 1200 x 5632 x 1024 169 / 133, 2048^3 191 / 150; 16 experts of 768 x 1024, 1766 rows 50 / 36, 600 rows 26 / 20.  What is left: a tile of 64 x 64 alone takes 24 us for a
// reduction of 1024, 18 of them products (one wave a SIMD multiplies 94 .. 115 TFLOP/s with 16x16x4, two 113 .. 131), and whole rounds of tiles.
#include "aria_device.h"
#include "aria_hip.h"
#include "elem.h"
#include "gemm_f32.h"
#include <algorithm>

namespace {
using namespace ad;

typedef AriaGemmF32 GemmF32;
constexpr int FIN_HEADS = 4, FIN_ROWS = 5;   // beside gemm_f32.h's: PLAIN with rows of A by index
// a product a head (blockIdx.y) of the latent attention's expansion: the result's row t of head h times its output gate over its softmax sum
struct Heads {
    const float *ml, *gate;   // [T, H, 2] (maximum, sum), gate logits [T, ldg]
    long long ldg;
    int H, cols;              // columns of a head's result in memory (zeros behind N)
};

// The (expert, rows) of row tile y where the tiles of all experts are one sequence; every wave finds it for itself.  false: behind the last one.
__device__ __forceinline__ bool find_rows(const GemmF32& p, int y, int rows, int& e, int& m0, int& m_end) {
    const int l = threadIdx.x & 63;
    for (int e0 = 0, seen = 0; e0 < p.E; e0 += 64) {
        const bool in = e0 + l < p.E;
        const int first = in ? p.offsets[e0 + l] : 0, end = in ? p.offsets[e0 + l + 1] : 0, tiles = (end - first + rows - 1) / rows;
        const int upto = seen + wave_incl_scan(tiles);
        const unsigned long long behind = ballot(in && upto > y);
        if (behind) {
            const int at = __builtin_ctzll(behind);
            e = e0 + at;
            m0 = read_lane(first, at) + (y - read_lane(upto - tiles, at)) * rows;
            m_end = read_lane(end, at);
            return true;
        }
        seen = read_lane(upto, 63);
    }
    return false;
}

// the row of A that row m of the result comes from (the others do not ask: a dependent load and a division in front of the first fetch, 0.5 us of the 10 of 17 x 1024 x 1024)
template <int FIN>
__device__ __forceinline__ long long row_of(const GemmF32& p, int m) {
    return FIN == FIN_ROWS || (FIN == ARIA_F32_PAIR && p.rows) ? p.rows[m] / p.per : m;
}

// What becomes of a sum (v2: the second weight's): as the launches of their own would have it, act_rows_kernel and dyt_stream_kernel
template <int FIN>
__device__ __forceinline__ float finished(const GemmF32& p, float v, float v2) {
    if (FIN == ARIA_F32_RELU2) return relu_squared(v);
    if (FIN == ARIA_F32_PAIR) return (p.relu_gate ? fmaxf(v, 0.f) : v * sigmoid_exact(v)) * v2;
    return v;
}
__device__ __forceinline__ void stream_step(const GemmF32& p, float v, float& x, float& h, int n) {
    x += dyt<float>(p.post, v, n);
    if (p.next.w) h = dyt<float>(p.next, x, n);
}

// ONCE: a step's weights come as the rows 0 .. 7 of a line, the next one's as the rows 8 .. 15 (the same bits)
template <int MT, int NT, int NW, int FIN, bool ONCE>
__global__ __launch_bounds__(NW * 64) void gemm_f32_kernel(GemmF32 p) {
    constexpr bool PAIR = FIN == ARIA_F32_PAIR;
    constexpr int WS = PAIR ? 2 : 1;
    // 16 x 16 outputs: a wave takes two neighbouring steps, whole lines of both operands (us, one / two: 4 x 64000 x 1536 84 / 78, 16 x 32000 x 1024 43.6 / 42.0, 4 x 12288 x 2048
    // 26.4 / 25.7, 2 x 8192 x 1024 13.1 / 13.0)
    constexpr int PER = MT * NT == 1 ? 2 : 1, LINE = 16 * PER;
    constexpr int DEPTH = MT + NT > 4 ? 2 : 4, TM = 16 * MT, TN = 16 * NT;
    ARIA_SMEM_STATIC float red[WS][NW][TM][TN + 1];
    const int t = threadIdx.x, l = t & 63, w = first_lane(t >> 6), q4 = l >> 4, c16 = l & 15;
    const unsigned ntn = unsigned(p.N + TN - 1) / TN;
    const int y = int(blockIdx.x / ntn), n0 = int(blockIdx.x % ntn) * TN;
    int m0 = y * TM, m_end = p.M, e = 0;
    if (p.offsets && !find_rows(p, y, TM, e, m0, m_end)) return;
    const float *ap[MT], *wp[WS][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) ap[i] = p.A + row_of<FIN>(p, min(m0 + 16 * i + c16, m_end - 1)) * p.lda + w * LINE + q4 * 4;
#pragma unroll
    for (int z = 0; z < WS; ++z)
#pragma unroll
        for (int j = 0; j < NT; ++j)   // ONCE: of the first of a line's two loads, rows 0 .. 7; the second's are those eight rows on
            wp[z][j] = (z ? p.W2 : p.W) + e * p.strideW + (long long)min(n0 + 16 * j + (ONCE ? c16 & 7 : c16), p.N - 1) * p.ldw + w * LINE + (ONCE ? q4 + 4 * (c16 >> 3) : q4) * 4;
    const long long eight = ONCE ? (long long)(min(n0 + (c16 & 7) + 8, p.N - 1) - min(n0 + (c16 & 7), p.N - 1)) * p.ldw - 16 : 0;   // (behind the step's own 16 columns)
    f32x4 acc[WS][MT][NT];
#pragma unroll
    for (int z = 0; z < WS; ++z)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[z][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // whole steps; this wave's are groups w, w + NW, .. of PER, the last of which may be short
    const int steps = p.K / 16, groups = (steps + PER - 1) / PER, own = (groups - w + NW - 1) / NW;
    const int mine = own * PER - (own > 0 && w + (own - 1) * NW == groups - 1 ? groups * PER - steps : 0);
    auto at = [](int s) __attribute__((always_inline)) { return (long long)((s / PER) * NW * LINE + (s % PER) * 16); };
    struct Step {
        f32x4 a[MT], b[WS][NT];
    };
    Step x[DEPTH];
    auto load = [&](long long k, Step& f, bool second) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i) f.a[i] = *reinterpret_cast<const f32x4*>(ap[i] + k);
#pragma unroll
        for (int z = 0; z < WS; ++z)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                if constexpr (ONCE)
                    f.b[z][j] = __builtin_bit_cast(f32x4, ld16_once(wp[z][j] + k + (second ? eight : 0)));
                else
                    f.b[z][j] = *reinterpret_cast<const f32x4*>(wp[z][j] + k);
            }
    };
    // ONCE: the two loads of a line become the fragments of its two steps
    auto exchange = [&](Step& f, Step& g) __attribute__((always_inline)) {
        if constexpr (ONCE) {
#pragma unroll
            for (int z = 0; z < WS; ++z) {
                u32x4 lo, hi;
                whole_lines(__builtin_bit_cast(u32x4, f.b[z][0]), __builtin_bit_cast(u32x4, g.b[z][0]), lo, hi);
                f.b[z][0] = __builtin_bit_cast(f32x4, lo), g.b[z][0] = __builtin_bit_cast(f32x4, hi);
            }
        }
    };
    auto use = [&](const Step& f) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int z = 0; z < WS; ++z)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[z][i][j] = mfma16_f32(f.a[i][c], f.b[z][j][c], acc[z][i][j]);
    };
#pragma unroll
    for (int u = 0; u < DEPTH; ++u)
        if (u < mine) load(at(u), x[u], u & 1);
    int s = 0;
    for (; s + 2 * DEPTH <= mine; s += DEPTH) {
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            if (u % 2 == 0) exchange(x[u], x[(u + 1) % DEPTH]);
            use(x[u]);
            load(at(s + u + DEPTH), x[u], u & 1);
            sched_fence();   // (left alone the compiler asks for all of them behind the last product)
        }
    }
    for (; s < mine; s += DEPTH) {   // the last DEPTH .. 2 DEPTH - 1 steps (or fewer altogether)
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            if (s + u >= mine) break;
            if (u % 2 == 0) exchange(x[u], x[(u + 1) % DEPTH]);
            use(x[u]);
            if (s + u + DEPTH < mine) load(at(s + u + DEPTH), x[u], u & 1);
        }
    }
    if (!ONCE && (p.K & 15) && w == steps % NW) {   // the rest of the row, K % 16 = 4, 8 or 12 columns: lanes behind it hold zeros in both operands
        const bool in = q4 * 4 < (p.K & 15);
        load(in ? steps * 16 - w * LINE : -(w * LINE + q4 * 4), x[0], false);   // (not in: a column of the same row)
        if (!in) {
#pragma unroll
            for (int i = 0; i < MT; ++i) x[0].a[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int z = 0; z < WS; ++z)
#pragma unroll
                for (int j = 0; j < NT; ++j) x[0].b[z][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        use(x[0]);
    }
#pragma unroll
    for (int z = 0; z < WS; ++z)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) red[z][w][16 * i + 4 * q4 + r][16 * j + c16] = acc[z][i][j][r];
    sync();
    for (int i = t; i < TM * TN; i += NW * 64) {
        const int m = i / TN, n = i % TN;
        float v[2] = {0.f, 0.f};
#pragma unroll
        for (int z = 0; z < WS; ++z)
#pragma unroll
            for (int ww = 0; ww < NW; ++ww) v[z] += red[z][ww][m][n];
        if (m0 + m >= m_end || n0 + n >= p.N) continue;
        const long long to = (long long)(m0 + m) * p.ldc + n0 + n;
        if (FIN == ARIA_F32_STREAM) {
            float xv = p.x[to], h = 0.f;
            stream_step(p, v[0], xv, h, n0 + n);
            p.x[to] = xv;
            if (p.next.w) p.C[to] = h;
        } else {
            p.C[to] = finished<FIN>(p, v[0], v[1]);
        }
    }
}

// Tiles of 32 MI x 32 NI outputs, 2 x 2 waves of 16 MI x 16 NI, both operands through the LDS: stages of 32 columns (whole lines of 128 bytes), four of them, filled
// by LDS-DMA.  The sums are gemm_f32_kernel's with four waves, bit for bit: a wave keeps four accumulators an output, for the 16-column steps 0, 4, 8 .., 1, 5, .. and
// so on, and adds them up in that order.
// PAIR: two weights, BN rows of each in a stage.
// A piece of 16 bytes of row r lies at slot (piece ^ (r >> 1 & 7)) of the row's 128 bytes: 16 lanes that read one piece of 16 rows touch every bank once.
template <int MI, int NI, int FIN>
__global__ __launch_bounds__(256) void gemm_f32_tiles_kernel(GemmF32 p, Heads hd, int vec) {
    constexpr bool HEADS = FIN == FIN_HEADS;
    constexpr int WS = FIN == ARIA_F32_PAIR ? 2 : 1, NB = WS * NI;   // NB: blocks of 16 weight rows of a wave, the second weight's behind the first's
    constexpr int BM = 32 * MI, BN = 32 * NI, STAGE = (BM + WS * BN) * 128, P = MI + NB;   // P: pieces of a wave a stage
    static_assert(P <= 8, "requested between the four sets of products");
    ARIA_DYN_SMEM(smem);
    const int t = threadIdx.x, l = t & 63, w = first_lane(t >> 6), q4 = l >> 4, c16 = l & 15, wm = w >> 1, wn = w & 1;
    if (HEADS) p.A += (long long)blockIdx.y * p.K, p.W += blockIdx.y * p.strideW, p.C += (long long)blockIdx.y * hd.cols;
    const int cols = HEADS ? hd.cols : p.N;
    const unsigned ntn = unsigned(cols + BN - 1) / BN;
    const int y = int(blockIdx.x / ntn), n0 = int(blockIdx.x % ntn) * BN;
    int m0 = y * BM, m_end = p.M, e = 0;
    if (p.offsets && !find_rows(p, y, BM, e, m0, m_end)) return;
    // this lane's pieces of a stage: rows 8 (w + 4 i) + l / 8 of [A's rows, W's rows], rows behind the end the last one again
    const float* src[P];
    int at[P];   // its column
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int r = 8 * (w + 4 * i) + (l >> 3);
        at[i] = ((l & 7) ^ (r >> 1 & 7)) * 4;
        const int rw = r < BM + BN ? r - BM : r - BM - BN;
        src[i] = r < BM ? p.A + row_of<FIN>(p, min(m0 + r, m_end - 1)) * p.lda : (r < BM + BN ? p.W : p.W2) + e * p.strideW + (long long)min(n0 + rw, p.N - 1) * p.ldw;
    }
    auto piece = [&](int s, int i) __attribute__((always_inline)) {   // of stage s (columns behind the row's end: its first ones; never used)
        const int k = 32 * s + at[i];
        glds16_raw(src[i] + (k < p.K ? k : 0), smem + (s & 3) * STAGE + (w + 4 * i) * 1024);
    };
    f32x4 acc[4][MI][NB];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[c][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int n = (p.K + 31) / 32, turn = c16 >> 1 & 7;
    const char *arow = smem + (wm * 16 * MI + c16) * 128, *brow = smem + (BM + wn * 16 * NI + c16) * 128;
    struct Half {   // 16 columns of a wave's rows
        f32x4 a[MI], b[NB];
    };
    auto load = [&](Half& f, int s, int half) __attribute__((always_inline)) {
        const int o = (s & 3) * STAGE + ((4 * half + q4) ^ turn) * 16;
#pragma unroll
        for (int i = 0; i < MI; ++i) f.a[i] = *reinterpret_cast<const f32x4*>(arow + o + i * 2048);
#pragma unroll
        for (int j = 0; j < NB; ++j) f.b[j] = *reinterpret_cast<const f32x4*>(brow + o + j / NI * (BN * 128) + j % NI * 2048);
        sched_fence();   // (left alone the compiler moves the reads down to their use)
    };
    // the products of 16 columns, and between them the requests of stage s (none behind the last one)
    auto use = [&](const Half& f, f32x4(&sum)[MI][NB], int s) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j) sum[i][j] = mfma16_f32(f.b[j][c], f.a[i][c], sum[i][j]);   // (a lane: row c16, columns 4 q4 .. + 3)
            if (c < P && s < n) piece(s, c);
            if (c + 4 < P && s < n) piece(s, c + 4);
        }
        sched_fence();
    };
    auto arrive = [&](int s) __attribute__((always_inline)) {   // stage s is there for all waves, stage s - 1 is free
        if (s == 0 && n > 3)
            wait_vm<3 * P>();
        else if (s + 2 < n)
            wait_vm<2 * P>();
        else if (s + 1 < n)
            wait_vm<P>();
        else
            wait_vm<0>();
        wait_lds();
        raw_barrier();
    };
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < P; ++i)
            if (s < n) piece(s, i);
    arrive(0);
    int s = 0;
    const int whole = p.K / 64 * 2;
    if (whole) {
        Half f0, f1;
        load(f0, 0, 0);
        for (; s < whole; s += 2) {   // (every read one set of products ahead of its use; behind the last stage it finds an old one's, which nothing uses)
            load(f1, s, 1);
            use(f0, acc[0], n);
            arrive(s + 1);
            load(f0, s + 1, 0);
            use(f1, acc[1], s + 4);
            load(f1, s + 1, 1);
            use(f0, acc[2], n);
            arrive(s + 2);
            load(f0, s + 2, 0);
            use(f1, acc[3], s + 5);
        }
    }
    if (s < n) {   // the rest of the rows: at most 60 columns
        const int rest = p.K - 32 * s;
        auto step = [&](int s, int half, f32x4(&sum)[MI][NB], int left) __attribute__((always_inline)) {   // left: columns that the rows have from here
            if (left <= 0) return;
            Half f;
            load(f, s, half);
            if (4 * q4 >= left) {
#pragma unroll
                for (int i = 0; i < MI; ++i) f.a[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < NB; ++j) f.b[j] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            use(f, sum, n);
        };
        step(s, 0, acc[0], rest);
        step(s, 1, acc[1], rest - 16);
        if (rest > 32) {
            arrive(s + 1);
            step(s + 1, 0, acc[2], rest - 32);
            step(s + 1, 1, acc[3], rest - 48);
        }
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int m = m0 + 16 * (wm * MI + i) + c16;
        if (m >= m_end) continue;
        float sum = 1.f, z = 0.f;
        if (HEADS) sum = hd.ml[((long long)m * hd.H + blockIdx.y) * 2 + 1], z = sigmoid_exact(hd.gate[m * hd.ldg + blockIdx.y]);
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const int c0 = n0 + 16 * (wn * NI + j) + 4 * q4;
            f32x4 v, v2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    v[r] += acc[c][i][j][r];
                    if (WS == 2) v2[r] += acc[c][i][(WS - 1) * NI + j][r];
                }
                if (HEADS)
                    v[r] = c0 + r < p.N ? v[r] / sum * z : 0.f;
                else
                    v[r] = finished<FIN>(p, v[r], v2[r]);
            }
            const long long to = (long long)m * p.ldc + c0;
            if (vec && c0 + 3 < cols) {
                if (FIN == ARIA_F32_STREAM) {
                    f32x4 x = *reinterpret_cast<const f32x4*>(p.x + to), h = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float xr = x[r], hr = 0.f;
                        stream_step(p, v[r], xr, hr, c0 + r);
                        x[r] = xr, h[r] = hr;
                    }
                    *reinterpret_cast<f32x4*>(p.x + to) = x;
                    v = h;
                    if (!p.next.w) continue;
                }
                *reinterpret_cast<f32x4*>(p.C + to) = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (c0 + r >= cols) continue;
                    if (FIN == ARIA_F32_STREAM) {
                        float x = p.x[to + r], h = 0.f;
                        stream_step(p, v[r], x, h, c0 + r);
                        p.x[to + r] = x;
                        if (p.next.w) p.C[to + r] = h;
                    } else {
                        p.C[to + r] = v[r];
                    }
                }
            }
        }
    }
}

template <int MT, int NT, int NW, int FIN>
int launch_f32(const GemmF32& p, void* stream) {
    const int64_t ntm = (int64_t(p.M) + 16 * MT - 1) / (16 * MT) + (p.offsets ? p.E : 0);   // (an expert's last tile may be ragged)
    const int64_t ntn = (int64_t(p.N) + 16 * NT - 1) / (16 * NT);
    if (ntm * ntn > 0x7fffffff) return ARIA_ERR_UNSUPPORTED;
    if constexpr (MT * NT == 1) {
        // Weights by whole lines, non-temporal (whole_lines): read once, and enough of them.  Us, half lines / whole: 4 x 32000 x 1024 29.9 / 26.9, 16 40.3 / 35.5, 16 x 64000 x 1536 120 / 99,
        // 4 x 2816 x 1024 5.7 / 5.4, 4 x 6656 x 2560 19.7 / 17.5; 4 x 1024 x 1024 5.0 / 5.0, 4 x 512 x 256 2.6 / 3.0;
        // By expert: 64 of 1664 x 2560, 2, 8, 16 rows each 204 / 188, 260 / 212, 334 / 275, a quarter of them with 40 rows and the rest with 2 (several tiles, each of which fetches the weights anew) 334 /
        // 305; 32 of 1024 x 1536 36.8 / 32.5, 49 / 40, 62 / 53, 62.6 / 58.2.  16 of 768 x 1024 (50 MB), which the Infinity Cache holds: 13.6 / 13.1, 15.0 / 14.6, 16.2 / 16.3, a quarter with 24 and the
        // rest with 8 16.1 / 16.7, with 40 and 2 18.0 / 18.5: there up to eight rows each on average.
        if (p.K % 32 == 0 && p.ldw % 32 == 0 && p.strideW % 32 == 0 &&
            (p.offsets ? p.M <= 8 * p.E || (long long)p.E * p.N * p.K >= 16 << 20 : (long long)p.N * p.K >= 3 << 19)) {
            ARIA_LAUNCH((gemm_f32_kernel<MT, NT, NW, FIN, true>), dim3(unsigned(ntm * ntn)), dim3(NW * 64), 0, stream, p);
            return aria_check_launch();
        }
    }
    ARIA_LAUNCH((gemm_f32_kernel<MT, NT, NW, FIN, false>), dim3(unsigned(ntm * ntn)), dim3(NW * 64), 0, stream, p);
    return aria_check_launch();
}

template <int MI, int NI, int FIN>
int launch_f32_tiles(const GemmF32& p, const Heads& hd, void* stream) {
    constexpr bool HEADS = FIN == FIN_HEADS;
    constexpr int BM = 32 * MI, BN = 32 * NI;
    const int64_t ntm = (int64_t(p.M) + BM - 1) / BM + (p.offsets ? p.E : 0);   // (an expert's last tile may be ragged)
    const int64_t ntn = ((HEADS ? hd.cols : p.N) + BN - 1) / BN;
    if (ntm * ntn > 0x7fffffff) return ARIA_ERR_UNSUPPORTED;
    const int vec = !(p.ldc & 3) && !((reinterpret_cast<uintptr_t>(p.C) | reinterpret_cast<uintptr_t>(p.x)) & 15) && !(HEADS && (hd.cols & 3));
    ARIA_LAUNCH((gemm_f32_tiles_kernel<MI, NI, FIN>), dim3(unsigned(ntm * ntn), unsigned(HEADS ? hd.H : 1)), dim3(256), 4 * (BM + (FIN == ARIA_F32_PAIR ? 2 : 1) * BN) * 128, stream, p, hd, vec);
    return aria_check_launch();
}

template <int FIN>
int product_f32(const GemmF32& p, void* stream) {
    if (p.offsets ? p.M <= 16 * p.E : p.M <= 16) return launch_f32<1, 1, 8, FIN>(p, stream);
    // Up to a round of 32 x 32 tiles, and of 64 x 32 ones, the reduction over the waves is the shorter chain (us, here / by stages: 48 x 1024 x 2816 22 / 24; 64 x 32: 300 x 1024 x 2816
    // 35 / 40, 500 x 768 x 2048 27 / 30, 100 x 2816 x 1024 15 / 17).  Beyond them the rounds of the chip decide, and of equal ones the larger tile (883 x 2112 x 1024, us as 64 x 64 / 32 x 64 / 32 x 32: 44 / 47 / 48; 883 x 2816 x 1024 61 / 53 / 55; 300 x 2112 x 1024
    // 24 / 25 / 20).  An expert's last tile stands half empty on average; for the first question every expert counts as one tile at least, which is what evenly spread rows come to (8 experts of
    // 768 x 1024, 200 rows: even 12 / 17, as a router spreads them 16 / 17).
    const int64_t M = p.M, N = p.N, round = 256;
    auto cols = [&](int ni) { return (N + 32 * ni - 1) / (32 * ni); };
    auto tiles = [&](int mi, int ni) { return ((M + 32 * mi - 1) / (32 * mi) + (p.offsets ? p.E / 2 : 0)) * cols(ni); };
    if ((p.offsets ? std::max<int64_t>((M + 31) / 32, p.E) * cols(1) : tiles(1, 1)) <= round) return launch_f32<2, 2, 4, FIN>(p, stream);
    if constexpr (FIN != ARIA_F32_PAIR) {   // (two weights' sums of 64 x 32 do not fit the static LDS)
        if (!p.offsets && tiles(2, 1) <= round) return launch_f32<4, 2, 4, FIN>(p, stream);
    }
    auto cost = [&](int mi, int ni, int more) { return (tiles(mi, ni) + round - 1) / round * mi * ni * (100 + more); };
    const int64_t c22 = cost(2, 2, 0), c12 = cost(1, 2, 5), c11 = cost(1, 1, 10);
    if (c22 <= c12 && c22 <= c11) return launch_f32_tiles<2, 2, FIN>(p, {}, stream);
    return c12 <= c11 ? launch_f32_tiles<1, 2, FIN>(p, {}, stream) : launch_f32_tiles<1, 1, FIN>(p, {}, stream);
}

}  // namespace

__attribute__((visibility("hidden"))) int aria_gemm_f32_heads(const float* part_o, const float* uv, float* out, const AriaLatentShape& s, const float* part_ml, const float* proj,
                                                              int64_t T, void* stream) {
    GemmF32 p{};
    p.A = part_o, p.W = uv, p.C = out, p.M = int(T), p.N = int(s.dv), p.K = int(s.R);
    p.lda = s.H * s.R, p.ldw = s.rp, p.ldc = s.H * s.dvp, p.E = 1, p.strideW = s.dv * s.rp;
    const Heads hd{part_ml, proj + s.g_off, (long long)s.ldp, int(s.H), int(s.dvp)};
    // (883 tokens, 8 heads of 128 x 256, us: 64 x 32 with the reduction over the waves 13.3, tiles of 32 x 32 10.9, 32 x 64 10.4, 64 x 64 11.6)
    return launch_f32_tiles<1, 2, FIN_HEADS>(p, hd, stream);
}

int aria_gemm_f32_finished(const AriaGemmF32& p, int finish, void* stream) {
    if (!p.A || !p.W || !p.C || p.M < 0 || p.N < 0 || p.K <= 0 || (p.offsets && p.E <= 0) || (p.rows && p.per <= 0) || (finish == ARIA_F32_PAIR && !p.W2) ||
        (finish == ARIA_F32_STREAM && (!p.x || !p.post.w || p.offsets)) || (p.rows && (finish == ARIA_F32_RELU2 || finish == ARIA_F32_STREAM)))
        return ARIA_ERR_INVALID;
    if (((reinterpret_cast<uintptr_t>(p.A) | reinterpret_cast<uintptr_t>(p.W) | reinterpret_cast<uintptr_t>(p.W2)) & 15) || (p.lda & 3) || (p.ldw & 3) || (p.K & 3) || (p.strideW & 3))
        return ARIA_ERR_ALIGN;
    if (p.M == 0 || p.N == 0) return ARIA_OK;
    if ((p.M + 63) / 64 > 65535 || p.E > 65535) return ARIA_ERR_UNSUPPORTED;
    switch (finish) {
        case ARIA_F32_RELU2: return product_f32<ARIA_F32_RELU2>(p, stream);
        case ARIA_F32_PAIR: return product_f32<ARIA_F32_PAIR>(p, stream);
        case ARIA_F32_STREAM: return product_f32<ARIA_F32_STREAM>(p, stream);
        default: return p.rows ? product_f32<FIN_ROWS>(p, stream) : product_f32<ARIA_F32_PLAIN>(p, stream);
    }
}

extern "C" {

int aria_gemm_f32(const float* A, const float* W, float* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t ldc,
                  const int32_t* offsets, int64_t E, int64_t strideW, void* stream) {
    if (!A || !W || !C || M < 0 || N < 0 || K <= 0 || (offsets && E <= 0)) return ARIA_ERR_INVALID;
    if (((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) & 15) || (lda & 3) || (ldw & 3) || (K & 3) || (strideW & 3)) return ARIA_ERR_ALIGN;
    if (M == 0 || N == 0) return ARIA_OK;
    if ((M + 63) / 64 > 65535 || E > 65535) return ARIA_ERR_UNSUPPORTED;
    AriaGemmF32 p{};
    p.A = A, p.W = W, p.C = C, p.M = int(M), p.N = int(N), p.K = int(K), p.lda = lda, p.ldw = ldw, p.ldc = ldc, p.offsets = offsets, p.E = int(offsets ? E : 1), p.strideW = strideW;
    return product_f32<ARIA_F32_PLAIN>(p, stream);
}

}  // extern "C"
