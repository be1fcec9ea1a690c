// C = A W^T in true 32-bit (v_mfma_f32_16x16x4_f32: 32-bit products, 32-bit sums, 256 multiply-adds a cycle and CU -- twice the vector pipe's unpacked rate).
//
// Both operands are k-contiguous, so fragments come straight from global memory: a lane loads 16 bytes of a row, four multiply steps whose reduction
// indices are whatever the four lanes of a row hold -- the same for both operands.  A workgroup computes a tile of 16 MT x 16 NT outputs, its NW waves on
// interleaved 16-column steps of the reduction, DEPTH steps in flight; the partial tiles meet in LDS once.  Splitting the REDUCTION over the waves is what
// fills the chip where a serving step has a few rows only (1 .. 16 rows of a 1024-wide layer are 16 tiles of 64 columns: 100 us a launch as one 64 x 64
// tile per workgroup with its waves side by side), and costs one pass over the tile in LDS.
// M x N x K, us as one 64 x 64 tile a workgroup on the vector pipe / now (relative error against 64 bits 5.7e-7 / 2.1e-7 at K = 1024): 4 x 2112 x 1024 57 / 10,
// 4 x 32000 x 1024 73 / 28, 16 x 1024 x 2816 152 / 12, 300 x 1024 x 1024 59 / 15, 883 x 1024 x 2816 176 / 76, 4096^3 1786 / 1480; 16 experts of 768 x 1024: 8
// rows 58 / 10, 1240 rows 136 / 43.  Tiles (rows x columns, waves): 16 x 16 x 8 up to 16 rows, where the weights' stream bounds it; 32 x 32 x 4 up to 64 rows, and
// for experts up to 128; 64 x 32 x 4 (620 x 2112 x 1024: 47 us, 32 x 32 x 4 49, 64 x 64 x 4 54); 64 x 64 x 4 from 512 tiles, where the L2's rate counts (4096^3:
// 1480 us, 64 x 32 x 4 1650).
#include "aria_device.h"
#include "aria_hip.h"
#include "elem.h"
#include <algorithm>

namespace {
using namespace ad;

struct GemmF32 {
    const float *A, *W;
    float* C;
    int M, N, K;
    long long lda, ldw, ldc;
    const int* offsets;   // rows grouped by expert, or NULL
    int E;
    long long strideW;
};
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

template <int MT, int NT, int NW, bool HEADS>
__global__ __launch_bounds__(NW * 64) void gemm_f32_kernel(GemmF32 p, Heads hd) {
    constexpr int DEPTH = MT + NT > 4 ? 2 : 4, TM = 16 * MT, TN = 16 * NT;
    ARIA_SMEM_STATIC float red[NW][TM][TN + 1];
    const int t = threadIdx.x, l = t & 63, w = first_lane(t >> 6), q4 = l >> 4, c16 = l & 15;
    if (HEADS) p.A += (long long)blockIdx.y * p.K, p.W += blockIdx.y * p.strideW, p.C += (long long)blockIdx.y * hd.cols;
    const unsigned ntn = unsigned((HEADS ? hd.cols : p.N) + TN - 1) / TN;
    const int y = int(blockIdx.x / ntn), n0 = int(blockIdx.x % ntn) * TN;
    int m0 = y * TM, m_end = p.M, e = 0;
    if (p.offsets && !find_rows(p, y, TM, e, m0, m_end)) return;
    const float *ap[MT], *wp[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) ap[i] = p.A + (long long)min(m0 + 16 * i + c16, m_end - 1) * p.lda;
#pragma unroll
    for (int j = 0; j < NT; ++j) wp[j] = p.W + e * p.strideW + (long long)min(n0 + 16 * j + c16, p.N - 1) * p.ldw;
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int steps = p.K / 16, mine = (steps - w + NW - 1) / NW;   // whole steps; this wave's: w, w + NW, ...
#pragma unroll
    for (int i = 0; i < MT; ++i) ap[i] += w * 16 + q4 * 4;
#pragma unroll
    for (int j = 0; j < NT; ++j) wp[j] += w * 16 + q4 * 4;
    f32x4 a[DEPTH][MT], b[DEPTH][NT];
    auto load = [&](int s, f32x4(&av)[MT], f32x4(&bv)[NT]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i) av[i] = *reinterpret_cast<const f32x4*>(ap[i] + s * NW * 16);
#pragma unroll
        for (int j = 0; j < NT; ++j) bv[j] = *reinterpret_cast<const f32x4*>(wp[j] + s * NW * 16);
    };
    auto use = [&](const f32x4(&av)[MT], const f32x4(&bv)[NT]) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = mfma16_f32(av[i][c], bv[j][c], acc[i][j]);
    };
#pragma unroll
    for (int u = 0; u < DEPTH; ++u)
        if (u < mine) load(u, a[u], b[u]);
    int s = 0;
    for (; s + 2 * DEPTH <= mine; s += DEPTH) {
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            use(a[u], b[u]);
            load(s + u + DEPTH, a[u], b[u]);
        }
    }
    for (; s < mine; s += DEPTH) {   // the last DEPTH .. 2 DEPTH - 1 steps (or fewer altogether)
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            if (s + u >= mine) break;
            use(a[u], b[u]);
            if (s + u + DEPTH < mine) load(s + u + DEPTH, a[u], b[u]);
        }
    }
    if ((p.K & 15) && w == steps % NW) {   // the rest of the row, K % 16 = 4, 8 or 12 columns: lanes behind it hold zeros in both operands
        const bool in = q4 * 4 < (p.K & 15);
        const int back = in ? mine * NW * 16 : -(w * 16 + q4 * 4);   // (a column of the same row)
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            a[0][i] = *reinterpret_cast<const f32x4*>(ap[i] + back);
            if (!in) a[0][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            b[0][j] = *reinterpret_cast<const f32x4*>(wp[j] + back);
            if (!in) b[0][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        use(a[0], b[0]);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[w][16 * i + 4 * q4 + r][16 * j + c16] = acc[i][j][r];
    sync();
    for (int i = t; i < TM * TN; i += NW * 64) {
        const int m = i / TN, n = i % TN;
        float v = 0.f;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) v += red[ww][m][n];
        if (HEADS) {
            if (m0 + m < m_end && n0 + n < hd.cols) {
                const float sum = hd.ml[((long long)(m0 + m) * hd.H + blockIdx.y) * 2 + 1], z = hd.gate[(m0 + m) * hd.ldg + blockIdx.y];
                p.C[(long long)(m0 + m) * p.ldc + n0 + n] = n0 + n < p.N ? v / sum * sigmoid_exact(z) : 0.f;
            }
        } else if (m0 + m < m_end && n0 + n < p.N) {
            p.C[(long long)(m0 + m) * p.ldc + n0 + n] = v;
        }
    }
}

template <int MT, int NT, int NW>
int launch_f32(const GemmF32& p, void* stream) {
    const int64_t ntm = (int64_t(p.M) + 16 * MT - 1) / (16 * MT) + (p.offsets ? p.E : 0);   // (an expert's last tile may be ragged)
    const int64_t ntn = (int64_t(p.N) + 16 * NT - 1) / (16 * NT);
    if (ntm * ntn > 0x7fffffff) return ARIA_ERR_UNSUPPORTED;
    ARIA_LAUNCH((gemm_f32_kernel<MT, NT, NW, false>), dim3(unsigned(ntm * ntn)), dim3(NW * 64), 0, stream, p, Heads{});
    return aria_check_launch();
}

}  // namespace

__attribute__((visibility("hidden"))) int aria_gemm_f32_heads(const float* part_o, const float* uv, float* out, const AriaLatentShape& s, const float* part_ml, const float* proj,
                                                              int64_t T, void* stream) {
    const GemmF32 p{part_o, uv, out, int(T), int(s.dv), int(s.R), (long long)(s.H * s.R), (long long)s.rp, (long long)(s.H * s.dvp), nullptr, 1, (long long)(s.dv * s.rp)};
    const Heads hd{part_ml, proj + s.g_off, (long long)s.ldp, int(s.H), int(s.dvp)};
    ARIA_LAUNCH((gemm_f32_kernel<4, 2, 4, true>), dim3(unsigned((T + 63) / 64 * ((s.dvp + 31) / 32)), unsigned(s.H)), dim3(256), 0, stream, p, hd);
    return aria_check_launch();
}

extern "C" {

int aria_gemm_f32(const float* A, const float* W, float* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t ldc,
                  const int32_t* offsets, int64_t E, int64_t strideW, void* stream) {
    if (!A || !W || !C || M < 0 || N < 0 || K <= 0 || (offsets && E <= 0)) return ARIA_ERR_INVALID;
    if (((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) & 15) || (lda & 3) || (ldw & 3) || (K & 3) || (strideW & 3)) return ARIA_ERR_ALIGN;
    if (M == 0 || N == 0) return ARIA_OK;
    if ((M + 63) / 64 > 65535 || E > 65535) return ARIA_ERR_UNSUPPORTED;
    const GemmF32 p{A, W, C, int(M), int(N), int(K), (long long)lda, (long long)ldw, (long long)ldc, (const int*)offsets, int(offsets ? E : 1), (long long)strideW};
    const int64_t rows = offsets ? (M + E - 1) / E : M;   // of an expert on average
    const int64_t tiles = (M + 63) / 64 * ((N + 63) / 64);
    if (rows <= 16) return launch_f32<1, 1, 8>(p, stream);
    if (rows <= (offsets ? 128 : 64)) return launch_f32<2, 2, 4>(p, stream);
    return tiles < 512 ? launch_f32<4, 2, 4>(p, stream) : launch_f32<4, 4, 4>(p, stream);
}

}  // extern "C"
