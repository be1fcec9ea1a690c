// The thin products of a low-rank adapter (rank 8 or 16) of a training step: result = base(x) + lora_B(lora_A(dropout(x))) * scaling
// (aria/lora/layers.py:129-139; for nn.Linear peft's adapter, the same line).  The base launch carries lora_B (the *_lora_* entries); here are
//   u:      scale * dropout(x) lora_A              (thin_product_kernel: the general tiles' bits) into the adapter's columns of the launch's extension
//   scale:  u * scaling                            where the general product computes u
//   down:   d_u = scale * dy W^T                   with lora_B
//   up:     dx += keep ? (d_u A) / (1 - p) : 0     the adapter's input gradient through its dropout mask, added where the base's gradient lies
//   wgrad:  dW = y^T u                             dense adapters' weight gradients (the experts' run as grouped products)
// The last three are bound by the bytes of the one wide operand; a 256-wide tile of the general kernels is 97 % padding here.  Rank 8, us a call with the launches:
// 4096 rows of 2560, down as a split 256 x 256 tile, its sum and three passes for the scaling 37, here 9 (the scaling alone 16 with its copy, here 3.5); up as a
// product and a masked add 22, here 10; wgrad as a split product and its sum 24, here 11 (64 rows a block: 12.5 us on cold rows, with 128 and four loads in flight a
// wave 15.5).  24 576 rows of 64 experts, 2560 wide: down 51 and 12 for the scaling, here 26; up 142, here 51 (6.1 TB/s would take 21 and 43).  An adapted training
// step of 4 x 1024 tokens 11 350 / 10 030.
#include "aria_device.h"
#include "aria_hip.h"
#include "elem.h"
#include "gemm_params.h"
#include <algorithm>
#include <type_traits>

namespace {
using namespace ad;

constexpr int ROWS = 32;                // rows of a block
constexpr int PAD = 32;                 // a row of the staged factor ends 64 bytes further: rows start on different banks
constexpr int64_t LDS_MAX = 112 << 10;  // the staged factor: rank 16 up to 3552 columns, 32 columns of 1728

// The rows of a block: block bid's tile of 32, or with offsets the bid-th of the tiles of 32 rows that start anew at every expert (collective; false: none left).
__device__ __forceinline__ bool rows_of(const int32_t* offsets, int E, int M, int bid, int& e, int& m0, int& m1) {
    if (!offsets) {
        e = 0, m0 = bid * ROWS, m1 = M;
        return m0 < M;
    }
    const int l = threadIdx.x & 63;
    int before = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
        const int n = e0 + l < E ? offsets[e0 + l + 1] - offsets[e0 + l] : 0, t = (n + ROWS - 1) / ROWS, incl = wave_incl_scan(t);
        const unsigned long long hit = ballot(before + incl > bid);
        if (hit) {
            const int j = __builtin_ctzll(hit);
            e = e0 + j;
            m0 = offsets[e] + (bid - before - wave_bcast(incl - t, j)) * ROWS;
            m1 = offsets[e + 1];
            return true;
        }
        before += wave_bcast(incl, 63);
    }
    return false;
}

__global__ __launch_bounds__(256) void lora_scale_kernel(const bf16_t* u, bf16_t* out, long long n, int pieces, long long ldo, float scale) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const u32x4 v = ld16(u + 8 * i);
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = pack2bf(bflo(v[q]) * scale, bfhi(v[q]) * scale);
    st16(out + i / pieces * ldo + 8 * (i % pieces), o);
}

// u[m][n] = scale * sum_k X[m][k] W[n][k], n < r.  W: [r][K], or with w_oc [K][r]; per expert where there are offsets.
// The factor is staged once a block, k-contiguous whichever way it lies; the eight waves take every eighth 64 columns of the reduction, four such steps of 32 rows
// in flight each, straight from global memory (16-row fragments of v_mfma_f32_16x16x32_bf16 read 64 bytes of a row, its neighbour the other half of the line).
// Splitting the reduction over the waves is what puts 4096 rows on 128 CUs with all of a block's bytes in flight at once.
__global__ __launch_bounds__(512) void lora_down_kernel(const bf16_t* X, const bf16_t* W, bf16_t* U, const int32_t* offsets, int E, int M, int K, int r, int w_oc,
                                                        long long ldx, long long ldu, float scale) {
    ARIA_DYN_SMEM(lds);
    bf16_t* wt = reinterpret_cast<bf16_t*>(lds);
    const int l = threadIdx.x & 63, lr = l & 15, kg = l >> 4, w = first_lane(int(threadIdx.x) >> 6), pitch = K + PAD, nch = K / 64;
    int e, m0, m1;
    if (!rows_of(offsets, E, M, blockIdx.x, e, m0, m1)) return;
    const bf16_t* xr[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) xr[h] = X + (long long)min(m0 + 16 * h + lr, m1 - 1) * ldx + 8 * kg;   // (rows past the end: the last one, never stored)
    s16x8 x[4][2][2];
    auto load = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (c0 + 8 * i < nch)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int s = 0; s < 2; ++s) x[i][h][s] = *reinterpret_cast<const s16x8*>(xr[h] + (c0 + 8 * i) * 64 + 32 * s);
    };
    load(w);
    const bf16_t* we = W + (long long)e * r * K;
    for (int i = threadIdx.x; i < r * K / 8; i += 512) {
        const u32x4 v = ld16(we + 8ll * i);
        if (w_oc) {
            const int k = i / (r / 8), n = 8 * (i % (r / 8));
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                wt[(n + 2 * q) * pitch + k] = bf16_t(v[q] & 0xffffu);
                wt[(n + 2 * q + 1) * pitch + k] = bf16_t(v[q] >> 16);
            }
        } else {
            const int n = i / (K / 8), k = 8 * (i % (K / 8));
            st16(wt + n * pitch + k, v);
        }
    }
    sync();
    f32x4 acc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) acc[h] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16_t* wr = wt + min(lr, r - 1) * pitch + 8 * kg;   // (past the last column: the last one again, never stored)
    for (int c0 = w; c0 < nch; c0 += 32) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (c0 + 8 * i < nch)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const s16x8 b = *reinterpret_cast<const s16x8*>(wr + (c0 + 8 * i) * 64 + 32 * s);
#pragma unroll
                    for (int h = 0; h < 2; ++h) acc[h] = mfma16(x[i][h][s], b, acc[h]);
                }
        if (c0 + 32 < nch) load(c0 + 32);
    }
    sync();
    float* red = reinterpret_cast<float*>(lds);   // [wave][row][16]
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[(w * ROWS + 16 * h + 4 * kg + i) * 16 + lr] = acc[h][i];
    sync();
    for (int i = threadIdx.x; i < ROWS * r; i += 512) {
        const int row = i / r, n = i % r;
        float s = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q) s += red[(q * ROWS + row) * 16 + n];
        if (m0 + row < m1) U[(long long)(m0 + row) * ldu + n] = f2bf(scale * s);
    }
}

// C[m][n] = sum_k X[m][k] W[n][k] in 32 bits, N <= 32 columns: the router's product of a mixture with up to 32 experts.
// The choice of experts hangs on its last bits, so they are those of the general tiles: an element is one chain of v_mfma_f32_32x32x16_bf16 over the reduction, in `cut` pieces
// for the rows from cut_row on, where those tiles would split it.  That chain (K / 16 products of one wave) and a block's own loads are the time; splitting the reduction
// over the waves adds in another order and is hardly ahead (us: 5580 rows of 1536 on 32 columns 9.9, here 9.6, in a prompt's step 11.6, here 12.3; 16 384 rows 16.2, here 16.1;
// 2000 rows of 3328 on 16 columns 10.1, here 15.2).  The eight waves stage W once a block and X in rounds of 512 columns, the next two in flight in registers (one: 15.3 in the
// step); the first wave multiplies.
// 5580 rows of 1536 on 32 columns as 128 x 128 tiles of the general kernel 25.8 us.
constexpr int XR = 512, XPITCH = XR + 8;   // (16 bytes: 16 rows' pieces lie on different banks)
// An adapter's u = bf16(scale * bf16(x W)) too (T = bf16_t; per expert where there are offsets, W_OC: W [K][N]): the forward's, in front of routers like the base products.  With the launches it takes
// the place of, us: cold rows, rank 8: 777 of 2560 27.6, here 21.5, 4096 32 / 19, 16 384 56 / 40; rows by expert, 4662 of 2560 58 / 19, 24 576 74 / 56, 98 304 174 / 151; where it
// is the slower one: lora_u_takes of ops.py.
template <bool W_OC, class T>
__global__ __launch_bounds__(512) void thin_product_kernel(const bf16_t* X, const bf16_t* W, T* C, const int32_t* offsets, int E, int M, int N, int K, long long ldx, long long ldc,
                                                           int cut_row, int cut, float scale) {
    ARIA_DYN_SMEM(lds);
    int e = 0, m0 = blockIdx.x * ROWS;
    if (sizeof(T) == 2 && !rows_of(offsets, E, M, blockIdx.x, e, m0, M)) return;   // (routers have no experts to ask for: 0.3 us of 7)
    const int t = threadIdx.x, l = t & 63, w = first_lane(t >> 6), pitch = K + 8, nch = K / 64, pieces = m0 >= cut_row ? cut : 1;
    bf16_t* xs = reinterpret_cast<bf16_t*>(lds);   // [32][XPITCH]
    bf16_t* ws = xs + ROWS * XPITCH;               // [N][pitch]
    u32x4 xa[4], xb[4];
    auto load = [&](u32x4 (&x)[4], int k0) __attribute__((always_inline)) {
        if (k0 + 8 * l < K)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = ld16(X + (long long)min(m0 + w + 8 * i, M - 1) * ldx + k0 + 8 * l);   // (rows past the end: the last one, never stored)
    };
    load(xa, 0);
    load(xb, XR);
#pragma unroll 6
    for (int i = t; i < N * K / 8; i += 512) {
        const u32x4 v = ld16(W + (long long)e * N * K + 8ll * i);
        if (W_OC) {
            const int k = i / (N / 8), n = 8 * (i % (N / 8));
#pragma unroll
            for (int q = 0; q < 4; ++q) ws[(n + 2 * q) * pitch + k] = bf16_t(v[q] & 0xffffu), ws[(n + 2 * q + 1) * pitch + k] = bf16_t(v[q] >> 16);
        } else {
            st16(ws + i / (K / 8) * pitch + 8 * (i % (K / 8)), v);
        }
    }
    f32x16 acc, sum;
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = sum[j] = 0.f;
    const bf16_t *xf = xs + (l & 31) * XPITCH + 8 * (l >> 5), *wf = ws + min(l & 31, N - 1) * pitch + 8 * (l >> 5);
    int piece = 0;
    auto round = [&](u32x4 (&x)[4], int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) st16(xs + (w + 8 * i) * XPITCH + 8 * l, x[i]);
        load(x, 64 * c0 + 2 * XR);
        sync();
        if (w == 0) {
#pragma unroll
            for (int cc = 0; cc < XR / 64; ++cc) {
                const int c = c0 + cc;
                if (c >= nch) break;
                if (piece + 1 < pieces && c == int((long long)nch * (piece + 1) / pieces)) {
#pragma unroll
                    for (int j = 0; j < 16; ++j) sum[j] = piece ? sum[j] + acc[j] : acc[j], acc[j] = 0.f;
                    ++piece;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc = mfma32(*reinterpret_cast<const s16x8*>(wf + c * 64 + 16 * i), *reinterpret_cast<const s16x8*>(xf + cc * 64 + 16 * i), acc);
            }
        }
        sync();
    };
    for (int c0 = 0; c0 < nch; c0 += 2 * XR / 64) {
        round(xa, c0);
        if (c0 + XR / 64 < nch) round(xb, c0 + XR / 64);
    }
    if (w || m0 + (l & 31) >= M) return;
    T* out = C + (long long)(m0 + (l & 31)) * ldc + 4 * (l >> 5);   // (a lane: a row, columns 8 q + 4 (l / 32) .. + 3)
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (8 * q < N)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float v = piece ? sum[4 * q + j] + acc[4 * q + j] : acc[4 * q + j];
                if constexpr (sizeof(T) == 4)
                    out[8 * q + j] = v;
                else
                    out[8 * q + j] = f2bf(rbf(v) * scale);
            }
}

__device__ __forceinline__ float half_of(const u32x4& v, int i) { return i & 1 ? bfhi(v[i >> 1]) : bflo(v[i >> 1]); }

// DX[m][k] += keep ? scale * sum_j DU[m][j] A[j][k] : 0.  A: [r][K] (a_oc), else [K][r]; per expert where there are offsets.  mask null: every element is kept.
// A lane holds eight columns of A and runs a wave's eight rows through them: a read and a write of DX, on the vector pipe in 32 bits, rounded once.
// GLU: DX is the gradient of silu(gate) up and stays as it is; its sum goes through the backward of that, H [M, 2 K] = [gate | up], DH its gradient (the bits of the two launches, which
// are the faster ones on few rows: lora_up_swiglu_pays of ops.py).
template <int R8, bool A_OC, bool GLU>
__global__ __launch_bounds__(256) void lora_up_kernel(const bf16_t* DU, const bf16_t* A, const unsigned char* mask, bf16_t* DX, const int32_t* offsets, int E, int M,
                                                      int K, long long ldu, float scale, const bf16_t* H, bf16_t* DH) {
    // rows at a time (by expert at rank 16 with GLU four: eight with their gate and up take 320 registers, one wave a SIMD; 4096 rows of 1664 34.8 / 30.6 us, 24 576 151 / 128, 98 304 562 /
    // 472; dense ones lose, the factor's rows being held for both halves: 2048 rows of 1664 13.6 / 14.8)
    constexpr int r = 8 * R8, NR = GLU && R8 == 2 && !A_OC ? ROWS / 8 : ROWS / 4;
    int e, m0, m1;
    if (!rows_of(offsets, E, M, blockIdx.x, e, m0, m1)) return;
    const int c = blockIdx.y * 64 + (threadIdx.x & 63), begin = m0 + ROWS / 4 * first_lane(int(threadIdx.x) >> 6);
    if (c >= K / 8) return;
    const bf16_t* ae = A + (long long)e * r * K;
#pragma unroll 1
    for (int first = begin; first < min(begin + ROWS / 4, m1); first += NR) {
        u32x4 old[NR];
        unsigned keep[NR];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const long long m = min(first + i, m1 - 1);
            old[i] = ld16(DX + m * K + 8 * c);
            keep[i] = mask ? mask[m * (K / 8) + c] : 255u;
        }
        float y[NR][8];
#pragma unroll
        for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int q = 0; q < 8; ++q) y[i][q] = 0.f;
#pragma unroll
        for (int jb = 0; jb < R8; ++jb) {
            u32x4 a[8];   // A_OC: eight columns of factor row 8 jb + i; else factor entries 8 jb .. of column 8 c + i
#pragma unroll
            for (int i = 0; i < 8; ++i) a[i] = A_OC ? ld16(ae + (long long)(8 * jb + i) * K + 8 * c) : ld16(ae + (8ll * c + i) * r + 8 * jb);
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const u32x4 d = ld16(DU + (long long)min(first + i, m1 - 1) * ldu + 8 * jb);
#pragma unroll
                for (int j = 0; j < 8; ++j)
#pragma unroll
                    for (int q = 0; q < 8; ++q) y[i][q] = fmaf(half_of(d, j), A_OC ? half_of(a[j], q) : half_of(a[q], j), y[i][q]);
            }
        }
        u32x4 gate[GLU ? NR : 1], up[GLU ? NR : 1];
        if (GLU)
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const bf16_t* h = H + (long long)min(first + i, m1 - 1) * 2 * K + 8 * c;
                gate[GLU ? i : 0] = ld16(h), up[GLU ? i : 0] = ld16(h + K);
            }
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            if (first + i >= m1) break;
            u32x4 o;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float lo = keep[i] >> (2 * q) & 1u ? scale * y[i][2 * q] : 0.f, hi = keep[i] >> (2 * q + 1) & 1u ? scale * y[i][2 * q + 1] : 0.f;
                o[q] = pack2bf(bflo(old[i][q]) + lo, bfhi(old[i][q]) + hi);
            }
            if (GLU) {
                u32x4 dg, du;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const u32x4 &g = gate[GLU ? i : 0], &u = up[GLU ? i : 0];
                    f32x2 da, db;
                    swiglu_bwd_pair(f32x2{bflo(g[q]), bfhi(g[q])}, f32x2{bflo(u[q]), bfhi(u[q])}, f32x2{bflo(o[q]), bfhi(o[q])}, da, db);
                    dg[q] = pack2bf(da.x, da.y), du[q] = pack2bf(db.x, db.y);
                }
                bf16_t* d = DH + (long long)(first + i) * 2 * K + 8 * c;
                st16(d, dg);
                st16(d + K, du);
            } else {
                st16(DX + (long long)(first + i) * K + 8 * c, o);
            }
        }
    }
}

// part[split][j][n] = sum over the split's rows of Y[m][n] U[m][j], j = 8 z .. 8 z + 7.  A lane holds 8 columns x 8 factor entries in 32 bits; the eight waves of a block take
// every eighth row of it and meet in LDS.  A split is `per` times 64 rows: 64 up to 16 384 rows, beyond them as many as keep 256 splits, so that the partial sums are no
// more than r N x 256 however many rows there are (65 536 x 6656, rank 8: 218 MB and 316 us with 64 each, 54 MB and 231 us here).
constexpr int WG_ROWS = 64, WG_SPLITS = 256;
int64_t wgrad_per(int64_t M) { return (M + int64_t(WG_ROWS) * WG_SPLITS - 1) / (int64_t(WG_ROWS) * WG_SPLITS); }
__global__ __launch_bounds__(512) void lora_wgrad_kernel(const bf16_t* Y, const bf16_t* U, float* part, int M, int N, int r, int per, long long ldy, long long ldu) {
    ARIA_DYN_SMEM(lds);
    float* red = reinterpret_cast<float*>(lds);   // [4 waves][64 sums][64 lanes]
    const int l = threadIdx.x & 63, w = first_lane(int(threadIdx.x) >> 6), c = blockIdx.y * 64 + l, cc = min(c, N / 8 - 1), jb = blockIdx.z;
    const int m1 = int(min((long long)M, ((long long)blockIdx.x + 1) * per * WG_ROWS));
    float acc[8][8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int q = 0; q < 8; ++q) acc[j][q] = 0.f;
    for (int m0 = int(blockIdx.x) * per * WG_ROWS; m0 < m1; m0 += WG_ROWS) {
        u32x4 y[WG_ROWS / 8], u[WG_ROWS / 8];   // (every load of the wave in flight at once)
#pragma unroll
        for (int i = 0; i < WG_ROWS / 8; ++i) {
            const int row = min(m0 + w + 8 * i, m1 - 1);
            y[i] = ld16(Y + (long long)row * ldy + 8 * cc);
            u[i] = ld16(U + (long long)row * ldu + 8 * jb);
        }
#pragma unroll
        for (int i = 0; i < WG_ROWS / 8; ++i) {
            if (m0 + w + 8 * i >= m1) break;
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int q = 0; q < 8; ++q) acc[j][q] = fmaf(half_of(u[i], j), half_of(y[i], q), acc[j][q]);
        }
    }
#pragma unroll
    for (int half = 4; half; half >>= 1) {
        if (w >= half && w < 2 * half)
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int q = 0; q < 8; ++q) red[((w - half) * 64 + 8 * j + q) * 64 + l] = acc[j][q];
        sync();
        if (w < half)
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int q = 0; q < 8; ++q) acc[j][q] += red[(w * 64 + 8 * j + q) * 64 + l];
        sync();
    }
    if (w || c >= N / 8) return;
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const f32x4 v = {acc[j][4 * h], acc[j][4 * h + 1], acc[j][4 * h + 2], acc[j][4 * h + 3]};
            *reinterpret_cast<f32x4*>(part + ((long long)blockIdx.x * r + 8 * jb + j) * N + 8ll * c + 4 * h) = v;
        }
}

// the splits' sum: out[j][n], or with n_first out[n][j].  Four threads share four columns' splits.
__global__ __launch_bounds__(256) void lora_wgrad_sum_kernel(const float* part, bf16_t* out, int splits, int N, int r, int n_first) {
    ARIA_SMEM_STATIC f32x4 red[4][64];
    const int t = threadIdx.x & 63, q = threadIdx.x >> 6, i = blockIdx.x * 64 + t;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    if (i < r * N / 4)
#pragma unroll 8
        for (int k = q; k < splits; k += 4) s += *reinterpret_cast<const f32x4*>(part + (long long)k * r * N + 4ll * i);
    red[q][t] = s;
    sync();
    if (q || i >= r * N / 4) return;
    s = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
    const int j = 4 * i / N, n = 4 * i % N;
    if (n_first) {
#pragma unroll
        for (int k = 0; k < 4; ++k) out[(long long)(n + k) * r + j] = f2bf(s[k]);
    } else {
        unsigned* dst = reinterpret_cast<unsigned*>(out + (long long)j * N + n);
        dst[0] = pack2bf(s[0], s[1]);
        dst[1] = pack2bf(s[2], s[3]);
    }
}

bool off16(const void* p) { return reinterpret_cast<uintptr_t>(p) & 15; }
bool thin(int64_t r) { return r == 8 || r == 16; }
unsigned row_tiles(int64_t M, const int32_t* offsets, int64_t E) { return unsigned(offsets ? M / ROWS + E : (M + ROWS - 1) / ROWS); }

}  // namespace

extern "C" {

int aria_lora_scale_bf16(const void* U, void* OUT, int64_t M, int64_t r, int64_t ldo, float scale, void* stream) {
    if (!U || !OUT || M < 0 || r <= 0) return ARIA_ERR_INVALID;
    if (off16(U) || off16(OUT) || (r & 7) || (ldo & 7)) return ARIA_ERR_ALIGN;
    if (M == 0) return ARIA_OK;
    const int64_t n = M * (r / 8);
    if (n >= (1ll << 38)) return ARIA_ERR_UNSUPPORTED;
    ARIA_LAUNCH(lora_scale_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, stream, static_cast<const bf16_t*>(U), static_cast<bf16_t*>(OUT), (long long)n,
                int(r / 8), (long long)ldo, scale);
    return aria_check_launch();
}

int aria_lora_down_bf16(const void* X, const void* W, int w_oc, void* U, const int32_t* offsets, int64_t E, int64_t M, int64_t K, int64_t r, int64_t ldx, int64_t ldu,
                        float scale, void* stream) {
    if (!X || !W || !U || M < 0 || K <= 0 || r <= 0 || (offsets && E <= 0)) return ARIA_ERR_INVALID;
    const int64_t lds = std::max<int64_t>(r * (K + PAD) * 2, 8 * ROWS * 16 * 4);
    if (!thin(r) || (K & 63) || lds > LDS_MAX || M >= (1ll << 30)) return ARIA_ERR_UNSUPPORTED;
    if (off16(X) || off16(W) || (ldx & 7)) return ARIA_ERR_ALIGN;
    if (M == 0) return ARIA_OK;
    ARIA_LAUNCH(lora_down_kernel, dim3(row_tiles(M, offsets, E)), dim3(512), unsigned(lds), stream, static_cast<const bf16_t*>(X), static_cast<const bf16_t*>(W),
                static_cast<bf16_t*>(U), offsets, int(E), int(M), int(K), int(r), w_oc, (long long)ldx, (long long)ldu, scale);
    return aria_check_launch();
}

int aria_thin_product_f32(const void* X, const void* W, float* C, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldc, void* stream) {
    if (!X || !W || !C || M < 0 || N <= 0 || K <= 0) return ARIA_ERR_INVALID;
    const int64_t lds = N * (K + 8) * 2 + ROWS * XPITCH * 2;
    if (N > 32 || (N & 7) || (K & 63) || N * (K + PAD) * 2 > LDS_MAX || M >= (1ll << 30)) return ARIA_ERR_UNSUPPORTED;
    if (off16(X) || off16(W) || (ldx & 7)) return ARIA_ERR_ALIGN;
    if (M == 0) return ARIA_OK;
    long long cut_row = 0;
    const int cut = aria_gemm3_cut(M, N, K, &cut_row);
    ARIA_LAUNCH((thin_product_kernel<false, float>), dim3(row_tiles(M, nullptr, 1)), dim3(512), unsigned(lds), stream, static_cast<const bf16_t*>(X), static_cast<const bf16_t*>(W),
                C, static_cast<const int32_t*>(nullptr), 1, int(M), int(N), int(K), (long long)ldx, (long long)ldc, int(cut_row), cut, 1.f);
    return aria_check_launch();
}

int aria_lora_u_bf16(const void* X, const void* W, int w_oc, void* U, const int32_t* offsets, int64_t E, int64_t M, int64_t K, int64_t r, int64_t ldx, int64_t ldu, float scale,
                     void* stream) {
    if (!X || !W || !U || M < 0 || K <= 0 || r <= 0 || (offsets && E <= 0)) return ARIA_ERR_INVALID;
    const int64_t lds = r * (K + 8) * 2 + ROWS * XPITCH * 2;
    if (!thin(r) || (K & 63) || r * (K + PAD) * 2 > LDS_MAX || M >= (1ll << 30)) return ARIA_ERR_UNSUPPORTED;
    if (off16(X) || off16(W) || (ldx & 7)) return ARIA_ERR_ALIGN;
    if (M == 0) return ARIA_OK;
    long long cut_row = 0;
    const int cut = offsets ? 1 : aria_gemm3_cut(M, r, K, &cut_row);   // (rows by expert are never cut)
    auto launch = [&](auto oc) {
        ARIA_LAUNCH((thin_product_kernel<decltype(oc)::value, bf16_t>), dim3(row_tiles(M, offsets, E)), dim3(512), unsigned(lds), stream, static_cast<const bf16_t*>(X),
                    static_cast<const bf16_t*>(W), static_cast<bf16_t*>(U), offsets, int(E), int(M), int(r), int(K), (long long)ldx, (long long)ldu, int(cut_row), cut, scale);
    };
    if (w_oc)
        launch(std::true_type{});
    else
        launch(std::false_type{});
    return aria_check_launch();
}

static int lora_up(const void* DU, const void* A, int a_oc, const void* mask, void* DX, const int32_t* offsets, int64_t E, int64_t M, int64_t K, int64_t r, int64_t ldu, float scale,
                   const void* H, void* DH, void* stream) {
    if (!DU || !A || !DX || M < 0 || K <= 0 || r <= 0 || (offsets && E <= 0)) return ARIA_ERR_INVALID;
    if (!thin(r) || (K & 7) || K >= (1ll << 24) || M >= (1ll << 30)) return ARIA_ERR_UNSUPPORTED;
    if (off16(DU) || off16(A) || off16(DX) || off16(H) || off16(DH) || (ldu & 7)) return ARIA_ERR_ALIGN;
    if (M == 0) return ARIA_OK;
    const dim3 grid(row_tiles(M, offsets, E), unsigned((K / 8 + 63) / 64)), block(256);
    auto launch = [&](auto r8, auto oc, auto glu) {
        ARIA_LAUNCH((lora_up_kernel<decltype(r8)::value, decltype(oc)::value, decltype(glu)::value>), grid, block, 0, stream, static_cast<const bf16_t*>(DU),
                    static_cast<const bf16_t*>(A), static_cast<const unsigned char*>(mask), static_cast<bf16_t*>(DX), offsets, int(E), int(M), int(K), (long long)ldu, scale,
                    static_cast<const bf16_t*>(H), static_cast<bf16_t*>(DH));
    };
    auto rank = [&](auto oc, auto glu) { r == 8 ? launch(std::integral_constant<int, 1>{}, oc, glu) : launch(std::integral_constant<int, 2>{}, oc, glu); };
    if (a_oc)
        H ? rank(std::true_type{}, std::true_type{}) : rank(std::true_type{}, std::false_type{});
    else
        H ? rank(std::false_type{}, std::true_type{}) : rank(std::false_type{}, std::false_type{});
    return aria_check_launch();
}

int aria_lora_up_bf16(const void* DU, const void* A, int a_oc, const void* mask, void* DX, const int32_t* offsets, int64_t E, int64_t M, int64_t K, int64_t r,
                      int64_t ldu, float scale, void* stream) {
    return lora_up(DU, A, a_oc, mask, DX, offsets, E, M, K, r, ldu, scale, nullptr, nullptr, stream);
}

int aria_lora_up_swiglu_bf16(const void* DU, const void* A, int a_oc, const void* mask, const void* D, const void* H, void* DH, const int32_t* offsets, int64_t E, int64_t M, int64_t K,
                             int64_t r, int64_t ldu, float scale, void* stream) {
    if (!H || !DH) return ARIA_ERR_INVALID;
    return lora_up(DU, A, a_oc, mask, const_cast<void*>(D), offsets, E, M, K, r, ldu, scale, H, DH, stream);
}

int aria_lora_wgrad_bf16(const void* Y, const void* U, void* out, int n_first, int64_t M, int64_t N, int64_t r, int64_t ldy, int64_t ldu, float* workspace,
                         int64_t workspace_floats, void* stream) {
    if (!Y || !U || !out || !workspace || M <= 0 || N <= 0 || r <= 0) return ARIA_ERR_INVALID;
    const int64_t per = wgrad_per(M), splits = (M + per * WG_ROWS - 1) / (per * WG_ROWS);
    if (!thin(r) || (N & 7) || M >= (1ll << 30) || N >= (1ll << 24)) return ARIA_ERR_UNSUPPORTED;
    if (workspace_floats < splits * r * N) return ARIA_ERR_INVALID;
    if (off16(Y) || off16(U) || off16(out) || off16(workspace) || (ldy & 7) || (ldu & 7)) return ARIA_ERR_ALIGN;
    ARIA_LAUNCH(lora_wgrad_kernel, dim3(unsigned(splits), unsigned((N / 8 + 63) / 64), unsigned(r / 8)), dim3(512), 65536, stream, static_cast<const bf16_t*>(Y),
                static_cast<const bf16_t*>(U), workspace, int(M), int(N), int(r), int(per), (long long)ldy, (long long)ldu);
    ARIA_LAUNCH(lora_wgrad_sum_kernel, dim3(unsigned((r * N / 4 + 63) / 64)), dim3(256), 0, stream, workspace, static_cast<bf16_t*>(out), int(splits), int(N), int(r),
                n_first);
    return aria_check_launch();
}

}  // extern "C"
