// Weight gradients of short reductions, dW = A^T dY: A [rows][M features], dY [rows][N], a few dozen to a few hundred rows for millions of outputs (an expert's tokens, the
// labelled tokens of one sample), so that the stores are the time: tiles of an output that each fetch both operands again spend longer on them than on their stores.
//
// A workgroup of four waves owns a strip of 256 columns and runs over tiles of 64 features; wave w owns columns [64 w, 64 w + 64) of the strip and holds dY's fragments of them
// for the whole reduction in registers (128 for 256 rows).  Only A moves: a tile's rows [up to 256][64] arrive by LDS-DMA in one of two buffers while the tile before is computed
// and stored, one barrier a tile, and every output line is written whole, eight lines a store instruction.  Two workgroups a CU (80 KiB each: the buffers, 4 KiB a wave in which
// 32 x 64 results are turned into rows).
//
// Longer reductions (an expert that most tokens want) are the 128 x 256 tiles', in the same launch (wgrad_strip_kernel, gemm4.hip).
//
// What bounds it is the stores: 64 experts of 2560 x 3328 outputs (1.09 GB) 196 us at 6 rows each and 206 at 26, where stores alone take 200 (5.5 TB/s; tiles of 128 x 256 took
// 240 and 265); 220 (361) at 73 rows each, where two waves a SIMD leave a part of a tile's reads and products uncovered.
//
// LDS images: [k][64 features or columns], 128 bytes a k-row; the 32-byte chunk c of k-row k lies at c ^ 2 ((k >> 1) & 1), so that the 32 lanes of a transposing read's half wave hit
// eight different 32-byte bank groups.  The products of an element come in the order of the other kernels' (sixteen rows a step, rows in order): the same bits.
#pragma once
#include "gemm_params.h"

namespace {
using namespace ad;

__device__ const uint32_t zero_page_wg[64] = {};   // the source of granules beyond the end of the reduction

constexpr int FT = 64, STRIP = 256, KC = 256, STAGE = KC * FT * 2, PARK = 4096, WGRAD_SMEM = 2 * STAGE + 4 * PARK;   // a tile's features; a strip's columns; rows held at once; bytes

// four fragments (steps kk .. kk + 3 of sixteen rows) of 32 columns of an image; `at`: this lane's address for kk = 0
__device__ __forceinline__ void frags4(s16x8 (&f)[4], const char* smem, uint32_t at) {
#ifdef ARIA_EMU
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const s16x4 a = ds_read_tr16(reinterpret_cast<const bf16_t*>(smem + at + j * 2048)), b = ds_read_tr16(reinterpret_cast<const bf16_t*>(smem + at + j * 2048 + 512));
        f[j] = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
    }
#else
    s16x4 r[8];
    const uint32_t a = uint32_t(reinterpret_cast<uintptr_t>(smem)) + at;
    asm volatile("ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:512\n\tds_read_b64_tr_b16 %2, %8 offset:2048\n\tds_read_b64_tr_b16 %3, %8 offset:2560\n\t"
                 "ds_read_b64_tr_b16 %4, %8 offset:4096\n\tds_read_b64_tr_b16 %5, %8 offset:4608\n\tds_read_b64_tr_b16 %6, %8 offset:6144\n\tds_read_b64_tr_b16 %7, %8 offset:6656\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
                 : "v"(a)
                 : "memory");
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] = __builtin_shufflevector(r[2 * j], r[2 * j + 1], 0, 1, 2, 3, 4, 5, 6, 7);
#endif
}

// Strip `wg` of `nwg`.  parts: pieces of a strip's feature tiles, per: tiles of one
template <bool GATHER>
__device__ __forceinline__ void wgrad_strip(const GemmParams& p, int wg, int nwg, int parts, int per, char* smem) {
    const bf16_t *A = p.A, *B = p.B;
    bf16_t* C = static_cast<bf16_t*>(p.C);
    const int32_t *offsets = p.offsets, *gather_rows = p.gather_rows;
    const int M = p.M, N = p.N, K = p.K;
    const long long lda = p.lda, ldb = p.ldb, ldc = p.ldc, strideC = p.strideC;
    const int t = threadIdx.x, l = t & 63, w = first_lane(t >> 6);
    // an XCD runs the strips of one expert after the other's: its rows are read into one L2
    const int q8 = nwg >> 3, r8 = nwg & 7, xcd = wg & 7, strips = N / STRIP;
    int id = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (wg >> 3);
    const int n0 = (id % strips) * STRIP;
    id /= strips;
    const int first = (id % parts) * per, last = min(first + per, M / FT), e = id / parts;
    int k_begin = 0, k_len = K;
    if (offsets) k_begin = first_lane(offsets[e]), k_len = first_lane(offsets[e + 1]) - k_begin;
    if (k_len > KC) return;   // (the tiles')
    C += e * strideC;
    if (k_len <= 0) {   // nothing but stores: two rows of the strip a wave's store
        bf16_t* out = C + (long long)(first * FT + (t >> 5)) * ldc + n0 + (t & 31) * 8;
        for (int row = first * FT; row < last * FT; row += 8, out += 8 * ldc) st16(out, zero16());
        return;
    }
    const uint32_t lda2 = uint32_t(2 * lda), ldb2 = uint32_t(2 * ldb);
    // this lane's k-row of a DMA piece of eight, its column (LDS images: the chunks' places swapped at the source)
    const int krow = l >> 3, col = ((((l & 7) >> 1) ^ (((l >> 4) & 1) << 1)) << 4) + (l & 1) * 8;
    const char* zeros = reinterpret_cast<const char*>(zero_page_wg) + 16 * (l & 15);
    // fragment addresses of the two 32-column halves of an image
    const int fk = 8 * (l >> 5) + ((l & 15) >> 2), swap = ((l & 15) >> 3) << 1;
    uint32_t fv[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) fv[g] = uint32_t(fk * 128 + 8 * (l & 3)) + uint32_t(((2 * g + ((l >> 4) & 1)) ^ swap) << 5);

    s16x8 held[KC / 16][2];   // dY's fragments
    uint32_t rows[KC / 32];   // byte offsets of this lane's rows of A

    // the kc rows of the reduction: dY's fragments through the buffers (16 KiB of them a wave), A's row offsets
    auto load_held = [&](int kc) __attribute__((always_inline)) {
        const char* b = reinterpret_cast<const char*>(B) + ((long long)k_begin * ldb + n0 + 64 * w + col) * 2;
        char* mine = smem + 16384 * w;
#pragma unroll
        for (int i = 0; i < KC / 32; ++i)
            if (32 * i < kc) {
                const int k = 32 * i + 8 * w + krow;
                rows[i] = GATHER ? mul24(uint32_t(gather_rows[k_begin + min(k, kc - 1)]), lda2) : mul24(uint32_t(k), lda2);
            }
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int left = kc - 128 * half;
            if (left <= 0) break;
            for (int j = 0; j < min(2 * ((left + 15) / 16), 16); ++j) {
                const int k = 128 * half + 8 * j + krow;
                const char* src = k < kc ? b + mul24(uint32_t(k), ldb2) : zeros;
                hold(src);   // (one piece for the whole wave, not one for each side of the choice)
                glds16_raw(src, mine + 1024 * j);
            }
            wait_vm<0>();
            wave_barrier();
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int k4 = 0; k4 < 2; ++k4)
                    if (64 * k4 < left) {
                        s16x8 f[4];
                        frags4(f, mine, fv[g] + uint32_t(k4 * 8192));
#pragma unroll
                        for (int j = 0; j < 4; ++j) held[8 * half + 4 * k4 + j][g] = f[j];
                    }
            wave_barrier();
        }
        raw_barrier();   // (A's pieces land in the other waves' places too)
    };
    auto fetch = [&](int tile, int kc, int buf) __attribute__((always_inline)) {
        const char* a = reinterpret_cast<const char*>(A) + (GATHER ? 0ll : 2 * (long long)k_begin * lda) + (tile * FT + col) * 2ll;
        char* d = smem + buf * STAGE + 1024 * w;
#pragma unroll
        for (int i = 0; i < KC / 32; ++i)
            if (32 * i < kc) {
                const char* src = 32 * i + 8 * w + krow < kc ? a + rows[i] : zeros;
                hold(src);
                glds16_raw(src, d + 4096 * i);
            }
    };
    // features 32 g .. of a buffer's tile times the held columns
    auto products = [&](f32x16 (&acc)[2], int g, int buf, int steps) __attribute__((always_inline)) {
#pragma unroll
        for (int k4 = 0; k4 < KC / 64; ++k4)
            if (4 * k4 < steps) {
                s16x8 f[4];
                frags4(f, smem, fv[g] + uint32_t(buf * STAGE + k4 * 8192));
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (4 * k4 + j < steps)
#pragma unroll
                        for (int n = 0; n < 2; ++n) acc[n] = mfma32(held[4 * k4 + j][n], f[j], acc[n]);
            }
    };
    // 32 features x 64 columns through this wave's 4 KiB (row r's 16-byte chunk c at c ^ ((r >> 1) & 7)): four store instructions of eight lines
    auto store = [&](const f32x16 (&acc)[2], int tile, int g) __attribute__((always_inline)) {
        char* park = smem + 2 * STAGE + PARK * w;
        const int r = l & 31, h = l >> 5;
        wave_barrier();
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<u32x2*>(park + r * 128 + (((4 * n + q) ^ ((r >> 1) & 7)) << 4) + 8 * h) =
                    u32x2{pack2bf(acc[n][4 * q], acc[n][4 * q + 1]), pack2bf(acc[n][4 * q + 2], acc[n][4 * q + 3])};
        wait_lds();
        wave_barrier();
        bf16_t* out = C + (long long)(tile * FT + 32 * g) * ldc + n0 + 64 * w + (l & 7) * 8;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 8 * i + (l >> 3);
            st16(out + row * ldc, *reinterpret_cast<const u32x4*>(park + row * 128 + (((l & 7) ^ ((row >> 1) & 7)) << 4)));
        }
    };
    auto clear = [&](f32x16 (&acc)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[n][i] = 0.f;
    };

    const int steps = (k_len + 15) / 16;
    load_held(k_len);
    fetch(first, k_len, 0);
    for (int tile = first; tile < last; ++tile) {
        const int buf = (tile - first) & 1;
        if (tile == first)
            wait_vm<0>();
        else
            wait_vm<8>();   // this wave's pieces of the tile; the eight stores of the tile before may be under way
        raw_barrier();      // everybody's, and the other buffer is free
        if (tile + 1 < last) fetch(tile + 1, k_len, buf ^ 1);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            f32x16 acc[2];
            clear(acc);
            products(acc, g, buf, steps);
            store(acc, tile, g);
        }
    }
}
}  // namespace
