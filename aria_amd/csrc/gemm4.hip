// GEMM with four waves, one a SIMD, for the products whose tiles of 256 x 256 leave CUs idle or stand half empty.  Three forms, by what bounds them:
//
//   tiles of 128 x 256, stages 64 deep, three of them (144 KiB), one workgroup a CU: outputs of up to one round, and rows by expert of a few dozen
//   tiles of 256 x 160 ([N, K] weights) or 128 x 320 ([K, N]): outputs of one round whose 256 x 256 tiles would fill only part of it
//   tiles of 128 x 256, stages 32 deep, two workgroups a CU: weight gradients with short reductions, where a tile's start and its stores are the time and the
//     other workgroup's work hides them
//
// Geometry.  Wave (wm, wn) of WM x WN owns rows {i * 32 WM + 32 wm + [0, 32)} x columns {b * 32 WN + 32 wn + [0, 32)} of the tile, i < MI, b < NI, as
// v_mfma_f32_32x32x16_bf16 tiles with transposed accumulators (mfma(B fragment, A fragment): a lane owns four consecutive columns of one row a register group).
// Large wave tiles keep the LDS reads below the matrix work: 128 x 64 a wave reads 24 KiB for 1024 cycles of products (eight waves of 64 x 64: 32 KiB).
//
// The reduction goes through S stages in the LDS, KD deep, filled by LDS-DMA, in sixteenths (one MFMA step).  While the products of one sixteenth run, the fragments
// of the next are read and pieces of stage t + S - 1 requested, one behind each product (in front of the products a wave's issue of the pieces took as long as the
// products).  Before the last sixteenth every wave holds its fragments, stage t + 1 has landed, and one s_barrier frees stage t's buffer.  A fragment never crosses a
// branch or the loop's back edge before it has arrived.
//
// What bounds the loop is the CU's rate of fetching lines: 777 x 2560 x 5120 on 70 CUs, a step of 32: the products alone 0.21 us, with every fragment read 0.22, with pieces
// from one fixed place 0.26, with the operands 0.30 .. 0.36.  A row operand ([rows][k]) in stages 32 deep fetches every 128-byte line twice (64 bytes, then the others): 0.355
// against 0.27 in stages 64 deep; 8192^3 1070 and 913 us.
//
// LDS images of a stage: A rows, then B rows.
//   rc operand ([rows][k]): a row = 2 KD bytes; its 16-byte chunk c lies at c ^ ((r >> 2) & 3) (KD 32) or c ^ ((r >> 1) & 7): the 16 rows of a ds_read_b128 group hit
//     16 different 16-byte bank groups.  A DMA piece (1 KiB) is 16 or 8 rows.
//   oc operand ([k][rows]): units of 64 rows, [KD][128 bytes]; 32-byte chunk c of k-row k lies at c ^ 2 ((k >> 1) & 1): the 32 lanes of a transposing read's half
//     wave (four k-rows, two chunks) hit eight different 32-byte bank groups.  A piece is 8 k-rows of a unit.
// The order of the products of an output element is that of the 256 x 256 kernel: the same bits where neither splits the reduction.
#include "aria_hip.h"
#include "gemm_params.h"
#include "wgrad.h"
#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <utility>

namespace {
using namespace ad;

__device__ const uint32_t zero_page4[64] = {};   // the source of granules beyond the end of the reduction

template <int OFF>
__device__ __forceinline__ s16x8 lds_b128(const char* smem, uint32_t at) {   // (the caller waits before the first use)
#ifdef ARIA_EMU
    return *reinterpret_cast<const s16x8*>(smem + at + OFF);
#else
    s16x8 f;
    const uint32_t a = uint32_t(reinterpret_cast<uintptr_t>(smem)) + at;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f) : "v"(a), "n"(OFF));
    return f;
#endif
}
template <int OFF>
__device__ __forceinline__ s16x8 lds_tr(const char* smem, uint32_t at) {   // eight k-rows of one column; the rows lie 128 bytes apart
#ifdef ARIA_EMU
    const s16x4 a0 = ds_read_tr16(reinterpret_cast<const bf16_t*>(smem + at + OFF)), a1 = ds_read_tr16(reinterpret_cast<const bf16_t*>(smem + at + OFF + 512));
#else
    s16x4 a0, a1;
    const uint32_t a = uint32_t(reinterpret_cast<uintptr_t>(smem)) + at;
    asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%3\n\tds_read_b64_tr_b16 %1, %2 offset:%4" : "=&v"(a0), "=&v"(a1) : "v"(a), "n"(OFF), "n"(OFF + 512));
#endif
    return __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
}

// fragment addresses of one operand in stages of KD: W waves side by side, this one at `wi`
template <bool OC, int W, int KD>
struct Frag {
    static constexpr int UNIT = KD * 128;   // bytes of 64 rows
    uint32_t v[2];
    __device__ __forceinline__ void init(int wi, int l) {
        if (!OC) {
            const int swap = KD == 32 ? (l >> 2) & 3 : (l >> 1) & 7;
            v[0] = uint32_t((wi * 32 + (l & 31)) * (2 * KD) + (((l >> 5) ^ swap) << 4));
            v[1] = 0;
        } else {
            const int k = 8 * (l >> 5) + ((l & 15) >> 2), f = ((l & 15) >> 3) << 1, first = wi * 32;
            const uint32_t at = uint32_t((first >> 6) * UNIT + k * 128 + 8 * (l & 3));
            v[0] = at + uint32_t(((((first & 32) >> 4) + ((l >> 4) & 1)) ^ f) << 5);
            v[1] = at + uint32_t(((2 + ((l >> 4) & 1)) ^ f) << 5);   // (W == 1: the odd 32-row tiles)
        }
    }
    // rows I * 32 W + 32 wi + (l & 31), k = 16 KK + 8 (l >> 5) + 0..7 of the image at `base`
    template <int I, int KK>
    __device__ __forceinline__ s16x8 read(const char* smem, uint32_t base) const {
        if (!OC) return lds_b128<I * W * 64 * KD>(smem, base + (v[0] ^ uint32_t(KK << 5)));
        constexpr int OFF = (I * W * 32 / 64) * UNIT + KK * 2048;
        return lds_tr<OFF>(smem, base + v[W == 1 ? I & 1 : 0]);
    }
};

template <class F, size_t... I>
__device__ __forceinline__ void each(F&& f, std::index_sequence<I...>) {
    (f(std::integral_constant<int, int(I)>{}), ...);
}

template <int WM, int WN, int MI, int NI, int KD, int S>
struct Shape4 {
    static constexpr int BM = WM * MI * 32, BN = WN * NI * 32, PA = BM * KD / 2048, PB = BN * KD / 2048;   // pieces a wave and stage
    static constexpr int STAGE = (BM + BN) * KD * 2, ROWP = BN * 2 + 16;                                   // bytes; pitch of the parked tile
    static constexpr size_t SMEM = std::max(size_t(S) * STAGE, size_t(BM) * ROWP);
};

// ONCE: B's pieces are non-temporal
// VER: what happens to the tile (the numbers of gemm3_kernel): 3 plain (bias, activation, accumulation, 32-bit results), 5 SwiGLU backward, 6 / 9 fused SwiGLU on two
// weight tensors (9: gathered rows), 8 on [K, N] weights with gathered rows, 14 on one [gate | up] tensor, 13 relu gate, 7 the interleaved rotation,
// 11 plain, with the reduction's rows of A reached through an index (per-expert weight gradients)
constexpr bool gathers(int ver) { return ver == 8 || ver == 9; }   // (11: gathered rows of the reduction)
constexpr bool gated(int ver) { return ver == 6 || ver == 8 || ver == 9 || ver == 13 || ver == 14; }

// one 16-byte piece (8 columns) of the parked tile on its way out
template <int VER, class P>
__device__ __forceinline__ void finish_piece(const P& p, char* C, const char* parked, int m, int n0, int cc) {
    u32x4 v = *reinterpret_cast<const u32x4*>(parked + cc * 2);
    bf16_t* out = reinterpret_cast<bf16_t*>(C);
    if (VER == 7) {   // interleaved rotation and the cache's rows (store_tile3_rows_rope of the 256 x 256 kernel)
        const int region = n0 / p.rope_D, col = n0 - region * p.rope_D + cc;
        const int seq = m / p.rope_S, ps = p.rope_pos ? p.rope_pos[m] : m - seq * p.rope_S;
        if (region < 2) {
            const u32x4 f = ld16(p.rope_fc + (long long)ps * p.rope_hd + col % p.rope_hd);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float x0 = bflo(v[q]), x1 = bfhi(v[q]), cs = bflo(f[q]), sn = bfhi(f[q]);
                v[q] = pack2bf(x0 * cs - x1 * sn, x1 * cs + x0 * sn);
            }
        }
        if (region == 0)
            st16(out + (long long)m * p.ldc + col, v);
        else if (unsigned(ps) < unsigned(p.cache_S))
            st16(static_cast<bf16_t*>(region == 1 ? p.kc : p.vc) + ((long long)seq * p.cache_S + ps) * p.ld_cache + col, v);
        return;
    }
    if (VER == 5) {   // v = d_act: gate and up of the same elements give their gradients
        const bf16_t* h = p.H + (long long)m * p.ldh + n0 + cc;
        const u32x4 g = ld16(h), u = ld16(h + p.N);
        u32x4 og, ou;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            f32x2 da, db;
            swiglu_bwd_pair(f32x2{bflo(g[q]), bfhi(g[q])}, f32x2{bflo(u[q]), bfhi(u[q])}, f32x2{bflo(v[q]), bfhi(v[q])}, da, db);
            og[q] = pack2bf(da.x, da.y), ou[q] = pack2bf(db.x, db.y);
        }
        bf16_t* d = out + (long long)m * p.ldc + n0 + cc;
        st16(d, og);
        st16(d + p.N, ou);
        return;
    }
    st16(out + (long long)m * p.ldc + n0 + cc, v);
}

// Where a workgroup's tile lies: row tile from m0 (rows end at m_end), column tile tn, its reduction, its expert's operand and result; slab >= 0: piece ks of a split reduction
struct Tile4 {
    int tn, m0, m_end, k_begin, k_len;
    long long b_off, c_off;
    int slab, ks;
};

template <bool A_OC, bool B_OC, int WM, int WN, int MI, int NI, int KD, int S, int VER, bool ONCE = false>
__device__ __forceinline__ void gemm4_tile(const GemmParams& p, const Tile4& place, char* smem) {
    using T = Shape4<WM, WN, MI, NI, KD, S>;
    constexpr int BM = T::BM, BN = T::BN, PA = T::PA, PB = T::PB, STAGE = T::STAGE, ROWP = T::ROWP, HALVES = KD / 16;
    constexpr bool GATHER = gathers(VER), GLU = gated(VER), GATHER_K = VER == 11, PLAIN = VER == 3 || VER == 11;
    constexpr int STEP = GLU ? BN / 2 : BN;
    const int t = threadIdx.x, l = t & 63, w = first_lane(t >> 6), wm = w / WN, wn = w % WN;
    const int tn = place.tn, m0 = place.m0, m_end = place.m_end, k_begin = place.k_begin, k_len = place.k_len, slab = place.slab, ks = place.ks;
    const long long b_off = place.b_off, c_off = place.c_off;
    const int n0 = tn * STEP;
    char* C = static_cast<char*>(p.C) + c_off * (p.c_f32 ? 4 : 2);

    // ---- the stages' sources
    int steps = (k_len + KD - 1) / KD, first_step = 0;
    const int tail_step = steps - 1, tail_k = k_len - tail_step * KD;
    if (slab >= 0) {
        first_step = int((long long)steps * ks / p.split);
        steps = int((long long)steps * (ks + 1) / p.split);
    }
    const uint32_t lda2 = uint32_t(2 * p.lda), ldb2 = uint32_t(2 * p.ldb);
    const char* gA = reinterpret_cast<const char*>(p.A) + (A_OC ? 2 * k_begin * p.lda : 2 * (long long)k_begin);
    const char* gB = reinterpret_cast<const char*>(p.B + b_off) + (B_OC ? 2 * k_begin * p.ldb : 2 * (long long)k_begin);
    const long long stepA = A_OC ? 2 * KD * p.lda : 2 * KD, stepB = B_OC ? 2 * KD * p.ldb : 2 * KD;
    // rc: a piece of 16 (KD 32) or 8 rows; oc: 8 k-rows of 64 columns -- this lane's row, chunk (bytes) and k-row, column of piece 0
    constexpr int RC = KD == 32 ? 16 : 8, OCU = KD / 32;   // rows of a piece; a wave's pieces of a 64-column unit
    const int rc_row = KD == 32 ? 16 * w + (l >> 2) : 8 * w + (l >> 3);
    const int rc_chunk = KD == 32 ? ((l & 3) ^ ((l >> 4) & 3)) * 16 : ((l & 7) ^ (4 * (w & 1) + (l >> 4))) * 16;
    const int oc_k = 8 * w + (l >> 3), oc_col = ((((l & 7) >> 1) ^ (((l >> 4) & 1) << 1)) << 4) + (l & 1) * 8;
    uint32_t offA[PA], offB[PB];
#pragma unroll
    for (int s = 0; s < PA; ++s) {
        if (A_OC) {
            offA[s] = (GATHER_K ? 0u : mul24(uint32_t(oc_k + 32 * (s % OCU)), lda2)) + 2u * uint32_t(min(m0 + 64 * (s / OCU) + oc_col, p.M - 8));
        } else {
            const int row = min(m0 + 4 * RC * s + rc_row, m_end - 1);
            offA[s] = mul24(uint32_t(GATHER ? p.gather_rows[row] : row), lda2) + uint32_t(rc_chunk);
        }
    }
    constexpr bool UP_ROWS = VER == 6 || VER == 9;   // up rows in a tensor of their own
#pragma unroll
    for (int s = 0; s < PB; ++s) {
        int first = n0 + (B_OC ? 64 * (s / OCU) : 4 * RC * s);
        if (GLU && s >= PB / 2) first += (UP_ROWS ? 0 : p.N / 2) - BN / 2;
        if (B_OC)
            offB[s] = mul24(uint32_t(oc_k + 32 * (s % OCU)), ldb2) + 2u * uint32_t(min(first + oc_col, p.N - 8));
        else
            offB[s] = mul24(uint32_t(UP_ROWS ? first + rc_row : min(first + rc_row, p.N - 1)), ldb2) + uint32_t(rc_chunk);
    }
    static_assert(!GATHER_K || (A_OC && OCU == 1), "one gathered row a lane and stage");
    // GATHER_K: the token row of this lane's k-row of a stage (past the end of the reduction: the last one, which meets zeros of B)
    auto row_of = [&](int step) __attribute__((always_inline)) { return p.gather_rows[k_begin + min(step * KD + oc_k, k_len - 1)]; };
    const char* A0 = reinterpret_cast<const char*>(p.A);
    // (up rows of a tensor of their own: as a distance from the gate rows' addresses)
    const long long up = UP_ROWS ? reinterpret_cast<const char*>(p.B_up) - reinterpret_cast<const char*>(p.B) : 0;
    // piece s of a stage (A's pieces first) from the step's operand addresses; the general form ends the reduction with zeros
    auto piece = [&](auto s, const char* a, const char* b, char* d) __attribute__((always_inline)) {
        constexpr int I = decltype(s)::value;
        if constexpr (I < PA)
            glds16(a + offA[I], d + 4096 * I);
        else if constexpr (ONCE)
            glds16_once(b + (I - PA >= PB / 2 ? up : 0) + offB[I - PA], d + 4096 * I);
        else
            glds16(b + (I - PA >= PB / 2 ? up : 0) + offB[I - PA], d + 4096 * I);
    };
    auto dma = [&](int step, uint32_t at) __attribute__((always_inline)) {
        const char* a = GATHER_K ? A0 + mul24(uint32_t(row_of(step)), lda2) : gA + step * stepA;
        const char* b = gB + step * stepB;
        char* d = smem + at + 1024 * w;
        if (step == tail_step && tail_k < KD) {
            const char* z = reinterpret_cast<const char*>(zero_page4) + 16 * (l & 15);
#pragma unroll
            for (int s = 0; s < PA + PB; ++s) {
                const int k = (s < PA ? A_OC : B_OC) ? oc_k + 32 * ((s < PA ? s : s - PA) % OCU) : rc_chunk >> 1;
                const char* src = k < tail_k ? (s < PA ? a + offA[s] : b + (s - PA >= PB / 2 ? up : 0) + offB[s - PA]) : z;
                hold(src);   // (one piece for the whole wave, not one for each side of the choice)
                glds16(src, d + 4096 * s);
            }
        } else {
            each([&](auto s) { piece(s, a, b, d); }, std::make_index_sequence<PA + PB>{});
        }
    };

    Frag<A_OC, WM, KD> fa;
    Frag<B_OC, WN, KD> fb;
    fa.init(wm, l);
    fb.init(wn, l);
    f32x16 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int b = 0; b < NI; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][b][r] = 0.f;
    s16x8 xa[MI], xb[NI], ya[MI], yb[NI];

    // fragment I (B's first: the first product needs one of each) of sixteenth KK
    auto frag = [&](auto kk, auto f, s16x8 (&ra)[MI], s16x8 (&rb)[NI], uint32_t at) __attribute__((always_inline)) {
        constexpr int KK = decltype(kk)::value, I = decltype(f)::value;
        if constexpr (I < NI)
            rb[I] = fb.template read<I, KK>(smem, at + BM * KD * 2);
        else
            ra[I - NI] = fa.template read<I - NI, KK>(smem, at);
    };
    constexpr auto FRAGS = std::make_index_sequence<MI + NI>{};
    constexpr auto PRODUCTS = std::make_index_sequence<MI * NI>{};
    auto product = [&](auto j, const s16x8 (&ra)[MI], const s16x8 (&rb)[NI]) __attribute__((always_inline)) {
        constexpr int J = decltype(j)::value;
        acc[J / NI][J % NI] = mfma32(rb[J % NI], ra[J / NI], acc[J / NI][J % NI]);
        sched_fence();
    };
    auto arrived = [&](s16x8 (&ra)[MI], s16x8 (&rb)[NI]) __attribute__((always_inline)) {
        wait_lds();
#pragma unroll
        for (int i = 0; i < MI; ++i) hold(ra[i]);
#pragma unroll
        for (int b = 0; b < NI; ++b) hold(rb[b]);
    };

    const int count = steps - first_step;
    if (count > 0) {
#pragma unroll
        for (int s = 0; s < S - 1; ++s)
            if (s < count) dma(first_step + s, uint32_t(s * STAGE));
        if (count >= S - 1)
            wait_vm<(S - 2) * (PA + PB)>();
        else
            wait_vm<0>();
        raw_barrier();
        each([&](auto f) { frag(std::integral_constant<int, 0>{}, f, xa, xb, 0u); }, FRAGS);
        arrived(xa, xb);
        int row = GATHER_K ? row_of(S - 1) : 0;
        uint32_t at = 0, fill = (S - 1) * STAGE;   // the stage in use; the one that was in use before it and is filled now
        // the products of sixteenth KK of the stage, with the reads of the next and a share of the DMA pieces one by one between them
        constexpr int QUOTA = (PA + PB + HALVES - 2) / (HALVES - 1);
        constexpr int READS = (MI + NI + MI * NI - 1) / (MI * NI), PIECES = (QUOTA + MI * NI - 1) / (MI * NI);   // behind one product (one each but in tiles of 32 rows)
        auto sixteenth = [&](auto kk, s16x8 (&ra)[MI], s16x8 (&rb)[NI], s16x8 (&na)[MI], s16x8 (&nb)[NI], uint32_t from, auto whole, const char* a, const char* b, char* d)
                             __attribute__((always_inline)) {
            constexpr int KK = decltype(kk)::value, NEXT = (KK + 1) % HALVES;
            each([&](auto j) {
                constexpr int J = decltype(j)::value;
                each([&](auto z) {
                    constexpr int F = J * READS + decltype(z)::value;
                    if constexpr (F < MI + NI) frag(std::integral_constant<int, NEXT>{}, std::integral_constant<int, F>{}, na, nb, from);
                }, std::make_index_sequence<READS>{});
                product(j, ra, rb);
                each([&](auto z) {
                    constexpr int Q = J * PIECES + decltype(z)::value;
                    if constexpr (decltype(whole)::value && KK < HALVES - 1 && Q < QUOTA && KK * QUOTA + Q < PA + PB) piece(std::integral_constant<int, KK * QUOTA + Q>{}, a, b, d);
                }, std::make_index_sequence<PIECES>{});
            }, PRODUCTS);
            arrived(na, nb);
        };
        auto stage = [&](int step, auto whole) __attribute__((always_inline)) {
            const uint32_t next = at + STAGE == S * STAGE ? 0u : at + STAGE;
            const char* a = GATHER_K ? A0 + mul24(uint32_t(row), lda2) : gA + (first_step + step + S - 1) * stepA;
            const char* b = gB + (first_step + step + S - 1) * stepB;
            char* d = smem + fill + 1024 * w;
            if (GATHER_K && decltype(whole)::value) row = row_of(step + S);   // (in front of this stage's pieces: waiting for it waits for none of them)
            if (!decltype(whole)::value && step + S - 1 < count) dma(first_step + step + S - 1, fill);
            each([&](auto kk) {
                constexpr int KK = decltype(kk)::value;
                if constexpr (KK % 2 == 0)
                    sixteenth(kk, xa, xb, ya, yb, at, whole, a, b, d);
                else
                    sixteenth(kk, ya, yb, xa, xb, at, whole, a, b, d);
            }, std::make_index_sequence<HALVES - 1>{});
            if (decltype(whole)::value || step + S - 1 < count)   // behind stage step + 1: stages up to step + S - 1
                wait_vm<(S - 2) * (PA + PB)>();
            else
                wait_vm<0>();
            raw_barrier();
            sixteenth(std::integral_constant<int, HALVES - 1>{}, ya, yb, xa, xb, next, whole, a, b, d);   // (behind the last step the reads are never used)
            fill = at;
            at = next;
        };
        static_assert(HALVES % 2 == 0, "a stage ends with the fragments that it began with");
        int step = 0;
        // steady steps: the stage that is filled exists and is whole
        const int steady = count - (S - 1) - (first_step + count - 1 == tail_step && tail_k < KD ? 1 : 0);
        for (; step < steady; ++step) stage(step, std::true_type{});
        for (; step < count; ++step) stage(step, std::false_type{});
    }

    const int c = l & 31, h = l >> 5;
    if (slab >= 0) {   // partial sums in the accumulators' order: 1 KiB contiguous a store
        float* dst = p.ws + (long long)slab * (BM * BN) + l * 4;
#pragma unroll
        for (int b = 0; b < NI; ++b)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<f32x4*>(dst + (((b * MI + i) * WM + wm) * WN + wn) * 1024 + q * 256) =
                        f32x4{acc[i][b][4 * q], acc[i][b][4 * q + 1], acc[i][b][4 * q + 2], acc[i][b][4 * q + 3]};
        return;
    }
    if (PLAIN && (p.c_f32 || !p.wide_store || (p.N & 7))) {   // straight from the registers
#pragma unroll
        for (int b = 0; b < NI; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = n0 + b * (WN * 32) + wn * 32 + 8 * q + 4 * h;
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    const int m = m0 + i * (WM * 32) + wm * 32 + c;
                    if (m >= m_end) continue;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if (n + j >= p.N) continue;
                        const float v = aria_epilogue_act(p, acc[i][b][4 * q + j] + (p.bias ? bf2f(p.bias[n + j]) : 0.f));
                        if (p.c_f32) {
                            float* d = reinterpret_cast<float*>(C) + (long long)m * p.ldc + n + j;
                            *d = p.accumulate ? *d + v : v;
                        } else {
                            bf16_t* d = reinterpret_cast<bf16_t*>(C) + (long long)m * p.ldc + n + j;
                            *d = f2bf(p.accumulate ? v + bf2f(*d) : v);
                        }
                    }
                }
            }
        return;
    }
    // ---- the tile is parked as bf16 rows and leaves in 16-byte pieces of them
    constexpr int CPR = BN / 8, ITS = BM * CPR / 256;
    const bool old = PLAIN && p.accumulate;
    raw_barrier();   // (the last stage's reads)
    if (old) {       // the old tile waits where the new values will be parked: they are added in 32 bits and rounded once
#pragma unroll 8
        for (int it = 0; it < ITS; ++it) {
            const int idx = it * 256 + t, row = idx / CPR, cc = (idx % CPR) * 8, m = m0 + row;
            const u32x4 o = m < m_end && n0 + cc < p.N ? ld16(reinterpret_cast<const bf16_t*>(C) + (long long)m * p.ldc + n0 + cc) : zero16();
            *reinterpret_cast<u32x4*>(smem + row * ROWP + cc * 2) = o;
        }
        sync();
    }
    auto park = [&](auto act) __attribute__((always_inline)) {
        constexpr int ACT = decltype(act)::value;
#pragma unroll
        for (int b = 0; b < NI; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int col = b * (WN * 32) + wn * 32 + 8 * q + 4 * h;
                float bv[4] = {0.f, 0.f, 0.f, 0.f};
                if (PLAIN && p.bias) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (n0 + col + j < p.N) bv[j] = bf2f(p.bias[n0 + col + j]);
                }
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; j += 2) {
                        const f32x2 pr = aria_epilogue_act2<ACT>(f32x2{acc[i][b][4 * q + j] + bv[j], acc[i][b][4 * q + j + 1] + bv[j + 1]});
                        v[j] = pr.x, v[j + 1] = pr.y;
                    }
                    u32x2* slot = reinterpret_cast<u32x2*>(smem + (i * (WM * 32) + wm * 32 + c) * ROWP + col * 2);
                    if (old) {
                        const u32x2 o = *slot;
                        v[0] += bflo(o[0]), v[1] += bfhi(o[0]), v[2] += bflo(o[1]), v[3] += bfhi(o[1]);
                    }
                    *slot = u32x2{pack2bf(v[0], v[1]), pack2bf(v[2], v[3])};
                }
            }
    };
    if (VER == 3 && p.act == 1)
        park(std::integral_constant<int, 1>{});
    else if (VER == 3 && !A_OC && !B_OC && p.act == 2)
        park(std::integral_constant<int, 2>{});
    else
        park(std::integral_constant<int, 0>{});
    sync();
    if (GLU) {   // rounding points as the unfused chain has them: h in bf16, silu(gate) in bf16, the product in bf16
        constexpr int HALF = BN / 2, GP = HALF / 8;
        const int I = p.N / 2;
        bf16_t *H = reinterpret_cast<bf16_t*>(C), *ACT = static_cast<bf16_t*>(p.C2);
#pragma unroll 4
        for (int it = 0; it < ITS / 2; ++it) {
            const int idx = it * 256 + t, row = idx / GP, cc = (idx % GP) * 8, m = m0 + row;
            if (m >= m_end) continue;
            const u32x4 g = *reinterpret_cast<const u32x4*>(smem + row * ROWP + cc * 2), u = *reinterpret_cast<const u32x4*>(smem + row * ROWP + (HALF + cc) * 2);
            u32x4 y;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float g0 = bflo(g[q]), g1 = bfhi(g[q]);
                y[q] = VER == 13 ? pack2bf(fmaxf(g0, 0.f) * bflo(u[q]), fmaxf(g1, 0.f) * bfhi(u[q]))
                                 : pack2bf(rbf(silu_fast(g0)) * bflo(u[q]), rbf(silu_fast(g1)) * bfhi(u[q]));
            }
            st16(ACT + (long long)m * p.ldc2 + n0 + cc, y);
            if (VER != 13 && H) {
                st16(H + (long long)m * p.ldc + n0 + cc, g);
                st16(H + (long long)m * p.ldc + I + n0 + cc, u);
            }
        }
        return;
    }
#pragma unroll 4
    for (int it = 0; it < ITS; ++it) {
        const int idx = it * 256 + t, row = idx / CPR, cc = (idx % CPR) * 8, m = m0 + row;
        if (m < m_end && n0 + cc < p.N) finish_piece<VER>(p, C, smem + row * ROWP, m, n0, cc);
    }
}

// LOW: rows by expert, of which most experts have fewer than a tile.  A tile that is its expert's only one holds as many blocks of 32 rows as there are rows, and its weights are non-temporal with
// ONCE: they are bound by the weights' stream, beside which the pieces of rows that are not there are up to a third of what a CU fetches and their products up to three quarters of the matrix
// work.  64 experts of 2560 x 1664, us with tiles of 128 rows / of what there is, rows an expert 8, 28, 73 evenly and 73, 100 as a router gives them: gate and up, gathered 190 181, 209 195, 235
// 219, 235 218, 252 244; down 105 97, 112 103, 125 117, 128 116, 129 118; SwiGLU backward 98 92, 115 107, 139 122, 140 131, 179 165; gate and up backward 202 180, 210 190, 222 210, 220 208, 229 216.
template <bool A_OC, bool B_OC, int WM, int WN, int MI, int NI, int KD, int S, int VER, int PER_CU, bool ONCE = false, bool LOW = false>
__global__ __launch_bounds__(256, PER_CU) void gemm4_kernel(GemmParams p) {
    constexpr int BM = Shape4<WM, WN, MI, NI, KD, S>::BM;
    ARIA_DYN_SMEM(smem);
    int tn = 0, tmi = 0, slab = -1, ks = 0;
    if (p.mode == 1) {
        // aria_grouped_tile below
    } else if (p.split > 1) {
        slab = blockIdx.x;
        ks = slab % p.split;
        if (!aria_tile_from_pos(p, slab / p.split, tmi, tn)) return;
    } else if (!aria_tile_coords(p, blockIdx.x, int(gridDim.x), tmi, tn)) {
        return;
    }
    long long b_off = 0, c_off = 0;
    int m0 = tmi * BM, m_end = p.M, k_begin = 0, k_len = p.K;
    bool alone = p.mode == 0 && p.M <= BM;   // the only tile of the rows, or of its expert's
    if (p.mode == 2) {
        k_begin = p.offsets[blockIdx.y];
        k_len = p.offsets[blockIdx.y + 1] - k_begin;
        c_off = (long long)blockIdx.y * p.strideC;
    } else if (p.mode == 1) {
        int expert = 0;
        if (!aria_grouped_tile<BM>(p, blockIdx.x, int(threadIdx.x) & 63, expert, m0, m_end, tn)) return;
        expert = first_lane(expert), m0 = first_lane(m0), m_end = first_lane(m_end), tn = first_lane(tn);
        b_off = (long long)(p.expert_mod > 0 ? expert % p.expert_mod : expert) * p.strideB;
        alone = m_end - m0 <= BM && m0 == p.offsets[expert];
    }
    const Tile4 place{tn, m0, m_end, k_begin, k_len, b_off, c_off, slab, ks};
    if constexpr (LOW) {
        static_assert(MI == 4 && WM == 1, "heights of 32 .. 128 rows");
        const int rows = m_end - m0;
        if (ONCE && !alone) return gemm4_tile<A_OC, B_OC, WM, WN, MI, NI, KD, S, VER>(p, place, smem);
        if (rows <= 32) return gemm4_tile<A_OC, B_OC, WM, WN, 1, NI, KD, S + 1, VER, ONCE>(p, place, smem);
        if (rows <= 64) return gemm4_tile<A_OC, B_OC, WM, WN, 2, NI, KD, S, VER, ONCE>(p, place, smem);
        if (rows <= 96) return gemm4_tile<A_OC, B_OC, WM, WN, 3, NI, KD, S, VER, ONCE>(p, place, smem);
    }
    gemm4_tile<A_OC, B_OC, WM, WN, MI, NI, KD, S, VER, ONCE>(p, place, smem);
}

// the sums of the slabs of gemm4_kernel<.., WM, WN, MI, NI, ..>: see gemm3_reduce_kernel; a block finishes 32 rows of 32 WN columns
template <int WM, int WN, int MI, int NI>
__global__ __launch_bounds__(256) void gemm4_reduce_kernel(GemmParams p) {
    constexpr int BM = WM * MI * 32, BN = WN * NI * 32, COLS = WN * 32, PITCH = COLS + 4;
    ARIA_SMEM_STATIC float sums[32 * PITCH];
    int tn, tmi;
    if (!aria_tile_from_pos(p, blockIdx.x, tmi, tn)) return;
    const int t = threadIdx.x, part = blockIdx.y, wm = part % WM, i = part / WM % MI, b = part / (WM * MI);
    const int l = t & 63, q = t >> 6;
    const float* ws = p.ws + (long long)blockIdx.x * p.split * (BM * BN) + part * (WN * 1024) + q * 256 + l * 4;
    f32x4 sum[WN];
#pragma unroll
    for (int k = 0; k < WN; ++k) sum[k] = *reinterpret_cast<const f32x4*>(ws + k * 1024);
    int s = 1;
    for (; s + 3 <= p.split; s += 3) {
        f32x4 v[3][WN];
#pragma unroll
        for (int z = 0; z < 3; ++z)
#pragma unroll
            for (int k = 0; k < WN; ++k) v[z][k] = *reinterpret_cast<const f32x4*>(ws + (long long)(s + z) * (BM * BN) + k * 1024);
#pragma unroll
        for (int z = 0; z < 3; ++z)
#pragma unroll
            for (int k = 0; k < WN; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[k][e] += v[z][k][e];
    }
    for (; s < p.split; ++s) {
        f32x4 v[WN];
#pragma unroll
        for (int k = 0; k < WN; ++k) v[k] = *reinterpret_cast<const f32x4*>(ws + (long long)s * (BM * BN) + k * 1024);
#pragma unroll
        for (int k = 0; k < WN; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[k][e] += v[k][e];
    }
#pragma unroll
    for (int k = 0; k < WN; ++k) *reinterpret_cast<f32x4*>(sums + (l & 31) * PITCH + k * 32 + 8 * q + 4 * (l >> 5)) = sum[k];
    sync();
    for (int idx = t; idx < 32 * COLS / 8; idx += 256) {
        const int row = idx / (COLS / 8), col = (idx % (COLS / 8)) * 8;
        aria_finish_sums(p, sums + row * PITCH + col, tmi * BM + i * (WM * 32) + wm * 32 + row, tn * BN + b * COLS + col);
    }
}


// the h-th expert of more than `rows` rows and its part of the reduction; false: there are fewer
__device__ __forceinline__ bool long_expert(const int* offsets, int E, int rows, int h, int l, int& e, int& k_begin, int& k_len) {
    for (int e0 = 0; e0 < E; e0 += 64) {
        const int begin = offsets[min(e0 + l, E)], n = offsets[min(e0 + l + 1, E)] - begin;
        unsigned long long m = ballot(n > rows);
        const int here = __builtin_popcountll(m);
        if (h >= here) {
            h -= here;
            continue;
        }
        for (; h > 0; --h) m &= m - 1;
        const int at = __builtin_ctzll(m);
        e = e0 + at, k_begin = first_lane(shfl(begin, at)), k_len = first_lane(shfl(n, at));
        return true;
    }
    return false;
}

// Weight gradients by strips (wgrad.h), and in front of them `tiling` workgroups that go through the tiles of the experts too long for strips; both kinds run side by side.
template <bool GATHER>
__global__ __launch_bounds__(256, 2) void wgrad_strip_kernel(GemmParams p, int tiling, int parts, int per) {
    ARIA_DYN_SMEM(smem);
    const int bid = blockIdx.x;
    if (bid >= tiling) {
        wgrad_strip<GATHER>(p, bid - tiling, int(gridDim.x) - tiling, parts, per, smem);
        return;
    }
    const int tiles = p.ntn * p.ntm, padded = (tiles + 7) & ~7;   // (an expert starts with XCD 0)
    for (int i = bid;; i += tiling) {
        int e = 0, k_begin = 0, k_len = 0, tmi = 0, tn = 0;
        if (!long_expert(p.offsets, p.E, KC, i / padded, int(threadIdx.x) & 63, e, k_begin, k_len)) return;
        if (i % padded >= tiles || !aria_tile_coords(p, i % padded, tiles, tmi, tn)) continue;
        sync();   // the rows that the tile before parked have left
        gemm4_tile<true, true, 1, 4, 4, 2, 32, 3, GATHER ? 11 : 3>(p, Tile4{tn, tmi * 128, p.M, k_begin, k_len, 0, (long long)e * p.strideC, -1, 0}, smem);
    }
}

template <bool A_OC, bool B_OC, int WM, int WN, int MI, int NI, int KD, int S, int VER, int PER_CU, bool ONCE = false, bool LOW = false>
int launch4(GemmParams q, int split, float* ws, void* stream) {
    using T = Shape4<WM, WN, MI, NI, KD, S>;
    constexpr int STEP = gated(VER) ? T::BN / 2 : T::BN;
    const int cols = gated(VER) ? q.N / 2 : q.N;
    q.ntn = (cols + STEP - 1) / STEP;
    q.ntm = q.mode == 1 ? q.M / T::BM + q.E : (q.M + T::BM - 1) / T::BM;
    q.split = split;
    q.ws = ws;
    if (q.ntn * q.ntm <= 0) return ARIA_OK;
    const unsigned grid = q.mode == 1 ? unsigned(q.ntn * q.ntm + 16) : unsigned(q.ntn * q.ntm * std::max(split, 1));
    static_assert(!LOW || Shape4<WM, WN, 1, NI, KD, S + 1>::SMEM <= T::SMEM, "the lowest tiles' stages");
    ARIA_LAUNCH((gemm4_kernel<A_OC, B_OC, WM, WN, MI, NI, KD, S, VER, PER_CU, ONCE, LOW>), dim3(grid, q.mode == 2 ? unsigned(q.E) : 1u), dim3(256), T::SMEM, stream, q);
    if (split > 1) ARIA_LAUNCH((gemm4_reduce_kernel<WM, WN, MI, NI>), dim3(unsigned(q.ntn * q.ntm), NI * MI * WM), dim3(256), 0, stream, q);
    return aria_check_launch();
}

constexpr long long ROUND = 256;   // CUs
long long cdiv(long long a, long long b) { return (a + b - 1) / b; }

// Time of a dense product, microseconds, as the kernels were measured on it (n: reduction in units of 64).  A round of the tiles named, whole workgroups a CU:
//   256 x 256 12 + 1.1 n (4096 x 2560: K 2560 57, 3328 69), split S times + 5 + 0.04 a slab (777 x 2560 x 2560, 40 tiles: 34)
//   128 x 128 5 + 1.25 n, three a CU
//   128 x 256 7 + 0.66 n (777 x 2560 x 2560 32.5, 1868 x 2560 x 2560 34, 777 x 7680 x 2560 36.5), split + 5 + 0.02 a slab (777 x 2560 x 2560 twice 27, 280 x 2560 x 2560 four
//     times 18.8)
//   256 x 160 9 + 0.85 n (4096 x 2560: K 2560 47.5, 3328 59; 5600 x 1536: K 1536 30.6, 4096 65.6)
//   128 x 320 9 + n (4096 x 2560: K 2560 51.3, 3328 63.4; K 7680 158 against 153: up to 4096)
double time_128(long long tiles, double n, int split) { return double(cdiv(tiles * split, ROUND)) * (7.0 + 0.66 * n / split) + (split > 1 ? 5.0 + 0.02 * double(tiles * split) : 0.0); }
double time_else(long long M, long long N, double n, int split) {
    const long long t3 = cdiv(M, 256) * cdiv(N, 256), t1 = cdiv(M, 128) * cdiv(N, 128);
    if (split > 1) return double(cdiv(t3 * split, ROUND)) * (12.0 + 1.1 * n / split) + 5.0 + 0.04 * double(t3 * split);
    return t3 >= 80 ? double(cdiv(t3, ROUND)) * (12.0 + 1.1 * n) : double(cdiv(t1, 3 * ROUND)) * (5.0 + 1.25 * n);
}

int split_128(long long M, long long N, long long K) {   // pieces of the reduction that tiles of 128 x 256 would take in one round
    const long long tiles = cdiv(M, 128) * cdiv(N, 256);
    const double n = double(K) / 64.0;
    int best = 1;
    for (int s = 2; s <= 8 && tiles * s <= ROUND && n / s >= 6.0; ++s)
        if (time_128(tiles, n, s) < 0.95 * time_128(tiles, n, best)) best = s;
    return best;
}
// outputs of at least four column tiles and reductions of at least 12 stages: what the figures above were taken on
bool dense_range(long long N, long long K) { return N >= 1024 && (N & 7) == 0 && K >= 768; }
// A dense product of one tile of rows with weights beyond the Infinity Cache (256 MB) is a stream of weights like an expert's.  100352 x 2560, us by the other tiles / by
// these: 17 rows 111 / 93, 32 118 / 98, 48 124 / 103, 64 125 / 108, 96 129 / 109, 112 135 / 116, 128 136 / 115 (two tiles of rows, 195, 154 / 193).  64000 x 1536, which the cache keeps, is level.
bool one_pass(const GemmParams& p, int a_oc, int b_oc) {
    return p.mode == 0 && !a_oc && !b_oc && p.M <= 128 && dense_range(p.N, p.K) && (long long)p.N * p.K >= 128 << 20 && aria_gemm3_workspace_bytes(p.M, p.N, p.K) == 0;
}

}  // namespace

long long aria_gemm4_workspace_bytes(long long M, long long N, long long K) {
    if (M <= 0 || !dense_range(N, K)) return 0;
    const int s = split_128(M, N, K);
    return s > 1 ? cdiv(M, 128) * cdiv(N, 256) * s * (128 * 256 * 4) : 0;
}

Gemm4Plan aria_plan_gemm4(const GemmParams& p, int a_oc, int b_oc, long long rows, int split3, long long workspace_bytes, bool own_cut) {
    Gemm4Plan none, plan;
    if (p.ext_k || p.rope_sn || (a_oc && !b_oc) || p.N < 8 || (a_oc && p.M < 8)) return none;   // (p.rope_sn: the entry takes whole rounds of 256 x 256 tiles only)
    const bool plain = !p.glu && !p.dglu && !p.rope_fc;
    if (const char* force = std::getenv("ARIA_GEMM_FORCE")) {   // "4": tiles of 128 x 256, "46": the wide ones, "47": strips, where there is such a form
        if (force[0] != '4') return none;
        plan.form = a_oc ? (force[1] == '7' && aria_wgrad_strips_take(p, rows, true) ? 4 : 3) : force[1] == '6' && plain && p.mode == 0 ? 2 : 1;
        plan.rows = rows;
        return plan;
    }
    if (a_oc && aria_wgrad_strips_take(p, rows)) {
        plan.form = 4, plan.rows = rows;
        return plan;
    }
    if (p.mode == 2) {   // rows: of all experts together, < 0: not known
        // Weight gradients by expert that strips do not take, 64 of them, 256 x 256 / 128 x 256 tiles: 2560 x 3328 at 6 rows each on average 283 / 222, 28 rows 301 / 237, 73 332 / 301, 140 405 / 392, 384
        // 641 / 634, 768 946 / 976; 1664 x 2560 139 / 114, 149 / 125, 171 / 161, 217 / 204, 328 / 328, 507 / 500.
        if (rows >= 0 && rows < 400ll * p.E) plan.form = 3;
        return plan;
    }
    if (a_oc) {   // 2560 x 2560, 7680 x 2560, 6656 x 2560: K 128 13 / 10, 21 / 18, 21 / 17; 784 24 / 18, 48 / 38, 49 / 39; 1568 39 / 27, 75 / 67, 68 / 66; 2048 45 / 33, 87 / 84, 77 / 82
        if (p.N >= 1024 && p.M >= 1024 && cdiv(p.M, 128) * cdiv(p.N, 256) <= 8 * ROUND && p.K >= 64 && p.K <= 1600) plan.form = 3;
        return plan;
    }
    if (p.mode == 1) {
        // Rows by expert.  Up to 100 an expert its tile of 256 rows is mostly empty and the weights' stream counts, of which three stages of 48 KiB keep more in flight.
        // 64 experts of 2560 x 1664, as a router gives the rows, 256 x 256 / these tiles, rows each on average 100, 120, 140: gate and up, gathered, [K, N] 287 / 244, 294 / 295, 298 / 338; down
        // [K, N] 144 / 118, 146 / 145, 151 / 154; SwiGLU backward 169 / 165, 176 / 188, 180 / 201; gate and up backward [N, K] 266 / 216, 271 / 253, 274 / 269.  And where all of it is one round:
        // 16 experts of 1024 x 768, 187 rows each, 32.6 / 20.2 and 25 / 16.
        if (p.K < 768 || p.N < 512) return none;
        const long long cols = p.glu ? p.N / 2 : p.N, ntn = cdiv(cols, p.glu ? 128 : 256);
        const bool few = p.M < 100ll * p.E, one_round = (p.M / 128 + p.E / 2) * ntn <= ROUND && p.M >= 16ll * p.E;
        if (few || one_round) plan.form = 1;
        return plan;
    }
    if (!dense_range(p.N, p.K)) return none;
    const double n = double(p.K) / 64.0;
    const long long t2 = cdiv(p.M, 128) * (p.glu ? cdiv(p.N / 2, 128) : cdiv(p.N, 256));
    if (!plain) {   // (these forms never split)
        if (t2 <= ROUND) plan.form = 1;
        return plan;
    }
    if (one_pass(p, a_oc, b_oc)) {
        plan.form = 1;
        return plan;
    }
    double best = 0.94 * time_else(p.M, p.N, n, split3);
    // A product's sums are cut where the 256 x 256 tiles cut them, and so have their bits.  Another cut rounds a few elements otherwise; in front of a router a near tie of a
    // token's last expert can turn, and in a short sample's gradient of the embedding, most of whose rows are zeros, single elements moved by 1.1 .. 1.9 of its root mean
    // square (64 .. 130 tokens; 0 with this cut, 777 tokens 5.15 -> 5.20 ms).  Given up for it, us: 777 x 2560 x 2560 in 3 pieces 27, in those tiles' 4 33; 4500 x 1536 x 4096
    // whole 57, in 2 68.  Aria's prompts of up to 288 tokens, which other kernels than the 256 x 256 tiles served before, are cut as it is fastest (own_cut; 280 tokens, four
    // layers: 1.014 times as fast as those with the 256 x 256 tiles' cut, 1.039 times with these tiles' own).
    int s = split3;
    if (own_cut) s = workspace_bytes >= aria_gemm4_workspace_bytes(p.M, p.N, p.K) ? split_128(p.M, p.N, p.K) : 1;
    if (t2 * s <= ROUND && time_128(t2, n, s) < best) best = time_128(t2, n, s), plan.form = 1, plan.split = s;
    const long long t6 = b_oc ? cdiv(p.M, 128) * cdiv(p.N, 320) : cdiv(p.M, 256) * cdiv(p.N, 160);
    const double time6 = 9.0 + (b_oc ? 1.0 : 0.85) * n;
    if (t6 <= ROUND && time6 < best && (own_cut || split3 == 1) && !(b_oc && p.K > 4096)) plan.form = 2, plan.split = 1;
    return plan;
}

// Where strips are the faster ones, us, 128 x 256 or 256 x 256 tiles / strips.  By expert, 64 of 2560 x 3328 (gathered) and 1664 x 2560, rows each on average, spread evenly, as a router
// does (the most wanted one four times the average) and with half of all rows on one expert: 6 254 / 200, 238 / 204, 238 / 198 and 124 / 109, 120 / 108, 122 / 108; 73 361 / 220, 336 / 225,
// 339 / 269 and 174 / 124, 166 / 126, 181 / 157; 144 471 / 292, 456 / 337, 446 / 344 and 225 / 160, 220 / 194, 244 / 207; beyond the line 192 456 / 322, 448 / 419 and 235 / 170, 237 / 218, 384 612 / 606,
// 624 / 615 and (a quarter on one) 628 / 749.  (Experts beyond 256 rows as strips too, 128 rows at a time: 73 rows, half on one, 339 / 794, 144 446 / 1386.)  All rows on six experts: 6
// 197 / 193 and 100 / 105, the rest zeros.  Dense: 100352 x 2560, 16 rows 266 / 106, 64 145 / 116, 200 209 / 163, 256 221 / 180; 64000 x 1536, 128
// rows 69 / 62, 256 91 / 82.  Outputs of a few rounds have too few strips: 7680 x 2560, 64 rows 18 / 22, 256 rows 25 / 34.  Dense ones of fewer than 64 rows are the others' slower
// kernels': 32000 x 1024, 8 rows 46 / 24, 2560 x 3328 15 / 20.
bool aria_wgrad_strips_take(const GemmParams& p, long long rows, bool any_size) {
    if (p.c_f32 || p.accumulate || p.bias || p.act || p.M % FT || p.N % STRIP || (reinterpret_cast<uintptr_t>(p.C) & 15) || (p.ldc & 7) || (p.strideC & 7)) return false;
    const long long experts = p.mode == 2 ? p.E : 1, outputs = experts * p.M * p.N;
    if (outputs <= (p.mode == 0 && p.K < 64 ? 16ll << 20 : 64ll << 20) && !any_size) return false;
    return p.mode == 2 ? rows >= 0 && rows <= 144 * experts : p.K <= KC;
}

static int launch_wgrad_strips(GemmParams p, long long rows, void* stream) {
    const int tiles = p.M / FT, experts = p.mode == 2 ? p.E : 1;
    // (ten tiles of 3.5 us to a start of 4; five or twenty 257 and 235 us for 240 at 73 rows, 207 and 219 for 206 at 26)
    const int parts = (tiles + 9) / 10, per = (tiles + parts - 1) / parts;
    using T = Shape4<1, 4, 4, 2, 32, 3>;
    p.ntm = (p.M + T::BM - 1) / T::BM, p.ntn = p.N / T::BN, p.order = 4, p.wide_store = 1, p.split = 1;
    // Experts of more than KC rows: at most rows / (KC + 1), whose tiles are a round of the chip's two workgroups a CU at a time.  (One at least: `rows` decides how many
    // workgroups look for them, never whether they are found.)
    const long long most = p.mode == 2 ? std::max<long long>(1, rows / (KC + 1)) : 0;
    const int tiling = int(std::min<long long>(2 * ROUND, most * ((p.ntm * p.ntn + 7) & ~7)));
    const dim3 grid(unsigned(tiling) + unsigned(experts) * unsigned(parts) * unsigned(p.N / STRIP));
    constexpr size_t SMEM = std::max(size_t(WGRAD_SMEM), T::SMEM);
    if (p.gather_rows)
        ARIA_LAUNCH((wgrad_strip_kernel<true>), grid, dim3(256), SMEM, stream, p, tiling, parts, per);
    else
        ARIA_LAUNCH((wgrad_strip_kernel<false>), grid, dim3(256), SMEM, stream, p, tiling, parts, per);
    return aria_check_launch();
}

int aria_launch_gemm4(const GemmParams& p, int a_oc, int b_oc, Gemm4Plan plan, float* ws, void* stream) {
    if (plan.form == 4) return launch_wgrad_strips(p, plan.rows, stream);
    GemmParams q = p;
    const char* wsd = std::getenv("ARIA_GEMM_WIDE_STORE");
    q.wide_store = !(wsd && wsd[0] == '0') && (reinterpret_cast<uintptr_t>(p.C) & 15) == 0 && (p.ldc & 7) == 0 && (p.strideC & 7) == 0;
    q.order = 4 | (p.glu && p.mode == 1 ? 512 : 0);
    const int split = ws && plan.split > 1 ? plan.split : 1;
    float* slabs = split > 1 ? ws : nullptr;
    if (plan.form == 3) {
        if (p.gather_rows) return launch4<true, true, 1, 4, 4, 2, 32, 3, 11, 2>(q, 1, nullptr, stream);
        return launch4<true, true, 1, 4, 4, 2, 32, 3, 3, 2>(q, 1, nullptr, stream);
    }
    if (plan.form == 2)
        return b_oc ? launch4<false, true, 2, 2, 2, 5, 32, 5, 3, 1>(q, 1, nullptr, stream) : launch4<false, false, 4, 1, 2, 5, 64, 3, 3, 1>(q, 1, nullptr, stream);
    // Weights by expert pass the caches where a tile is the only one of its expert's rows (gemm4_kernel): a stream of 500 MB at 6.9 TB/s for 6.2.  Tensors that the Infinity Cache keeps from one use to
    // the next lose by it: 16 experts of 1024 x 768 (25 MB) 13.8 us and 16.7; their pairs (50 MB), held 11.5 and 13.6, in turn with others 15.1 and 15.5.
    const bool once = p.mode == 1 ? p.expert_mod <= 0 && (long long)p.E * p.N * p.K >= 32 << 20 : one_pass(p, 0, b_oc);
#define ARIA_G4(BOC, VER) launch4<false, BOC, 1, 4, 4, 2, 64, 3, VER, 1>(q, split, slabs, stream)
#define ARIA_G4E(BOC, VER) \
    (once ? launch4<false, BOC, 1, 4, 4, 2, 64, 3, VER, 1, true, true>(q, split, slabs, stream) \
          : p.mode == 1 ? launch4<false, BOC, 1, 4, 4, 2, 64, 3, VER, 1, false, true>(q, split, slabs, stream) : ARIA_G4(BOC, VER))
    if (p.rope_fc) return ARIA_G4(false, 7);
    if (p.glu == 2) return ARIA_G4(false, 13);
    if (p.glu && p.gather_rows) return p.glu_up_rows > 0 ? ARIA_G4E(false, 9) : ARIA_G4E(true, 8);
    if (p.glu && p.glu_up_rows > 0) return ARIA_G4E(false, 6);
    if (p.glu) return b_oc ? ARIA_G4E(true, 14) : ARIA_G4(false, 14);
    if (p.dglu) return b_oc ? ARIA_G4(true, 5) : ARIA_G4E(false, 5);
    return b_oc ? ARIA_G4E(true, 3) : ARIA_G4E(false, 3);
#undef ARIA_G4E
#undef ARIA_G4
}
