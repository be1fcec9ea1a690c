// Products of 17 .. a few hundred tokens that are bound by their weights: short prompts, and the experts of somewhat longer ones.
//
// A 256 x 256 tile of the matrix product leaves most of the chip idle there: 280 tokens x 7680 outputs are 60 tiles, each with the whole reduction to itself
// (44 us for 39 MB of weights).  The row-streaming kernels of the decode step (rows.h) split the reduction over a workgroup's waves instead and take
// up to 64 tokens at a time past the weights; further tokens find the weights in the L2 / MALL.  Weights from HBM, us as tiles / here: 64 tokens: q | k | v
// 29 / 17, gate and up with SwiGLU (2 x 3328) 48 / 18, 2560 x 2560 27 / 13; 280: 44 / 37, 49 / 39, 30 / 21; 352: 45 / 44, 52 / 40, 30 / 21; 400: 46 / 54,
// 57 / 48, 31 / 24; lm_head of one token 140 / 86.
// Routed experts: with n tokens an expert's matrix meets n k / E rows (26 at 280 tokens, 6 of 64 experts); its rows are read once per 64 of them, by whole lines that are non-temporal
// (rows.h).  Up pairs (64 experts of 2 x 1664 x 2560), half lines / whole: 24 tokens 174 / 151, 64 204 / 172, 128 220 / 180, 280 238 / 193 (5.6 TB/s of weights); 32 of 2 x 1024 x 1536, 4 a
// token: 64 tokens 43 / 34, 280 58 / 52.  Down (2560 x 1664): 24 tokens 93 / 77, 64 109 / 89, 280 130 / 116.  The line to the tiles: aria_rows_experts_most.
#include "rows.h"

namespace {
using namespace ad;

template <class T>
struct Store {
    static constexpr bool SUMSQ = false, WAVES = false;
    T* out;
    long long ld;
    float* sums = nullptr;
    __device__ __forceinline__ float operator()(float v, int tok, int n, int) const {
        stf(out + tok * ld + n, v);
        return 0.f;
    }
};
struct SwiGlu {   // rounded where the unfused chain has bf16 tensors
    static constexpr bool SUMSQ = false, WAVES = false;
    bf16_t* act;
    long long ld;
    float* sums = nullptr;
    __device__ __forceinline__ void operator()(float g, float u, int tok, int n) const { act[tok * ld + n] = f2bf(rbf(silu_fast(rbf(g))) * rbf(u)); }
};
// q rotated to its own rows, k rotated and v into the cache: row pos of the slot (slot NULL: slot 0, position = token)
struct QkvCache {
    static constexpr bool SUMSQ = false, WAVES = true;
    bf16_t *q, *kc, *vc;
    const bf16_t* fc;
    const int32_t *slot, *pos;
    long long S;
    int D, hd;
    float* sums = nullptr;
    __device__ __forceinline__ void operator()(float v, int tok, int n, bool in) const {
        const float mine = rbf(v), other = xor1(mine);   // (interleaved pairs: neighbouring columns, neighbouring lanes)
        if (!in) return;
        const int ps = pos ? pos[tok] : tok, part = n / D, col = n - part * D;
        const long long row = ((slot ? slot[tok] * S : 0) + ps) * D + col;
        if (part == 2) {
            vc[row] = f2bf(mine);
            return;
        }
        const uint32_t cs = *reinterpret_cast<const uint32_t*>(fc + (long long)ps * hd + (col % hd & ~1));
        const float c = bflo(cs), s = bfhi(cs);
        const bf16_t y = f2bf(col & 1 ? mine * c + other * s : mine * c - other * s);
        if (part)
            kc[row] = y;
        else
            q[(long long)tok * D + col] = y;
    }
};

struct ExpertRows {   // rows sorted by expert: X row of place i is rows[i] (rows NULL: i)
    const bf16_t *W, *W2, *X;
    const int32_t *rows, *offsets;
    long long ldx;
    int E, K, N;
};
// upto[e]: tiles of up to ROWS rows that experts 0 .. e have together; the sum of all
template <int ROWS>
__device__ __forceinline__ int count_tiles(const int32_t* offsets, int E, int* upto) {
    const int l = threadIdx.x & 63;
    int seen = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = min(e0 + l, E - 1), n = e0 + l < E ? offsets[e + 1] - offsets[e] : 0;
        const int at = seen + wave_incl_scan((n + ROWS - 1) / ROWS);
        if (int(threadIdx.x) == l && e0 + l < E) upto[e] = at;   // (the first wave; all waves hold the same numbers)
        seen = read_lane(at, 63);
    }
    return seen;
}
// The weight row groups of all token tiles of all experts are one sequence, cut into equal pieces for the workgroups (experts.h): an expert with more rows than a
// tile holds is further work in the sequence.  (As further work of the workgroups that own its weight rows it held up the launch: 64 experts of
// 2 x 1664 x 2560, 280 tokens, 80 rows for the most popular one: 361 us, now 245; 55 rows 234 in both.)  e(value, up value, place, row)
template <int KS, int MT, class Ep, bool PAIR, bool ONCE>
__global__ __launch_bounds__(512) void sorted_rows_kernel(ExpertRows in, Ep e) {
    ARIA_SMEM_STATIC RowsRed<8, MT> red;
    ARIA_SMEM_STATIC int upto[256];
    constexpr int OUT = PAIR ? 8 : 16, ROWS = 16 * MT;
    const int t = threadIdx.x, l = t & 63, c16 = t & 15, groups = (in.N + OUT - 1) / OUT;
    const int total = count_tiles<ROWS>(in.offsets, in.E, upto) * groups;
    const int per = (total + int(gridDim.x) - 1) / int(gridDim.x), end = min(total, (int(blockIdx.x) + 1) * per);
    int g = int(blockIdx.x) * per;
    sync();
    while (g < end) {
        const int tile = g / groups, g0 = g - tile * groups, g1 = min(groups, g0 + end - g);
        int id = 0;
        for (int e0 = 0; e0 < in.E; e0 += 64) {   // the first expert with tiles beyond this one's number
            const unsigned long long behind = ballot(e0 + l < in.E && upto[min(e0 + l, in.E - 1)] > tile);
            id = e0 + (behind ? __builtin_ctzll(behind) : 0);
            if (behind) break;
        }
        const int first = in.offsets[id], m = in.offsets[id + 1] - first, t0 = (tile - (id ? upto[id - 1] : 0)) * ROWS;
        const long long at = (long long)id * in.N * in.K;
        sync();   // (the sums of the piece before are read)
        stream_rows<8, KS, MT, ONCE>(
            in.K, [&](int gg, int r) { return (PAIR && r >= 8 ? in.W2 : in.W) + at + (long long)min(gg * OUT + (PAIR ? r & 7 : r), in.N - 1) * in.K; },
            [&](int i) {
                const int at = first + min(t0 + 16 * i + c16, m - 1);
                return in.X + (long long)(in.rows ? in.rows[at] : at) * in.ldx;
            },
            g0, g1, red, [&](float v, int tok, int n, int gg) {
                const float u = PAIR ? shfl_xor(v, 8) : 0.f;
                if (t0 + tok < m && gg * OUT + n < in.N && n < OUT) e(v, u, first + t0 + tok, gg * OUT + n);
            });
        g += g1 - g0;
    }
}
struct ExpertAct {
    bf16_t* act;
    long long ld;
    __device__ __forceinline__ void operator()(float g, float u, int at, int n) const { act[at * ld + n] = f2bf(rbf(silu_fast(rbf(g))) * rbf(u)); }
};
struct ExpertOut {
    bf16_t* out;
    long long ld;
    __device__ __forceinline__ void operator()(float v, float, int at, int n) const { out[at * ld + n] = f2bf(v); }
};
template <bool PAIR, class Ep>
int launch_sorted_rows(const ExpertRows& in, int64_t M, const Ep& e, void* stream) {
    const int64_t rows = (M + in.E - 1) / in.E, most = int64_t((in.N + (PAIR ? 7 : 15)) / (PAIR ? 8 : 16)) * std::min<int64_t>(in.E, M);
    const int mt = rows_tiles(in.K, 4 * rows);   // (loads differ: tiles for four times the average -- 280 tokens, 26 rows an expert on average, 63 at most)
    const dim3 grid(unsigned(std::min<int64_t>(mt > 2 ? 256 : 512, most)));
    const bool once = experts_once(in.E, in.N * (PAIR ? 2 : 1), in.K, 16);
#define ARIA_SORTED(KS, MT)                                                                                  \
    if (once)                                                                                                \
        ARIA_LAUNCH((sorted_rows_kernel<KS, MT, Ep, PAIR, true>), grid, dim3(512), 0, stream, in, e);        \
    else                                                                                                     \
        ARIA_LAUNCH((sorted_rows_kernel<KS, MT, Ep, PAIR, false>), grid, dim3(512), 0, stream, in, e)
#define ARIA_SORTED_TILES(KS) \
    if (mt == 1) {            \
        ARIA_SORTED(KS, 1);   \
    } else if (mt == 2) {     \
        ARIA_SORTED(KS, 2);   \
    } else {                  \
        ARIA_SORTED(KS, 4);   \
    }
    if (in.K <= 1024) {
        ARIA_SORTED_TILES(4);
    } else if (in.K <= 1536) {
        ARIA_SORTED_TILES(6);
    } else if (in.K <= 1792) {
        ARIA_SORTED_TILES(7);
    } else {
        ARIA_SORTED_TILES(10);
    }
#undef ARIA_SORTED
#undef ARIA_SORTED_TILES
    return aria_check_launch();
}
bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

extern "C" {

int aria_rows_gemm(const void* X, const void* W, void* out, int out_f32, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldo, void* stream) {
    if (!X || !W || !out || M < 0 || N < 0) return ARIA_ERR_INVALID;
    if (!al16(X) || !al16(W) || (ldx & 7) || (K & 7)) return ARIA_ERR_ALIGN;
    if (K < 128 || K > 4096) return ARIA_ERR_UNSUPPORTED;
    if (M == 0 || N == 0) return ARIA_OK;
    const RowsIn in{static_cast<const bf16_t*>(W), nullptr, static_cast<const bf16_t*>(X), (long long)ldx, int(K), int(N)};
    if (out_f32) return launch_rows_wide<false>(in, M, Store<float>{static_cast<float*>(out), (long long)ldo}, stream);
    return launch_rows_wide<false>(in, M, Store<bf16_t>{static_cast<bf16_t*>(out), (long long)ldo}, stream);
}

int aria_rows_swiglu(const void* X, const void* Wg, const void* Wu, void* act, int64_t M, int64_t I, int64_t K, int64_t ldx, int64_t ldact, void* stream) {
    if (!X || !Wg || !Wu || !act || M < 0 || I < 0) return ARIA_ERR_INVALID;
    if (!al16(X) || !al16(Wg) || !al16(Wu) || (ldx & 7) || (K & 7)) return ARIA_ERR_ALIGN;
    if (K < 128 || K > 4096) return ARIA_ERR_UNSUPPORTED;
    if (M == 0 || I == 0) return ARIA_OK;
    const RowsIn in{static_cast<const bf16_t*>(Wg), static_cast<const bf16_t*>(Wu), static_cast<const bf16_t*>(X), (long long)ldx, int(K), int(I)};
    return launch_rows_wide<true>(in, M, SwiGlu{static_cast<bf16_t*>(act), (long long)ldact}, stream);
}

int aria_rows_qkv_rope_cache(const void* X, const void* Wqkv, void* Q, void* Kc, void* Vc, const void* freqs_cis, const int32_t* slot, const int32_t* pos,
                             int64_t M, int64_t D, int64_t K, int64_t hd, int64_t S_cache, int64_t ldx, void* stream) {
    if (!X || !Wqkv || !Q || !Kc || !Vc || !freqs_cis || M < 0 || D <= 0 || hd <= 0 || S_cache <= 0 || !slot != !pos) return ARIA_ERR_INVALID;
    if (!al16(X) || !al16(Wqkv) || (ldx & 7) || (K & 7)) return ARIA_ERR_ALIGN;
    if (K < 128 || K > 4096 || (D & 15) || (hd & 1) || D % hd || (!pos && M > S_cache)) return ARIA_ERR_UNSUPPORTED;
    if (M == 0) return ARIA_OK;
    const RowsIn in{static_cast<const bf16_t*>(Wqkv), nullptr, static_cast<const bf16_t*>(X), (long long)ldx, int(K), int(3 * D)};
    return launch_rows_wide<false>(in, M, QkvCache{static_cast<bf16_t*>(Q), static_cast<bf16_t*>(Kc), static_cast<bf16_t*>(Vc),
                                                   static_cast<const bf16_t*>(freqs_cis), slot, pos, (long long)S_cache, int(D), int(hd)}, stream);
}

// The line between rows by expert and tiles.  Gate and up, launches of one kind in turn, us by rows / tiles: 64 experts of 1664 x 2560: 6 rows an expert 162 / 182, 12 180 / 184, 16 180 / 186, 20
// 200 / 187, 28 205 / 192, 40 230 / 199; 32 of 1024 x 1536: 8 33.1 / 34.3, 10 39.2 / 35.0, 20 42.6 / 35.8, 40 48.8 / 36.9.  Fewer weights are a launch's ramp: 16 of 768 x 1024: 12 14.1 / 16.0, 28
// 15.9 / 17.2, 40 16.4 / 18.3.  Down: 64 experts 6 88.0 / 89.5, 10 89.3 / 90.6, 12 93.8 / 90.7, 16 114 / 92; 32: 8 19.5 / 19.0, 12 23.4 / 19.5; 16: 10 10.5 / 11.4, 16 13.1 / 11.7.
// A prompt's outputs hold to where the line lay when the tiles were slower, 8 and 4 rows: rows add in another order, which moves an Aria prompt's logits by 0.7 % at the same error against 64 bits.
// Its four layers by rows up to 27 and 10 rows / by this line: 86 tokens 1706 / 1768, 130 1833 / 1858, 200 1890 / 1932, 240 1926 / 1973, 280 2060 / 2038 and, of another draw, 1978 / 2034.
int64_t aria_rows_experts_most(int64_t E, int64_t N, int64_t K, int which) {
    if (which == ARIA_ROWS_DOWN) return 4 * E;
    return which == ARIA_ROWS_PAIR && E * N * K >= 1 << 25 ? 8 * E : 27 * E;
}

int aria_rows_experts(const void* X, const int32_t* rows, const int32_t* offsets, const void* W, const void* Wu, void* out, int64_t E, int64_t M, int64_t N,
                      int64_t K, int64_t ldx, int64_t ldo, void* stream) {
    if (!X || !offsets || !W || !out || E <= 0 || M < 0 || N <= 0) return ARIA_ERR_INVALID;
    if (!al16(X) || !al16(W) || (Wu && !al16(Wu)) || (ldx & 7) || (K & 7)) return ARIA_ERR_ALIGN;
    if (K < 128 || K > 2560 || E > 256) return ARIA_ERR_UNSUPPORTED;
    if (M == 0) return ARIA_OK;
    const ExpertRows in{static_cast<const bf16_t*>(W), static_cast<const bf16_t*>(Wu), static_cast<const bf16_t*>(X), rows, offsets, (long long)ldx, int(E),
                        int(K), int(N)};
    if (Wu) return launch_sorted_rows<true>(in, M, ExpertAct{static_cast<bf16_t*>(out), (long long)ldo}, stream);
    return launch_sorted_rows<false>(in, M, ExpertOut{static_cast<bf16_t*>(out), (long long)ldo}, stream);
}

}  // extern "C"
