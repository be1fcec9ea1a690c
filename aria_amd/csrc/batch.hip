// The decode step of several sequences of the gptfast (Aria) decoder: one token each, every weight read once for all of them.
//
// Running the sequences one after the other through decode.hip reads the whole model once per sequence (8 sequences at 28 layers: 62 GB).  Here a
// projection streams its rows past all tokens on the matrix pipe (rows.h) and a routed expert is read once for the tokens that chose it (experts.h); the
// shared expert is one more expert that every token chose.  RMS norms take no launch: the kernel that writes the residual stream leaves h = x w beside
// partial sums of x^2, the one that reads h scales its results by 1 / rms.  Nine launches a layer: qkv | attention (RoPE and cache write inside) | merge
// | wo + residual | router logits | routing and lists | up pairs + SwiGLU | down | weighted sum + residual.
// Tensors that the tile path materialises in bf16 are rounded here too (projections, SwiGLU, expert outputs, their weighted sum, residuals); norms, scores,
// softmax and sums are fp32.
#include "decode.h"
#include "experts.h"

namespace {
using namespace ad;

constexpr int STREAM_COLS = 256;   // stream columns per workgroup of the kernels that write the residual themselves
inline int stream_parts(int64_t D) { return int((D + STREAM_COLS - 1) / STREAM_COLS); }

// sum over a workgroup of 256 threads, in thread 0
__device__ __forceinline__ float block_sum(float v, float* red) {
    const float s = wave_sum_bcast(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    sync();
    return (red[0] + red[1]) + (red[2] + red[3]);
}
__global__ __launch_bounds__(256) void embedding_rows_kernel(const bf16_t* rows, const bf16_t* norm, bf16_t* x, bf16_t* h, float* sums, int D) {
    ARIA_SMEM_STATIC float red[4];
    const int n = blockIdx.x * STREAM_COLS + threadIdx.x, tok = blockIdx.y;
    float v = 0.f;
    if (n < D) {
        const bf16_t b = rows[(long long)tok * D + n];
        v = bf2f(b);
        x[(long long)tok * D + n] = b;
        h[(long long)tok * D + n] = f2bf(v * bf2f(norm[n]));
    }
    const float s = block_sum(v * v, red);
    if (threadIdx.x == 0) sums[tok * gridDim.x + blockIdx.x] = s;
}

struct StoreBf16 {
    static constexpr bool SUMSQ = false, WAVES = false;
    bf16_t* out;
    long long ld;
    float* sums = nullptr;
    __device__ __forceinline__ float operator()(float v, int tok, int n, int) const {
        out[tok * ld + n] = f2bf(v);
        return 0.f;
    }
};
struct StoreF32 {
    static constexpr bool SUMSQ = false, WAVES = false;
    float* out;
    long long ld;
    float* sums = nullptr;
    __device__ __forceinline__ float operator()(float v, int tok, int n, int) const {
        out[tok * ld + n] = v;
        return 0.f;
    }
};
struct Residual {   // x += the rounded product; the next norm's input beside it
    static constexpr bool SUMSQ = true, WAVES = false;
    bf16_t *x, *h;
    const bf16_t* norm;
    long long D;
    float* sums;
    __device__ __forceinline__ float operator()(float v, int tok, int n, int) const {
        const float y = rbf(bf2f(x[tok * D + n]) + rbf(v));
        x[tok * D + n] = f2bf(y);
        h[tok * D + n] = f2bf(y * bf2f(norm[n]));
        return y * y;
    }
};
// routing of T tokens (a wave each), the lists of the experts in use -- slots k .. k + ns - 1 of a token are the shared expert's slices -- and 1 / rms of h
__global__ __launch_bounds__(1024) void route_lists_kernel(const bf16_t* logits, int E, int k, int ns, int T, float* scores, float* rinv, RowsIn norm, ExpertLists lists) {
    ARIA_SMEM_STATIC ListsLds sl;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, ks = k + ns;
    for (int tok = w; tok < T; tok += 16) {
        float ss = 0.f;
        for (int j = l; j < norm.sq_n; j += 64) ss += norm.sq[(long long)tok * norm.sq_n + j];
        float score;
        int id;
        route_one_token(logits + (long long)tok * E, E, k, l, 0, score, id);
        if (l < ks) sl.idx[tok * ks + l] = l < k ? id : E + l - k;
        if (l < k) scores[tok * k + l] = rbf(score);
        ss = wave_sum_bcast(ss);
        if (l == 0) rinv[tok] = 1.f / sqrtf(ss * norm.inv_n + norm.eps);
    }
    write_lists(lists, sl, T * ks);
}
struct GatedAct {
    bf16_t* act;
    const float* rinv;
    int F, div;
    __device__ __forceinline__ void operator()(float g, float u, int entry, int n) const {
        const float r = rinv[entry / div];
        act[(long long)entry * F + n] = f2bf(rbf(silu_fast(rbf(g * r))) * rbf(u * r));
    }
};
struct Partial {
    float* out;
    long long D;
    __device__ __forceinline__ void operator()(float v, float, int entry, int n) const { out[entry * D + n] = v; }
};
// x += (the experts' weighted sum + the shared expert); the next norm's input beside it
__global__ __launch_bounds__(256) void moe_sum_kernel(const float* part, const float* scores, int k, int ns, bf16_t* x, bf16_t* h, const bf16_t* norm, float* sums,
                                                      int D) {
    ARIA_SMEM_STATIC float red[4];
    const int n = blockIdx.x * STREAM_COLS + threadIdx.x, tok = blockIdx.y, ks = k + ns;
    float y = 0.f;
    if (n < D) {
        const float* p = part + (long long)tok * ks * D + n;
        float v[8], routed = 0.f, shared = 0.f;   // k <= 8
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = p[(long long)min(j, k - 1) * D];
        for (int i = k; i < ks; ++i) shared += p[(long long)i * D];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j < k) routed += rbf(rbf(v[j]) * scores[tok * k + j]);
        const long long at = (long long)tok * D + n;
        y = rbf(bf2f(x[at]) + rbf(rbf(routed) + rbf(shared)));
        x[at] = f2bf(y);
        h[at] = f2bf(y * bf2f(norm[n]));
    }
    const float s = block_sum(y * y, red);
    if (threadIdx.x == 0) sums[tok * gridDim.x + blockIdx.x] = s;
}

struct Scratch {
    bf16_t *x, *h, *qkv, *ao, *logits, *act;
    float *sums, *part, *scores, *rinv, *eo;
    int32_t *table, *list;
    int64_t bytes;
};
Scratch layout(const int64_t* d, int64_t T, int64_t max_len, char* base) {
    const int64_t D = d[1], H = d[2], hd = d[3], E = d[4], k = d[5], I = d[6], ns = d[7] / d[6], ks = k + ns;
    Scratch z{};
    int64_t at = 0;
    auto take = [&](int64_t bytes) {
        char* p = base + at;
        at += (bytes + 255) & ~int64_t(255);
        return p;
    };
    z.x = reinterpret_cast<bf16_t*>(take(2 * T * D));
    z.h = reinterpret_cast<bf16_t*>(take(2 * T * D));
    z.qkv = reinterpret_cast<bf16_t*>(take(6 * T * D));
    z.ao = reinterpret_cast<bf16_t*>(take(2 * T * D));
    z.logits = reinterpret_cast<bf16_t*>(take(2 * T * E));
    z.act = reinterpret_cast<bf16_t*>(take(2 * T * ks * I));
    z.sums = reinterpret_cast<float*>(take(4 * T * std::max(rows_parts(T, D), stream_parts(D))));
    z.part = reinterpret_cast<float*>(take(4 * T * H * aria_decode_rows_splits(H, T, max_len, d[9]) * (hd + 2)));
    z.scores = reinterpret_cast<float*>(take(4 * T * k));
    z.rinv = reinterpret_cast<float*>(take(4 * T));
    z.eo = reinterpret_cast<float*>(take(4 * T * ks * D));
    z.table = reinterpret_cast<int32_t*>(take(4 * ExpertLists::table_ints(E + ns)));
    z.list = reinterpret_cast<int32_t*>(take(4 * T * ks));
    z.bytes = at;
    return z;
}
bool batch_ok(const int64_t* d, int64_t T) {
    const int64_t ns = d[7] / d[6];
    return d[5] >= 1 && expert_rows_can(d[1], d[6], d[4] + ns, d[5] + ns, T);
}

}  // namespace

extern "C" {

int64_t aria_decode_step_scratch(const int64_t* dims, int64_t T, int64_t max_len) {
    if (!dims || T <= 0 || max_len <= 0 || aria_decode_dims_ok(dims) != ARIA_OK) return 0;
    if (T == 1) return aria_decode_one_scratch(dims);
    return batch_ok(dims, T) ? layout(dims, T, max_len, nullptr).bytes : 0;
}

int aria_decode_step(const void* const* ptrs, const int64_t* dims, float eps, int64_t T, const void* x, const int32_t* slot, const int32_t* pos,
                     int64_t max_len, float* logits, void* scratch, int64_t scratch_bytes, void* stream) {
    if (!ptrs || !dims || !x || !slot || !pos || !logits || !scratch || T < 0 || max_len <= 0) return ARIA_ERR_INVALID;
    if (T == 0) return ARIA_OK;
    if ((reinterpret_cast<uintptr_t>(scratch) | reinterpret_cast<uintptr_t>(x)) & 15) return ARIA_ERR_ALIGN;
    const int64_t need = aria_decode_step_scratch(dims, T, max_len);
    if (need == 0) return ARIA_ERR_UNSUPPORTED;
    const int64_t L = dims[0], D = dims[1], H = dims[2], hd = dims[3], E = dims[4], k = dims[5], I = dims[6], Is = dims[7], V = dims[8], Smax = dims[9];
    if (scratch_bytes < need || max_len > Smax) return ARIA_ERR_INVALID;
    if (const int bad = aria_decode_table_ok(ptrs, L)) return bad;
    if (T == 1) return aria_decode_one(ptrs, dims, eps, x, slot, pos, max_len, logits, static_cast<char*>(scratch), stream);
    const Scratch z = layout(dims, T, max_len, static_cast<char*>(scratch));
    auto weight = [&](int64_t i) { return static_cast<const bf16_t*>(ptrs[i]); };
    const int64_t ns = Is / I;
    const int parts = stream_parts(D), splits = aria_decode_rows_splits(H, T, max_len, Smax);
    const dim3 stream_grid = dim3(unsigned(parts), unsigned(T));
    const float inv_n = 1.f / float(D);
    int sq_n = parts;   // partial sums a token has beside h
    auto input = [&](const bf16_t* W, int64_t N) { return RowsIn{W, nullptr, z.h, (long long)D, int(D), int(N), z.sums, sq_n, inv_n, eps}; };
    auto rows = [&](const RowsIn& in, const auto& e) { return launch_rows(RowsPair{{in, in}}, 1, T, e, stream); };
    ARIA_LAUNCH(embedding_rows_kernel, stream_grid, dim3(256), 0, stream, static_cast<const bf16_t*>(x), weight(ARIA_DECODE_STEP_PTRS), z.x, z.h, z.sums,
                int(D));
    int rc = aria_check_launch();
    const ExpertLists lists{z.table, z.list, int(E + ns)};
    for (int64_t li = 0; li < L && rc == ARIA_OK; ++li) {
        const int64_t p = ARIA_DECODE_STEP_PTRS + ARIA_DECODE_LAYER_PTRS * li;
        bf16_t *kc = const_cast<bf16_t*>(weight(p + 11)), *vc = const_cast<bf16_t*>(weight(p + 12));
        rc = rows(input(weight(p + 1), 3 * D), StoreBf16{z.qkv, 3 * D});
        if (rc == ARIA_OK) rc = aria_decode_rows_attn(z.qkv, weight(0), slot, pos, kc, vc, z.ao, z.part, H, hd, Smax, T, splits, max_len, stream);
        RowsIn wo{weight(p + 2), nullptr, z.ao, (long long)D, int(D), int(D)};
        if (rc == ARIA_OK) rc = rows(wo, Residual{z.x, z.h, weight(p + 3), (long long)D, z.sums});
        sq_n = rows_parts(T, D);
        if (rc == ARIA_OK) rc = rows(input(weight(p + 4), E), StoreBf16{z.logits, (long long)E});
        if (rc != ARIA_OK) break;
        ARIA_LAUNCH(route_lists_kernel, dim3(1), dim3(1024), 0, stream, (const bf16_t*)z.logits, int(E), int(k), int(ns), int(T), z.scores, z.rinv,
                    input(nullptr, 0), lists);
        const ExpertIn up{weight(p + 5), weight(p + 6), z.h, (long long)D, int(k + ns), int(D), int(I), weight(p + 8), weight(p + 9), (long long)(I * D),
                          (long long)D, int(E)};
        const ExpertIn down{weight(p + 7), nullptr, z.act, (long long)I, 1, int(I), int(D), weight(p + 10), nullptr, (long long)I, (long long)Is, int(E)};
        rc = aria_check_launch();
        if (rc == ARIA_OK) rc = launch_expert_rows<true>(up, lists, k + ns, T, GatedAct{z.act, z.rinv, int(I), int(k + ns)}, stream);
        if (rc == ARIA_OK) rc = launch_expert_rows<false>(down, lists, k + ns, T, Partial{z.eo, (long long)D}, stream);
        if (rc != ARIA_OK) break;
        sq_n = parts;
        ARIA_LAUNCH(moe_sum_kernel, stream_grid, dim3(256), 0, stream, (const float*)z.eo, (const float*)z.scores, int(k), int(ns), z.x, z.h,
                    li + 1 < L ? weight(p + ARIA_DECODE_LAYER_PTRS) : weight(1), z.sums, int(D));
        rc = aria_check_launch();
    }
    if (rc != ARIA_OK) return rc;
    return rows(input(weight(2), V), StoreF32{logits, (long long)V});
}

}  // extern "C"
