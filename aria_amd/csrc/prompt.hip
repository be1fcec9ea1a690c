// A serving step over short prompts of the gptfast (Aria) decoder in one call: packed tokens of one or several sequences, the products by the row-streaming kernels
// of wide.hip, by the tiles of gemm4.hip from 193 tokens on, the experts' from 9 (down-projections: five) rows an expert on.  At these sizes a layer is fifteen launches of 5 .. 230 us;
// enqueued one by one from Python they take longer than they run (four layers, 280 tokens: 3.2 ms of host time for 2.5 ms of kernels).
// Served: what wide.hip's products take, up to 27 rows an expert on average (6 of 64 experts: 288 tokens).
#include "decode.h"
#include "gemm_params.h"
#include "rows.h"
#include <algorithm>

namespace {
using namespace ad;

__global__ __launch_bounds__(256) void clear_counts_kernel(int32_t* counts, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) counts[i] = 0;
}

struct Scratch {
    bf16_t *x, *y, *h, *qkv, *ao, *d, *logits, *scores, *act, *eo, *sact, *sh;
    int32_t *idx, *counts, *offsets, *src, *inv, *rows;
    char* ws;
    int64_t ws_bytes, bytes;
};
// A dense product x [T, K] w [N, K]^T as tiles (its reduction in pieces).  Weights from HBM, us by rows / tiles: 7680 x 2560: 128 tokens 23.7 / 23.7, 200 32.0 / 28.1, 256 34.6 /
// 30.2, 288 38.0 / 34.8; 2560 x 2560: 200 19.0 / 19.0, 288 21.1 / 20.0; 2560 x 3328: 200 23.2 / 18.9, 288 31.2 / 21.6.  Narrower: 4096 x 1536: 288 19.3 / 18.9.
bool tiles_ahead(int64_t T, int64_t N, int64_t K) { return T > 192 && K >= 2048 && N * K >= (6 << 20) && K % 64 == 0 && N % 8 == 0; }
Scratch layout(const int64_t* dims, int64_t T, char* base) {
    const int64_t L = dims[0], D = dims[1], E = dims[4], k = dims[5], I = dims[6], Is = dims[7];
    Scratch z{};
    int64_t at = 0;
    auto take = [&](int64_t bytes) {
        char* p = base + at;
        at += (bytes + 255) & ~int64_t(255);
        return p;
    };
    auto rows = [&](int64_t n) { return reinterpret_cast<bf16_t*>(take(2 * T * n)); };
    z.x = rows(D), z.y = rows(D), z.h = rows(D), z.qkv = rows(3 * D), z.ao = rows(D), z.d = rows(D), z.logits = rows(E), z.scores = rows(k);
    z.act = rows(k * I), z.eo = rows(k * D), z.sact = rows(Is), z.sh = rows(D);
    auto ints = [&](int64_t n) { return reinterpret_cast<int32_t*>(take(4 * n)); };
    z.idx = ints(T * k), z.counts = ints(L * E), z.offsets = ints(E + 1), z.src = ints(T * k), z.inv = ints(T * k), z.rows = ints(T * k);
    const int64_t shapes[3][2] = {{3 * D, D}, {D, D}, {D, Is}};
    for (const auto& nk : shapes)
        if (tiles_ahead(T, nk[0], nk[1])) z.ws_bytes = std::max(z.ws_bytes, aria_gemm_own_cut_bytes(T, nk[0], nk[1]));
    z.ws = take(z.ws_bytes);
    z.bytes = at;
    return z;
}
bool prompt_ok(const int64_t* d, int64_t T) {
    const int64_t D = d[1], E = d[4], k = d[5], I = d[6], Is = d[7];
    return aria_decode_dims_ok(d) == ARIA_OK && E <= 64 && k >= 1 && k <= E && T * k <= std::min<int64_t>(8192, aria_rows_experts_most(E, I, D, ARIA_ROWS_PAIR_ONLY)) && D >= 512 && D <= 2560 && I >= 512 && I <= 2560 && Is <= 4096 &&
           D % 16 == 0;
}

}  // namespace

extern "C" {

int64_t aria_prompt_step_scratch(const int64_t* dims, int64_t T) {
    return dims && T > 0 && prompt_ok(dims, T) ? layout(dims, T, nullptr).bytes : 0;
}

int aria_prompt_step(const void* const* ptrs, const int64_t* dims, float eps, int64_t T, const void* embedded, const int32_t* slot, const int32_t* pos,
                     const int32_t* cu, int64_t n_seq, int64_t longest, const int32_t* wanted, int64_t n_wanted, float* logits, void* scratch,
                     int64_t scratch_bytes, void* stream) {
    if (!ptrs || !dims || !embedded || !slot || !pos || !cu || !scratch || T < 0 || n_seq <= 0 || longest <= 0 || n_wanted < 0 || (n_wanted && (!wanted || !logits)))
        return ARIA_ERR_INVALID;
    if (T == 0) return ARIA_OK;
    if ((reinterpret_cast<uintptr_t>(scratch) | reinterpret_cast<uintptr_t>(embedded)) & 15) return ARIA_ERR_ALIGN;
    const int64_t need = aria_prompt_step_scratch(dims, T);
    if (need == 0) return ARIA_ERR_UNSUPPORTED;
    const int64_t L = dims[0], D = dims[1], H = dims[2], hd = dims[3], E = dims[4], k = dims[5], I = dims[6], Is = dims[7], V = dims[8], Smax = dims[9];
    if (scratch_bytes < need || longest > Smax || n_wanted > T) return ARIA_ERR_INVALID;
    if (const int bad = aria_decode_table_ok(ptrs, L)) return bad;
    const Scratch z = layout(dims, T, static_cast<char*>(scratch));
    ARIA_LAUNCH(clear_counts_kernel, dim3(unsigned((L * E + 255) / 256)), dim3(256), 0, stream, z.counts, int(L * E));
    int rc = aria_check_launch();
    const bf16_t *x = static_cast<const bf16_t*>(embedded), *delta = nullptr;   // the residual before the sum that comes next; y: behind it
    bf16_t *y = z.x, *spare = z.y;
    auto summed = [&] {
        x = y;
        std::swap(y, spare);
    };
    auto product = [&](const bf16_t* a, const void* w, bf16_t* out, int64_t N, int64_t K) {
        if (tiles_ahead(T, N, K)) return aria_gemm_own_cut(a, w, out, T, N, K, z.ws_bytes ? z.ws : nullptr, z.ws_bytes, stream);
        return aria_rows_gemm(a, w, out, 0, T, N, K, K, N, stream);
    };
    // (the line between rows and tiles by expert: wide.hip)
    auto expert_pairs = [&](const void* gate, const void* up) {
        int r = ARIA_ERR_UNSUPPORTED;
        if (T * k > aria_rows_experts_most(E, I, D, ARIA_ROWS_PAIR)) r = aria_expert_pair_tiles(z.h, z.rows, T, gate, up, z.act, z.offsets, E, T * k, I, D, D, stream);
        return r != ARIA_ERR_UNSUPPORTED ? r : aria_rows_experts(z.h, z.rows, z.offsets, gate, up, z.act, E, T * k, I, D, D, I, stream);
    };
#define ARIA_TRY(call) \
    if (rc == ARIA_OK) rc = (call)
    for (int64_t li = 0; li < L; ++li) {
        const void* const* p = ptrs + ARIA_DECODE_STEP_PTRS + ARIA_DECODE_LAYER_PTRS * li;
        void *kc = const_cast<void*>(p[11]), *vc = const_cast<void*>(p[12]);
        if (delta) {
            ARIA_TRY(aria_rmsnorm_fwd(delta, x, p[0], y, z.h, nullptr, T, D, eps, stream));
            summed();
        } else {
            ARIA_TRY(aria_rmsnorm_fwd(x, nullptr, p[0], nullptr, z.h, nullptr, T, D, eps, stream));
        }
        ARIA_TRY(product(z.h, p[1], z.qkv, 3 * D, D));
        ARIA_TRY(aria_rope_cache_rows(z.qkv, ptrs[0], slot, pos, kc, vc, T, H, hd, Smax, stream));
        ARIA_TRY(aria_attn_varlen_sized_fwd(z.qkv, z.qkv + D, z.qkv + 2 * D, z.ao, cu, nullptr, n_seq, longest, H, H, hd, hd, 3 * D, 3 * D, 3 * D, D, 0,
                                            1.0f / sqrtf(float(hd)), T, stream));
        ARIA_TRY(product(z.ao, p[2], z.d, D, D));
        ARIA_TRY(aria_rmsnorm_fwd(z.d, x, p[3], y, z.h, nullptr, T, D, eps, stream));
        summed();
        ARIA_TRY(aria_rows_gemm(z.h, p[4], z.logits, 0, T, E, D, D, E, stream));
        ARIA_TRY(aria_route_and_sort(z.logits, z.scores, z.idx, z.counts + li * E, z.offsets, z.src, z.inv, z.rows, int(T), int(E), int(k), stream));
        ARIA_TRY(expert_pairs(p[5], p[6]));
        if (T * k <= aria_rows_experts_most(E, D, I, ARIA_ROWS_DOWN)) {
            ARIA_TRY(aria_rows_experts(z.act, nullptr, z.offsets, p[7], nullptr, z.eo, E, T * k, D, I, I, D, stream));
        } else {
            ARIA_TRY(aria_grouped_gemm_bf16(z.act, p[7], z.eo, z.offsets, E, T * k, D, I, 0, I, I, D * I, D, stream));
        }
        ARIA_TRY(aria_rows_swiglu(z.h, p[8], p[9], z.sact, T, Is, D, D, Is, stream));
        ARIA_TRY(product(z.sact, p[10], z.sh, D, Is));
        ARIA_TRY(aria_moe_unpermute(z.eo, z.inv, z.scores, z.sh, z.d, T, D, k, stream));
        delta = z.d;
    }
    if (n_wanted == 0) return rc;
    ARIA_TRY(aria_rmsnorm_fwd(delta, x, ptrs[1], y, z.h, nullptr, T, D, eps, stream));
    ARIA_TRY(aria_moe_permute(z.h, wanted, z.ao, n_wanted, D, 1, D, stream));
    if (rows_ahead(n_wanted, V, D) || (V & 1)) {   // (the tiles store pairs of columns)
        ARIA_TRY(aria_rows_gemm(z.ao, ptrs[2], logits, 1, n_wanted, V, D, D, V, stream));
    } else {
        ARIA_TRY(aria_gemm_bf16(z.ao, ptrs[2], logits, nullptr, n_wanted, V, D, 0, 0, D, D, V, 1, 0, stream));
    }
#undef ARIA_TRY
    return rc;
}

}  // extern "C"
