// Masked mean cross-entropy over the vocabulary (aria/model/modeling_aria.py:301-323), fused forward + backward:
// one workgroup per token row, online logsumexp in fp32 over bf16 logits, then dlogits = (softmax - onehot) * scale
// written in place of the logits if the caller aliases them.  HBM-bound: 2 reads + 1 write of the row.
// Four waves a row, whose order of sums the gradients of a model hold to (sixteen waves: those of a sample of 777 tokens 0.4 % away, at equal errors against 64 bits), eight chunks of a thread in
// flight, and three rows a CU, so that many rows' second reads find them nearer.  Rows of 100352, us by one chunk in flight and eight rows a CU / here: 16 53 / 36, 195 53 / 35, 656 69 / 66, 1024
// 108 / 92, 4096 450 / 345; 300 of 32000 34 / 30.  Two rows a CU: 656 73, 4096 336; four: 66, 364; four chunks ahead: 16 37.5, 4096 374; sixteen waves a row: 16 34, 195 31, 656 69, 4096 331.
#include "aria_device.h"
#include "aria_hip.h"

namespace {
using namespace ad;

constexpr int NW = 4, NT = NW * 64, AHEAD = 8;
constexpr int ROWS_A_CU = 41 << 10;   // bytes of LDS that nobody uses: room for three workgroups in 160 KB

// use(chunk, its place) over a thread's chunks of a row, every NT-th, in order, AHEAD of them in flight
template <class Use>
__device__ __forceinline__ void each_chunk(const bf16_t* row, int nch, int tid, const Use& use) {
    const int full = nch / NT;   // chunks that every thread has
    u32x4 v[AHEAD];
    auto load = [&](int i) __attribute__((always_inline)) { return ld16(row + (long long)(tid + i * NT) * 8); };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
        if (u < full) v[u] = load(u);
    int i = 0;
    for (; i + 2 * AHEAD <= full; i += AHEAD)
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            use(v[u], tid + (i + u) * NT);
            v[u] = load(i + u + AHEAD);
        }
    for (; i < full; i += AHEAD)
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (i + u >= full) break;
            use(v[u], tid + (i + u) * NT);
            if (i + u + AHEAD < full) v[u] = load(i + u + AHEAD);
        }
    if (tid < nch - full * NT) use(load(full), tid + full * NT);
}

__global__ __launch_bounds__(NT) void ce_kernel(const bf16_t* logits, const int32_t* labels, float* loss_sum, int32_t* count,
                                                bf16_t* dlogits, float grad_scale, const int32_t* count_in, int V, long long ld) {
    ARIA_SMEM_STATIC float red_m[NW];
    ARIA_SMEM_STATIC float red_s[NW];
    const int t = blockIdx.x, tid = threadIdx.x, l = tid & 63, w = tid >> 6;
    const int label = labels[t];
    const bf16_t* row = logits + (long long)t * ld;
    const int nch = V >> 3;
    if (label < 0) {  // ignored position (block-uniform)
        if (dlogits) {
            bf16_t* drow = dlogits + (long long)t * ld;
            for (int c = tid; c < nch; c += NT) st16(drow + c * 8, zero16());
        }
        return;
    }
    const float at_label = tid == 0 ? bf2f(row[label]) : 0.f;   // (before the barrier: the gradient may take the logits' place)
    float m = -INFINITY, s = 0.f;
    each_chunk(row, nch, tid, [&](const u32x4& v, int) __attribute__((always_inline)) {
        float x[8];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            x[2 * q] = bflo(v[q]);
            x[2 * q + 1] = bfhi(v[q]);
        }
        float cm = x[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) cm = fmaxf(cm, x[i]);
        const float nm = fmaxf(m, cm);
        float cs = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) cs += __expf(x[i] - nm);
        s = s * __expf(m - nm) + cs;
        m = nm;
    });
    const float wm = wave_max(m);
    s = wave_sum(m == -INFINITY ? 0.f : s * __expf(m - wm));  // lanes (or whole waves) without data carry m = -inf
    if (l == 0) {
        red_m[w] = wm;
        red_s[w] = s;
    }
    sync();
    const float M = fmaxf(fmaxf(red_m[0], red_m[1]), fmaxf(red_m[2], red_m[3]));
    const float S = red_s[0] * __expf(red_m[0] - M) + red_s[1] * __expf(red_m[1] - M) + red_s[2] * __expf(red_m[2] - M) +
                    red_s[3] * __expf(red_m[3] - M);
    const float lse = M + logf(S);
    if (tid == 0) {
        atomic_add(loss_sum, lse - at_label);
        atomic_add(count, 1);
    }
    if (dlogits) {
        float scale = grad_scale;
        if (count_in) scale /= float(max(1, *count_in));
        bf16_t* drow = dlogits + (long long)t * ld;
        each_chunk(row, nch, tid, [&](const u32x4& v, int c) __attribute__((always_inline)) {
            u32x4 o;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float p0 = __expf(bflo(v[q]) - lse), p1 = __expf(bfhi(v[q]) - lse);
                if (c * 8 + 2 * q == label) p0 -= 1.f;
                if (c * 8 + 2 * q + 1 == label) p1 -= 1.f;
                o[q] = pack2bf(p0 * scale, p1 * scale);
            }
            st16(drow + (long long)c * 8, o);
        });
    }
}

}  // namespace

extern "C" int aria_cross_entropy(const void* logits, const int32_t* labels, float* loss_sum, int32_t* count, void* dlogits,
                                  float grad_scale, const int32_t* count_in, int64_t T, int64_t V, int64_t ld, void* stream) {
    if (!logits || !labels || !loss_sum || !count || T < 0 || V <= 0) return ARIA_ERR_INVALID;
    if ((V & 7) || (ld & 7)) return ARIA_ERR_ALIGN;
    if (T == 0) return ARIA_OK;
    ARIA_LAUNCH(ce_kernel, dim3(int(T)), dim3(NT), ROWS_A_CU, stream, static_cast<const bf16_t*>(logits), labels, loss_sum, count,
                static_cast<bf16_t*>(dlogits), grad_scale, count_in, int(V), (long long)ld);
    return aria_check_launch();
}
