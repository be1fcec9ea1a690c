// One float32 step of a Duguzen or Kozipel stack as one call: the launches of the step's sublayers (latent.hip, chunk.hip, linear.hip, mix.hip, norm.hip, moe.hip,
// gemm_f32.hip), enqueued in order from here.  The results are those of the step run sublayer by sublayer, bit for bit.
//
// What follows a product element by element is its epilogue (gemm_f32.h): the dynamic-tanh steps of the stream, squared relu, gate times up of a pair of weights;
// rows by expert and the rows that logits are asked for are read where they lie.  A decoded token's step of three Duguzen layers 1024 wide is 46 launches
// one by one and 30 so, of about 4.5 us each whatever they do.
//
// Why: the host bounded these steps.  Three layers 1024 wide: 46 launches that keep the device busy for 0.32 ms took 1.2 ms, most of it the operations' own checks
// and allocations around each launch.  A session of four prompts of up to 250 tokens and four decoded tokens took the host 3.1 ms (6 on a slower one), now 1.2.
#include "aria_device.h"
#include "aria_hip.h"
#include "gemm_f32.h"
#include <algorithm>

__attribute__((visibility("hidden"))) int aria_route_groups_sorted(const float* logits, const float* correction, float* weights, int32_t* indices, int32_t* offsets, int32_t* src,
                                                                   int32_t* inv, int64_t T, int64_t E, int64_t ldl, int64_t groups, int64_t keep, int64_t k, void* stream);

namespace {

// a walk over the scratch: offsets only where base is null
struct Walk {
    char* base;
    int64_t at = 0, most = 0;
    template <class T = float>
    T* take(int64_t n) {
        T* p = base ? reinterpret_cast<T*>(base + at) : nullptr;
        at += (n * int64_t(sizeof(T)) + 255) & ~int64_t(255);
        most = std::max(most, at);
        return p;
    }
};

AriaGemmF32 dense(const float* a, const void* w, float* c, int64_t M, int64_t N, int64_t K) {
    AriaGemmF32 p{};
    p.A = a, p.W = static_cast<const float*>(w), p.C = c, p.M = int(M), p.N = int(N), p.K = int(K), p.lda = K, p.ldw = K, p.ldc = N, p.E = 1;
    return p;
}
int product(const float* a, const void* w, float* c, int64_t M, int64_t N, int64_t K, void* stream) {
    return aria_gemm_f32_finished(dense(a, w, c, M, N, K), ARIA_F32_PLAIN, stream);
}
// x += post(a w^T), h = next(x)
int product_into_stream(const float* a, const void* w, float* x, float* h, const AriaDyT& post, const AriaDyT& next, int64_t M, int64_t D, int64_t K, void* stream) {
    AriaGemmF32 p = dense(a, w, h, M, D, K);
    p.x = x, p.post = post, p.next = next;
    return aria_gemm_f32_finished(p, ARIA_F32_STREAM, stream);
}

// what lives through the whole step; the sublayers' own buffers follow, one sublayer's over the other's
struct Common {
    float *x, *h;
};
Common common(Walk& z, int64_t T, int64_t D) { return {z.take(T * D), z.take(T * D)}; }

struct Latent {
    float *proj, *qa, *part_o, *part_ml, *ao;
};
Latent latent(Walk& z, const AriaLatentShape& s, int64_t T, int64_t splits) {
    return {z.take(T * s.ldp), z.take(T * s.H * s.cw), z.take(T * splits * s.H * s.R), z.take(T * splits * s.H * 2), z.take(T * s.H * s.dvp)};
}
struct Mixture {
    float *logits, *weights, *act, *eo;
    int32_t *idx, *counts, *offsets, *src, *inv, *ws;
};
Mixture mixture(Walk& z, const AriaLatentLayer& y, int64_t T, int64_t D) {
    const int64_t M = T * y.k;
    return {z.take(T * ((y.E + 7) & ~int64_t(7))), z.take(M), z.take(M * y.ff), z.take(M * D), z.take<int32_t>(M),
            z.take<int32_t>(y.E), z.take<int32_t>(y.E + 1), z.take<int32_t>(M), z.take<int32_t>(M), z.take<int32_t>(std::max<int64_t>(1, (M + 2047) / 2048) * 128 + 64)};
}

struct Chunk {
    float* out;
};
struct Linear {
    float *out, *gated;
};

// the rows whose logits are asked for (W < 0: every row), times the head
int head(const float* h, const int32_t* wanted, int64_t W, int64_t T, int64_t D, int64_t V, const void* w, float* logits, void* stream) {
    if (W == 0) return ARIA_OK;
    AriaGemmF32 p = dense(h, w, logits, W < 0 ? T : W, V, D);
    if (W > 0) p.rows = wanted, p.per = 1;
    return aria_gemm_f32_finished(p, ARIA_F32_PLAIN, stream);
}

}  // namespace

extern "C" {

int64_t aria_latent_step_f32_scratch(const AriaLatentStack* st, const AriaLatentLayer* L, int64_t T, int64_t max_len, int64_t W) {
    if (!st || !L || T <= 0) return 0;
    Walk z{nullptr};
    common(z, T, st->D);
    const int64_t own = z.at;
    for (int64_t i = 0; i < st->n_layers; ++i) {
        z.at = own, latent(z, L[i].mix, T, aria_latent_splits_f32(&L[i].mix, T, max_len));
        z.at = own;
        if (L[i].mlp == 1) z.take(T * L[i].ff);
        if (L[i].mlp == 2) mixture(z, L[i], T, st->D);
    }
    return z.most;
}

int aria_latent_step_f32(const AriaLatentStack* st, const AriaLatentLayer* L, int64_t T, const int32_t* ids, const int32_t* slot, const int32_t* pos, int64_t max_len,
                         const int32_t* wanted, int64_t W, float* logits, void* scratch, int64_t scratch_bytes, void* stream) {
    if (!st || !L || !ids || !slot || !pos || (!logits && W != 0) || (!wanted && W > 0) || !scratch || T < 0 || max_len <= 0 || st->n_layers <= 0) return ARIA_ERR_INVALID;
    if (T == 0) return ARIA_OK;
    if ((reinterpret_cast<uintptr_t>(scratch) & 15) || (st->D & 7)) return ARIA_ERR_ALIGN;
    if (scratch_bytes < aria_latent_step_f32_scratch(st, L, T, max_len, W)) return ARIA_ERR_INVALID;
    for (int64_t i = 0; i < st->n_layers; ++i) {
        if (max_len > L[i].mix.S_cap) return ARIA_ERR_INVALID;
        if (L[i].mlp == 2 && (L[i].E <= 0 || L[i].k <= 0)) return ARIA_ERR_INVALID;
        if (L[i].mlp && (L[i].ff & 7)) return ARIA_ERR_ALIGN;
    }
    const int64_t D = st->D;
    Walk z{static_cast<char*>(scratch)};
    const Common c = common(z, T, D);
    const int64_t own = z.at;
    const AriaDyT none{0.f, nullptr, nullptr};
    int rc = aria_dyt_stream(ids, st->embed, nullptr, nullptr, nullptr, 0, &none, c.x, &st->first, c.h, T, D, 0, 1, stream);
    for (int64_t i = 0; i < st->n_layers && rc == ARIA_OK; ++i) {
        const AriaLatentLayer& y = L[i];
        const AriaLatentShape& s = y.mix;
        z.at = own;
        const int64_t ns = aria_latent_splits_f32(&s, T, max_len);
        const Latent a = latent(z, s, T, ns);
        rc = product(c.h, y.w_in, a.proj, T, s.ldp, D, stream);
        if (rc == ARIA_OK) rc = aria_latent_absorb(a.proj, &s, slot, pos, y.rope, y.kv_norm, y.w_uk, y.cache, a.qa, T, 1, stream);
        if (rc == ARIA_OK) rc = aria_latent_attn(a.qa, y.cache, &s, slot, pos, a.part_o, a.part_ml, T, ns, 1, stream);
        if (rc == ARIA_OK) rc = aria_latent_expand(a.part_o, a.part_ml, &s, a.proj, y.w_uv, a.ao, T, ns, 1, stream);
        if (rc == ARIA_OK) rc = product_into_stream(a.ao, y.w_o, c.x, c.h, y.norm1b, y.mlp ? y.norm2 : y.next, T, D, s.H * s.dvp, stream);
        if (rc != ARIA_OK || y.mlp == 0) continue;
        z.at = own;
        if (y.mlp == 1) {
            float* act = z.take(T * y.ff);
            rc = aria_gemm_f32_finished(dense(c.h, y.w_up, act, T, y.ff, D), ARIA_F32_RELU2, stream);
            if (rc == ARIA_OK) rc = product_into_stream(act, y.w_down, c.x, c.h, y.norm2b, y.next, T, D, y.ff, stream);
            continue;
        }
        const Mixture m = mixture(z, y, T, D);
        const int64_t ldl = (y.E + 7) & ~int64_t(7), M = T * y.k;
        rc = product(c.h, y.w_router, m.logits, T, ldl, D, stream);
        if (rc == ARIA_OK) {
            rc = aria_route_groups_sorted(m.logits, y.correction, m.weights, m.idx, m.offsets, m.src, m.inv, T, y.E, ldl, y.groups, y.keep, y.k, stream);
            if (rc == ARIA_ERR_UNSUPPORTED) {   // more tokens, more experts
                rc = aria_moe_route_groups(m.logits, y.correction, m.weights, m.idx, m.counts, T, y.E, ldl, y.groups, y.keep, y.k, stream);
                if (rc == ARIA_OK) rc = aria_moe_sort(m.idx, m.counts, m.offsets, m.src, m.inv, m.ws, T, y.E, y.k, stream);
            }
        }
        AriaGemmF32 up = dense(c.h, y.w_gate, m.act, M, y.ff, D), down = dense(m.act, y.w_down, m.eo, M, D, y.ff);
        up.W2 = static_cast<const float*>(y.w_up), up.rows = m.src, up.per = int(y.k), up.offsets = down.offsets = m.offsets, up.E = down.E = int(y.E);
        up.strideW = down.strideW = y.ff * D;
        if (rc == ARIA_OK) rc = aria_gemm_f32_finished(up, ARIA_F32_PAIR, stream);
        if (rc == ARIA_OK) rc = aria_gemm_f32_finished(down, ARIA_F32_PLAIN, stream);
        if (rc == ARIA_OK) rc = aria_dyt_stream(nullptr, nullptr, m.eo, m.inv, m.weights, y.k, &y.norm2b, c.x, &y.next, c.h, T, D, D, 1, stream);
    }
    if (rc != ARIA_OK) return rc;
    return head(c.h, wanted, W, T, D, st->V, st->head, logits, stream);
}

int64_t aria_mix_step_f32_scratch(const AriaMixStack* st, const AriaMixLayer* R, int64_t T, int64_t W) {
    if (!st || !R || T <= 0) return 0;
    Walk z{nullptr};
    common(z, T, st->D), z.take(T * st->D), z.take(T * st->D);
    const int64_t own = z.at;
    for (int64_t i = 0; i < st->n_runs; ++i) {
        const AriaLinearShape& s = R[i].right;
        z.at = own, z.take(T * s.ldp), z.take(T * s.H * s.dvp), z.take(T * s.H * s.dvp);
        if (R[i].kind) z.take(T * R[i].left.H * R[i].left.dvp);
        z.at = own, z.take(T * R[i].ff);
    }
    return z.most;
}

int aria_mix_step_f32(const AriaMixStack* st, const AriaMixLayer* R, int64_t T, const int32_t* ids, const int32_t* slot, const int32_t* pos, const int32_t* seq,
                      const int32_t* cu, int64_t n_seq, int64_t max_len, const int32_t* wanted, int64_t W, float* logits, void* scratch, int64_t scratch_bytes, void* stream) {
    if (!st || !R || !ids || !slot || !pos || !seq || !cu || (!logits && W != 0) || (!wanted && W > 0) || !scratch || T < 0 || n_seq <= 0 || max_len <= 0 || st->n_runs <= 0)
        return ARIA_ERR_INVALID;
    if (T == 0) return ARIA_OK;
    if ((reinterpret_cast<uintptr_t>(scratch) & 15) || (st->D & 7)) return ARIA_ERR_ALIGN;
    if (scratch_bytes < aria_mix_step_f32_scratch(st, R, T, W)) return ARIA_ERR_INVALID;
    for (int64_t i = 0; i < st->n_runs; ++i) {
        if (R[i].kind && std::min(R[i].left.size, max_len) > R[i].left.cap) return ARIA_ERR_INVALID;
        if (R[i].norm2 && (R[i].ff & 7)) return ARIA_ERR_ALIGN;
    }
    const int64_t D = st->D;
    Walk z{static_cast<char*>(scratch)};
    const Common c = common(z, T, D);
    float *const out = z.take(T * D), *const out2 = z.take(T * D);   // the sublayers' results
    const int64_t own = z.at;
    auto stream_pass = [&](const int32_t* i, const float* y, const float* y2, const float* w, const float* w2, const float* next) {
        const AriaRmsStream a{i, i ? st->embed : nullptr, i ? st->embedding_scale : 1.f, y ? st->mult : 1.f, st->eps, st->n, y ? D : 0, y, y2, w, w2, c.x, next, c.h};
        return aria_rms_stream(&a, T, D, 1, stream);
    };
    int rc = stream_pass(ids, nullptr, nullptr, nullptr, nullptr, st->first);
    for (int64_t i = 0; i < st->n_runs && rc == ARIA_OK; ++i) {
        const AriaMixLayer& y = R[i];
        const AriaLinearShape& s = y.right;
        const int64_t C = s.H * s.dvp, groups = y.kind ? s.H : 1;
        z.at = own;
        float* proj = z.take(T * s.ldp);
        const Linear b{z.take(T * C), z.take(T * C)};
        rc = product(c.h, y.w_in, proj, T, s.ldp, D, stream);
        if (rc == ARIA_OK && y.kind) {
            const Chunk a{z.take(T * y.left.H * y.left.dvp)};
            rc = aria_chunk_attn_any(proj, y.ring, &y.left, slot, pos, seq, cu, a.out, T, 1, stream);
            if (rc == ARIA_OK) rc = aria_chunk_rows(proj, y.ring, &y.left, slot, pos, seq, cu, T, 1, stream);
            if (rc == ARIA_OK) rc = product(a.out, y.w_o_left, out, T, D, y.left.H * y.left.dvp, stream);
        }
        if (rc == ARIA_OK) rc = aria_linear_step(proj, &s, y.state, slot, pos, cu, n_seq, b.out, 1, stream);
        // (kind 0: one norm over all heads, a sigmoid gate; kind 1: a norm per head with a shared weight, a silu gate)
        if (rc == ARIA_OK)
            rc = aria_norm_gate(b.out, proj + y.g_off, s.ldp, y.norm, y.kind ? 0 : C, b.gated, T, groups, C / groups, y.kind ? s.dv : s.H * s.dv, st->eps, y.kind ? 1 : 0, 1, stream);
        if (rc == ARIA_OK) rc = product(b.gated, y.w_o, y.kind ? out2 : out, T, D, C, stream);
        const float *y2 = y.kind ? out2 : nullptr, *w = y.kind ? y.out_left : nullptr, *w2 = y.kind ? y.out_right : nullptr;
        const int32_t* again = y.next_embedding ? ids : nullptr;
        if (rc == ARIA_OK && y.norm2) {
            rc = stream_pass(nullptr, out, y2, w, w2, y.norm2);
            z.at = own;
            float* act = z.take(T * y.ff);
            AriaGemmF32 up = dense(c.h, y.w_gate, act, T, y.ff, D);   // (gate rows, then up rows)
            up.W2 = up.W + y.ff * D, up.relu_gate = 1;
            if (rc == ARIA_OK) rc = aria_gemm_f32_finished(up, ARIA_F32_PAIR, stream);
            if (rc == ARIA_OK) rc = product(act, y.w_down, out, T, D, y.ff, stream);
            if (rc == ARIA_OK) rc = stream_pass(again, out, nullptr, nullptr, nullptr, y.next);
        } else if (rc == ARIA_OK) {
            rc = stream_pass(again, out, y2, w, w2, y.next);
        }
    }
    if (rc != ARIA_OK) return rc;
    rc = head(c.h, wanted, W, T, D, st->V, st->head, logits, stream);
    const int64_t rows = W < 0 ? T : W;
    return rc != ARIA_OK || rows == 0 ? rc : aria_softcap(logits, rows * st->V, st->cap, stream);
}

}  // extern "C"
