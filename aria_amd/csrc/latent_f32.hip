// Latent attention in 32-bit on v_mfma_f32_16x16x4_f32: softmax(q . cache row) over a sequence's cached latents, whose first R columns are the values too.
//
// The heads of a token share its sequence's latents, so one workgroup takes 16 (token, head) columns -- the heads of 16 / H neighbouring tokens, or 16 heads of one
// -- and reads each latent row once for all of them.  Its waves take tiles of 16 keys in turn: a wave stages its tile in the LDS (the next tile's rows are in flight
// in registers meanwhile), computes S^T = K Q^T, whose accumulators are the probabilities' operand of O^T += V^T P^T as they lie (key 4 (lane / 16) + r in register r),
// and keeps its own running maximum and sums; the waves' states meet once at the end.
//
// Bound by the matrix pipe's 32-bit rate at (cw + R) / 4 multiply steps a tile, and by the tiles a wave walks.  As one (token, head) a workgroup on the vector
// pipe the latents were read once for every head: 883 tokens of four prompts, 8 heads, 320-column rows 185 us, now 55; 4 single tokens of 250 keys 22 us, now 15 (four splits).
// The first keys requested before the queries are staged, and columns dealt to threads without divisions: those 4 tokens 15.3 -> 12.6, 614 tokens of four prompts 40 -> 32.
#include "aria_device.h"
#include "aria_hip.h"
#include <algorithm>

namespace {
using namespace ad;
typedef AriaLatentShape Shape;

template <int NW>
constexpr size_t lds_bytes(int64_t cw) { return size_t(16 + 16 * NW) * size_t(cw + 4) * 4 + size_t(NW) * 32 * 4; }

// NB: blocks of 16 value columns held; PF: 16-byte pieces of a key tile a lane holds in flight (cw <= 16 PF); tpb: tokens of a workgroup, hp: columns each
template <int NB, int PF, int NW>
__global__ __launch_bounds__(NW * 64) void latent_attn_f32_kernel(const float* qa, const float* cache, Shape s, const int32_t* slot, const int32_t* pos, float* part_o,
                                                                  float* part_ml, int T, int tpb, int hs, int splits) {
    ARIA_DYN_SMEM(smem);
    const int cw = int(s.cw), P = cw + 4, R = int(s.R), H = int(s.H);
    const int t = threadIdx.x, l = t & 63, w = first_lane(t >> 6), q4 = l >> 4, c = l & 15;
    float* sQ = reinterpret_cast<float*>(smem);            // [16 columns][P]
    float* sK = sQ + 16 * P + w * 16 * P;                  // this wave's keys [16][P]
    float* state = sQ + (16 + 16 * NW) * P;                // [NW][16] maxima, [NW][16] sums
    const int t0 = blockIdx.y * tpb, h0 = blockIdx.x << hs, hp = 1 << hs, z = blockIdx.z;
    const int tok = t0 + (c >> hs), head = h0 + (c & (hp - 1));
    const bool real = tok < T && head < H && c < tpb * hp;
    // a column of 16 to a thread where the columns are gone through one by one, LANES threads each
    constexpr int LANES = NW * 4;
    const int col = t / LANES, lane = t % LANES, col_tok = t0 + (col >> hs), col_head = h0 + (col & (hp - 1));
    const bool col_real = col_tok < T && col_head < H && col < tpb * hp;
    const float scale2 = s.scale * 1.4426950408889634f;
    float m = -INFINITY, lsum = 0.f;
    f32x4 o[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};

    f32x4 next[PF];
    const int row0 = l >> 3, col0 = (l & 7) * 4, pieces = cw / 16;   // piece i: rows row0 + 8 (i & 1), columns col0 + 32 (i >> 1)
    auto request = [&](const float* base, int k0, int k_end) __attribute__((always_inline)) {   // (rows behind the end: the last one again)
#pragma unroll
        for (int i = 0; i < PF; ++i) {
            if (i < pieces) next[i] = *reinterpret_cast<const f32x4*>(base + (long long)min(k0 + row0 + 8 * (i & 1), k_end - 1) * cw + col0 + 32 * (i >> 1));
        }
    };
    // keys [first, end) of the rows at `base`, all of them seen by the columns with `mine` and by no other; tiles counted on from `tiles`
    int tiles = 0;
    auto walk = [&](const float* base, int first, int end, bool mine, bool everyone, bool requested) __attribute__((always_inline)) {
        const int n = (end - first + 15) / 16, turns = NW * splits, me = z * NW + w;
        int u = (me - tiles % turns + turns) % turns;
        tiles += n;
        if (u < n && !requested) request(base, first + 16 * u, end);
        for (; u < n; u += turns) {
            const int k0 = first + 16 * u;
            wave_barrier();
#pragma unroll
            for (int i = 0; i < PF; ++i) {
                if (i < pieces) *reinterpret_cast<f32x4*>(sK + (row0 + 8 * (i & 1)) * P + col0 + 32 * (i >> 1)) = next[i];
            }
            wave_barrier();
            if (u + turns < n) request(base, k0 + 16 * turns, end);
            f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
            for (int j = 0; j < cw; j += 32) {   // (cw is a multiple of 64)
                const f32x4 ka = *reinterpret_cast<const f32x4*>(sK + c * P + j + 4 * q4), qa0 = *reinterpret_cast<const f32x4*>(sQ + c * P + j + 4 * q4);
                const f32x4 kb = *reinterpret_cast<const f32x4*>(sK + c * P + j + 16 + 4 * q4), qb = *reinterpret_cast<const f32x4*>(sQ + c * P + j + 16 + 4 * q4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s0 = mfma16_f32(ka[e], qa0[e], s0);
                    s1 = mfma16_f32(kb[e], qb[e], s1);
                }
            }
            float x[4], mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                x[r] = mine && k0 + 4 * q4 + r < end ? (s0[r] + s1[r]) * scale2 : -INFINITY;
                mx = fmaxf(mx, x[r]);
            }
            mx = fmaxf(mx, shfl_xor(mx, 16));
            mx = max_halves(mx);
            const float mn = fmaxf(m, mx), safe = mn == -INFINITY ? 0.f : mn, alpha = exp2f(m - safe);
            float sum = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                x[r] = exp2f(x[r] - safe);
                sum += x[r];
            }
            if (mine) {
                m = mn;
                lsum = lsum * alpha + sum;
            }
#pragma unroll
            for (int n16 = 0; n16 < NB; ++n16) {
                if (16 * n16 < R) {
                    f32x4 a = o[n16];
#pragma unroll
                    for (int r = 0; r < 4; ++r) a[r] *= alpha;
#pragma unroll
                    for (int e = 0; e < 4; ++e) a = mfma16_f32(sK[(4 * q4 + e) * P + 16 * n16 + c], x[e], a);
                    // (a column that does not see the tile keeps its sums: zero times a value that is no number is none)
                    if (everyone || mine) o[n16] = a;
                }
            }
        }
    };
    // neighbouring tokens of one sequence together: what all of them see, then what is one's alone
    int j = 0, common = 0;
    auto group_from = [&](int i) __attribute__((always_inline)) {
        const int sl = slot[t0 + i];
        j = i + 1, common = pos[t0 + i] + 1;
        for (; j < tpb && t0 + j < T && slot[t0 + j] == sl; ++j) common = min(common, pos[t0 + j] + 1);
        return cache + (long long)sl * s.S_cap * cw;
    };
    const float* base = group_from(0);
    if (16 * (z * NW + w) < common) request(base, 16 * (z * NW + w), common);   // (the first keys come while the queries are staged)
    for (int at = 4 * lane; at < cw; at += 4 * LANES)
        *reinterpret_cast<f32x4*>(sQ + col * P + at) =
            col_real ? *reinterpret_cast<const f32x4*>(qa + ((long long)col_tok * H + col_head) * cw + at) : f32x4{0.f, 0.f, 0.f, 0.f};
    sync();
    for (int i = 0; i < tpb && t0 + i < T;) {
        if (i) base = group_from(i);
        const bool group = real && tok >= t0 + i && tok < t0 + j;
        walk(base, 0, common, group, i == 0 && j == min(tpb, T - t0), i == 0);
        for (int b = i; b < j; ++b)
            if (pos[t0 + b] + 1 > common) walk(base, common, pos[t0 + b] + 1, real && tok == t0 + b, false, false);
        i = j;
    }
    // ---- the waves' states meet
    lsum += shfl_xor(lsum, 16);
    lsum += shfl_xor(lsum, 32);
    if (q4 == 0) state[w * 16 + c] = m, state[NW * 16 + w * 16 + c] = lsum;
    sync();
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < NW; ++i) top = fmaxf(top, state[i * 16 + c]);
    const float f = m == -INFINITY ? 0.f : exp2f(m - top);
#pragma unroll
    for (int n16 = 0; n16 < NB; ++n16)
        if (16 * n16 < R) *reinterpret_cast<f32x4*>(sK + c * P + 16 * n16 + 4 * q4) = m == -INFINITY ? f32x4{0.f, 0.f, 0.f, 0.f}
                                                                                                     : f32x4{o[n16][0] * f, o[n16][1] * f, o[n16][2] * f, o[n16][3] * f};
    sync();
    const float* all = sQ + 16 * P;
    if (col_real) {
        float* out = part_o + (((long long)col_tok * splits + z) * H + col_head) * R;
        auto sums = [&](auto v, int d) __attribute__((always_inline)) {
            using V = decltype(v);
            v = *reinterpret_cast<const V*>(all + col * P + d);
#pragma unroll
            for (int k = 1; k < NW; ++k) v += *reinterpret_cast<const V*>(all + k * 16 * P + col * P + d);
            *reinterpret_cast<V*>(out + d) = v;
        };
        if ((R & 3) || (reinterpret_cast<uintptr_t>(part_o) & 15))   // (a caller's buffer may start at any float)
            for (int d = lane; d < R; d += LANES) sums(0.f, d);
        else
            for (int d = 4 * lane; d < R; d += 4 * LANES) sums(f32x4{}, d);
    }
    if (w == 0 && q4 == 0 && real) {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < NW; ++i) sum += state[i * 16 + c] == -INFINITY ? 0.f : state[NW * 16 + i * 16 + c] * exp2f(state[i * 16 + c] - top);
        float* ml = part_ml + (((long long)tok * splits + z) * H + head) * 2;
        ml[0] = top;
        ml[1] = sum;
    }
}

}  // namespace

// whether the rows fit the kernel's registers and LDS
__attribute__((visibility("hidden"))) bool aria_latent_f32_takes(const AriaLatentShape& s) { return (s.cw & 63) == 0 && ((s.R <= 256 && s.cw <= 384) || (s.R <= 512 && s.cw <= 640)); }

// Tokens a workgroup shares latents between only where many follow one another (prompts): single tokens belong to different sequences.
__attribute__((visibility("hidden"))) int aria_latent_f32_attn(const float* qa, const float* cache, const AriaLatentShape& s, const int32_t* slot, const int32_t* pos, float* part_o, float* part_ml, int64_t T,
                         int64_t splits, void* stream) {
    int hs = 4;   // 2^hs columns a token
    while (hs > 0 && (1 << hs >> 1) >= s.H) --hs;
    const int hp = 1 << hs, tpb = T > 64 ? 16 / hp : 1;
    const dim3 grid(unsigned((s.H + hp - 1) / hp), unsigned((T + tpb - 1) / tpb), unsigned(splits));
#define ARIA_LATENT32(NB, PF, NW)                                                                                                                                   \
    ARIA_LAUNCH((latent_attn_f32_kernel<NB, PF, NW>), grid, dim3(NW * 64), lds_bytes<NW>(s.cw), stream, qa, cache, s, slot, pos, part_o, part_ml, int(T), tpb, hs, \
                int(splits))
    if (s.R <= 256 && s.cw <= 384)
        ARIA_LATENT32(16, 24, 4);
    else
        ARIA_LATENT32(32, 40, 2);
#undef ARIA_LATENT32
    return aria_check_launch();
}

extern "C" int64_t aria_latent_splits_f32(const AriaLatentShape* s, int64_t T, int64_t max_len) {
    // a tile of 16 keys a wave, for the few single tokens that leave the chip empty; every split is a slab of sums for the expansion to add up
    if (!s || T <= 0 || T > 16 || !aria_latent_f32_takes(*s)) return 1;
    return std::min<int64_t>(8, std::max<int64_t>(1, (max_len + 63) / 64));
}
