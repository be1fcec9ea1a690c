// Routed experts of a few tokens (bf16): every expert that somebody chose has its weight rows read ONCE, for all the tokens that chose it.  A launch per
// (token, slot) reads an expert again for each of its tokens: 16 tokens with 6 of 64 experts each are 96 reads of about 51 different experts.
//
// A list kernel turns the choices into: which experts are in use, and which (token, slot) pairs each of them serves.  The projections then run
// stream_rows (rows.h) on the gathered token rows of one expert after the other.
#pragma once
#include "rows.h"

namespace ad {

// table: [0] experts in use, [1 + a] their ids in rising order, [1 + E + a] the place in `list` where the a-th one's entries begin (and their end);
// list: entries token * k + slot
struct ExpertLists {
    int32_t *table, *list;
    int E;
    static int64_t table_ints(int64_t E) { return 2 * E + 2; }
};
constexpr int LISTS_MAX = 1024;   // entries, i.e. tokens x slots

// Run by one workgroup of 16 waves whose threads have left the choices in sidx[n] (entries in order): the table and the list (E <= 256).  A wave looks for
// one expert in 64 entries at a time; places come from a scan with a thread per expert.
struct ListsLds {
    int idx[LISTS_MAX], count[256], place[256], scan[4][2];
};
__device__ __forceinline__ void write_lists(const ExpertLists& x, ListsLds& s, int n) {
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    sync();
    for (int e = w; e < x.E; e += 16) {
        int c = 0;
        for (int i = l; i - l < n; i += 64) c += __builtin_popcountll(ballot(i < n && s.idx[i] == e));
        if (l == 0) s.count[e] = c;
    }
    sync();
    const int count = t < x.E ? s.count[t] : 0;
    const unsigned long long used = ballot(count > 0);
    const int upto = wave_incl_scan(count);
    if (t < 256 && l == 63) {
        s.scan[w][0] = __builtin_popcountll(used);
        s.scan[w][1] = upto;
    }
    sync();
    if (t < x.E) {
        int a = __builtin_popcountll(used & ((1ull << l) - 1)), first = upto - count;
        for (int i = 0; i < w; ++i) {
            a += s.scan[i][0];
            first += s.scan[i][1];
        }
        if (count) {
            x.table[1 + a] = t;
            x.table[1 + x.E + a] = first;
            x.table[2 + x.E + a] = first + count;   // (the next one in use writes the same number there)
        }
        s.place[t] = first;
    }
    if (t == 0) x.table[0] = s.scan[0][0] + s.scan[1][0] + s.scan[2][0] + s.scan[3][0];
    sync();
    for (int e = w; e < x.E; e += 16) {
        if (s.count[e] == 0) continue;
        int at = s.place[e];
        for (int i = l; i - l < n; i += 64) {
            const bool mine = i < n && s.idx[i] == e;
            const unsigned long long who = ballot(mine);
            if (mine) x.list[at + __builtin_popcountll(who & ((1ull << l) - 1))] = i;
            at += __builtin_popcountll(who);
        }
    }
}

struct ExpertIn {
    const bf16_t *W, *W2;   // [E, N, K]; W2: the up matrices of a gated pair
    const bf16_t* X;        // row of an entry: X + (entry / div) ldx
    long long ldx;
    int div, K, N;
    // experts that every token uses, E, E + 1, ... in the lists: their rows have the stride s_ld, the next one begins s_step further on
    const bf16_t *S = nullptr, *S2 = nullptr;
    long long s_step = 0, s_ld = 0;
    int E = 1 << 30;
};

namespace {
// e(value, up value, entry, row).  The row groups of all experts in use are one sequence, cut into equal pieces for the workgroups: how many experts are in
// use is known on the device only, and a grid over (expert, rows) left the last round of workgroups nearly empty (29 experts x 18 pieces = 522 on
// 512 places: 110 us; as one sequence 93).
template <int NW, int KS, class Ep, bool PAIR, bool ONCE>
__global__ __launch_bounds__(NW * 64) void expert_rows_kernel(ExpertIn in, ExpertLists lists, Ep e) {
    ARIA_SMEM_STATIC RowsRed<NW, 1> red;
    ARIA_SMEM_STATIC int entries[16];
    constexpr int OUT = PAIR ? 8 : 16;
    const int groups = (in.N + OUT - 1) / OUT, total = lists.table[0] * groups, per = (total + int(gridDim.x) - 1) / int(gridDim.x), t = threadIdx.x;
    const int end = min(total, (int(blockIdx.x) + 1) * per), c16 = t & 15;
    int g = int(blockIdx.x) * per;
    while (g < end) {
        const int a = g / groups, g0 = g - a * groups, g1 = min(groups, g0 + end - g);
        const int first = lists.table[1 + lists.E + a], m = lists.table[2 + lists.E + a] - first;
        const int id = lists.table[1 + a];
        const bool all = id >= in.E;
        const long long at = all ? (id - in.E) * in.s_step : (long long)id * in.N * in.K, ldw = all ? in.s_ld : (long long)in.K;
        const bf16_t *W = (all ? in.S : in.W) + at, *W2 = PAIR ? (all ? in.S2 : in.W2) + at : W;
        for (int t0 = 0; t0 < m; t0 += 16) {   // (more than 16 only where tokens chose an expert several times: NaN logits)
            sync();                            // (red and entries of the piece before are read)
            const int mine = lists.list[first + min(t0 + c16, m - 1)];
            if (t < 16) entries[t] = mine;     // (published by the first group's barrier)
            stream_rows<NW, KS, 1, ONCE>(
                in.K, [&](int gg, int r) { return (PAIR && r >= 8 ? W2 : W) + (long long)min(gg * OUT + (PAIR ? r & 7 : r), in.N - 1) * ldw; },
                [&](int) { return in.X + (long long)(mine / in.div) * in.ldx; }, g0, g1, red, [&](float v, int tok, int n, int gg) {
                    const float u = PAIR ? shfl_xor(v, 8) : 0.f;
                    if (t0 + tok < m && gg * OUT + n < in.N && n < OUT) e(v, u, entries[tok], gg * OUT + n);
                });
        }
        g += g1 - g0;
    }
}

// Whether T tokens' choices go through lists (K0, K1: the reductions of the two projections).  A list and the weighted sum as launches of their own cost
// about 11 us, a projection per (token, slot) reads every expert once more for each further token: worth it when on average a sixth of the T k
// choices fall on an expert that another token has chosen already.  Up + down + the extra launches against a projection per choice, us: 64 experts of
// 2560 x 1664, 6 a token: 4 tokens (13 % fall together) 114 / 107, 6 (20 %) 149 / 157, 16 (50 %) 220 / 394; 32 of 1536 x 1024, 4 a token: 8 tokens
// 54 / 60, 16 67 / 103; 16 of 1024 x 768, 2 a token: 12 tokens 29 / 31, 16 30 / 36.  At 16 tokens the weights of the experts in use arrive at 5.9 TB/s.
inline bool expert_rows_can(int64_t K0, int64_t K1, int64_t E, int64_t k, int64_t T) {
    return T * k <= LISTS_MAX && E <= 256 && k <= E && std::min(K0, K1) >= 128 && std::max(K0, K1) <= 6656;
}
inline bool expert_rows_take(int64_t K0, int64_t K1, int64_t E, int64_t k, int64_t T) {
    if (T < 2 || !expert_rows_can(K0, K1, E, k, T)) return false;
    const double reached = double(E) * (1.0 - std::pow(1.0 - double(k) / double(E), double(T)));
    return reached * 6.0 <= 5.0 * double(T * k);
}

template <bool PAIR, class Ep>
int launch_expert_rows(const ExpertIn& in, const ExpertLists& lists, int64_t k, int64_t T, const Ep& e, void* stream) {
    const int64_t most = (in.N + (PAIR ? 7 : 15)) / (PAIR ? 8 : 16) * std::min<int64_t>(lists.E, T * k);
    const dim3 grid(unsigned(std::min<int64_t>(512, most)));   // two workgroups a CU are resident
    const bool once = in.s_ld % 64 == 0 && experts_once(lists.E, in.N * (PAIR ? 2 : 1), in.K, 32);
#define ARIA_ROWS(NW, KS)                                                                                                 \
    {                                                                                                                     \
        if (once)                                                                                                         \
            ARIA_LAUNCH((expert_rows_kernel<NW, KS, Ep, PAIR, true>), grid, dim3(NW * 64), 0, stream, in, lists, e);      \
        else                                                                                                              \
            ARIA_LAUNCH((expert_rows_kernel<NW, KS, Ep, PAIR, false>), grid, dim3(NW * 64), 0, stream, in, lists, e);     \
    }
    ARIA_ROWS_SHAPE(in.K, ARIA_ROWS, return ARIA_ERR_UNSUPPORTED;)
#undef ARIA_ROWS
    return aria_check_launch();
}
}  // namespace
}  // namespace ad
