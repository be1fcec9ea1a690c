// What the one-token decode engine (decode.hip) and the routing share with the steps of several sequences (batch.hip, prompt.hip).  Hidden: not part of the C ABI.
#pragma once
#include "aria_device.h"
#include "aria_hip.h"
#include <algorithm>

#define ARIA_HIDDEN __attribute__((visibility("hidden")))

// Splits of the keys of one head: a round of eight workgroups a CU over all heads and tokens, one pass of 128 keys at least.  Up to 256 keys one workgroup
// of 16 waves per head is as fast and needs no merge.  8 sequences of 750 .. 3000 keys, 20 heads of 128: 5 splits 49 + 5 us, 13 splits 42 + 5 (165 MB of keys
// and values: 3.9 TB/s).  One sequence of 600 keys: 5 splits 5.7 + 4.5 us, unsplit 12.5.  ARIA_DECODE_SPLIT_KV, where it is set, decides as for aria_decode_token.
ARIA_HIDDEN int aria_decode_rows_splits(int64_t H, int64_t T, int64_t max_len, int64_t Smax);
// RoPE, cache write and attention of T tokens of T sequences: qkv [T, 3 H hd], caches [slots, Smax, H hd], part: T H splits (hd + 2) floats, out [T, H hd]
ARIA_HIDDEN int aria_decode_rows_attn(const ad::bf16_t* qkv, const ad::bf16_t* freqs, const int32_t* slot, const int32_t* pos, ad::bf16_t* kc, ad::bf16_t* vc,
                                      ad::bf16_t* out, float* part, int64_t H, int64_t hd, int64_t Smax, int64_t T, int splits, int64_t max_len, void* stream);
ARIA_HIDDEN int aria_route_and_sort(const ad::bf16_t* logits, ad::bf16_t* scores, int32_t* idx, int32_t* counts, int32_t* offsets, int32_t* src, int32_t* inv,
                                    int32_t* rows, int T, int E, int k, void* stream);
ARIA_HIDDEN int aria_decode_dims_ok(const int64_t* dims);
// ARIA_OK where every tensor of a step's table is there and starts at 16 bytes
ARIA_HIDDEN int aria_decode_table_ok(const void* const* ptrs, int64_t layers);
// One sequence's step by the engine's kernels
ARIA_HIDDEN int64_t aria_decode_one_scratch(const int64_t* dims);
ARIA_HIDDEN int aria_decode_one(const void* const* ptrs, const int64_t* dims, float eps, const void* x, const int32_t* slot, const int32_t* pos,
                                int64_t max_len, float* logits, char* scratch, void* stream);
