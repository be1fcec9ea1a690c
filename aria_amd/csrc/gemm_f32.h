// 32-bit products with what follows them (gemm_f32.hip), for the steps of steps32.hip.  Hidden: not part of the C ABI.
#pragma once
#include "aria_hip.h"

enum {
    ARIA_F32_PLAIN = 0,
    ARIA_F32_RELU2 = 1,    // max(v, 0)^2
    ARIA_F32_PAIR = 2,     // silu (relu_gate: max(., 0)) of the product with W times the product with W2
    ARIA_F32_STREAM = 3,   // x += post(v), C = next(x), where next.w is given; x [M, ldc] like C
};
struct AriaGemmF32 {
    const float *A, *W, *W2;
    float* C;
    int M, N, K;
    long long lda, ldw, ldc;
    const int* offsets;   // rows grouped by expert, or NULL
    int E;
    long long strideW;
    const int* rows;      // row m of the result from row rows[m] / per of A; NULL: from row m
    int per;
    int relu_gate;
    AriaDyT post, next;
    float* x;
};
__attribute__((visibility("hidden"))) int aria_gemm_f32_finished(const AriaGemmF32& p, int finish, void* stream);
