// Arguments of the prefill's fp16 products (gemm_f16.hip, gemm_f16_split.hip).
#pragma once

#include <type_traits>

#include "pe_common.h"

namespace pe {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));

struct GemmF16Args {
    const float* a;   // (M, K), row stride lda (fp32 A)
    const _Float16* ah;  // (M, K), row stride lda (fp16 A, AH)
    int64_t lda;
    const _Float16* w;  // (N, K) row-major
    const float* bias;  // (N) or NULL
    const float* res;   // (M, N), row stride ldr, or NULL
    int64_t ldr;
    float* c;           // (M, N), row stride ldc
    _Float16* ch;       // (M, N / 2), row stride ldc (fp16 SiLU output, CH)
    int64_t ldc;
    int64_t M, N, K;
    int round_wgs;      // k_gemm_h16_silu_dl: workgroups per round (a multiple of 8)
    int by_columns;     // k_gemm_h16_silu_dl: few row tiles, XCDs take column tiles
};

// gemm_f16_split.hip: the product of few tiles (false: not a shape for it). added: with a bias or a
// residual; wide: k_gemm_h16_dl would take the product.
bool gemm_split_ok(int64_t M, int64_t N, int64_t K, bool added, bool wide);
int gemm_split_launch(const GemmF16Args& p, bool silu, hipStream_t s);

}  // namespace pe
