// 16-bit MFMA GEMM with the LoRA term in its epilogue (gemm16.hip).
#pragma once

#include "common.hpp"

namespace grpo {

// C[m, n] = dt(sum_k A[m, k] B[n, k]), both operands contiguous along k, then
//   GEMM16_ADD   C = dt(C + dt(t low^T))
//   GEMM16_LORA  C = dt(dt(C [+ bias]) + dt(dt(t low^T) * dt(scaling)))
enum Gemm16Mode { GEMM16_ADD, GEMM16_LORA };

struct Gemm16 {
  const uint16_t* a;  // [M][K], row stride lda
  int64_t lda;
  const uint16_t* b;  // [N][K], row stride ldb
  int64_t ldb;
  uint16_t* c;        // [M][N], row stride ldc
  int64_t ldc;
  int M, N, K;
  const uint16_t* t;    // [M][32], ranks >= r zero
  const uint16_t* low;  // [N] rows of r 16-bit values, row stride ldl
  int64_t ldl;
  const uint16_t* bias;  // GEMM16_LORA: [N] or null
  int r;                 // 1..32
  float scaling;         // GEMM16_LORA
};

// K % 32 == 0 and N % 8 == 0; rows of a, b and c 16-byte aligned; row strides of
// a and b below 2^22 elements (32-bit offsets within a tile).
bool gemm16_ok(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb);
int gemm16_launch(const Gemm16& g, Gemm16Mode mode, bool f16, hipStream_t st);

}  // namespace grpo
