// The persistent 256-row GEMM of gemm_big.hip: tile configs 15 (256 x 256) and 25 (256 x 192) of mx_gemm_bf16.
#pragma once
#include "common.h"

// The operands of a checked mx_gemm_bf16 call without split-K.
struct BigGemm {
  const uint16_t* A;
  long lda;
  const uint16_t* W;
  long ldw;
  const float* bias;
  const uint16_t* R;
  long ldr;
  int r_rows;
  uint16_t* C;
  long ldc;
  int M, N, K, Kw, act_ncols;
};
// Whether launch_gemm_big takes the call: rows of C (and R) of whole aligned 16-byte chunks, at least 4 k-steps, and
// 256 rows of every operand within the 31-bit offsets of a buffer resource.
bool gemm_big_fits(int act, const BigGemm& g);
hipError_t launch_gemm_big(hipStream_t st, int bn, int act, const BigGemm& g);
