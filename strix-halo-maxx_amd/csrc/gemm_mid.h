// The 128-row GEMM of gemm_mid.hip for grids of about one tile per CU: tile configs 19 (128 x 128), 27 (128 x 192) and 17
// (128 x 256) of mx_gemm_bf16 and mx_gemm_bf16_partial.
#pragma once
#include "gemm_big.h"

// Whether launch_gemm_mid takes the call (without partials): rows of C (and R) of whole aligned 16-byte chunks, and a
// tile's rows of every operand within the 31-bit offsets of a buffer resource.
bool gemm_mid_fits(int act, const BigGemm& g);
// P: raw partials of `splits` k ranges (row stride ldp, split stride p_split) instead of C.
hipError_t launch_gemm_mid(hipStream_t st, int bn, int act, const BigGemm& g, int splits = 1, float* P = nullptr,
                           long ldp = 0, long p_split = 0);
