// dense16.h — what other files call of dense16's products.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

// epilogues: fp32 stored, fp32 added to, 16-bit, 16-bit after GELU, a gated unit beside fp32 columns, a part of K
enum { D16_F32 = 0, D16_ADD = 1, D16_ACT = 2, D16_GELU = 3, D16_GLU = 4, D16_PART = 5 };

// 16-bit products of the model's activation type (dense16_enc.hip): epi D16_ACT / D16_GELU: Y [M, N] (ldy) = act(A B^T + bias); D16_PART: `parts` parts
// of K to part [parts][M][N]. K % 64 == 0, N % 8 == 0, all pointers and rows 16-byte aligned, rows below 2^23 bytes.
int mx_dense16_enc(int epi, int tile, const uint16_t* A, int lda, const uint16_t* B, int M, int N, int K, const uint16_t* bias, uint16_t* Y, int ldy,
                   int parts, float* part, hipStream_t st);
