// The matrix-core MatMulNBits kernels, called by the dispatch in mnb.hip.
#pragma once

#include "common.h"

namespace ortmi {

// Y[M, N] = A[M, K] . dequant(B)^T for BITS-bit weights in blocks of 32, 64 or 128;
// with SWI the SwiGLU of interleaved gate/up columns, Y[M, N / 2] (fp16, 4-bit).
// Returns an ORTMI_* status, or -1 (nothing launched) for a form it does not take:
// another block size, a tensor not 16-byte aligned, rows of A that are not whole
// 16-byte vectors, a tensor past 32-bit buffer offsets, or a K whose scales do not
// fit LDS beside one column tile.
template <typename T, int BITS, bool SWI = false>
int mnb_blk(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y, int M, int N, int K,
            int bs, hipStream_t st);

// Rows up to which 4-bit weights with fp16 or bf16 activations take mnb_blk; more
// rows take the prefill GEMM's shared weight tiles. On MI355X, GEMM against mnb_blk in
// fp16: 8 rows of 4096 x 14336 24.7 -> 12.6 us, 32 rows 25.1 -> 16.5 us, 64 rows 25.1
// -> 24.3 us; 64 rows of 4096 x 4096 21.7 -> 10.4 us.
constexpr int kBlkRows = 64;

// The prefill GEMM (mnb_gemm.hip): bs in {32, 64, 128}, A and B 16-byte aligned,
// K % 8 == 0, tensors within 32-bit buffer offsets (the caller checks).
template <typename T, bool SWI = false>
int mnb_gemm(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y, int M, int N, int K,
             int bs, hipStream_t st);

}  // namespace ortmi
