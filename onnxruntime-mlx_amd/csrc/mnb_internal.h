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

// Shapes of 4-bit weights with fp16 or bf16 activations that take mnb_blk; larger ones take
// the prefill GEMM's shared weight tiles. On MI355X, GEMM against mnb_blk in fp16: 8 rows of
// 4096 x 14336 24.7 -> 12.6 us, 64 rows of 4096 x 4096 21.7 -> 10.4 us. Past 64 rows the GEMM
// has too few tiles for the chip while M * N is below about 2^20: 128 rows of 8960 x 1536
// 43.3 -> 16.6 us, 256 rows 44.1 -> 24.8 us, 128 rows of 4096 x 4096 21.4 -> 13.6 us; level
// at 512 x 8960 x 1536 (46.0, 45.6 us) and at 384 x 4096 x 4096 (34.8, 34.1 us), and behind
// at 512 x 4096 x 4096 (33.4, 40.4 us) and 1024 x 896 x 1152 (11.3, 13.3 us).
inline bool mnb_takes_blk(int64_t M, int64_t N) {
    return M <= 64 || (M <= 512 && M * N < (1 << 20));
}

// The prefill GEMM (mnb_gemm.hip): bs in {32, 64, 128}, A and B 16-byte aligned,
// K % 8 == 0, tensors within 32-bit buffer offsets (the caller checks).
template <typename T, bool SWI = false>
int mnb_gemm(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y, int M, int N, int K,
             int bs, hipStream_t st);

}  // namespace ortmi
