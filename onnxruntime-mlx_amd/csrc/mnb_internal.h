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
// the prefill GEMM's shared weight tiles. Up to 32 rows the GEMM's tiles are mostly padding
// (MI355X, GEMM against mnb_blk in fp16: 8 rows of 4096 x 14336 21.7 -> 11.7 us). Beyond,
// mnb_blk gains while its tiles of 32 x 64 outputs all run at once, a CU to each: the GEMM has
// a quarter of the tiles and leaves CUs idle (240 tiles, 96 rows of K 4096, N 5120: 1.5 times
// as fast as the GEMM; 256 tiles, 512 rows of K 896 to 14336, N 1024: 1.2 to 1.7 times). From
// 257 tiles on, each CU dequantises for two: 320 (128 rows of N 5120) 1.12 times at K 4096 but
// 0.92 at K 8960, 448 (64 rows of N 14336) 0.75 to 0.97.
inline bool mnb_takes_blk(int64_t M, int64_t N) {
    return M <= 32 || (M <= 512 && ((M + 31) / 32) * ((N + 63) / 64) <= device_cu_count());
}

// The prefill GEMM (mnb_gemm.hip): bs in {32, 64, 128}, A and B 16-byte aligned,
// K % 8 == 0, tensors within 32-bit buffer offsets (the caller checks).
template <typename T, bool SWI = false>
int mnb_gemm(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y, int M, int N, int K,
             int bs, hipStream_t st);

}  // namespace ortmi
