// MatMulNBits prefill GEMM (4-bit weights, fp16 or bf16 activations) on the matrix
// cores of gfx950: v_mfma_f32_32x32x16_f16 / _bf16 over a weight tile dequantised to
// the activation type (fp16((q - zp) * s) or bf16((q - zp) * s), one rounding) and an
// activation tile staged in LDS; fp32 accumulation, one rounding of Y.
#include "common.h"
#include "mnb_internal.h"

namespace ortmi {

// k-steps of 64 codes. LDS rows hold 64 halfs padded to 72 (144 bytes): 16-byte
// reads of 8 consecutive rows fall in 8 different bank groups (144/16 = 9 = 1 mod 8).
constexpr int kBK = 64;
constexpr int kLdsRow = 72;

// Dequantise one 32-bit word (codes k0..k7 of a chunk) to four fp16 pairs
// (k0,k4) (k1,k5) (k2,k6) (k3,k7): (w >> 4j) & 0x000F000F | 0x6400 6400 is the
// pair (1024 + q) exactly; subtracting (1024 + zp) is exact, and the multiply by
// the scale rounds once, giving fp16((q - zp) * s).
__device__ __forceinline__ uint4 dequant_word_pairs(uint32_t w, half2_t zoff, half2_t s2) {
    uint32_t r[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t m = ((w >> (4 * j)) & 0x000F000Fu) | 0x64006400u;
        half2_t h = __builtin_bit_cast(half2_t, m);
        h = (h - zoff) * s2;
        r[j] = __builtin_bit_cast(uint32_t, h);
    }
    return make_uint4(r[0], r[1], r[2], r[3]);
}


// bf16 weights, in the codes' own order (the activations then need no permutation): a byte
// 0000qqqq read as fp8 (e4m3) is q * 2^-9 exactly, the convert's scale makes it q, and q * s -
// zp * s is exact in fp32 (s has 8 mantissa bits), so that only the conversion rounds:
// bf16((q - zp) * s). 19 vector instructions per 8 codes; by way of fp16 pairs, widened and scaled in fp32, 32 (1999 x
// 17920 x 1536, block 128: 159 us, 143 us now).
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
__device__ __forceinline__ uint4 dequant_word_bf16(uint32_t w, float s, float zs) {
    const uint32_t ev = w & 0x0F0F0F0Fu, od = (w >> 4) & 0x0F0F0F0Fu;
    uint32_t r[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const auto e = h ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8((int)ev, 512.f, true)
                         : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8((int)ev, 512.f, false);
        const auto o = h ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8((int)od, 512.f, true)
                         : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8((int)od, 512.f, false);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bf16x2_t v = {(__bf16)fmaf(e[i], s, zs), (__bf16)fmaf(o[i], s, zs)};
            r[2 * h + i] = __builtin_bit_cast(uint32_t, v);
        }
    }
    return make_uint4(r[0], r[1], r[2], r[3]);
}

// Per-element-type pieces of the MFMA GEMM: T = half_t (fp16) or uint16_t (bf16
// bits). A block's dequantisation parameters, one word of codes to four operand
// pairs, and the 32x32x16 matrix-core step.
template <typename T>
struct GemmDq {
    half2_t zoff, s2;  // fp16: 1024 + zero point and the scale, as pairs
    float s, zs;       // bf16: scale, -zero point * scale
};
template <typename T>
__device__ __forceinline__ GemmDq<T> gemm_dq(float zf, uint16_t sbits) {
    GemmDq<T> d{};
    if constexpr (std::is_same<T, half_t>::value) {
        const half_t sh = __builtin_bit_cast(half_t, sbits);
        d.zoff = half2_t{(half_t)(1024.f + zf), (half_t)(1024.f + zf)};
        d.s2 = half2_t{sh, sh};
    } else {
        d.s = to_f32(sbits);
        d.zs = -zf * to_f32(sbits);
    }
    return d;
}
template <typename T>
__device__ __forceinline__ uint4 gemm_dequant(uint32_t w, const GemmDq<T>& d) {
    if constexpr (std::is_same<T, half_t>::value) return dequant_word_pairs(w, d.zoff, d.s2);
    else return dequant_word_bf16(w, d.s, d.zs);
}
template <typename T>
__device__ __forceinline__ float16_t gemm_mfma(half8_t a, half8_t b, float16_t c) {
    if constexpr (std::is_same<T, half_t>::value)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0,
                                                       0);
}

// One k-step's loads, kept raw until they are stored to LDS (a conversion at load
// time would make the compiler wait for this load, and so for every earlier one).
template <int BM, int BN, int BS>
struct GemmStage {
    static constexpr int A_VEC = BM * kBK / 8 / 256;  // 16-byte activation vectors per thread
    uint4 a[A_VEC];
    uint4 b;         // 32 codes (one 32-code chunk of one weight row)
    // Whole registers for the small fields: packed as 16 + 8 + 8 bits, the stage
    // was carried across the loop as byte pieces, and splitting a freshly loaded
    // scale into them waited on that load (loads complete in order, so on all of
    // the stage's loads, issued only one step before) at the end of every odd
    // step, which left one step of prefetch instead of two.
    uint32_t s;      // fp16 bits of that chunk's block scale
    uint32_t z;      // zero-point byte of the block pair
    uint32_t zhi;    // 1: the block's zero point is the byte's high nibble
};

// KS = 2 splits the k-steps of a tile between two groups of 4 waves (512 threads,
// own LDS buffers, common barriers: both halves run the same number of steps),
// whose accumulators are summed through LDS at the end: 2 waves per SIMD to hide
// the load latency when the grid has only about one tile per CU.
//
// BR (weights in registers, BN = 128): the 4 waves sit side by side, each with
// all BM rows and 32 columns. Lane l of a wave loads chunk 2s + (l >> 5) of
// column (l & 31) of k-step s and dequantises it straight into its MFMA B
// operands (word kk of the chunk for sub-step kk). Only the activation tile goes
// through LDS, read at column 32 (l >> 5) + 8 kk so that both operands take the
// same codes in each k slot.
template <typename T, int BM, int BN, int BS, int KS = 1, bool SWI = false, bool BR = false>
__global__ __launch_bounds__(256 * KS) void mnb_gemm4_kernel(const T* __restrict__ A,
                                                             const uint8_t* __restrict__ B,
                                                             const T* __restrict__ S,
                                                             const uint8_t* __restrict__ Z,
                                                             T* __restrict__ Y, int M,
                                                             int N, int K, int nb, int tiles_m,
                                                             int tiles_n) {
    static_assert(sizeof(T) == 2, "fp16 or bf16 (16-bit storage)");
    // Each k-step stages BN weight rows x 2 chunks of 32 codes: one chunk per thread
    // (BN = 128) or half a chunk per thread (BN = 64).
    static_assert(BN == 128 || BN == 64, "weight tile rows");
    static_assert(KS == 1 || KS == 2, "k split");
    static_assert(!BR || BN == 128, "weights in registers: 4 waves x 32 columns");
    constexpr int WM = BR ? BM : BM / 2, WN = BR ? 32 : BN / 2;
    constexpr int TM = WM / 32, TN = WN / 32;
    using Stage = GemmStage<BM, BN, BS>;
    constexpr int A_VEC = Stage::A_VEC;
    __shared__ half_t sAall[KS][2][BM * kLdsRow];
    __shared__ half_t sBall[KS][2][BR ? 8 : BN * kLdsRow];
    const int half_id = KS == 2 ? (int)(threadIdx.x >> 8) : 0;
    half_t (&sA)[2][BM * kLdsRow] = sAall[half_id];
    auto& sB = sBall[half_id];

    // XCD-aware order: workgroups are dealt round-robin to the 8 XCDs; give each
    // XCD a contiguous range of tiles (m fastest) so tiles sharing weight columns
    // share that XCD's L2.
    const int nwg = gridDim.x;
    int tile = blockIdx.x;
    if (nwg % 8 == 0) tile = (blockIdx.x % 8) * (nwg / 8) + blockIdx.x / 8;
    const int tm = tile % tiles_m, tn = tile / tiles_m;
    const int m0 = tm * BM, n0 = tn * BN;

    const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
    const int wm = BR ? 0 : (wave & 1) * WM, wn = BR ? wave * 32 : (wave >> 1) * WN;
    const int Kp = nb * BS;
    const int ksteps_all = (Kp + kBK - 1) / kBK;
    // This half's k-steps: [kbase, kbase + ksteps); steps past the end read zeros.
    const int ksteps = (ksteps_all + KS - 1) / KS;
    const int kbase = half_id * ksteps;
    const int chunks = Kp / 32;
    const size_t row_bytes = (size_t)Kp / 2;
    const int zp_cols = (nb + 1) / 2;
    // Raw buffer loads with range checks: a row past M or N, or a chunk past the
    // row, reads zeros without touching memory, so no load sits behind a branch
    // and the two-step prefetch is never drained by a conservative wait. (A's
    // rows are whole 16-byte vectors: the caller guarantees K % 8 == 0.)
    const uint32_t a_end = (uint32_t)((size_t)M * K * sizeof(half_t));
    const uint32_t b_end = (uint32_t)((size_t)N * row_bytes);
    const uint32_t s_end = (uint32_t)((size_t)N * nb * sizeof(half_t));
    const uint32_t z_end = Z ? (uint32_t)((size_t)N * zp_cols) : 0u;
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(A), 0, (int)a_end, kBufferWord3);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(B), 0, (int)b_end, kBufferWord3);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(S), 0, (int)s_end, kBufferWord3);
    const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(Z ? Z : B), 0, (int)z_end, kBufferWord3);

    auto gload = [&](Stage& st, int ks_local) {
        // Steps past this half's range read zeros (they may lie inside the other
        // half's range).
        const bool live = ks_local < ksteps;
        const int ks = kbase + ks_local;
        const int k0 = ks * kBK;
#pragma unroll
        for (int p = 0; p < A_VEC; ++p) {
            const int idx = tid + p * 256;
            const int r = idx >> 3, c = (idx & 7) * 8;
            const int m = m0 + r, k = k0 + c;
            const uint32_t off = (live && m < M && k < K)
                                     ? (uint32_t)(((size_t)m * K + k) * sizeof(half_t))
                                     : a_end;
            const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(ra, off, 0, 0);
            st.a[p] = make_uint4(v.x, v.y, v.z, v.w);
        }
        constexpr int TPR = 256 / BN;  // threads per weight row: 2 (one chunk) or 4 (half)
        // BR: column (lane & 31) of this wave's 32, chunk (lane >> 5) of the step.
        const int r = BR ? wn + (lane & 31) : tid / TPR;
        const int chunk = 2 * ks + (BR ? (lane >> 5) : (tid % TPR) * 2 / TPR);
        const int n = n0 + r;
        const bool ok = live && n < N && chunk < chunks;
        const int blk = (chunk * 32) / BS;
        if constexpr (BN == 128) {
            const uint32_t boff =
                ok ? (uint32_t)((size_t)n * row_bytes + (size_t)chunk * 16) : b_end;
            const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rb, boff, 0, 0);
            st.b = make_uint4(v.x, v.y, v.z, v.w);
        } else {
            const uint32_t boff =
                ok ? (uint32_t)((size_t)n * row_bytes + (size_t)chunk * 16 + (tid & 1) * 8)
                   : b_end;
            const uint2 v = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rb, boff, 0, 0));
            st.b = make_uint4(v.x, v.y, 0u, 0u);
        }
        const uint32_t soff = ok ? (uint32_t)(((size_t)n * nb + blk) * sizeof(half_t)) : s_end;
        st.s = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, soff, 0, 0);  // 0 out of range
        const uint32_t zoff = ok ? (uint32_t)((size_t)n * zp_cols + blk / 2) : z_end;
        st.z = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(rz, zoff, 0, 0);
        st.zhi = (uint32_t)(blk & 1);
    };
    auto sstore = [&](const Stage& st, int buf) {
#pragma unroll
        for (int p = 0; p < A_VEC; ++p) {
            const int idx = tid + p * 256;
            const int r = idx >> 3, c = (idx & 7) * 8;
            *reinterpret_cast<uint4*>(&sA[buf][r * kLdsRow + c]) =
                std::is_same<T, half_t>::value ? permute_act8(st.a[p]) : st.a[p];
        }
        if constexpr (!BR) {
            const float zf = Z ? (float)nibble(st.z, st.zhi) : 8.f;
            const GemmDq<T> dq = gemm_dq<T>(zf, st.s);
            if constexpr (BN == 128) {
                const int r = tid >> 1, h = tid & 1;
                uint4* dst = reinterpret_cast<uint4*>(&sB[buf][r * kLdsRow + h * 32]);
                dst[0] = gemm_dequant<T>(st.b.x, dq);
                dst[1] = gemm_dequant<T>(st.b.y, dq);
                dst[2] = gemm_dequant<T>(st.b.z, dq);
                dst[3] = gemm_dequant<T>(st.b.w, dq);
            } else {
                const int r = tid >> 2, h = (tid >> 1) & 1, q = tid & 1;
                uint4* dst = reinterpret_cast<uint4*>(&sB[buf][r * kLdsRow + h * 32 + q * 16]);
                dst[0] = gemm_dequant<T>(st.b.x, dq);
                dst[1] = gemm_dequant<T>(st.b.y, dq);
            }
        }
    };

    float16_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    const int lrow = lane & 31, lk = (lane >> 5) * 8;
    // BR: the B operands of the current step, dequantised from its stage.
    uint4 bq[BR ? 4 : 1];
    auto dequant_b = [&](const Stage& st) {
        const float zf = Z ? (float)nibble(st.z, st.zhi) : 8.f;
        const GemmDq<T> dq = gemm_dq<T>(zf, st.s);
        bq[0] = gemm_dequant<T>(st.b.x, dq);
        if constexpr (BR) {
            bq[1] = gemm_dequant<T>(st.b.y, dq);
            bq[2] = gemm_dequant<T>(st.b.z, dq);
            bq[3] = gemm_dequant<T>(st.b.w, dq);
        }
    };
    auto compute = [&](int buf) {
#pragma unroll
        for (int kk = 0; kk < kBK / 16; ++kk) {
            half8_t af[TM], bf[TN];
            const int acol = BR ? 4 * lk + kk * 8 : kk * 16 + lk;
#pragma unroll
            for (int i = 0; i < TM; ++i)
                af[i] = *reinterpret_cast<const half8_t*>(
                    &sA[buf][(wm + i * 32 + lrow) * kLdsRow + acol]);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (BR)
                    bf[j] = __builtin_bit_cast(half8_t, bq[kk]);
                else
                    bf[j] = *reinterpret_cast<const half8_t*>(
                        &sB[buf][(wn + j * 32 + lrow) * kLdsRow + kk * 16 + lk]);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = gemm_mfma<T>(af[i], bf[j], acc[i][j]);
        }
    };

    // Pipeline: loads for step s are issued two steps ahead (register sets r0/r1
    // alternate), stored to the LDS buffer of step s at the end of step s-1.
    // Loads and stores past the last step are issued too (they read zeros and
    // fill a buffer nobody reads), so the loop has no branch around a load. The
    // loop runs an even number of steps (an odd count gets one all-zero step):
    // a mid-body exit made the compiler copy all accumulators every iteration.
    Stage r0, r1;
    gload(r0, 0);
    gload(r1, 1);
    sstore(r0, 0);
    __syncthreads();
    const int ksteps2 = (ksteps + 1) & ~1;
    for (int ks = 0; ks < ksteps2; ks += 2) {
        // even step ks: LDS buf 0 holds it; r1 holds step ks+1. (BR: r0's weights
        // become the B operands before r0 is reloaded.)
        if constexpr (BR) dequant_b(r0);
        gload(r0, ks + 2);
        compute(0);
        sstore(r1, 1);
        __syncthreads();
        // odd step ks+1: LDS buf 1; r0 holds step ks+2.
        if constexpr (BR) dequant_b(r1);
        gload(r1, ks + 3);
        compute(1);
        sstore(r0, 0);
        __syncthreads();
    }

    if constexpr (KS == 2) {
        // Half 1 hands its accumulators to half 0 through LDS (the loop ended on a
        // barrier, so the tile buffers are free).
        float* xch = BR ? reinterpret_cast<float*>(&sAall[0][0][0])
                        : reinterpret_cast<float*>(&sBall[0][0][0]);
        static_assert(4 * TM * TN * 16 * 64 * sizeof(float) <= (BR ? sizeof(sAall) : sizeof(sBall)),
                      "exchange space");
        if (half_id == 1) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        xch[((wave * TM * TN + i * TN + j) * 16 + e) * 64 + lane] = acc[i][j][e];
        }
        __syncthreads();
        if (half_id == 1) return;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    acc[i][j][e] += xch[((wave * TM * TN + i * TN + j) * 16 + e) * 64 + lane];
    }
    // D layout of a 32x32 MFMA: lane holds column (lane & 31); accumulator e holds
    // row 8*(e/4) + 4*(lane/32) + (e%4).
    if constexpr (SWI) {
        // Interleaved gate/up columns (2i, 2i+1) sit in lanes (2l, 2l+1): the even
        // lane takes its partner's value and writes column i of the [M, N/2] output,
        // (g * sigmoid(g)) * u with each op rounded to fp16 as the unfused ops store.
        const int Nh = N / 2;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n0 + wn + j * 32 + (lane & 31);
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float y = round_to<T>(acc[i][j][e]);
                    const float partner = dpp_mov<0xB1>(y);  // quad_perm [1,0,3,2]
                    const int m = m0 + wm + i * 32 + 8 * (e / 4) + 4 * (lane >> 5) + (e % 4);
                    if ((lane & 1) == 0 && m < M && n < N) {
                        const float sig = round_to<T>(1.0f / (1.0f + __expf(-y)));
                        Y[(size_t)m * Nh + n / 2] = from_f32<T>(round_to<T>(y * sig) * partner);
                    }
                }
            }
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + wn + j * 32 + (lane & 31);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + wm + i * 32 + 8 * (e / 4) + 4 * (lane >> 5) + (e % 4);
                if (m < M && n < N) Y[(size_t)m * N + n] = from_f32<T>(acc[i][j][e]);
            }
        }
}

template <typename T, int BM, int BN, int BS, int KS = 1, bool SWI = false, bool BR = false>
static int launch_gemm4(const T* A, const uint8_t* B, const T* S, const uint8_t* Z,
                        T* Y, int M, int N, int K, int nb, hipStream_t st) {
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    hipLaunchKernelGGL((mnb_gemm4_kernel<T, BM, BN, BS, KS, SWI, BR>), dim3(tiles_m * tiles_n),
                       dim3(256 * KS), 0, st, A, B, S, Z, Y, M, N, K, nb, tiles_m, tiles_n);
    return check_launch("mnb_gemm4");
}

template <typename T, int BS, bool SWI = false>
static int dispatch_gemm4(const T* A, const uint8_t* B, const T* S, const uint8_t* Z,
                          T* Y, int M, int N, int K, int nb, hipStream_t st) {
    // 128x128 tiles once they fill the CUs twice over; below that, the k-steps are
    // split over two wave groups, with 64x128 tiles while those still give every
    // CU a tile and 64x64 tiles under that (M=512 on MI355X: K=N=4096 41.6 us
    // with 64x128; N=1536 K=8960 66.4 -> 49.7 us, N=2048 K=1536 15.1 -> 11.5 us
    // with 64x64).
    const int cus = device_cu_count();
    const long big = (long)((M + 127) / 128) * ((N + 127) / 128);
    // 128x128 tiles take their weights in registers (gate/up 512x17920x1536:
    // 52-54 -> 46-47 us); at 64x128 the LDS form measured equal or faster.
    if (big >= 2L * cus)
        return launch_gemm4<T, 128, 128, BS, 1, SWI, true>(A, B, S, Z, Y, M, N, K, nb, st);
    const long mid = (long)((M + 63) / 64) * ((N + 127) / 128);
    if (mid >= cus) return launch_gemm4<T, 64, 128, BS, 2, SWI>(A, B, S, Z, Y, M, N, K, nb, st);
    return launch_gemm4<T, 64, 64, BS, 2, SWI>(A, B, S, Z, Y, M, N, K, nb, st);
}

template <typename T, bool SWI>
int mnb_gemm(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y, int M, int N, int K,
             int bs, hipStream_t st) {
    const int nb = (K + bs - 1) / bs;
    if (bs == 32) return dispatch_gemm4<T, 32, SWI>(A, B, S, Z, Y, M, N, K, nb, st);
    if (bs == 64) return dispatch_gemm4<T, 64, SWI>(A, B, S, Z, Y, M, N, K, nb, st);
    return dispatch_gemm4<T, 128, SWI>(A, B, S, Z, Y, M, N, K, nb, st);
}

#define ORTMI_GEMM(T, SWI)                                                                  \
    template int mnb_gemm<T, SWI>(const T*, const uint8_t*, const T*, const uint8_t*, T*, int, \
                                  int, int, int, hipStream_t);
ORTMI_GEMM(half_t, false)
ORTMI_GEMM(half_t, true)
ORTMI_GEMM(uint16_t, false)

}  // namespace ortmi
