// MatMulNBits (com.microsoft) for gfx950.
//
// ORT layout, read in place (no repack): B is [N, nb, bs*bits/8] uint8 with
// blocks consecutive along K, so row n is nb*bs*bits/8 contiguous bytes and each
// byte holds k (low nibble) and k+1 (high nibble). Scales are [N, nb] in the
// activation dtype; 4-bit zero points are packed [N, ceil(nb/2)], low nibble for
// even blocks.
//
// Kernels:
//  * mnb_gemv4  - decode (M == 1), bits 4, bs in {32, 64, 128}. HBM-bound: each
//    lane owns a contiguous run of 32-code chunks of K and keeps the matching
//    activations in VGPRs (staged once per workgroup through LDS), then streams
//    rows of B with 128-bit range-checked buffer loads, a ring of row groups in
//    flight per wave. fp32/bf16 activations: zero points folded as
//    s*(sum(a*q) - zp*sum(a)), one byte-convert and one FMA per code. fp16
//    activations: codes become exact fp16 (q - zp) pairs and v_dot2_f32_f16
//    takes two codes per instruction.
//  * the prefill GEMM (mnb_gemm.hip) - prompts, fp16 or bf16, bits 4, bs in {32, 64,
//    128}: matrix-core tiles over dequantised weights staged in LDS.
//  * mnb_blk.hip - smaller products of those (mnb_takes_blk), and bits 8 or fp32 activations at any M:
//    matrix cores fed from registers, K split over the waves of a workgroup.
//  * mnb_generic - every other form (bs 16, unaligned tensors): fp32 dequant to LDS
//    and a VALU tile product.
#include "common.h"
#include "mnb_internal.h"

namespace ortmi {

// -------------------------------------------------------------- GEMV (M=1) --

// Dot product of 32 activations with the 32 4-bit codes of one 16-byte chunk.
// Code i of the chunk is nibble (i & 1) of byte i/2, i.e. bits [4i, 4i+4) of the
// little-endian 128-bit word.
//
// The codes are converted two at a time by the fp8 (e4m3) pack convert: a byte
// 0000qqqq read as e4m3 is q * 2^-9 exactly (a subnormal m * 2^-9 for q < 8,
// (8 + m) * 2^-9 with exponent field 1 for q >= 8), so the sum comes out scaled
// by the exact power of two code_unit() and the caller scales it back. Scaling
// by a power of two commutes with every rounding here, so the result equals the
// unscaled sum bit for bit. One instruction per two codes, against a bit-field
// extract plus a byte convert per code.
__device__ __forceinline__ float dot32_codes(const float* a, uint4 w) {
    const uint32_t words[4] = {w.x, w.y, w.z, w.w};
    float d0 = 0.f, d1 = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t lo = words[i] & 0x0F0F0F0Fu;         // codes 8i+0,2,4,6
        const uint32_t hi = (words[i] >> 4) & 0x0F0F0F0Fu;  // codes 8i+1,3,5,7
        const float* ai = a + 8 * i;
        const auto l01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, false);
        const auto l23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, true);
        const auto h01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, false);
        const auto h23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, true);
        d0 = fmaf(ai[0], l01[0], d0);
        d1 = fmaf(ai[1], h01[0], d1);
        d0 = fmaf(ai[2], l01[1], d0);
        d1 = fmaf(ai[3], h01[1], d1);
        d0 = fmaf(ai[4], l23[0], d0);
        d1 = fmaf(ai[5], h23[0], d1);
        d0 = fmaf(ai[6], l23[1], d0);
        d1 = fmaf(ai[7], h23[1], d1);
    }
    return d0 + d1;
}
// The value dot32_codes gives code 1 (2^-9 for e4m3), read from the hardware.
__device__ __forceinline__ float code_unit() {
    return __builtin_amdgcn_cvt_pk_f32_fp8(1, false)[0];
}

// Activations live in LDS as fp32 in 16-byte units. Lane l reads the 8*CPL
// consecutive units of its chunks; unit u of lane l is stored at
// u ^ ((u / (8*CPL)) & 7), so the 8 lanes of one read phase hit 8 bank groups.
template <int CPL>
__device__ __forceinline__ int act_unit(int u) {
    return u ^ ((u / (8 * CPL)) & 7);
}

// Zero-point bytes that cover the blocks of one lane's CPL chunks, worst case
// over the 64 lanes (4-bit zero points: two blocks per byte).
constexpr int zp_window(int BS, int CPL) {
    int most = 1;
    for (int l = 0; l < 64; ++l) {
        const int c0 = l * CPL;
        const int b0 = (32 * c0) / BS / 2, b1 = (32 * (c0 + CPL - 1)) / BS / 2;
        if (b1 - b0 + 1 > most) most = b1 - b0 + 1;
    }
    return most;
}

// One group of R rows as loaded: weights, scales and zero-point bytes are kept
// raw and converted only when the group is reduced, so no instruction consumes a
// prefetched value before its row is needed (a conversion at load time would
// make the compiler wait for the prefetch there).
template <typename T, int R, int CPL, int ZB>
struct GemvGroup {
    uint4 w[R][CPL];
    T s[R][CPL];
    uint8_t z[R][ZB];
};

// Lane l owns the CPL consecutive 32-code chunks [l*CPL, (l+1)*CPL) of every row,
// so a row costs one 16*CPL-byte weight run, CPL adjacent scales and one or two
// zero-point bytes per lane; or (IL, fp16 rows of whole 64-chunk runs at block 32)
// chunks l, l + 64, ..., so each of the row's CPL weight loads reads 1 KB
// contiguous, each scale load 128 bytes, with one zero-point byte per chunk. The
// activation loads are issued first, then the weight loads of the wave's first D
// row groups; the activations go through LDS
// (one copy per workgroup) into VGPRs while the weights are in flight. Row groups
// of R rows are dealt to waves round-robin; a ring of D groups keeps the next
// D - 1 groups' loads in flight while one group is reduced.
// Activations in VGPRs: fp32 (32 per chunk) for fp32/bf16, fp16 pairs (16 VGPRs
// per chunk, v_dot2 products) for fp16 (H2).
// Optional fusions of the decoder's neighbours into the GEMV (decode only):
//  * prologue: the activation row is (Skip)SimplifiedLayerNorm(x [+ skip]) * gamma,
//    computed by every workgroup from x (K elements) before staging; workgroup 0
//    also writes the residual x + skip. Rounding as the unfused ops: the sum is
//    rounded to T, the normalised value once more.
//  * SwiGLU pairs: rows come interleaved (gate row i, up row i), a wave takes both
//    rows of a pair and writes Y[i] = (g * sigmoid(g)) * u, each op rounded to T as
//    the Sigmoid/Mul/Mul graph stores it.
//  * split merge (MRG): the activation row is attention output still held as
//    split partials [heads][splits][hd + 2] (o, max, sum) by the one-token decode;
//    each workgroup merges them as the merge kernel would, rounding to T.
template <typename T>
struct GemvPrologue {
    const T* skip;
    const T* gamma;
    T* residual;
    float eps;
    const float* part = nullptr;
    int splits = 0;
    int hd = 0;
};

// One scale, or an aligned pair of scales, through a buffer load.
template <typename T>
__device__ __forceinline__ T load_scale(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
    } else {
        return __builtin_bit_cast(T, (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
    }
}
template <typename T>
__device__ __forceinline__ void load_scale_pair(__amdgpu_buffer_rsrc_t r, uint32_t off, T& a, T& b) {
    if constexpr (sizeof(T) == 4) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
        a = __builtin_bit_cast(T, (uint32_t)v[0]);
        b = __builtin_bit_cast(T, (uint32_t)v[1]);
    } else {
        const uint32_t v = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
        a = __builtin_bit_cast(T, (uint16_t)(v & 0xffffu));
        b = __builtin_bit_cast(T, (uint16_t)(v >> 16));
    }
}

// Split-merge prologue bounds: partial floats per workgroup (one batch of
// float4 loads, kMergeVec per thread).
constexpr int kMergeVec = kDecodeMergeMaxFloats / (256 * 4);

// LDS bytes of the staged activation row (fp16 pairs or fp32 units).
template <typename T, bool H2>
constexpr size_t gemv_stage_bytes(int Kp) {
    return (size_t)Kp * (H2 ? sizeof(half_t) : sizeof(float));
}
// LDS bytes of the split-merge prologue: partials, split weights, 1/L per head.
static inline size_t gemv_merge_bytes(int K, int hd, int splits) {
    const size_t nh = (size_t)K / hd, nparts = nh * splits * (hd + 2);
    return (((nparts + 3) & ~(size_t)3) + nh * splits + nh) * sizeof(float);
}

template <typename T, int BS, int CPL, int R, int D, bool PRO = false, bool PAIR = false,
          bool SV = false, bool H2 = std::is_same<T, half_t>::value, bool NT = true,
          bool MRG = false, int RW = 1, bool IL = false>
__global__ __launch_bounds__(256) void mnb_gemv4_kernel(const T* __restrict__ A,
                                                        const uint8_t* __restrict__ B,
                                                        const T* __restrict__ S,
                                                        const uint8_t* __restrict__ Z,
                                                        T* __restrict__ Y, int N, int K,
                                                        int nb, GemvPrologue<T> pro) {
    static_assert(!PAIR || R == 2, "SwiGLU pairs take two rows per group");
    static_assert(!H2 || std::is_same<T, half_t>::value, "fp16 pairs need fp16 activations");
    static_assert(D >= 1, "ring depth");
    static_assert(!IL || (H2 && !SV && BS == 32), "interleaved chunks: fp16 pairs, block 32");
    extern __shared__ float4 sA[];
    __shared__ float s_red[4];
    constexpr int ZB = IL ? CPL : zp_window(BS, CPL);
    using Group = GemvGroup<T, R, CPL, ZB>;
    const int Kp = nb * BS;
    const int C = Kp / 32;  // 32-code chunks per row
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int waves_total = gridDim.x * 4;
    // A wave works on RW units of R rows at once, LR = 64 / RW lanes per unit
    // (RW > 1 when a row has few chunks, so that no lane idles); a group is RW
    // consecutive units.
    constexpr int LR = 64 / RW;
    const int li = lane % LR, slot = lane / LR;
    const int nunits = (N + R - 1) / R;
    const int ngroups = (nunits + RW - 1) / RW;
    const size_t row_bytes = (size_t)Kp / 2;
    const int zp_cols = (nb + 1) / 2;
    const int c0 = li * CPL;
    // Chunk j of this lane: CPL consecutive chunks, or (IL) chunks li + j * LR, so
    // that each load instruction of a unit reads one contiguous run.
    auto chunk = [&](int j) { return IL ? li + j * LR : c0 + j; };

    // 1. activation loads (16 bytes each), all in flight before anything else.
    constexpr int EPL = 16 / sizeof(T);
    // Kp <= 64 lanes * CPL * 32 codes, so 256 threads need ceil(8 * CPL / EPL) vectors each.
    constexpr int AV = (8 * CPL + EPL - 1) / EPL;
    const int nvec = Kp / EPL;
    const bool vec_ok = (K % EPL) == 0 && (reinterpret_cast<uintptr_t>(A) % 16) == 0;
    uint4 av[AV];
    auto load_vec = [&](const T* src, int u) -> uint4 {
        const int vi = threadIdx.x + u * 256;
        const int k0 = vi * EPL;
        if (vi < nvec && vec_ok && k0 + EPL <= K) return *reinterpret_cast<const uint4*>(src + k0);
        T t[EPL];
#pragma unroll
        for (int e = 0; e < EPL; ++e)
            t[e] = (vi < nvec && k0 + e < K) ? src[k0 + e] : from_f32<T>(0.f);
        return *reinterpret_cast<const uint4*>(t);
    };
    // Split merge: the whole partial array in one batch of loads (at most
    // kMergeVec float4 per thread; the launcher checks the size).
    float4 pbuf[MRG ? kMergeVec : 1];
    float ptail = 0.f;
    if constexpr (MRG) {
        const int nparts = (K / pro.hd) * pro.splits * (pro.hd + 2);
#pragma unroll
        for (int u = 0; u < kMergeVec; ++u) {
            const int idx = threadIdx.x + 256 * u;
            pbuf[u] = idx < nparts / 4 ? reinterpret_cast<const float4*>(pro.part)[idx]
                                       : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        if (threadIdx.x < (nparts & 3)) ptail = pro.part[(nparts & ~3) + threadIdx.x];
    } else {
#pragma unroll
        for (int u = 0; u < AV; ++u) av[u] = load_vec(A, u);
    }
    uint4 skv[PRO ? AV : 1], gmv[PRO ? AV : 1];
    if constexpr (PRO) {
#pragma unroll
        for (int u = 0; u < AV; ++u) {
            skv[u] = pro.skip ? load_vec(pro.skip, u) : make_uint4(0, 0, 0, 0);
            gmv[u] = load_vec(pro.gamma, u);
        }
    }

    // 2. weights of the first D row groups, issued after the activation loads (a
    // wait on a load also waits on every load issued before it). Loads never
    // branch, which keeps every wait on a prefetch exact: they are buffer loads,
    // and a group past the end, or a chunk past the row end, gets an offset past
    // the buffer's range, which returns zeros without a memory access (a zero chunk
    // meets zero activations, a missing group is never reduced). The last group's
    // second row, when N is odd, repeats row N - 1 (in bounds).
    const int g0 = blockIdx.x * 4 + wave;
    const int blk0 = (32 * min(c0, C - 1)) / BS;
    const uint32_t b_end = (uint32_t)((size_t)N * row_bytes);
    const uint32_t s_end = (uint32_t)((size_t)N * nb * sizeof(T));
    const uint32_t z_end = (uint32_t)((size_t)N * zp_cols);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(B), 0, (int)b_end, kBufferWord3);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(S), 0, (int)s_end, kBufferWord3);
    const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(Z ? Z : B), 0, Z ? (int)z_end : 0, kBufferWord3);
    // A unit past the end in a live group repeats the last unit (in bounds; its
    // lanes then store the same values to the same rows).
    auto unit_of = [&](int gi) { return min(gi * RW + slot, nunits - 1); };
    auto load_group = [&](Group& g, int gi) {
        const bool live = gi < ngroups;
        const int unit = unit_of(gi);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int n = min(unit * R + r, N - 1);
            const uint32_t zoff = live ? (uint32_t)(n * zp_cols) : z_end;
#pragma unroll
            for (int t = 0; t < ZB; ++t) {
                // Loaded either way (no records without Z): no load behind a branch.
                const int zcol = IL ? min(chunk(t), C - 1) / 2 : blk0 / 2 + t;
                const uint8_t zb = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(
                    rz, zoff + (uint32_t)min(zcol, zp_cols - 1), 0, 0);
                g.z[r][t] = Z ? zb : (uint8_t)0x88;
            }
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int c = chunk(j);
                const bool ok = live && c < C;
                const uint32_t boff = ok ? (uint32_t)((size_t)n * row_bytes) + 16u * c : b_end;
                // Streamed once: optionally non-temporal (cache policy nt).
                const u32x4_t v =
                    __builtin_amdgcn_raw_buffer_load_b128(rb, boff, 0, NT ? kCachePolicyNT : 0);
                g.w[r][j] = make_uint4(v.x, v.y, v.z, v.w);
                if constexpr (!SV) {
                    const uint32_t soff =
                        ok ? (uint32_t)(((size_t)n * nb + (32 * c) / BS) * sizeof(T)) : s_end;
                    g.s[r][j] = load_scale<T>(rs, soff);
                }
            }
            if constexpr (SV) {
                // Block 32 and an even CPL: the lane's scales are CPL/2 aligned pairs.
#pragma unroll
                for (int j = 0; j < CPL; j += 2) {
                    const int c = c0 + j;
                    const uint32_t soff =
                        live && c < C ? (uint32_t)(((size_t)n * nb + c) * sizeof(T)) : s_end;
                    load_scale_pair(rs, soff, g.s[r][j], g.s[r][j + 1]);
                }
            }
        }
    };
    Group g[D];
#pragma unroll
    for (int d = 0; d < D; ++d) load_group(g[d], g0 + d * waves_total);

    if constexpr (MRG) {
        // Partials -> LDS (after the staging area), then per head h the split
        // weights e^(m_i - M) and 1 / sum_i w_i l_i, then activation k = h*hd + d
        // as (sum_i w_i o_i[d]) / L, rounded to T as the merge kernel stores it.
        const int nh = K / pro.hd, ns = pro.splits, stride = pro.hd + 2;
        const int nparts = nh * ns * stride;
        float* sP = reinterpret_cast<float*>(reinterpret_cast<char*>(sA) + gemv_stage_bytes<T, H2>(Kp));
        float* sW = sP + ((nparts + 3) & ~3);
        float* sInv = sW + nh * ns;
#pragma unroll
        for (int u = 0; u < kMergeVec; ++u) {
            const int idx = threadIdx.x + 256 * u;
            if (idx < nparts / 4) reinterpret_cast<float4*>(sP)[idx] = pbuf[u];
        }
        if (threadIdx.x < (nparts & 3)) sP[(nparts & ~3) + threadIdx.x] = ptail;
        __syncthreads();
        for (int h = threadIdx.x; h < nh; h += 256) {
            const float* ph = sP + h * ns * stride;
            float M = -INFINITY;
            for (int i = 0; i < ns; ++i) M = fmaxf(M, ph[i * stride + pro.hd]);
            float L = 0.f;
            for (int i = 0; i < ns; ++i) {
                const float mi = ph[i * stride + pro.hd];
                const float w = mi == -INFINITY ? 0.f : __expf(mi - M);
                sW[h * ns + i] = w;
                L += w * ph[i * stride + pro.hd + 1];
            }
            sInv[h] = L > 0.f ? 1.0f / L : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < AV; ++u) {
            const int vi = threadIdx.x + u * 256;
            const int k0 = vi * EPL;
            T t[EPL];
#pragma unroll
            for (int e = 0; e < EPL; ++e) t[e] = from_f32<T>(0.f);
            if (vi < nvec && k0 < K) {
                const int h = k0 / pro.hd, d0 = k0 % pro.hd;
                const float* ph = sP + h * ns * stride + d0;
                const float* wh = sW + h * ns;
                float acc[EPL];
#pragma unroll
                for (int e = 0; e < EPL; ++e) acc[e] = 0.f;
                for (int i = 0; i < ns; ++i) {
                    const float w = wh[i];
#pragma unroll
                    for (int e = 0; e < EPL; ++e) acc[e] = fmaf(ph[i * stride + e], w, acc[e]);
                }
#pragma unroll
                for (int e = 0; e < EPL; ++e) t[e] = from_f32<T>(acc[e] * sInv[h]);
            }
            av[u] = *reinterpret_cast<const uint4*>(t);
        }
    }

    // 3. activations (normalised first when fused) -> LDS -> VGPRs.
    float scale_all = 1.f;
    if constexpr (PRO) {
        float ss = 0.f;
#pragma unroll
        for (int u = 0; u < AV; ++u) {
            const int vi = threadIdx.x + u * 256;
            if (vi >= nvec) continue;
            T* t = reinterpret_cast<T*>(&av[u]);
            const T* k = reinterpret_cast<const T*>(&skv[u]);
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                float v = to_f32(t[e]);
                if (pro.skip) v = round_to<T>(v + to_f32(k[e]));
                t[e] = from_f32<T>(v);
                ss += v * v;
            }
            if (pro.residual && blockIdx.x == 0) {
                const int k0 = vi * EPL;
                if (vec_ok && k0 + EPL <= K) {
                    *reinterpret_cast<uint4*>(pro.residual + k0) = av[u];
                } else {
                    for (int e = 0; e < EPL; ++e)
                        if (k0 + e < K) pro.residual[k0 + e] = t[e];
                }
            }
        }
        ss = wave_sum(ss);
        if (lane == 0) s_red[wave] = ss;
        __syncthreads();
        scale_all = 1.0f / sqrtf((s_red[0] + s_red[1] + s_red[2] + s_red[3]) / (float)K + pro.eps);
    }
#pragma unroll
    for (int u = 0; u < AV; ++u) {
        const int vi = threadIdx.x + u * 256;
        if (vi >= nvec) continue;
        T* t = reinterpret_cast<T*>(&av[u]);
        if constexpr (H2) {
            // 8 halfs = one 8-code word: one 16-byte unit in pair order.
            if constexpr (PRO) {
                const T* gm = reinterpret_cast<const T*>(&gmv[u]);
#pragma unroll
                for (int e = 0; e < EPL; ++e)
                    t[e] = from_f32<T>(to_f32(t[e]) * scale_all * to_f32(gm[e]));
            }
            reinterpret_cast<uint4*>(sA)[vi] = permute_act8(av[u]);
        } else {
            float f[EPL];
#pragma unroll
            for (int e = 0; e < EPL; ++e) f[e] = to_f32(t[e]);
            if constexpr (PRO) {
                const T* gm = reinterpret_cast<const T*>(&gmv[u]);
#pragma unroll
                for (int e = 0; e < EPL; ++e) f[e] = round_to<T>(f[e] * scale_all * to_f32(gm[e]));
            }
#pragma unroll
            for (int e = 0; e < EPL; e += 4) {
                const int q = (vi * EPL + e) / 4;
                sA[act_unit<CPL>(q)] = make_float4(f[e], f[e + 1], f[e + 2], f[e + 3]);
            }
        }
    }
    __syncthreads();
    // fp32 form: a[j][*] and asum[j]; fp16 pairs: ah[j][*] (the other form is unused).
    float a[H2 ? 1 : CPL][32];
    float asum[H2 ? 1 : CPL];
    uint4 ah[H2 ? CPL : 1][4];
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
        const int c = chunk(j);
        if constexpr (H2) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                ah[j][i] = c < C ? reinterpret_cast<const uint4*>(sA)[4 * c + i]
                                 : make_uint4(0, 0, 0, 0);
        } else {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float4 v =
                    c < C ? sA[act_unit<CPL>(8 * c + i)] : make_float4(0.f, 0.f, 0.f, 0.f);
                a[j][4 * i + 0] = v.x;
                a[j][4 * i + 1] = v.y;
                a[j][4 * i + 2] = v.z;
                a[j][4 * i + 3] = v.w;
                s += (v.x + v.y) + (v.z + v.w);
            }
            asum[j] = s * code_unit();  // in dot32_codes' scaled units (exact)
        }
    }
    // Back from dot32_codes' units: an exact power of two.
    const float code_scale = H2 ? 1.f : 1.0f / code_unit();

    auto reduce_store = [&](const Group& gr, int gi) {
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float total = 0.f;
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int blk = (32 * min(chunk(j), C - 1)) / BS;
                const int d = blk / 2 - blk0 / 2;
                uint8_t zbyte = gr.z[r][0];
                if constexpr (IL) {
                    zbyte = gr.z[r][j];
                } else {
#pragma unroll
                    for (int t = 1; t < ZB; ++t)
                        if (d == t) zbyte = gr.z[r][t];
                }
                const int zq = nibble(zbyte, blk & 1);
                if constexpr (H2) {
                    const half_t zo = (half_t)(1024 + zq);
                    const half2_t zoff = {zo, zo};
                    total = fmaf(to_f32(gr.s[r][j]), dot32_pairs(ah[j], gr.w[r][j], zoff), total);
                } else {
                    const float d32 = dot32_codes(a[j], gr.w[r][j]);
                    total = fmaf(to_f32(gr.s[r][j]), d32 - (float)zq * asum[j], total);
                }
            }
            acc[r] = total * code_scale;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = group_sum<LR>(acc[r]);
        // Every lane of a unit holds its sums and every lane stores (same-address
        // writes of a wave coalesce).
        const int unit = unit_of(gi);
        if constexpr (PAIR) {
            const float gv = round_to<T>(acc[0]), up = round_to<T>(acc[1]);
            const float sig = round_to<T>(1.0f / (1.0f + __expf(-gv)));
            Y[unit] = from_f32<T>(round_to<T>(gv * sig) * up);
            return;
        }
        const int r = li % R;
        float v = acc[0];
#pragma unroll
        for (int i = 1; i < R; ++i)
            if (r == i) v = acc[i];
        Y[min(unit * R + r, N - 1)] = from_f32<T>(v);
    };

    for (int gi = g0; gi < ngroups; gi += D * waves_total) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int idx = gi + d * waves_total;
            if (idx >= ngroups) return;
            reduce_store(g[d], idx);
            load_group(g[d], idx + D * waves_total);
        }
    }
}

// Launch of one kernel instance: `grid` workgroups of 4 waves.
template <typename T, int BS, int CPL, int R, int D, bool PRO, bool PAIR, bool SV, bool H2,
          bool NT = true, bool MRG = false, int RW = 1, bool IL = false>
static int launch_gemv4_inst(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y,
                             int N, int K, int nb, const GemvPrologue<T>& pro, long grid,
                             hipStream_t st) {
    size_t lds = gemv_stage_bytes<T, H2>(nb * BS);
    if constexpr (MRG) lds += gemv_merge_bytes(K, pro.hd, pro.splits);
    hipLaunchKernelGGL((mnb_gemv4_kernel<T, BS, CPL, R, D, PRO, PAIR, SV, H2, NT, MRG, RW, IL>),
                       dim3((unsigned)grid), dim3(256), lds, st, A, B, S, Z, Y, N, K, nb, pro);
    return check_launch("mnb_gemv4");
}

// Grid, ring depth and cache policy per shape, from sweeps on MI355X with the
// weights streamed from HBM (the decoder's N x K = 2048 x 1536, 1536 x 1536,
// 17920 x 1536 in pairs, 1536 x 8960 and 151936 x 1536 in fp16, and 11008 x 4096
// in fp32). Groups per wave: 1 while the groups fit about 10 waves per CU, 2 for
// K > 4096 fp16 (activations fill the VGPRs), about 3.6 (3 workgroups per CU) for
// K = 4096, 3 up to about 80 groups per CU, 16 beyond. A ring of 2, of 1 when
// the activations fill the VGPRs, of 4 for the long walks. Weights non-temporal
// except for those two cases, which measured faster with cached loads.
template <typename T, int BS, int CPL, bool PRO, bool PAIR, bool MRG>
static int launch_gemv4_cpl(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y,
                            int N, int K, int nb, const GemvPrologue<T>& pro, hipStream_t st) {
    constexpr int R = PAIR ? 2 : 1;
    constexpr bool H2 = std::is_same<T, half_t>::value;
    const long groups = ((long)N + R - 1) / R;
    const long cus = device_cu_count();
    const bool longwalk = groups > 80 * cus;
    long grid;
    if (longwalk) grid = (groups + 63) / 64;
    else if (CPL >= 3) grid = (groups + 7) / 8;
    // With the split-merge prologue every workgroup merges the whole activation
    // row first: fewer, fuller workgroups (o_proj 1536x1536: 384 -> 256
    // workgroups, 5.13 -> 4.87 us).
    else if (MRG && groups <= 10 * cus) grid = (groups + 5) / 6;
    else if (groups <= 10 * cus) grid = (groups + 3) / 4;
    // Three workgroups per CU: K = 4096, N = 11008 measured 8.1 us against 8.6 us at
    // four (fp32 and fp16 alike); grids that are not a multiple of the CU count
    // (2.5 or 3.5 per CU) measured slowest.
    else if (CPL >= 2) grid = std::min((groups + 3) / 4, 3 * cus);
    else grid = (groups + 11) / 12;
    bool sv = false;
    if constexpr (BS == 32 && CPL % 2 == 0)  // scale pairs as one load when every lane's pair is aligned
        sv = nb % 2 == 0 && (reinterpret_cast<uintptr_t>(S) % (2 * sizeof(T))) == 0 && nb >= 2;
    constexpr bool kSV = BS == 32 && CPL % 2 == 0;
#define ORTMI_GEMV_INST(DV, SVV, NTV)                                                              \
    return launch_gemv4_inst<T, BS, CPL, R, DV, PRO, PAIR, SVV, H2, NTV, MRG>(A, B, S, Z, Y, N, K, \
                                                                             nb, pro, grid, st)
    // Interleaved chunks (lane l owns chunks l, l + 64, ...: every weight load of a
    // row one contiguous 1 KB run) for fp16 rows of a whole number of 64-chunk runs,
    // with non-temporal loads. Measured on MI355X in graph replay against the
    // consecutive chunks: 4096 x 14336 13.4 -> 11.8 us, 3072 x 8192 9.1 -> 6.8 us,
    // 8192 x 8192 (zero points) 14.8 -> 13.3 us, 4096 x 4096 4.9 -> 4.6 us; equal at
    // 6144 and 11008 x 4096 (kept consecutive above 16 row groups per CU at two
    // chunks per lane); 1536 x 8960 (280 chunks) 5.8 -> 6.2 us, so rows with a
    // partial run keep consecutive chunks.
    const bool il = H2 && BS == 32 && nb % 64 == 0 && (CPL >= 3 || groups <= 16 * cus);
#define ORTMI_GEMV_IL(DV)                                                                         \
    return launch_gemv4_inst<T, BS, CPL, R, DV, PRO, PAIR, false, H2, true, MRG, 1, H2 && BS == 32>( \
        A, B, S, Z, Y, N, K, nb, pro, grid, st)
    if constexpr (CPL >= 6 && H2) {
        // fp16 rows of K > 10240 (6-8 chunks per lane): two rows in flight per wave
        // (Mistral-7B's down_proj 4096 x 14336: 14.3 -> 13.1 us; 16 rows per
        // workgroup instead of 8 measured 14.7 us).
        if (il) ORTMI_GEMV_IL(2);
        if (sv) ORTMI_GEMV_INST(2, kSV, false);
        ORTMI_GEMV_INST(2, false, false);
    } else if constexpr (CPL >= 3) {
        if (il) ORTMI_GEMV_IL(1);
        if (sv) ORTMI_GEMV_INST(1, kSV, false);
        ORTMI_GEMV_INST(1, false, false);
    } else {
        if (il && !longwalk) ORTMI_GEMV_IL(2);
        if (longwalk) {
            if (sv) ORTMI_GEMV_INST(4, kSV, false);
            ORTMI_GEMV_INST(4, false, false);
        }
        if (sv) ORTMI_GEMV_INST(2, kSV, true);
        ORTMI_GEMV_INST(2, false, true);
    }
#undef ORTMI_GEMV_INST
#undef ORTMI_GEMV_IL
}

template <typename T, int BS, bool PRO = false, bool PAIR = false, bool MRG = false>
static int launch_gemv4(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y, int N,
                        int K, int nb, hipStream_t st,
                        const GemvPrologue<T>& pro = GemvPrologue<T>{nullptr, nullptr, nullptr, 0.f}) {
    const int C = nb * BS / 32;
    const int cpl = (C + 63) / 64;
    if ((long)nb * BS > 2048L * (16 / (long)sizeof(T))) return -1;  // activation staging bound
    if ((size_t)N * nb * BS / 2 > 0xFFFFFF00ull) return -1;  // buffer offsets are 32-bit
    // Long walks over short rows (lm_head: 151936 x 1536): 4 rows per wave, 16
    // lanes x ceil(C/16) chunks each, so no lane idles on a 48-chunk row; cached
    // loads, ring of 2, 8 groups (32 rows) per wave: 33.6 us against 39 us with
    // a row per wave.
    constexpr int R = PAIR ? 2 : 1;
    const long units = ((long)N + R - 1) / R;
    if (units > 80L * device_cu_count() && C <= 48) {
        constexpr bool H2 = std::is_same<T, half_t>::value;
        const long grid = (units + 127) / 128;  // 4 waves x 32 rows per workgroup
        switch ((C + 15) / 16) {
            case 1: return launch_gemv4_inst<T, BS, 1, R, 2, PRO, PAIR, false, H2, false, MRG, 4>(
                        A, B, S, Z, Y, N, K, nb, pro, grid, st);
            case 2: return launch_gemv4_inst<T, BS, 2, R, 2, PRO, PAIR, false, H2, false, MRG, 4>(
                        A, B, S, Z, Y, N, K, nb, pro, grid, st);
            default: return launch_gemv4_inst<T, BS, 3, R, 2, PRO, PAIR, false, H2, false, MRG, 4>(
                        A, B, S, Z, Y, N, K, nb, pro, grid, st);
        }
    }
    switch (cpl) {
        case 1: return launch_gemv4_cpl<T, BS, 1, PRO, PAIR, MRG>(A, B, S, Z, Y, N, K, nb, pro, st);
        case 2: return launch_gemv4_cpl<T, BS, 2, PRO, PAIR, MRG>(A, B, S, Z, Y, N, K, nb, pro, st);
        case 3: return launch_gemv4_cpl<T, BS, 3, PRO, PAIR, MRG>(A, B, S, Z, Y, N, K, nb, pro, st);
        case 4: return launch_gemv4_cpl<T, BS, 4, PRO, PAIR, MRG>(A, B, S, Z, Y, N, K, nb, pro, st);
        case 5: return launch_gemv4_cpl<T, BS, 5, PRO, PAIR, MRG>(A, B, S, Z, Y, N, K, nb, pro, st);
        default: break;
    }
    // fp16 activations held as pairs (16 VGPRs per chunk) also take K up to 16384
    // (the down_proj of 7B-class decoders, K = 11008 or 14336); fp32 and bf16 hold
    // 32 VGPRs per chunk and stop at 10240.
    if constexpr (std::is_same<T, half_t>::value) {
        switch (cpl) {
            case 6: return launch_gemv4_cpl<T, BS, 6, PRO, PAIR, MRG>(A, B, S, Z, Y, N, K, nb, pro, st);
            case 7: return launch_gemv4_cpl<T, BS, 7, PRO, PAIR, MRG>(A, B, S, Z, Y, N, K, nb, pro, st);
            case 8: return launch_gemv4_cpl<T, BS, 8, PRO, PAIR, MRG>(A, B, S, Z, Y, N, K, nb, pro, st);
            default: break;
        }
    }
    return -1;  // the caller falls back
}

// ----------------------------------------------------------------- generic --

// Any bits/block/dtype: 64x64 output tile, 256 threads, 4x4 outputs per thread,
// fp32 dequantisation of a 64x32 weight tile into LDS.
template <typename T>
__global__ __launch_bounds__(256) void mnb_generic_kernel(const T* __restrict__ A,
                                                          const uint8_t* __restrict__ B,
                                                          const T* __restrict__ S,
                                                          const uint8_t* __restrict__ Z,
                                                          T* __restrict__ Y, int M, int N, int K,
                                                          int nb, int bits, int bs) {
    __shared__ float sA[64][33];
    __shared__ float sW[64][33];
    const int tid = threadIdx.x;
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    const int tr = tid / 16, tc = tid % 16;
    const size_t blob = (size_t)bs * bits / 8;
    const int zp_cols = bits == 4 ? (nb + 1) / 2 : nb;
    const int zdef = 1 << (bits - 1);
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += 32) {
        for (int i = tid; i < 64 * 32; i += 256) {
            const int r = i / 32, c = i % 32;
            const int m = m0 + r, k = k0 + c;
            sA[r][c] = (m < M && k < K) ? to_f32(A[(size_t)m * K + k]) : 0.f;
            const int n = n0 + r;
            float wv = 0.f;
            if (n < N && k < K) {
                const int blk = k / bs, within = k % bs;
                int q, z;
                if (bits == 4) {
                    const uint8_t byte = B[((size_t)n * nb + blk) * blob + within / 2];
                    q = nibble(byte, within & 1);
                    z = Z ? nibble(Z[(size_t)n * zp_cols + blk / 2], blk & 1) : zdef;
                } else {
                    q = B[((size_t)n * nb + blk) * blob + within];
                    z = Z ? Z[(size_t)n * zp_cols + blk] : zdef;
                }
                wv = (float)(q - z) * to_f32(S[(size_t)n * nb + blk]);
            }
            sW[r][c] = wv;
        }
        __syncthreads();
#pragma unroll 8
        for (int kk = 0; kk < 32; ++kk) {
            float av[4], wv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = sA[tr * 4 + i][kk];
#pragma unroll
            for (int j = 0; j < 4; ++j) wv[j] = sW[tc * 4 + j][kk];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int m = m0 + tr * 4 + i, n = n0 + tc * 4 + j;
            if (m < M && n < N) Y[(size_t)m * N + n] = from_f32<T>(acc[i][j]);
        }
}

template <typename T>
static int launch_generic(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y, int M,
                          int N, int K, int nb, int bits, int bs, hipStream_t st) {
    dim3 grid((N + 63) / 64, (M + 63) / 64);
    hipLaunchKernelGGL((mnb_generic_kernel<T>), grid, dim3(256), 0, st, A, B, S, Z, Y, M, N, K, nb,
                       bits, bs);
    return check_launch("mnb_generic");
}

template <typename T>
static int run_mnb(const void* A, const uint8_t* B, const void* S, const uint8_t* Z, void* Y,
                   int M, int N, int K, int bits, int bs, hipStream_t st) {
    const int nb = (K + bs - 1) / bs;
    const T* a = static_cast<const T*>(A);
    const T* s = static_cast<const T*>(S);
    T* y = static_cast<T*>(Y);
    const bool aligned = (reinterpret_cast<uintptr_t>(B) % 16) == 0;
    const bool fast_form = bits == 4 && (bs == 32 || bs == 64 || bs == 128) && aligned;
    const size_t kmax = std::is_same<T, half_t>::value ? 16384 : 10240;
    if (fast_form && M == 1 && (size_t)nb * bs <= kmax) {
        int rc = -1;
        if (bs == 32) rc = launch_gemv4<T, 32>(a, B, s, Z, y, N, K, nb, st);
        if (bs == 64) rc = launch_gemv4<T, 64>(a, B, s, Z, y, N, K, nb, st);
        if (bs == 128) rc = launch_gemv4<T, 128>(a, B, s, Z, y, N, K, nb, st);
        if (rc >= 0) return rc;
    }
    // The prefill GEMM's forms: fp16 and bf16, 32-bit buffer offsets.
    const bool gemm_form = sizeof(T) == 2 && fast_form && M > 1 &&
                           (reinterpret_cast<uintptr_t>(A) % 16) == 0 && K % 8 == 0 &&
                           (size_t)M * K * 2 <= 0xFFFFFF00ull &&
                           (size_t)N * nb * bs / 2 <= 0xFFFFFF00ull;
    if (!gemm_form || mnb_takes_blk(M, N)) {
        const int rc = bits == 4 ? mnb_blk<T, 4>(a, B, s, Z, y, M, N, K, bs, st)
                                 : mnb_blk<T, 8>(a, B, s, Z, y, M, N, K, bs, st);
        if (rc >= 0) return rc;
    }
    if constexpr (sizeof(T) == 2) {
        if (gemm_form) return mnb_gemm<T>(a, B, s, Z, y, M, N, K, bs, st);
    }
    return launch_generic<T>(a, B, s, Z, y, M, N, K, nb, bits, bs, st);
}

}  // namespace ortmi

using namespace ortmi;

namespace ortmi {
template <typename T, bool PRO, bool PAIR>
static int run_fused_gemv(const void* x, const void* skip, const void* gamma, float eps,
                          void* residual, const uint8_t* B, const void* S, const uint8_t* Z,
                          void* Y, int N, int K, int bs, hipStream_t st) {
    const int nb = (K + bs - 1) / bs;
    GemvPrologue<T> pro{static_cast<const T*>(skip), static_cast<const T*>(gamma),
                        static_cast<T*>(residual), eps};
    const T* a = static_cast<const T*>(x);
    const T* s = static_cast<const T*>(S);
    T* y = static_cast<T*>(Y);
    if (bs == 32) return launch_gemv4<T, 32, PRO, PAIR>(a, B, s, Z, y, N, K, nb, st, pro);
    if (bs == 64) return launch_gemv4<T, 64, PRO, PAIR>(a, B, s, Z, y, N, K, nb, st, pro);
    return launch_gemv4<T, 128, PRO, PAIR>(a, B, s, Z, y, N, K, nb, st, pro);
}

template <typename T>
static int dispatch_fused_gemv(const void* x, const void* skip, const void* gamma, float eps,
                               void* residual, const uint8_t* B, const void* S,
                               const uint8_t* Z, void* Y, int N, int K, int bs, bool norm,
                               bool pair, hipStream_t st) {
    if (norm && pair)
        return run_fused_gemv<T, true, true>(x, skip, gamma, eps, residual, B, S, Z, Y, N, K, bs, st);
    if (norm)
        return run_fused_gemv<T, true, false>(x, skip, gamma, eps, residual, B, S, Z, Y, N, K, bs, st);
    if (pair)
        return run_fused_gemv<T, false, true>(x, skip, gamma, eps, residual, B, S, Z, Y, N, K, bs, st);
    return run_fused_gemv<T, false, false>(x, skip, gamma, eps, residual, B, S, Z, Y, N, K, bs, st);
}
}  // namespace ortmi

extern "C" int ortmi_matmul_nbits_decode_fused(const void* x, const void* skip, const void* gamma,
                                               float epsilon, void* residual, const uint8_t* B,
                                               const void* scales, const uint8_t* zero_points,
                                               void* Y, int64_t N, int64_t K, int64_t block_size,
                                               int32_t flags, int32_t dtype, void* stream) {
    const bool norm = (flags & ORTMI_FUSE_RMS_NORM) != 0;
    const bool pair = (flags & ORTMI_FUSE_SWIGLU_PAIRS) != 0;
    ORTMI_REQUIRE((flags & ~(ORTMI_FUSE_RMS_NORM | ORTMI_FUSE_SWIGLU_PAIRS)) == 0,
                  "MatMulNBits fused: unknown flags");
    ORTMI_REQUIRE(block_size == 32 || block_size == 64 || block_size == 128,
                  "MatMulNBits fused: block_size must be 32, 64 or 128");
    ORTMI_REQUIRE(N > 0 && K > 0 && N < (1LL << 31), "MatMulNBits fused: bad shape");
    ORTMI_REQUIRE(!pair || N % 2 == 0, "MatMulNBits fused: SwiGLU pairs need an even N");
    ORTMI_REQUIRE(x && B && scales && Y, "MatMulNBits fused: null tensor");
    ORTMI_REQUIRE(!norm || gamma, "MatMulNBits fused: the norm needs gamma");
    ORTMI_REQUIRE(!residual || (norm && skip), "MatMulNBits fused: residual needs the skip norm");
    ORTMI_REQUIRE((reinterpret_cast<uintptr_t>(B) & 15) == 0,
                  "MatMulNBits fused: B must be 16-byte aligned");
    const int64_t nb = (K + block_size - 1) / block_size;
    const int64_t limit = 2048LL * (dtype == ORTMI_F32 ? 4 : 8);
    ORTMI_REQUIRE(nb * block_size <= std::min<int64_t>(limit, dtype == ORTMI_F16 ? 16384 : 10240),
                  "MatMulNBits fused: K too large for the decode kernel");
    hipStream_t st = as_stream(stream);
    int rc;
    switch (dtype) {
        case ORTMI_F16:
            rc = dispatch_fused_gemv<half_t>(x, skip, gamma, epsilon, residual, B, scales,
                                             zero_points, Y, (int)N, (int)K, (int)block_size, norm,
                                             pair, st);
            break;
        case ORTMI_BF16:
            rc = dispatch_fused_gemv<uint16_t>(x, skip, gamma, epsilon, residual, B, scales,
                                               zero_points, Y, (int)N, (int)K, (int)block_size,
                                               norm, pair, st);
            break;
        default:
            return fail(ORTMI_E_INVALID, "MatMulNBits fused: fp16 or bf16 activations only");
    }
    // The launcher declines shapes beyond its staging or 32-bit buffer range.
    if (rc < 0) return fail(ORTMI_E_INVALID, "MatMulNBits fused: shape has no decode kernel");
    return rc;
}

namespace ortmi {
template <typename T>
static int run_merge_gemv(const float* part, int splits, int hd, const uint8_t* B, const void* S,
                          const uint8_t* Z, void* Y, int N, int K, int bs, hipStream_t st) {
    const int nb = (K + bs - 1) / bs;
    GemvPrologue<T> pro{nullptr, nullptr, nullptr, 0.f, part, splits, hd};
    const T* s = static_cast<const T*>(S);
    T* y = static_cast<T*>(Y);
    if (bs == 32) return launch_gemv4<T, 32, false, false, true>(nullptr, B, s, Z, y, N, K, nb, st, pro);
    if (bs == 64) return launch_gemv4<T, 64, false, false, true>(nullptr, B, s, Z, y, N, K, nb, st, pro);
    return launch_gemv4<T, 128, false, false, true>(nullptr, B, s, Z, y, N, K, nb, st, pro);
}
}  // namespace ortmi

extern "C" int ortmi_matmul_nbits_decode_merge(const float* partials, int64_t splits,
                                               int64_t head_size, const uint8_t* B,
                                               const void* scales, const uint8_t* zero_points,
                                               void* Y, int64_t N, int64_t K, int64_t block_size,
                                               int32_t dtype, void* stream) {
    ORTMI_REQUIRE(partials && B && scales && Y, "MatMulNBits merge: null tensor");
    ORTMI_REQUIRE(splits >= 1 && splits <= 4096, "MatMulNBits merge: bad split count");
    ORTMI_REQUIRE(head_size == 64 || head_size == 128,
                  "MatMulNBits merge: head_size must be 64 or 128");
    ORTMI_REQUIRE(K > 0 && K % head_size == 0 && N > 0 && N < (1LL << 31),
                  "MatMulNBits merge: K must be a whole number of heads");
    ORTMI_REQUIRE(block_size == 32 || block_size == 64 || block_size == 128,
                  "MatMulNBits merge: block_size must be 32, 64 or 128");
    ORTMI_REQUIRE((reinterpret_cast<uintptr_t>(B) & 15) == 0,
                  "MatMulNBits merge: B must be 16-byte aligned");
    const int64_t nb = (K + block_size - 1) / block_size;
    ORTMI_REQUIRE(nb * block_size <= 10240, "MatMulNBits merge: K too large for the decode kernel");
    ORTMI_REQUIRE((reinterpret_cast<uintptr_t>(partials) & 15) == 0,
                  "MatMulNBits merge: partials must be 16-byte aligned");
    const size_t stage = (size_t)nb * block_size * (dtype == ORTMI_F16 ? 2 : 4);
    if ((K / head_size) * splits * (head_size + 2) > kDecodeMergeMaxFloats ||
        gemv_merge_bytes((int)K, (int)head_size, (int)splits) + stage > 65536)
        return fail(ORTMI_E_INVALID, "MatMulNBits merge: too many split partials for one workgroup");
    hipStream_t st = as_stream(stream);
    int rc = -1;
    if (dtype == ORTMI_F16)
        rc = run_merge_gemv<half_t>(partials, (int)splits, (int)head_size, B, scales, zero_points,
                                    Y, (int)N, (int)K, (int)block_size, st);
    else if (dtype == ORTMI_BF16)
        rc = run_merge_gemv<uint16_t>(partials, (int)splits, (int)head_size, B, scales,
                                      zero_points, Y, (int)N, (int)K, (int)block_size, st);
    else
        return fail(ORTMI_E_INVALID, "MatMulNBits merge: fp16 or bf16 activations only");
    if (rc < 0) return fail(ORTMI_E_INVALID, "MatMulNBits merge: shape has no decode kernel");
    return rc;
}

extern "C" int ortmi_matmul_nbits_swiglu_pairs(const void* A, const uint8_t* B,
                                               const void* scales, const uint8_t* zero_points,
                                               void* Y, int64_t M, int64_t N, int64_t K,
                                               int64_t block_size, int32_t dtype, void* stream) {
    ORTMI_REQUIRE(M >= 0 && N >= 0 && K > 0 && N % 2 == 0 && M < (1LL << 31) &&
                      N < (1LL << 31) && K < (1LL << 31),
                  "MatMulNBits SwiGLU pairs: bad shape (N must be even)");
    if (M == 0 || N == 0) return ORTMI_OK;
    ORTMI_REQUIRE(A && B && scales && Y, "MatMulNBits SwiGLU pairs: null tensor");
    const int nb = (int)((K + block_size - 1) / block_size);
    const bool ok = dtype == ORTMI_F16 && (block_size == 32 || block_size == 64 ||
                                           block_size == 128) &&
                    (reinterpret_cast<uintptr_t>(B) % 16) == 0 &&
                    (reinterpret_cast<uintptr_t>(A) % 16) == 0 && K % 8 == 0 &&
                    (size_t)M * K * 2 <= 0xFFFFFF00ull &&
                    (size_t)N * nb * block_size / 2 <= 0xFFFFFF00ull;
    if (!ok)
        return fail(ORTMI_E_INVALID,
                    "MatMulNBits SwiGLU pairs: needs fp16, 4-bit block 32/64/128, 16-byte "
                    "aligned A and B, K % 8 == 0");
    const half_t* a = static_cast<const half_t*>(A);
    const half_t* s = static_cast<const half_t*>(scales);
    half_t* y = static_cast<half_t*>(Y);
    hipStream_t st = as_stream(stream);
    const int m = (int)M, n = (int)N, k = (int)K;
    if (m > 1 && mnb_takes_blk(m, n)) {  // the rule of ortmi_matmul_nbits: the same sums
        const int rc = mnb_blk<half_t, 4, true>(a, B, s, zero_points, y, m, n, k, (int)block_size, st);
        if (rc >= 0) return rc;
    }
    return mnb_gemm<half_t, true>(a, B, s, zero_points, y, m, n, k, (int)block_size, st);
}

extern "C" int ortmi_matmul_nbits(const void* A, const uint8_t* B, const void* scales,
                                  const uint8_t* zero_points, void* Y, int64_t M, int64_t N,
                                  int64_t K, int64_t bits, int64_t block_size, int32_t dtype,
                                  void* stream) {
    // Claim contract of rust/src/ops/quant.rs:1655-1711 plus shape checks.
    ORTMI_REQUIRE(bits == 4 || bits == 8, "MatMulNBits: only 4-bit and 8-bit weights are supported");
    ORTMI_REQUIRE(block_size == 16 || block_size == 32 || block_size == 64 || block_size == 128,
                  "MatMulNBits: block_size must be 16, 32, 64, or 128");
    ORTMI_REQUIRE(M >= 0 && N >= 0 && K >= 0, "MatMulNBits: negative dimension");
    ORTMI_REQUIRE(M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31),
                  "MatMulNBits: dimension too large");
    if (M == 0 || N == 0) return ORTMI_OK;
    ORTMI_REQUIRE(K > 0, "MatMulNBits: K must be positive");
    ORTMI_REQUIRE(A && B && scales && Y, "MatMulNBits: null tensor");
    hipStream_t st = as_stream(stream);
    switch (dtype) {
        case ORTMI_F32:
            return run_mnb<float>(A, B, scales, zero_points, Y, (int)M, (int)N, (int)K, (int)bits,
                                  (int)block_size, st);
        case ORTMI_F16:
            return run_mnb<half_t>(A, B, scales, zero_points, Y, (int)M, (int)N, (int)K, (int)bits,
                                   (int)block_size, st);
        case ORTMI_BF16:
            return run_mnb<uint16_t>(A, B, scales, zero_points, Y, (int)M, (int)N, (int)K,
                                     (int)bits, (int)block_size, st);
        default:
            return fail(ORTMI_E_INVALID,
                        "MatMulNBits: activation/scales must be float (fp32/fp16/bf16)");
    }
}

// --------------------------------------------------- GatherBlockQuantized --

namespace ortmi {

// Rows of an int4 block-quantised table gathered by index: data [V, D/2] (two
// codes per byte, low nibble first, the MatMulNBits row layout), scales
// [V, ceil(D/block)], optional packed zero points [V, ceil(nblocks/2)] (low nibble
// = even block; 8 when absent). out[i, k] = (q - zp) * scale in fp32, rounded
// once to the output type. One thread per data byte (two codes); an index outside
// [-V, V) yields a zero row (the host reports no error from device data).
template <typename T, typename I>
__global__ void gbq_kernel(const uint8_t* __restrict__ data, const T* __restrict__ scales,
                           const uint8_t* __restrict__ zp, const I* __restrict__ idx,
                           T* __restrict__ out, int64_t n_idx, int64_t V, int D, int block) {
    const int bytes = D / 2;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_idx * bytes) return;
    const int64_t i = t / bytes;
    const int j = (int)(t % bytes);
    int64_t row = (int64_t)idx[i];
    if (row < 0) row += V;
    const bool ok = row >= 0 && row < V;
    const int nb = (D + block - 1) / block;
    const int zcols = (nb + 1) / 2;
    float v[2] = {0.f, 0.f};
    if (ok) {
        const uint8_t b = data[row * bytes + j];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = 2 * j + h;
            const int blk = k / block;
            const float s = to_f32(scales[row * nb + blk]);
            const int z = zp ? nibble(zp[row * zcols + blk / 2], blk & 1) : 8;
            v[h] = (float)(nibble(b, h) - z) * s;
        }
    }
    out[i * D + 2 * j] = from_f32<T>(v[0]);
    out[i * D + 2 * j + 1] = from_f32<T>(v[1]);
}

template <typename T>
static int launch_gbq(const uint8_t* data, const void* scales, const uint8_t* zp,
                      const void* idx, int idx_is_i64, void* out, int64_t n_idx, int64_t V,
                      int64_t D, int64_t block, hipStream_t st) {
    const int64_t threads = n_idx * (D / 2);
    if (threads == 0) return ORTMI_OK;
    const unsigned grid = (unsigned)((threads + 255) / 256);
    if (idx_is_i64)
        hipLaunchKernelGGL((gbq_kernel<T, int64_t>), dim3(grid), dim3(256), 0, st, data,
                           static_cast<const T*>(scales), zp, static_cast<const int64_t*>(idx),
                           static_cast<T*>(out), n_idx, V, (int)D, (int)block);
    else
        hipLaunchKernelGGL((gbq_kernel<T, int32_t>), dim3(grid), dim3(256), 0, st, data,
                           static_cast<const T*>(scales), zp, static_cast<const int32_t*>(idx),
                           static_cast<T*>(out), n_idx, V, (int)D, (int)block);
    return check_launch("gather_block_quantized");
}

}  // namespace ortmi

extern "C" int ortmi_gather_block_quantized(const uint8_t* data, const void* scales,
                                            const uint8_t* zero_points, const void* indices,
                                            int32_t indices_are_int64, void* output,
                                            int64_t num_indices, int64_t rows, int64_t D,
                                            int64_t block_size, int64_t bits, int32_t dtype,
                                            void* stream) {
    // Claim contract of rust/src/ops/quant.rs:1713-1749: 4-bit codes, gather axis 0,
    // quantize axis 1, block >= 16; data/zero points uint8, scales = output dtype.
    ORTMI_REQUIRE(bits == 4, "GatherBlockQuantized: only 4-bit data is supported");
    ORTMI_REQUIRE(block_size >= 16, "GatherBlockQuantized: block_size must be at least 16");
    ORTMI_REQUIRE(num_indices >= 0 && rows > 0 && D > 0 && D % 2 == 0 && D < (1LL << 30),
                  "GatherBlockQuantized: bad shape");
    ORTMI_REQUIRE(num_indices == 0 || (data && scales && indices && output),
                  "GatherBlockQuantized: null tensor");
    hipStream_t st = as_stream(stream);
    switch (dtype) {
        case ORTMI_F32:
            return launch_gbq<float>(data, scales, zero_points, indices, indices_are_int64, output,
                                     num_indices, rows, D, block_size, st);
        case ORTMI_F16:
            return launch_gbq<half_t>(data, scales, zero_points, indices, indices_are_int64,
                                      output, num_indices, rows, D, block_size, st);
        case ORTMI_BF16:
            return launch_gbq<uint16_t>(data, scales, zero_points, indices, indices_are_int64,
                                        output, num_indices, rows, D, block_size, st);
        default:
            return fail(ORTMI_E_INVALID, "GatherBlockQuantized: scales must be fp32, fp16 or bf16");
    }
}
