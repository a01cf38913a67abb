// MatMulNBits on the matrix cores without a shared weight tile, for gfx950: small
// batches of 4-bit weights, and every shape of 8-bit weights and of fp32 activations
// (blocks of 32, 64 or 128).
//
// 4-bit weights with fp16 or bf16 activations of more than one row are dequantised to the
// activation type ((q - zp) * s, one rounding), the weights the prefill GEMM multiplies. In
// the other forms, and for a single row (K past the GEMV's, whose weights are not rounded
// either), no weight is rounded: the codes enter the matrix cores as whole numbers
// (q - zp), exact in fp16 and (up to a power of two) in bf16, v_mfma 16x16x32 sums the
// 32 products of one chunk in fp32, and the chunk's sum takes its block's scale in
// fp32. fp32 activations are split into three bf16 pieces of 8 mantissa bits each,
// whose products with the codes are exact: three matrix steps carry the whole 24-bit
// mantissa. Error against 64-bit arithmetic: 5.3e-7 relative at 512 x 896 x 1152 fp32
// with the VALU tile product these forms took before, 1.3e-7 here.
//
// Bound: the weight stream and, from about 16 rows, the dequantisation (about 17
// vector instructions per 8 codes). Measured on MI355X, before (VALU tile product, or
// the prefill GEMM's tiles for 4-bit fp16) and now: one row of 3072 x 32064 8-bit 497
// -> 23.6 us (4.4 TB/s), 8 rows of 4096 x 14336 4-bit 21.7 -> 11.5 us (2.9 TB/s), 512
// x 896 x 1152 fp32 185 -> 14.8 us, 512 x 4096 x 4096 fp32 866 -> 98 us.
#include <algorithm>

#include "common.h"
#include "mnb_internal.h"

namespace ortmi {
namespace {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

struct U32Pair {
    uint32_t a, b;
};
__device__ __forceinline__ U32Pair swap16u(uint32_t x, uint32_t y) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    return {(uint32_t)r[0], (uint32_t)r[1]};
}
__device__ __forceinline__ U32Pair swap32u(uint32_t x, uint32_t y) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    return {(uint32_t)r[0], (uint32_t)r[1]};
}

// The pieces of an activation vector: 1 (fp16, bf16) or 3 (fp32).
template <typename T>
constexpr int blk_pieces() { return sizeof(T) == 4 ? 3 : 1; }

// Forms with dequantised weights (one rounding to T) instead of whole codes, at M > 1.
template <typename T, int BITS>
constexpr bool blk_scaled() { return sizeof(T) == 2 && BITS == 4; }

// A code enters bf16 operands as (q - zp) times this power of two (exact), so that a
// chunk's 32 products sum to no more than the largest activation: no overflow that
// the scaled weights would not have had. The sums stay in this unit to the end, where
// the scale of no block can overflow either. fp16 sums cannot overflow fp32.
template <typename T, int BITS, bool SC>
constexpr float blk_unit() {
    if (std::is_same<T, half_t>::value || SC) return 1.f;
    return BITS == 4 ? 1.f / 512.f : 1.f / 8192.f;
}

template <typename T>
__device__ __forceinline__ float4_t blk_mfma(u32x4_t a, u32x4_t b, float4_t c) {
    if constexpr (std::is_same<T, half_t>::value)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a),
                                                      __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// The high halves of two fp32 words as one bf16 pair (truncation; exact where the
// low halves are zero).
__device__ __forceinline__ uint32_t high_halves(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// 8 codes of 4 bits as 8 weights (q - zp) * s rounded once to T. fp16 comes in pair
// order (0,4) (1,5) (2,6) (3,7), the activations permuted alike: (1024 + q) -
// (1024 + zp) is exact, the product rounds. bf16 comes in order: a byte 0000qqqq read
// as fp8 (e4m3) is q * 2^-9 exactly, the convert's scale makes it q, and both products of
// the fused multiply-add are exact in fp32, so only the conversion rounds.
template <typename T>
__device__ __forceinline__ u32x4_t scaled_codes(uint32_t w, uint32_t zp, uint32_t sbits,
                                                uint32_t magic) {
    u32x4_t r;
    if constexpr (std::is_same<T, half_t>::value) {
        const half_t zo = __builtin_bit_cast(half_t, (uint16_t)(0x6400u | zp));  // 1024 + zp
        const half_t sh = __builtin_bit_cast(half_t, (uint16_t)sbits);
        const half2_t z2 = {zo, zo}, s2 = {sh, sh};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t m = ((w >> (4 * j)) & 0x000F000Fu) | magic;
            r[j] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(half2_t, m) - z2) * s2);
        }
    } else {
        const float s = to_f32((uint16_t)sbits), zo = -(float)zp * s;
        const uint32_t ev = w & 0x0F0F0F0Fu, od = (w >> 4) & 0x0F0F0F0Fu;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const auto e = h ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8((int)ev, 512.f, true)
                             : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8((int)ev, 512.f, false);
            const auto o = h ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8((int)od, 512.f, true)
                             : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8((int)od, 512.f, false);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const bf16x2_t v = {(__bf16)fmaf(e[i], s, zo), (__bf16)fmaf(o[i], s, zo)};
                r[2 * h + i] = __builtin_bit_cast(uint32_t, v);
            }
        }
    }
    return r;
}

// 8 codes as the 8 operand halves (q - zp) * blk_unit, in order; 4-bit codes of fp16 in the
// pair order of scaled_codes.
template <typename T, int BITS>
__device__ __forceinline__ u32x4_t blk_codes(uint32_t w0, uint32_t w1, uint32_t zp) {
    u32x4_t r;
    if constexpr (std::is_same<T, half_t>::value) {
        const half_t zo = __builtin_bit_cast(half_t, (uint16_t)(0x6400u | zp));
        const half2_t z2 = {zo, zo};
        const uint32_t w[2] = {w0, w1};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t m = BITS == 4 ? ((w0 >> (4 * j)) & 0x000F000Fu) | 0x64006400u
                                         : __builtin_amdgcn_perm(0x64646464u, w[j / 2],
                                                                 j % 2 ? 0x04030402u : 0x04010400u);
            r[j] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, m) - z2);
        }
    } else if constexpr (BITS == 4) {
        const float zo = (float)zp * (1.f / 512.f);
        const uint32_t ev = w0 & 0x0F0F0F0Fu, od = (w0 >> 4) & 0x0F0F0F0Fu;
        const auto e01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)ev, false);
        const auto e23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)ev, true);
        const auto o01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)od, false);
        const auto o23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)od, true);
        r[0] = high_halves(e01[0] - zo, o01[0] - zo);
        r[1] = high_halves(e01[1] - zo, o01[1] - zo);
        r[2] = high_halves(e23[0] - zo, o23[0] - zo);
        r[3] = high_halves(e23[1] - zo, o23[1] - zo);
    } else {
        constexpr float u = 1.f / 8192.f;
        const float zo = -(float)zp * u;
        const uint32_t w[2] = {w0, w1};
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float f0 = fmaf((float)(w[j] & 0xffu), u, zo);
            const float f1 = fmaf((float)((w[j] >> 8) & 0xffu), u, zo);
            const float f2 = fmaf((float)((w[j] >> 16) & 0xffu), u, zo);
            const float f3 = fmaf((float)(w[j] >> 24), u, zo);
            r[2 * j] = high_halves(f0, f1);
            r[2 * j + 1] = high_halves(f2, f3);
        }
    }
    return r;
}

// An activation vector of 8 as matrix operands: fp16 (4-bit) in the codes' pair
// order; bf16 as is; fp32 as three bf16 pieces: the high 16 bits, the high 16 bits
// of the exact remainder, and the rest (8 bits each). The remainder of an infinity
// would be NaN: it is held to a finite value (below any overflow, above every real
// remainder), so an infinity stays one, and a NaN without payload in its high half turns
// into one (the kernel's end sees to those).
template <typename T, int BITS>
__device__ __forceinline__ void blk_acts(const u32x4_t* raw, u32x4_t* op) {
    if constexpr (sizeof(T) == 4) {
        constexpr float lim = 0x1p122f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float lo[2], hi[2];
            uint32_t x[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                x[e] = raw[j / 2][(j % 2) * 2 + e];
                const float h = __uint_as_float(x[e] & 0xffff0000u);
                hi[e] = __builtin_amdgcn_fmed3f(__uint_as_float(x[e]) - h, -lim, lim);
                lo[e] = hi[e] - __uint_as_float(__float_as_uint(hi[e]) & 0xffff0000u);
            }
            op[0][j] = __builtin_amdgcn_perm(x[1], x[0], 0x07060302u);
            op[1][j] = high_halves(hi[0], hi[1]);
            op[2][j] = high_halves(lo[0], lo[1]);
        }
    } else if constexpr (std::is_same<T, half_t>::value && BITS == 4) {
        op[0] = u32x4_t{__builtin_amdgcn_perm(raw[0][2], raw[0][0], 0x05040100u),
                        __builtin_amdgcn_perm(raw[0][2], raw[0][0], 0x07060302u),
                        __builtin_amdgcn_perm(raw[0][3], raw[0][1], 0x05040100u),
                        __builtin_amdgcn_perm(raw[0][3], raw[0][1], 0x07060302u)};
    } else {
        op[0] = raw[0];
    }
}

// One step of a wave: 128 (4-bit) or 64 (8-bit) codes of its columns, with the
// activations of its rows. A step's activations go through LDS in SUB parts of PPR
// 16-byte pieces per row (fp32 rows of 128 in two halves).
template <typename T, int BITS, int MT, int NT>
struct BlkStage {
    static constexpr int CH = BITS == 4 ? 4 : 2;  // 32-code chunks per step
    static constexpr int KSTEP = 32 * CH;
    static constexpr int SUB = sizeof(T) == 4 && BITS == 4 ? 2 : 1;
    static constexpr int PPR = KSTEP / SUB * (int)sizeof(T) / 16;
    static constexpr int AI = 16 * PPR / 64;  // vectors per lane, row tile and part
    static constexpr int WAVE_LDS = NT * 1024 + MT * 16 * PPR * 16;
    u32x4_t b[NT];
    u32x4_t a[SUB][MT][AI];
};

// LDS of a workgroup: the waves' exchange regions (reused for the final sum), then
// the tile's scales and zero points as they lie in memory, 16-byte units permuted
// inside groups of 16 (a row of the image is often a multiple of 256 bytes, which
// would put a column's entry of every row in one bank).
__device__ __host__ constexpr uint32_t image_bytes(uint32_t n) { return ((n + 255) & ~255u) + 256; }
__device__ __forceinline__ uint32_t image_at(uint32_t x) { return x ^ ((x >> 4) & 0xF0u); }
template <typename T, int BITS, int MT, int NT, int NW>
constexpr uint32_t blk_fixed_lds() {
    return (uint32_t)NW * (uint32_t)std::max(BlkStage<T, BITS, MT, NT>::WAVE_LDS, MT * NT * 1024);
}
template <typename T, int BITS, int MT, int NT, int NW>
uint32_t blk_lds(int nb) {
    const uint32_t zc = BITS == 4 ? (nb + 1) / 2 : nb;
    return blk_fixed_lds<T, BITS, MT, NT, NW>() + image_bytes(16u * NT * nb * (uint32_t)sizeof(T)) +
           image_bytes(16u * NT * zc);
}

// A workgroup owns a tile of 16*MT rows by 16*NT columns; its NW waves split K
// between them (steps dealt round-robin, so that the lines of weights that
// neighbouring steps share are wanted at the same time), each streaming its own
// weights and activations into registers a step ahead and no barrier until the end, where the
// partial tiles are summed through LDS in wave order.
//
// Matrix layout (16x16x32): lane l holds column (or row) l & 15 and the eight k of
// group g = l >> 4; accumulator e is row 4g + e of column l & 15. Loaded in that
// layout, neighbouring lanes would read different rows: the address unit took about a
// cycle per lane (M = 2, 4096 x 14336, fp16: 19.0 us). So four neighbouring lanes
// load 64 contiguous bytes (of a column; a whole row part of the activations), and
// each wave passes what it loaded through an LDS region of its own (same-wave LDS
// accesses stay in order: no workgroup barrier). The scales and zero points of the tile, a few
// bytes per column and step, are copied to LDS whole before the first step.
//
// Lane (column, g) then reads chunk 4s + g (4-bit) or half chunk 4s + g (8-bit) of its
// column. Dequantised weights (SC) need no exchange: matrix step c takes word
// c of every group's own chunk and the activations at the same k. Whole codes must be
// summed a chunk at a time: row swaps (v_permlane16/32_swap) give every lane group
// its eight codes of each chunk in turn, so that one matrix step covers exactly one
// chunk and its sum can take one scale; the chunk's scale and zero point are spread
// to all groups the same way.
template <typename T, int BITS, int MT, int NT, int NW, bool SWI, bool SC>
__global__ __launch_bounds__(64 * NW, 2) void mnb_blk_kernel(
    const T* __restrict__ A, const uint8_t* __restrict__ B, const T* __restrict__ S,
    const uint8_t* __restrict__ Z, T* __restrict__ Y, int M, int N, int K, int nb, int bshift,
    int tiles_m, int tiles_n) {
    using Stage = BlkStage<T, BITS, MT, NT>;
    constexpr int CH = Stage::CH, P = blk_pieces<T>(), SUB = Stage::SUB, PPR = Stage::PPR,
                  AI = Stage::AI, KSTEP = Stage::KSTEP, KSUB = KSTEP / SUB;
    extern __shared__ uint4 blk_smem[];
    uint8_t* const smem = reinterpret_cast<uint8_t*>(blk_smem);

    // Tiles sharing weight columns (m fastest) stay on one XCD where the grid divides.
    const int nwg = gridDim.x;
    int tile = blockIdx.x;
    if (nwg % kXcds == 0) tile = (blockIdx.x % kXcds) * (nwg / kXcds) + blockIdx.x / kXcds;
    const int m0 = (tile % tiles_m) * 16 * MT, n0 = (tile / tiles_m) * 16 * NT;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // scalar
    const int li = lane & 15, g = lane >> 4;

    const int chunks = nb << (bshift - 5);
    const uint32_t row_bytes = (uint32_t)chunks * (BITS == 4 ? 16u : 32u);
    const uint32_t zp_cols = BITS == 4 ? (uint32_t)((nb + 1) / 2) : (uint32_t)nb;
    const int steps = (chunks + CH - 1) / CH;
    const int sh = bshift - 5;  // chunks per block, log2

    // Scales and zero points: whole 16-byte vectors of the tile's contiguous range, the
    // first ones requested before anything else.
    uint8_t* const s_img = smem + blk_fixed_lds<T, BITS, MT, NT, NW>();
    uint8_t* const z_img = s_img + image_bytes(16u * NT * (uint32_t)nb * (uint32_t)sizeof(T));
    const uint32_t cols = (uint32_t)min(N - n0, 16 * NT);
    const uint32_t s_bytes = cols * (uint32_t)nb * (uint32_t)sizeof(T);
    const uint32_t z_bytes = Z ? cols * zp_cols : 0u;
    const uint8_t* const s_src = reinterpret_cast<const uint8_t*>(S + (size_t)n0 * nb);
    const uint8_t* const z_src = Z ? Z + (size_t)n0 * zp_cols : B;
    constexpr int NTHR = 64 * NW;
    constexpr int SV = 4;  // scale vectors per thread requested up front
    u32x4_t sv0[SV], zv0;
    {
        const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(s_src, s_bytes & ~15u);
        const __amdgpu_buffer_rsrc_t rz = buffer_rsrc(z_src, z_bytes & ~15u);
#pragma unroll
        for (int u = 0; u < SV; ++u)
            sv0[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, 16u * (threadIdx.x + u * NTHR), 0, 0);
        zv0 = __builtin_amdgcn_raw_buffer_load_b128(rz, 16u * threadIdx.x, 0, 0);
    }

    // Every load of the loop is range-checked by its buffer resource, whose base moves
    // with the step (scalar arithmetic only): a row or column past the end has an
    // offset past any range, and a step past the last gets an empty resource; both read
    // zeros without touching memory, so that no load sits behind a branch and the
    // vector unit computes no addresses. A chunk past the row's end (the last step)
    // reads the next row's codes against activations that read zero; its scale is
    // taken as zero too.
    constexpr uint32_t kOut = 0xFFFFFFF0u;
    const uint32_t a_end = (uint32_t)((size_t)M * K * sizeof(T));
    const uint32_t b_end = (uint32_t)((size_t)N * row_bytes);
    const int gch = BITS == 4 ? g : g >> 1;  // this lane's chunk of a step
    uint32_t b_off[NT], a_off[MT][AI];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const uint32_t n = (uint32_t)(n0 + 16 * t + (lane >> 2));
        b_off[t] = (int)n < N ? n * row_bytes + 16u * (uint32_t)(lane & 3) : kOut;
    }
    const int apos = lane % PPR;  // this lane's piece of a row part
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < AI; ++j) {
            const int m = m0 + 16 * i + (64 * j + lane) / PPR;
            a_off[i][j] = m < M ? (uint32_t)m * (uint32_t)K * (uint32_t)sizeof(T) + 16u * apos : kOut;
        }
    auto part = [](const void* base, uint32_t off, uint32_t end, bool live) {
        // The scalar moves keep the compiler from treating the resource as divergent.
        const uint32_t o = (uint32_t)__builtin_amdgcn_readfirstlane((int)off);
        const uint32_t n = (uint32_t)__builtin_amdgcn_readfirstlane(
            (int)(((int)live & (int)(off < end)) ? end - off : 0u));
        return buffer_rsrc(static_cast<const uint8_t*>(base) + o, n);
    };

    // 0x64006400 in a register of its own: with the mask in a scalar register the
    // pair's AND and OR are one instruction (two literals are not).
    uint32_t magic;
    asm("v_mov_b32 %0, 0x64006400" : "=v"(magic));
    // Without zero points: the middle code (bit arithmetic, no branch on Z in the loop).
    const uint32_t zmask = Z ? (BITS == 4 ? 15u : 255u) : 0u, zdef = Z ? 0u : (BITS == 4 ? 8u : 128u);

    auto load = [&](Stage& st, int step) {
        const __amdgpu_buffer_rsrc_t rb = part(B, 64u * (uint32_t)step, b_end, step < steps);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            st.b[t] = __builtin_amdgcn_raw_buffer_load_b128(rb, b_off[t], 0,
                                                            MT == 1 ? kCachePolicyNT : 0);
#pragma unroll
        for (int h = 0; h < SUB; ++h) {
            const int k = step * KSTEP + KSUB * h;
            const __amdgpu_buffer_rsrc_t ra =
                part(A, (uint32_t)k * (uint32_t)sizeof(T), a_end, step < steps);
            const uint32_t past = apos * (16 / (int)sizeof(T)) < K - k ? 0u : kOut;
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < AI; ++j)
                    st.a[h][i][j] =
                        __builtin_amdgcn_raw_buffer_load_b128(ra, a_off[i][j] | past, 0, 0);
        }
    };
    // The wave's LDS region: NT column tiles of 16 x 64 bytes, then MT row tiles of
    // 16 x PPR pieces. Pieces are permuted by the row (column) number so that the
    // operand reads, which walk the rows, spread over the banks.
    uint8_t* const wreg = smem + wave * (uint32_t)Stage::WAVE_LDS;
    uint8_t* const areg = wreg + NT * 1024;
    constexpr int AM = (PPR < 16 ? PPR : 16) - 1;
    const uint32_t b_put = 64u * (lane >> 2) + 16u * ((lane & 3) ^ ((lane >> 4) & 3));
    const uint32_t b_get = 64u * li + 16u * (g ^ ((li >> 2) & 3));
    auto put_a = [&](const Stage& st, int h) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < AI; ++j) {
                const int row = (64 * j + lane) / PPR;
                *reinterpret_cast<u32x4_t*>(areg + 16 * (PPR * (16 * i + row) + (apos ^ (row & AM)))) =
                    st.a[h][i][j];
            }
    };
    auto get_a = [&](int i, int piece) {
        return *reinterpret_cast<const u32x4_t*>(areg + 16 * (PPR * (16 * i + li) + (piece ^ (li & AM))));
    };

    float4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = float4_t{0.f, 0.f, 0.f, 0.f};

    // Between a wave's accesses of its region by one lane and those by another: the hardware
    // keeps them in order, and this keeps the compiler from moving one past the other.
    auto exchange = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
    };

    // Multiplies a stage; its registers take the loads of step `next` as soon as their
    // contents are in LDS.
    auto process = [&](Stage& st, int step, int next) {
        exchange();
#pragma unroll
        for (int t = 0; t < NT; ++t)
            *reinterpret_cast<u32x4_t*>(wreg + 1024 * t + b_put) = st.b[t];
        put_a(st, 0);
        exchange();
        uint32_t w[NT][4];
        // Scale and zero point, of the lane's chunk (SC) or of each chunk.
        constexpr int NS = SC ? 1 : CH;
        uint32_t sv[NT][NS], zv[NT][NS];
        const uint32_t blk = (uint32_t)(CH * step + gch) >> sh;
        const bool in_row = gch < chunks - CH * step;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const u32x4_t b = *reinterpret_cast<const u32x4_t*>(wreg + 1024 * t + b_get);
            const uint32_t col = 16u * t + li;
            const uint32_t sx = image_at((col * (uint32_t)nb + blk) * (uint32_t)sizeof(T));
            const uint32_t zx = image_at(col * zp_cols + (BITS == 4 ? blk >> 1 : blk));
            uint32_t sq;
            if constexpr (sizeof(T) == 4) sq = *reinterpret_cast<const uint32_t*>(s_img + sx);
            else sq = *reinterpret_cast<const uint16_t*>(s_img + sx);
            sq = in_row ? sq : 0u;
            uint32_t zq = z_img[zx];
            if constexpr (BITS == 4) zq >>= (blk & 1) * 4;
            zq = (zq & zmask) | zdef;
            if constexpr (SC) {
#pragma unroll
                for (int c = 0; c < 4; ++c) w[t][c] = b[c];
                sv[t][0] = sq;
                zv[t][0] = zq;
            } else if constexpr (BITS == 4) {
                // 4x4 transposition of words over lane groups: w[t][c] = word g of chunk c.
                const U32Pair p02 = swap32u(b[0], b[2]), p13 = swap32u(b[1], b[3]);
                const U32Pair q01 = swap16u(p02.a, p13.a), q23 = swap16u(p02.b, p13.b);
                w[t][0] = q01.a;
                w[t][1] = q01.b;
                w[t][2] = q23.a;
                w[t][3] = q23.b;
            } else {
                // w[t][2c], w[t][2c + 1]: words 2g and 2g + 1 of chunk c.
                const U32Pair p02 = swap16u(b[0], b[2]), p13 = swap16u(b[1], b[3]);
                const U32Pair q0 = swap32u(p02.a, p02.b), q1 = swap32u(p13.a, p13.b);
                w[t][0] = q0.a;
                w[t][1] = q1.a;
                w[t][2] = q0.b;
                w[t][3] = q1.b;
            }
            if constexpr (!SC) {
                auto spread = [&](uint32_t x, uint32_t* out) {
                    if constexpr (BITS == 4) {
                        const U32Pair h = swap16u(x, x);
                        const U32Pair e = swap32u(h.a, h.a), o = swap32u(h.b, h.b);
                        out[0] = e.a;
                        out[1] = o.a;
                        out[2] = e.b;
                        out[3] = o.b;
                    } else {
                        const U32Pair e = swap32u(x, x);
                        out[0] = e.a;
                        out[1] = e.b;
                    }
                };
                if constexpr (sizeof(T) == 4) {
                    spread(sq, sv[t]);
                    spread(zq, zv[t]);
                } else {
                    spread(sq | (zq << 16), sv[t]);
#pragma unroll
                    for (int c = 0; c < CH; ++c) zv[t][c] = sv[t][c] >> 16;
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SUB == 1) load(st, next);
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            // One chunk at a time: scheduled together, the chunks' operands spill.
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (SUB == 2) {
                if (c == CH / 2) {
                    exchange();
                    put_a(st, 1);
                    exchange();
                    load(st, next);
                }
            }
            u32x4_t ao[MT][P];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                // Pieces of matrix step c: word c of the lane's chunk (SC), or the
                // lane's eight k of chunk c.
                constexpr int AV = sizeof(T) == 4 ? 2 : 1;
                const int piece = SC ? 4 * g + c : (4 * (c % (CH / SUB)) + g) * AV;
                u32x4_t raw[AV];
#pragma unroll
                for (int v = 0; v < AV; ++v) raw[v] = get_a(i, piece + v);
                blk_acts<T, BITS>(raw, ao[i]);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if constexpr (SC) {
                    const u32x4_t bo = scaled_codes<T>(w[t][c], zv[t][0], sv[t][0], magic);
#pragma unroll
                    for (int i = 0; i < MT; ++i) acc[i][t] = blk_mfma<T>(ao[i][0], bo, acc[i][t]);
                } else {
                    float sc;
                    if constexpr (sizeof(T) == 4)
                        sc = __uint_as_float(sv[t][c]);
                    else if constexpr (std::is_same<T, half_t>::value)
                        sc = (float)__builtin_bit_cast(half_t, (uint16_t)(sv[t][c] & 0xffffu));
                    else
                        sc = to_f32((uint16_t)(sv[t][c] & 0xffffu));
                    constexpr int W = BITS / 4;  // words per chunk and lane
                    const u32x4_t bo =
                        blk_codes<T, BITS>(w[t][W * c], w[t][W * c + W - 1], zv[t][c]);
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        float4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int p = P - 1; p >= 0; --p) d = blk_mfma<T>(ao[i][p], bo, d);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][t][e] = fmaf(sc, d[e], acc[i][t][e]);
                    }
                }
            }
        }
    };

    Stage st;
    // After the image's loads: loads complete in order, and the waits in the loop have
    // to hold for its first round too.
    __builtin_amdgcn_sched_barrier(0);
    load(st, wave);
    __builtin_amdgcn_sched_barrier(0);
    // The image beyond the vectors already here, and the last bytes of the tensor when
    // they are no whole vector.
    auto fill = [&](uint8_t* img, const uint8_t* src, uint32_t bytes, uint32_t from) {
        for (uint32_t u = from + threadIdx.x; u < bytes / 16; u += NTHR)
            *reinterpret_cast<u32x4_t*>(img + image_at(16 * u)) =
                *reinterpret_cast<const u32x4_t*>(src + 16 * u);
        if (threadIdx.x < (bytes & 15u)) {
            const uint32_t x = (bytes & ~15u) + threadIdx.x;
            img[image_at(x)] = src[x];
        }
    };
#pragma unroll
    for (int u = 0; u < SV; ++u) {
        const uint32_t at = threadIdx.x + u * NTHR;
        if (at < s_bytes / 16) *reinterpret_cast<u32x4_t*>(s_img + image_at(16 * at)) = sv0[u];
    }
    if (threadIdx.x < z_bytes / 16)
        *reinterpret_cast<u32x4_t*>(z_img + image_at(16 * threadIdx.x)) = zv0;
    fill(s_img, s_src, s_bytes, SV * NTHR);
    fill(z_img, z_src, z_bytes, NTHR);
    __syncthreads();
    for (int s = wave; s < steps; s += NW) process(st, s, s + NW);

    // Partial tiles [wave][tile][e][lane] in place of the exchange regions.
    float* const red = reinterpret_cast<float*>(smem);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                red[((wave * MT * NT + i * NT + t) * 4 + e) * 64 + lane] = acc[i][t][e];
    __syncthreads();
    for (int q = wave; q < MT * NT * 4; q += NW) {
        const int e = q & 3, it = q >> 2;
        float v = 0.f;
#pragma unroll
        for (int j = 0; j < NW; ++j) v += red[((j * MT * NT + it) * 4 + e) * 64 + lane];
        v *= 1.f / blk_unit<T, BITS, SC>();
        const int m = m0 + 16 * (it / NT) + 4 * g + e, n = n0 + 16 * (it % NT) + li;
        if constexpr (sizeof(T) == 4) {
            // A NaN whose payload lies in the low 16 bits alone entered as an infinity (its
            // first piece), which left no finite sum: an infinite one looks for NaN in its row.
            if (__builtin_isinf(v) && m < M)
                for (int k = 0; k < K; ++k) {
                    const float x = A[(size_t)m * K + k];
                    if (x != x) v = x;
                }
        }
        if constexpr (SWI) {
            // Interleaved gate/up columns (2i, 2i + 1) in adjacent lanes: the even lane
            // writes column i of the [M, N / 2] output, (g * sigmoid(g)) * u with each
            // op rounded to T as the unfused ops store it.
            const float y = round_to<T>(v);
            const float up = dpp_mov<0xB1>(y);  // quad_perm [1,0,3,2]
            if ((lane & 1) == 0 && m < M && n < N) {
                const float sig = round_to<T>(1.0f / (1.0f + __expf(-y)));
                Y[(size_t)m * (N / 2) + n / 2] = from_f32<T>(round_to<T>(y * sig) * up);
            }
        } else if (m < M && n < N) {
            Y[(size_t)m * N + n] = from_f32<T>(v);
        }
    }
}

// A tile shape and its launch. LDS allows 160 KB per workgroup; a K whose scales do
// not fit takes fewer columns, and past one column tile none (-1).
constexpr uint32_t kBlkLds = 160 * 1024;
template <typename T, int BITS, int MT, int NT, int NW, bool SWI, bool SC>
int launch_blk(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y, int M, int N,
               int K, int nb, int bshift, hipStream_t st) {
    const int tiles_m = (M + 16 * MT - 1) / (16 * MT), tiles_n = (N + 16 * NT - 1) / (16 * NT);
    const uint32_t lds = blk_lds<T, BITS, MT, NT, NW>(nb);
    if ((long)tiles_m * tiles_n > 0x7fffffffL || lds > kBlkLds) return -1;
    hipLaunchKernelGGL((mnb_blk_kernel<T, BITS, MT, NT, NW, SWI, SC>), dim3(tiles_m * tiles_n),
                       dim3(64 * NW), lds, st, A, B, S, Z, Y, M, N, K, nb, bshift, tiles_m, tiles_n);
    return check_launch("mnb_blk");
}

}  // namespace

template <typename T, int BITS, bool SWI>
int mnb_blk(const T* A, const uint8_t* B, const T* S, const uint8_t* Z, T* Y, int M, int N, int K,
            int bs, hipStream_t st) {
    const int nb = (K + bs - 1) / bs;
    constexpr int EPL = 16 / (int)sizeof(T);
    if (bs != 32 && bs != 64 && bs != 128) return -1;
    // Whole 16-byte vectors, and 32-bit buffer offsets.
    auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    if (K % EPL || !aligned(A) || !aligned(B) || !aligned(S) || !aligned(Z) ||
        (size_t)M * K * sizeof(T) > 0xFFFFFF00ull ||
        (size_t)N * nb * bs * BITS / 8 > 0xFFFFFF00ull || (size_t)N * nb * sizeof(T) > 0xFFFFFF00ull)
        return -1;
    const int bshift = bs == 32 ? 5 : bs == 64 ? 6 : 7;
    // Tile shapes: 16 rows for up to 16, else 32; 1, 2 or 4 column tiles; 8 waves, or 4
    // where 8 waves' exchange regions would leave one workgroup per CU. The choice is
    // the least of rounds * (start + work), in units of about 0.05 us fitted to a sweep
    // of all shapes on MI355X: a round starts and drains in about 92, a step of one
    // column tile takes 1 per workgroup that shares the CU (1.6 for two row tiles,
    // twice that in fp32). Measured against the other choices: 8 x 4096 x 14336 fp16
    // 12.4 us (NT 2) against 12.8 (4) and 14.9 (1); 8 x 4096 x 4096 6.5 (1) against 8.2
    // (2); 32 x 4096 x 14336 15.8 (4, 8 waves) against 19.8 (2); 64 x 4096 x 14336 23.3
    // (4, 4 waves) against 27.6 (8 waves); 512 x 896 x 1152 fp32 15.1 (2, 4 waves)
    // against 20.3 (4, 8 waves).
    struct Shape {
        int mt, nt, nw;
        uint32_t lds;
        int (*launch)(const T*, const uint8_t*, const T*, const uint8_t*, T*, int, int, int, int,
                      int, hipStream_t);
    };
    constexpr bool SC = blk_scaled<T, BITS>();
#define ORTMI_SHAPE(MT, NT, NW) \
    {MT, NT, NW, blk_lds<T, BITS, MT, NT, NW>(nb), launch_blk<T, BITS, MT, NT, NW, SWI, SC>}
    const Shape shapes[] = {ORTMI_SHAPE(1, 1, 8), ORTMI_SHAPE(1, 2, 8), ORTMI_SHAPE(1, 4, 8),
                            ORTMI_SHAPE(2, 1, 8), ORTMI_SHAPE(2, 2, 8), ORTMI_SHAPE(2, 4, 8),
                            ORTMI_SHAPE(2, 2, 4), ORTMI_SHAPE(2, 4, 4)};
#undef ORTMI_SHAPE
    const long cus = device_cu_count();
    const int steps = (nb * bs + BlkStage<T, BITS, 1, 1>::KSTEP - 1) / BlkStage<T, BITS, 1, 1>::KSTEP;
    const Shape* best = nullptr;
    double least = 0;
    for (const Shape& c : shapes) {
        if (c.lds > kBlkLds || (c.mt == 1) != (M <= 16)) continue;
        const long tiles = ((M + 16 * c.mt - 1L) / (16 * c.mt)) * ((N + 16 * c.nt - 1L) / (16 * c.nt));
        // Two 8-wave workgroups fill a CU's wave slots at the kernels' register use.
        const long fit = std::min<long>(kBlkLds / c.lds, 16 / c.nw);
        const long share = std::min(fit, (tiles + cus - 1) / cus);
        const long rounds = (tiles + cus * share - 1) / (cus * share);
        const double step = (c.mt == 1 ? 1.0 : 1.6) * (sizeof(T) == 4 ? 2.0 : 1.0);
        const double cost = rounds * (92.0 + share * steps * step * (c.nt + (c.mt == 1 ? 0.0 : 0.5)));
        if (!best || cost < least) best = &c, least = cost;
    }
    if (!best) return -1;
    if constexpr (SC && !SWI) {
        // One row keeps its weights unrounded, as the GEMV does at smaller K. MI355X, 4096
        // columns: bf16 K 14336 15.0 us (scaled weights 13.8, VALU tile product 1764), fp16 K
        // 17920 18.2 us (17.3, 2278).
        if (M == 1) {
            auto* launch = best->nt == 1   ? launch_blk<T, BITS, 1, 1, 8, false, false>
                           : best->nt == 2 ? launch_blk<T, BITS, 1, 2, 8, false, false>
                                           : launch_blk<T, BITS, 1, 4, 8, false, false>;
            return launch(A, B, S, Z, Y, M, N, K, nb, bshift, st);
        }
    }
    return best->launch(A, B, S, Z, Y, M, N, K, nb, bshift, st);
}

#define ORTMI_BLK(T, BITS, SWI)                                                            \
    template int mnb_blk<T, BITS, SWI>(const T*, const uint8_t*, const T*, const uint8_t*, \
                                       T*, int, int, int, int, hipStream_t);
ORTMI_BLK(half_t, 4, false)
ORTMI_BLK(half_t, 4, true)
ORTMI_BLK(half_t, 8, false)
ORTMI_BLK(uint16_t, 4, false)
ORTMI_BLK(uint16_t, 8, false)
ORTMI_BLK(float, 4, false)
ORTMI_BLK(float, 8, false)

}  // namespace ortmi
