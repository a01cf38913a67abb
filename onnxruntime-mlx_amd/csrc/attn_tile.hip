// Attention tiles on the matrix cores of gfx950: GroupQueryAttention prompts, fp16 and bf16.
//
// One workgroup of 8 waves takes 128 query rows of one KV head: 4 row waves of 32 rows,
// twice, the two halves of the waves ("key groups") taking every other block of 64
// keys; the groups' states are merged through LDS at the end. (A call whose keys all lie in
// one block has workgroups of 4 waves, one group.) Everything a query needs stays in its
// lanes:
//   S^T = K Q^T     (v_mfma 32x32x16; A = 32 keys x 16 dims from LDS, B = 16 dims x 32
//                    queries, held in registers for the whole tile)
//   O^T += V^T P^T  (A = 32 head dims x 16 keys, B = this lane's own probabilities)
// In the accumulator layout a lane holds one query (column lane % 32) and 16 keys (or
// head dims) of it; lanes l and l ^ 32 share a query. The online softmax is register
// arithmetic plus one permlane32 swap per block, and P never goes through LDS: the
// k-order of the second product is the keys a lane already holds (4h..4h+3 and
// 8+4h..8+4h+3 of each 16 for lane half h).
//
// Bound: the instructions issued. A step (128 rows x 64 keys per key group) takes the
// matrix cores 2048 cycles per SIMD and the vector units about 2800 (250 instructions and 32
// exponentials per wave), and the two overlap in part only: 2.6 us. So that little else takes
// issue slots, K and V blocks go from memory to LDS without passing registers
// (global_load_lds, two buffers of each per key group, one step ahead), V is transposed by
// the LDS read itself (ds_read_b64_tr_b16), and Q is read once and rotated in registers.
// LDS holds rows of 128 or 256 bytes whose 16-byte pieces are permuted by the row number, so
// that both kinds of read spread over all banks (no conflict measured).
// Measured on MI355X, 2048 tokens, 32 heads of 128 on 8: 105 us with tiles of 256 rows and
// keys passing registers, with 22 us of rotation before and 32 us of merging after it; 62 us
// and 7 us now, without a merge. 64 rows per wave (one wave per SIMD, half the LDS reads): 80.
#include <type_traits>

#include "attn_internal.h"

namespace ortmi {
namespace {

typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef u32x4_t u32x4_any_t __attribute__((aligned(2)));  // at any element
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(1))) void global_void;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;

template <typename T>
__device__ __forceinline__ float16_t tile_mfma(u32x4_t a, u32x4_t b, float16_t c) {
    if constexpr (std::is_same<T, half_t>::value)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a),
                                                      __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
// Two floats rounded to T (nearest even) as one word.
template <typename T>
__device__ __forceinline__ uint32_t tile_round2(float x, float y) {
    if constexpr (std::is_same<T, half_t>::value) {
        const half2_t v = {(half_t)x, (half_t)y};
        return __builtin_bit_cast(uint32_t, v);
    } else {
        const bf16x2_t v = {(__bf16)x, (__bf16)y};
        return __builtin_bit_cast(uint32_t, v);
    }
}
template <typename T>
__device__ __forceinline__ float tile_lo(uint32_t w) {
    if constexpr (std::is_same<T, half_t>::value)
        return (float)__builtin_bit_cast(half_t, (uint16_t)(w & 0xffffu));
    else
        return __uint_as_float(w << 16);
}
template <typename T>
__device__ __forceinline__ float tile_hi(uint32_t w) {
    if constexpr (std::is_same<T, half_t>::value)
        return (float)__builtin_bit_cast(half_t, (uint16_t)(w >> 16));
    else
        return __uint_as_float(w & 0xffff0000u);
}
// Sum of two T values (the halves of w) added to acc in fp32, exactly widened.
template <typename T>
__device__ __forceinline__ float tile_pair_sum(uint32_t w, float acc) {
    if constexpr (std::is_same<T, half_t>::value) {
        const half2_t one2 = {(half_t)1.f, (half_t)1.f};
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, w), one2, acc, false);
    } else {
        const bf16x2_t one2 = {(__bf16)1.f, (__bf16)1.f};
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w), one2, acc, false);
    }
}

struct TileDesc {
    int tok0;      // first token (packed row) of the tile
    int ntok;      // tokens in the tile
    int qpos0;     // absolute position of the first query token
};

constexpr int kKeys = 64;       // keys per block
constexpr int kRowWaves = kAttnRows / 32;  // waves of 32 query rows
// KG: groups of waves that share the key blocks, 1 or 2.

// Pieces of P in the second product. The kernel that took head 96 before had fp32
// probabilities: three bf16 pieces carry their 24 bits, two fp16 pieces 22 bits down to 2^-17
// of a row's largest and below that an error of 2^-39 of it (less than the error of the
// exponential, a few 2^-22, down to 2^-18).
template <typename T, int HD>
constexpr int p_pieces() { return HD != 96 ? 1 : std::is_same<T, half_t>::value ? 2 : 3; }

// 16-byte pieces of an LDS row (96 dims take a row of 128), and the permutation: piece c
// of row r lies at place c ^ swizzle(r). Any 16 consecutive rows of one piece (the key
// reads), and any aligned 4 rows of an aligned 4 pieces (the transposed reads), fall in
// different banks.
constexpr int lds_pieces(int hd) { return hd == 64 ? 8 : 16; }
template <int CPR>
__device__ __forceinline__ int swizzle(int r) {
    return CPR == 16 ? ((r & 3) << 2) | ((r >> 2) & 3) : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
}

template <typename T, int HD, int KG, bool A16>
__device__ void attn_tile(const TileDesc& t, int kvh, int G, int H, const QueryRows<T>& qr,
                          const T* __restrict__ kd, const T* __restrict__ vd,
                          float scale, int k0, int k1,
                          T* __restrict__ out, int64_t out_tok_stride, float* __restrict__ part,
                          int nsplit, int split) {
    static_assert(sizeof(T) == 2 && HD % 32 == 0, "tile shape");
    constexpr int KC = lds_pieces(HD);
    constexpr int DT = HD / 32;         // head-dim tiles of O^T
    constexpr int KI = KC / kRowWaves;  // loads per wave and block, of K and of V
    constexpr int P = p_pieces<T, HD>();
    // Two buffers of K and V blocks per key group, arrays of their own so that a read of
    // one is known not to wait for the load in flight into the other.
    __shared__ __attribute__((aligned(1024))) uint16_t sK0[KG][kKeys * KC * 8];
    __shared__ __attribute__((aligned(1024))) uint16_t sK1[KG][kKeys * KC * 8];
    __shared__ __attribute__((aligned(1024))) uint16_t sV0[KG][kKeys * KC * 8];
    __shared__ __attribute__((aligned(1024))) uint16_t sV1[KG][kKeys * KC * 8];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int rw = wave % kRowWaves, kg = wave / kRowWaves;
    const int lrow = lane & 31, hh = lane >> 5;
    const int rows = t.ntok * G;
    // This lane's query row: token and head of the group.
    const int q = rw * 32 + lrow;
    const bool qlive = q < rows;
    const int qtok = qlive ? q / G : 0, qhead = qlive ? q - qtok * G : 0;
    // Earliest position among the wave's queries: a block up to it is visible to all.
    const int qpos_wave = t.qpos0 + (rw * 32) / G;

    // Scores are kept in the log2 domain (exp2 is the hardware exponential). The scale is
    // applied inside the exponent, after the block maximum of the raw scores, which
    // needs it positive: a negative scale flips the sign of Q.
    constexpr float kLog2e = 1.4426950408889634f;
    const float sc2 = fabsf(scale) * kLog2e;
    const uint32_t qsign = scale < 0.f ? 0x80008000u : 0u;

    float m, lsum;
    float16_t oT[DT];
    m = -INFINITY;
    lsum = 0.f;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) oT[d][e] = 0.f;

    // --- staging: this lane's rows of a block -------------------------------------
    // Load i of a wave fills LDS bytes [1024 * (rw * KI + i), + 1024) in lane order, so a
    // lane picks which piece of its row it fetches. Rows past the range end load its last
    // row; their keys are masked and their values zeroed in LDS once the loads are in.
    // Addresses are formed anew in each block (a few instructions) from a value that the
    // compiler cannot see through: kept across blocks for all loads and buffers they would
    // take over 40 registers, and a spilled register's reload waits for the row loads.
    // Rows that are not 16-byte aligned pass through registers to the same places.
    auto opaque = [](int x) {
        asm volatile("" : "+v"(x));
        return x;
    };
    const int per_load = 64 / KC;  // rows
    auto load_rows = [&](uint16_t (&buf)[KG][kKeys * KC * 8], const T* base, int kb) {
        const uint32_t ln = (uint32_t)opaque(lane);
        const int r0 = (int)(ln / KC), x = (int)(ln % KC) ^ swizzle<KC>(r0);
        int past_end = 0;
        u32x4_t w[A16 ? 1 : KI];
#pragma unroll
        for (int i = 0; i < KI; ++i) {
            // The first row of a load is a multiple of 4 (of 8 at 8 pieces), so that
            // swizzle(row) = swizzle(r0) ^ swizzle(first).
            const int first = (rw * KI + i) * per_load;
            int c = x ^ swizzle<KC>(first);
            if (HD != 8 * KC && c >= HD / 8) c -= 8;  // 96 dims: the row's unused pieces
            const int r = first + r0, rc = min(r, k1 - 1 - kb);
            // A uniform base and a 32-bit offset inside the block.
            const T* src = base + (int64_t)kb * HD + (uint32_t)(rc * HD + c * 8);
            if constexpr (A16)
                __builtin_amdgcn_global_load_lds((global_void*)(void*)src,
                                                 (lds_void*)&buf[kg][(rw * KI + i) * 512], 16, 0, 0);
            else
                w[i] = *reinterpret_cast<const u32x4_any_t*>(src);
            past_end |= (int)(r != rc) << i;
        }
        if constexpr (!A16) {
#pragma unroll
            for (int i = 0; i < KI; ++i)
                *reinterpret_cast<u32x4_t*>(&buf[kg][(rw * KI + i) * 512 + ln * 8]) = w[i];
        }
        return past_end;
    };
    int vbad = 0;  // rows of the V block in flight that are to be zeroed
    auto stage_k = [&](uint16_t (&buf)[KG][kKeys * KC * 8], int kb) {
        if (kb < k1) load_rows(buf, kd, kb);
    };
    auto stage_v = [&](uint16_t (&buf)[KG][kKeys * KC * 8], int kb) {
        if (kb < k1) vbad = load_rows(buf, vd, kb);
    };
    // Waits for this wave's loads and zeroes the value rows that are not there.
    auto arrive = [&](uint16_t (&buf)[KG][kKeys * KC * 8]) {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        if (__any(vbad)) {
            const int ln = opaque(lane);
#pragma unroll
            for (int i = 0; i < KI; ++i)
                if ((vbad >> i) & 1)
                    *reinterpret_cast<u32x4_t*>(&buf[kg][(rw * KI + i) * 512 + ln * 8]) =
                        u32x4_t{0u, 0u, 0u, 0u};
            vbad = 0;
        }
    };

    // Blocks of this group: k0 + (2 s + kg) * 64 in step s.
    const int nblocks = k1 > k0 ? (k1 - k0 + kKeys - 1) / kKeys : 0;
    const int steps = (nblocks + KG - 1) / KG;
    auto block = [&](int s) { return k0 + (KG * s + kg) * kKeys; };
    // --- queries ------------------------------------------------------------------
    // B operand of step s2: dims 16 s2 + 8 hh .. + 7 of the lane's query, rotated here
    // (one rounding to T) when the call has not staged rotated rows. Their loads go out
    // first, then those of the first blocks, which arrive during the rotation.
    constexpr int QS = HD / 16;
    u32x4_t qf[QS], cw[QS / 2], sw[QS / 2];
    const T* row = qr.q + (int64_t)(t.tok0 + qtok) * qr.tok_stride +
                   (int64_t)(kvh * G + qhead) * HD + 8 * hh;
#pragma unroll
    for (int s2 = 0; s2 < QS; ++s2)
        qf[s2] = *reinterpret_cast<const u32x4_t*>(row + 16 * s2);
    if (qr.cos) {
        // Half-split pairs (i, i + hd/2): entries 16 j + 8 hh .. + 7 for dims of step j
        // and j + QS/2. Interleaved pairs (2i, 2i + 1): entries 8 s2 + 4 hh .. + 3 for
        // step s2, two steps to a vector.
        const int64_t row = (int64_t)(t.qpos0 + qtok) * (HD / 2);
#pragma unroll
        for (int j = 0; j < QS / 2; ++j) {
            const T *c = qr.cos + row + 16 * j, *s = qr.sin + row + 16 * j;
            if (qr.interleaved) {
                const u32x2_t c0 = *reinterpret_cast<const u32x2_t*>(c + 4 * hh);
                const u32x2_t c1 = *reinterpret_cast<const u32x2_t*>(c + 8 + 4 * hh);
                const u32x2_t s0 = *reinterpret_cast<const u32x2_t*>(s + 4 * hh);
                const u32x2_t s1 = *reinterpret_cast<const u32x2_t*>(s + 8 + 4 * hh);
                cw[j] = u32x4_t{c0[0], c0[1], c1[0], c1[1]};
                sw[j] = u32x4_t{s0[0], s0[1], s1[0], s1[1]};
            } else {
                cw[j] = *reinterpret_cast<const u32x4_t*>(c + 8 * hh);
                sw[j] = *reinterpret_cast<const u32x4_t*>(s + 8 * hh);
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (steps > 0) {
        stage_k(sK0, block(0));
        stage_v(sV0, block(0));
        stage_k(sK1, block(1));
    }
    __builtin_amdgcn_sched_barrier(0);
    if (qr.cos) {
        if (qr.interleaved) {
#pragma unroll
            for (int s2 = 0; s2 < QS; ++s2)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t ce = cw[s2 / 2][2 * (s2 % 2) + j / 2];
                    const uint32_t se = sw[s2 / 2][2 * (s2 % 2) + j / 2];
                    const float c = j & 1 ? tile_hi<T>(ce) : tile_lo<T>(ce);
                    const float s = j & 1 ? tile_hi<T>(se) : tile_lo<T>(se);
                    const float a = tile_lo<T>(qf[s2][j]), b = tile_hi<T>(qf[s2][j]);
                    qf[s2][j] = tile_round2<T>(a * c - b * s, b * c + a * s);
                }
        } else {
#pragma unroll
            for (int s2 = 0; s2 < QS / 2; ++s2)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t x = qf[s2][j], y = qf[s2 + QS / 2][j];
                    const float c0 = tile_lo<T>(cw[s2][j]), c1 = tile_hi<T>(cw[s2][j]);
                    const float s0 = tile_lo<T>(sw[s2][j]), s1 = tile_hi<T>(sw[s2][j]);
                    const float a0 = tile_lo<T>(x), a1 = tile_hi<T>(x);
                    const float b0 = tile_lo<T>(y), b1 = tile_hi<T>(y);
                    qf[s2][j] = tile_round2<T>(a0 * c0 - b0 * s0, a1 * c1 - b1 * s1);
                    qf[s2 + QS / 2][j] =
                        tile_round2<T>(b0 * c0 + a0 * s0, b1 * c1 + a1 * s1);
                }
        }
    }
#pragma unroll
    for (int s2 = 0; s2 < QS; ++s2)
        qf[s2] = qlive ? qf[s2] ^ qsign : u32x4_t{0u, 0u, 0u, 0u};

    // --- the two products ---------------------------------------------------------
    const int kx0 = hh ^ swizzle<KC>(lrow);  // piece 2 s2 + hh of row lrow lies at kx ^ 2 s2
    auto key_operand = [&](const uint16_t (&buf)[KG][kKeys * KC * 8], int kx, int s2,
                           int kt) {
        return *reinterpret_cast<const u32x4_t*>(&buf[kg][(kt * 32 * KC + (kx ^ (2 * s2))) * 8]);
    };
    // Transposed read: the 16 lanes of a group name 4 rows (keys) x 16 dims, 8 bytes
    // each, and lane i of them receives dim i of the 4 rows. Lane groups 0 and 1 (2 and
    // 3) take dims 0-15 and 16-31 of a tile for keys 4h.. (second read: 8 + 4h..).
    const int vr = (lane & 15) >> 2;
    const int vlow = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    auto voff = [&](int sec) {  // dim tile 0; tile d lies at voff ^ 32 d
        const int r = 4 * hh + 8 * sec + vr;
        return (r * KC + (vlow ^ swizzle<KC>(r))) * 8 + 4 * (lane & 1);
    };
    const int v0 = voff(0), v1 = voff(1);
    auto value_operand = [&](const uint16_t (&buf)[KG][kKeys * KC * 8], int o0, int o1,
                             int kk, int d) {
        const uint16_t* b = &buf[kg][kk * 16 * KC * 8];
        const u32x2_t lo = __builtin_bit_cast(
            u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(b + (o0 ^ (32 * d)))));
        const u32x2_t hi = __builtin_bit_cast(
            u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(b + (o1 ^ (32 * d)))));
        return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
    };

    // --- the key walk, software-pipelined across blocks -------------------------------
    // Step s issues the scores of block s + 1, then runs the softmax and the P V product of
    // block s. Its V(s) and K(s + 1) were requested a step earlier; it requests V(s + 1)
    // and K(s + 2) into the buffers that step s - 1 left. The two waves of a SIMD drift
    // apart, so that one's vector instructions run beside the other's matrix instructions;
    // the walk is bound by the instructions issued (interleaving both kinds inside a wave,
    // by halves of a block, issued more of them: 61 -> 66 us at 2048 tokens, 32 heads).
    float16_t stA[2], stB[2];
    auto scores = [&](const uint16_t (&buf)[KG][kKeys * KC * 8], float16_t (&st)[2]) {
        const int kx = opaque(lrow * KC + kx0);
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int e = 0; e < 16; ++e) st[kt][e] = 0.f;
#pragma unroll
        for (int s2 = 0; s2 < QS; ++s2)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
                st[kt] = tile_mfma<T>(key_operand(buf, kx, s2, kt), qf[s2], st[kt]);
    };
    auto step = [&](int s, float16_t (&cur)[2], float16_t (&nxt)[2],
                    uint16_t (&kfill)[KG][kKeys * KC * 8],
                    uint16_t (&knext)[KG][kKeys * KC * 8],
                    uint16_t (&vcur)[KG][kKeys * KC * 8],
                    uint16_t (&vfill)[KG][kKeys * KC * 8]) {
        const int kb = block(s);
        arrive(vcur);
        __syncthreads();
        stage_v(vfill, block(s + 1));
        stage_k(kfill, block(s + 2));
        if (kb >= k1) return;  // the other key group's last block
        __builtin_amdgcn_sched_barrier(0);
        // Past the last block this scores what the buffer holds; nothing reads it.
        scores(knext, nxt);
        // Keys that are past the range or causally hidden (only in blocks that are not wholly
        // visible).
        if (kb + kKeys > k1 || kb + kKeys - 1 > qpos_wave) {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                // Keys of the lane: 4h + a constant; the last one it may see.
                const int last = min(k1 - 1, t.qpos0 + qtok) - kb - 32 * kt - 4 * hh;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int kk = 8 * (e / 4) + (e & 3);
                    cur[kt][e] = kk <= last ? cur[kt][e] : -INFINITY;
                }
            }
        }
        // Block max of the raw scores. Scaling by sc2 > 0 keeps the maximum (and rounds it
        // alike), so the scale joins the exponent's argument in one fma.
        float bmax = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int e = 0; e < 16; ++e) bmax = fmaxf(bmax, cur[kt][e]);
        {
            const LanePair pr = swap32(bmax);
            bmax = fmaxf(pr.a, pr.b);
        }
        // The reference point m moves only when the block max passes it by more than kLazy
        // (log2 units), so P = exp2(s - m) stays below 2^kLazy (exact in fp16's range) and
        // O is rarely rescaled; neither the final O / l nor a merge of (m, l, O) states
        // depends on where m sits. With P in two fp16 pieces it sits 14 below the maximum and
        // follows it closely: the second piece is subnormal, its error 2^-25, from P = 2^-3
        // down, which is 2^-17 of the largest probability or less.
        constexpr bool two16 = P == 2;
        constexpr float kLazy = two16 ? 15.f : 8.f, kBelow = two16 ? 14.f : 0.f;
        const float bm = bmax * sc2;
        const float m_new = bm > m + kLazy ? bm - kBelow : m;
        // v_exp_f32 directly: results below 2^-126 flush to zero, which the softmax weights
        // can afford.
        const float alpha = (m == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
        const float mref = m_new == -INFINITY ? 0.f : m_new;  // exp2(-inf - 0) = 0
        m = m_new;
        if (__any(alpha != 1.f)) {
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int e = 0; e < 16; ++e) oT[d][e] *= alpha;
        }
        // P^T operands: k-step kk takes e in [8 (kk % 2), 8 (kk % 2) + 8) of tile kk / 2.
        u32x4_t pb[P][4];
        float ls[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            ls[kk] = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = 8 * (kk % 2) + 2 * j;
                float x = __builtin_amdgcn_exp2f(fmaf(cur[kk / 2][e], sc2, -mref));
                float y = __builtin_amdgcn_exp2f(fmaf(cur[kk / 2][e + 1], sc2, -mref));
                if constexpr (P > 1) ls[kk] += x + y;
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    const uint32_t w = tile_round2<T>(x, y);
                    pb[p][kk][j] = w;
                    if constexpr (P > 1) {
                        x -= tile_lo<T>(w);
                        y -= tile_hi<T>(w);
                    }
                }
                // One piece: the sum takes the rounded values that weight V.
                if constexpr (P == 1) ls[kk] = tile_pair_sum<T>(pb[0][kk][j], ls[kk]);
            }
        }
        lsum = fmaf(lsum, alpha, (ls[0] + ls[1]) + (ls[2] + ls[3]));
        const int o0 = opaque(v0), o1 = opaque(v1);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const u32x4_t a = value_operand(vcur, o0, o1, kk, d);
#pragma unroll
                for (int p = P - 1; p >= 0; --p) oT[d] = tile_mfma<T>(a, pb[p][kk], oT[d]);
            }
    };
    if (steps > 0) {
        arrive(sV0);
        __syncthreads();
        scores(sK0, stA);
    }
    for (int s = 0; s < steps; s += 2) {
        step(s, stA, stB, sK0, sK1, sV0, sV1);
        if (s + 1 < steps) step(s + 1, stB, stA, sK1, sK0, sV1, sV0);
    }
    {
        const LanePair pr = swap32(lsum);
        lsum = pr.a + pr.b;
    }
    if constexpr (HD == 96) {
        // A value that is not finite must neither reach a row that does not see its key
        // (through 0 * infinity) nor turn NaN between the pieces of P: the kernel that took
        // these prompts before read visible keys only, in fp32. Every such product leaves a
        // NaN in O; a wave that ends with one adds up P V again, a key at a time (m and the
        // sum of P stand, they do not depend on V).
        float z = 0.f;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int e = 0; e < 16; ++e) z = fmaf(oT[d][e], 0.f, z);
        if (__any(z != 0.f)) {
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int e = 0; e < 16; ++e) oT[d][e] = 0.f;
            const int last = min(k1 - 1, t.qpos0 + qtok);
            const float mref = m == -INFINITY ? 0.f : m;
            for (int n = 0; n < steps * kKeys; ++n) {
                const int j = block(n / kKeys) + n % kKeys;
                if (!__any(j <= last)) break;
                const T *kr = kd + (int64_t)j * HD + 8 * hh, *vr = vd + (int64_t)j * HD + 4 * hh;
                float dot = 0.f;
#pragma unroll
                for (int s2 = 0; s2 < QS; ++s2) {
                    const u32x4_t w = *reinterpret_cast<const u32x4_t*>(kr + 16 * s2);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        dot = fmaf(tile_lo<T>(qf[s2][i]), tile_lo<T>(w[i]), dot);
                        dot = fmaf(tile_hi<T>(qf[s2][i]), tile_hi<T>(w[i]), dot);
                    }
                }
                const LanePair pr = swap32(dot);
                const float p = __builtin_amdgcn_exp2f(fmaf(pr.a + pr.b, sc2, -mref));
                if (j > last) continue;
#pragma unroll
                for (int d = 0; d < DT; ++d)
#pragma unroll
                    for (int e4 = 0; e4 < 4; ++e4) {
                        const u32x2_t w =
                            *reinterpret_cast<const u32x2_t*>(vr + 32 * d + 8 * e4);
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            const int e = 4 * e4 + 2 * i;
                            oT[d][e] = fmaf(p, tile_lo<T>(w[i]), oT[d][e]);
                            oT[d][e + 1] = fmaf(p, tile_hi<T>(w[i]), oT[d][e + 1]);
                        }
                    }
            }
        }
    }

    // --- the key groups' states, merged by the first (which alone has a single block) ----
    if (KG == 1 || nblocks <= 1) {
        if (kg == 1 || !qlive) return;
    } else {
        constexpr int DK = KC / 8;  // head-dim tiles per K buffer pair (16 KB each)
        static_assert(DT <= 2 * DK, "exchange space");
        float* const x0 = reinterpret_cast<float*>(&sK0[0][0]);
        float* const x1 = reinterpret_cast<float*>(&sK1[0][0]);
        float* const xm = reinterpret_cast<float*>(&sV0[0][0]);
        auto at = [&](int d, int e) {
            return (d < DK ? x0 : x1) +
                   (((d % DK) * kRowWaves + rw) * 16 + e) * 64 + lane;
        };
        __syncthreads();
        if (kg == 1) {
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int e = 0; e < 16; ++e) *at(d, e) = oT[d][e];
            xm[rw * 128 + lane] = m;
            xm[rw * 128 + 64 + lane] = lsum;
        }
        __syncthreads();
        if (kg == 1 || !qlive) return;
        const float m1 = xm[rw * 128 + lane];
        const float l1 = xm[rw * 128 + 64 + lane];
        const float mm = fmaxf(m, m1);
        const float a0 = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mm);
        const float a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - mm);
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                oT[d][e] = fmaf(*at(d, e), a1, oT[d][e] * a0);
        lsum = fmaf(l1, a1, lsum * a0);
        m = mm;
    }
    float l = lsum;
    float mn = m == -INFINITY ? m : m / kLog2e;  // the merge's natural-log domain
    const int tok = t.tok0 + qtok, h = kvh * G + qhead;
    if (part) {
        float* dst = part + (((int64_t)tok * H + h) * nsplit + split) * (HD + 2);
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                dst[d * 32 + 8 * (e / 4) + 4 * hh + (e & 3)] = oT[d][e];
        if (hh == 0) {
            dst[HD] = mn;
            dst[HD + 1] = l;
        }
        return;
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
    T* dst = out + (int64_t)tok * out_tok_stride + (int64_t)h * HD;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
            const u32x2_t w = {
                tile_round2<T>(oT[d][4 * e4] * inv, oT[d][4 * e4 + 1] * inv),
                tile_round2<T>(oT[d][4 * e4 + 2] * inv, oT[d][4 * e4 + 3] * inv)};
            *reinterpret_cast<u32x2_t*>(dst + d * 32 + 8 * e4 + 4 * hh) = w;
        }
}

// Grid B * KV * tiles * nsplit, the (sequence, KV head) fastest: with a multiple of 8 of
// them the tiles that read the same keys run on one XCD. Tiles of later tokens, which
// walk more keys, come first, so that the short ones fill the last round.
template <typename T, int HD, int KG, bool A16>
__global__ __launch_bounds__(64 * kRowWaves * KG, 1) void gqa_tile_kernel(
    QueryRows<T> q, const T* __restrict__ k, const T* __restrict__ v, int64_t cap, int B, int S,
    int QT, int tiles, int G, int H, int KV, int vp, float scale, T* __restrict__ out, int chunk,
    int nsplit, float* __restrict__ part, int* __restrict__ nsplit_row) {
    const int bkv = (int)(blockIdx.x % (unsigned)(B * KV));
    const int rest = (int)(blockIdx.x / (unsigned)(B * KV));
    const int split = rest % nsplit, tile = tiles - 1 - rest / nsplit;
    const int b = bkv / KV, kvh = bkv % KV;
    TileDesc t;
    const int s0 = tile * QT;
    t.ntok = min(QT, S - s0);
    t.tok0 = b * S + s0;
    t.qpos0 = vp + s0;
    const int k1 = t.qpos0 + t.ntok;  // causal bound of the tile
    // Key splits of `chunk` keys (the last takes the rest); rows of a tile that needs one
    // split are written directly and marked 0 for the merge.
    const int ns = min(nsplit, max(1, (k1 + chunk - 1) / chunk));
    if (split == 0 && nsplit > 1) {
        for (int r = threadIdx.x; r < t.ntok * G; r += blockDim.x)
            nsplit_row[(int64_t)(t.tok0 + r / G) * H + kvh * G + r % G] = ns > 1 ? ns : 0;
    }
    if (split >= ns) return;
    const int64_t slab = (int64_t)bkv * cap * HD;
    const int k0 = split * chunk;
    const int ks1 = split == ns - 1 ? k1 : min(k1, k0 + chunk);
    attn_tile<T, HD, KG, A16>(t, kvh, G, H, q, k + slab, v + slab, scale, k0, ks1, out,
                              (int64_t)H * HD, ns > 1 ? part : nullptr, nsplit, split);
}

}  // namespace

template <typename T>
int gqa_tile(const QueryRows<T>& q, const T* k, const T* v, int64_t cap, int B, int S, int H,
             int KV, int hd, int vp, float scale, T* out, int chunk, int nsplit, float* part,
             int* nsplit_row, hipStream_t st) {
    const int G = H / KV, QT = std::max(1, kAttnRows / G), tiles = (S + QT - 1) / QT;
    const int64_t grid = (int64_t)B * KV * tiles * nsplit;
    if (grid > 0x7fffffffLL) return fail(ORTMI_E_INVALID, "GroupQueryAttention: grid too large");
    auto launch = [&](auto kernel, int kg) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * kRowWaves * kg), 0, st, q, k, v,
                           cap, B, S, QT, tiles, G, H, KV, vp, scale, out, chunk, nsplit, part,
                           nsplit_row);
        return check_launch("gqa_tile");
    };
    // Present tensors that are not 16-byte aligned pass through registers: 2048 tokens, 32
    // heads of 128 on 8, 101 us off by one element (a workgroup per query row 4380), 73 aligned.
    if ((reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15) {
        if (hd == 64) return launch(gqa_tile_kernel<T, 64, 2, false>, 2);
        if (hd == 128) return launch(gqa_tile_kernel<T, 128, 2, false>, 2);
        return fail(ORTMI_E_INVALID, "GroupQueryAttention: unaligned present tensor");
    }
    // All keys in one block: a second key group would have no work, and its waves and LDS
    // would only lengthen the start. 32 heads of 128 on 8, 8, 32 and 64 tokens: 9.6, 12.0, 12.1
    // us with two groups, 9.2, 11.1, 11.2 with one; 32 heads on 32, 32 tokens: 10.2 and 9.6.
    if (vp + S <= kKeys) {
        if (hd == 64) return launch(gqa_tile_kernel<T, 64, 1, true>, 1);
        if (hd == 96) return launch(gqa_tile_kernel<T, 96, 1, true>, 1);
        return launch(gqa_tile_kernel<T, 128, 1, true>, 1);
    }
    if (hd == 64) return launch(gqa_tile_kernel<T, 64, 2, true>, 2);
    if (hd == 96) return launch(gqa_tile_kernel<T, 96, 2, true>, 2);
    return launch(gqa_tile_kernel<T, 128, 2, true>, 2);
}

#define ORTMI_GQA_TILE(T)                                                                        \
    template int gqa_tile<T>(const QueryRows<T>&, const T*, const T*, int64_t, int, int, int,    \
                             int, int, int, float, T*, int, int, float*, int*, hipStream_t);
ORTMI_GQA_TILE(half_t)
ORTMI_GQA_TILE(uint16_t)

}  // namespace ortmi
