// GroupQueryAttention for the forms the fused fp16/bf16 kernels do not take:
// fp32 tensors, per-head QK RMS-norm (inputs 14/15), an additive attention_bias
// (input 10) and head sizes other than 64/128 (multiples of 16 up to 256).
//
// Three kernels:
//  - gqa_ex_prep_kernel: one wave per (token, head) vector. Q heads: optional
//    RMS-norm, optional RoPE at position valid_past + s, each step rounded to the
//    op dtype as the reference materialises it (rust/src/ops/attention.rs:663-708),
//    written to an fp32 workspace. K heads: the same, written to present_key at row
//    valid_past + s. V heads: copied to present_value.
//  - gqa_ex_attn_kernel: one workgroup of 16 teams x 16 lanes per (token, query
//    head). Team t scores keys t, t+16, ... (a 16-lane dot product reduced inside a
//    DPP row), adds the bias, and keeps an online softmax; the 16 team states are
//    merged through LDS. Causal: query s attends keys [0, valid_past + s].
//  - gqa_f32_tile_kernel: fp32 at head sizes 64, 96 and 128 without a bias, on the fp32
//    matrix cores, where rows and keys are many enough (f32_tiles_pay).
// The KV contract (shared buffer vs growing, attention.rs:636-651) is that of
// ortmi_group_query_attention.
//
// The sliding-window cache (sliding_window_cache = 1, attention.rs:725-880) adds
// two: gqa_sw_attn_kernel (the same teams, keys read from the cached rows and the
// new rows of the query's window) and gqa_sw_present_kernel (the compacted
// present: the last cache_end(length) rows, zeros after). The prep kernel then
// takes per-sequence positions from seqlens_k and writes the new K/V rows to a
// workspace instead of present.

#include <algorithm>
#include <cmath>

#include "common.h"

namespace ortmi {
namespace {

constexpr int kTeamLanes = 16;
constexpr int kTeams = 16;
constexpr int kMaxHead = 256;
constexpr int kMaxPerLane = kMaxHead / kTeamLanes;  // 16

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Copies the first `rows` rows of every [cap, row_words] head block of src into
// the [dst_cap, row_words] block of dst (32-bit words).
__global__ __launch_bounds__(256) void kv_rows_copy_kernel(const uint32_t* __restrict__ src,
                                                           uint32_t* __restrict__ dst,
                                                           int64_t src_cap, int64_t dst_cap,
                                                           int64_t rows, int row_words,
                                                           int64_t total) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t per_head = rows * row_words;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int64_t bh = i / per_head;
        const int64_t rem = i - bh * per_head;
        dst[bh * dst_cap * row_words + rem] = src[bh * src_cap * row_words + rem];
    }
}

// grid (B*S, H + 2*KV), block 64 (one wave per head vector of hd <= 256 dims;
// lane l holds dims l, l+64, l+128, l+192).
template <typename T>
__global__ __launch_bounds__(64) void gqa_ex_prep_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, int64_t q_stride,
    int64_t kv_stride, const T* __restrict__ cos_c, const T* __restrict__ sin_c, int half,
    int interleaved, const T* __restrict__ qw, const T* __restrict__ kw, float eps,
    float* __restrict__ qf, T* __restrict__ pk, T* __restrict__ pv, int S, int H, int KV, int hd,
    int64_t pcap, int vp, const int* __restrict__ seqlens, int max_pos) {
    __shared__ float sx[kMaxHead];
    const int bs = blockIdx.x;
    const int b = bs / S, s = bs % S;
    const int head = blockIdx.y;
    const int lane = threadIdx.x;
    // Rotary position and destination row: valid_past + s for the dense contracts;
    // with seqlens (the sliding-window cache) the sequence's own past length
    // max(seqlens_k + 1 - S, 0) + s, clamped to the cos/sin rows, and row s of the
    // [B, KV, S, hd] new-row workspace.
    int64_t pos = vp + s, row = vp + s;
    if (seqlens) {
        pos = min(max((int64_t)seqlens[b] + 1 - S, (int64_t)0) + s, (int64_t)max(max_pos - 1, 0));
        row = s;
    }
    if (head >= H + KV) {  // V head: copied as is
        const int kh = head - H - KV;
        const T* src = v + (int64_t)bs * kv_stride + (int64_t)kh * hd;
        T* dst = pv + (((int64_t)b * KV + kh) * pcap + row) * hd;
        for (int d = lane; d < hd; d += 64) dst[d] = src[d];
        return;
    }
    const bool is_q = head < H;
    const int kh = head - H;
    const T* src = is_q ? q + (int64_t)bs * q_stride + (int64_t)head * hd
                        : k + (int64_t)bs * kv_stride + (int64_t)kh * hd;
    const T* w = is_q ? qw : kw;
    float x[4];
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int d = lane + 64 * e;
        x[e] = d < hd ? to_f32(src[d]) : 0.f;
        ss += x[e] * x[e];
    }
    if (w) {  // QK-norm: y = x / sqrt(mean(x^2) + eps) * w, in the op dtype
        const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)hd + eps);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int d = lane + 64 * e;
            if (d < hd) x[e] = round_to<T>(x[e] * inv * to_f32(w[d]));
        }
    }
    if (cos_c) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int d = lane + 64 * e;
            if (d < hd) sx[d] = x[e];
        }
        __syncthreads();
        const T* crow = cos_c + pos * half;
        const T* srow = sin_c + pos * half;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int d = lane + 64 * e;
            if (d >= 2 * half) continue;  // dims past the rotary span pass through
            if (interleaved) {
                const int i = d >> 1;
                const float c = to_f32(crow[i]), sn = to_f32(srow[i]);
                const float a = sx[d & ~1], bb = sx[d | 1];
                x[e] = round_to<T>((d & 1) ? bb * c + a * sn : a * c - bb * sn);
            } else {
                const int i = d < half ? d : d - half;
                const float c = to_f32(crow[i]), sn = to_f32(srow[i]);
                const float a = sx[i], bb = sx[i + half];
                x[e] = round_to<T>(d < half ? a * c - bb * sn : bb * c + a * sn);
            }
        }
    }
    if (is_q) {
        float* dst = qf + ((int64_t)bs * H + head) * hd;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int d = lane + 64 * e;
            if (d < hd) dst[d] = x[e];
        }
    } else {
        T* dst = pk + (((int64_t)b * KV + kh) * pcap + row) * hd;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int d = lane + 64 * e;
            if (d < hd) dst[d] = from_f32<T>(x[e]);
        }
    }
}

// Rows a sliding-window cache of capacity cap holds after `length` tokens: once
// full it drops its oldest gap = cap - window + 1 rows at a time
// (attention.rs:736-745).
__device__ __forceinline__ int64_t sw_cache_end(int64_t length, int64_t cap, int64_t gap) {
    if (length <= cap) return length;
    return length - gap * ((length - cap + gap - 1) / gap);
}

// Sliding-window attention, grid (B*S*H), block 256 (the teams of
// gqa_ex_attn_kernel). The sequence's p = max(seqlens_k + 1 - S, 0) earlier
// tokens sit in cache rows [0, before), the last `before` of them; query s (position
// t = p + s) attends positions (t - window, t]: cached rows first, then the new
// rows (the workspace written by the prep kernel). Equal to the reference's
// working buffer with its causal window mask (attention.rs:786-839).
template <typename T>
__global__ __launch_bounds__(256) void gqa_sw_attn_kernel(
    const float* __restrict__ qf, const T* __restrict__ past_k, const T* __restrict__ past_v,
    const T* __restrict__ knew, const T* __restrict__ vnew, const int* __restrict__ seqlens,
    T* __restrict__ out, int S, int H, int KV, int hd, int cap, int window, float scale) {
    __shared__ float s_m[kTeams], s_l[kTeams];
    __shared__ float s_acc[kTeams][kMaxHead];
    const int row = blockIdx.x;  // (b*S + s)*H + h
    const int h = row % H;
    const int bs = row / H;
    const int b = bs / S, s = bs % S;
    const int kh = h / (H / KV);
    const int team = threadIdx.x / kTeamLanes;
    const int lt = threadIdx.x % kTeamLanes;
    const int E = hd / kTeamLanes;
    const int64_t p = max((int64_t)seqlens[b] + 1 - S, (int64_t)0);
    const int64_t before = sw_cache_end(p, cap, cap - window + 1);
    const int64_t t = p + s;
    const int64_t lo = max(t - window + 1, (int64_t)0);
    const int npast = (int)max(p - lo, (int64_t)0);      // cached keys, rows [before - npast, before)
    const int first_new = (int)max(lo - p, (int64_t)0);  // new keys [first_new, s]
    const int nk = npast + s - first_new + 1;
    const int64_t slab = (int64_t)b * KV + kh;
    const T* kc = past_k + (slab * cap + (before - npast)) * hd;
    const T* vc = past_v + (slab * cap + (before - npast)) * hd;
    const T* kn = knew + (slab * S + first_new) * hd;
    const T* vn = vnew + (slab * S + first_new) * hd;
    const float* qrow = qf + (int64_t)row * hd;

    float qv[kMaxPerLane], acc[kMaxPerLane];
#pragma unroll
    for (int e = 0; e < kMaxPerLane; ++e) {
        qv[e] = e < E ? qrow[lt + kTeamLanes * e] : 0.f;
        acc[e] = 0.f;
    }
    float m = -INFINITY, l = 0.f;
    for (int base = 0; base < nk; base += kTeams) {
        const int j = base + team;
        if (j >= nk) continue;  // uniform over the team's 16 lanes
        const bool cached = j < npast;
        const T* kr = cached ? kc + (int64_t)j * hd : kn + (int64_t)(j - npast) * hd;
        const T* vr = cached ? vc + (int64_t)j * hd : vn + (int64_t)(j - npast) * hd;
        float dot = 0.f;
#pragma unroll
        for (int e = 0; e < kMaxPerLane; ++e)
            if (e < E) dot += qv[e] * to_f32(kr[lt + kTeamLanes * e]);
        const float sc = group_sum<kTeamLanes>(dot) * scale;
        const float mn = fmaxf(m, sc);
        const float corr = __expf(m - mn);  // m = -inf -> 0
        const float pe = __expf(sc - mn);
        l = l * corr + pe;
#pragma unroll
        for (int e = 0; e < kMaxPerLane; ++e)
            if (e < E) acc[e] = acc[e] * corr + pe * to_f32(vr[lt + kTeamLanes * e]);
        m = mn;
    }
    if (lt == 0) {
        s_m[team] = m;
        s_l[team] = l;
    }
#pragma unroll
    for (int e = 0; e < kMaxPerLane; ++e)
        if (e < E) s_acc[team][lt + kTeamLanes * e] = acc[e];
    __syncthreads();
    float M = -INFINITY;
    for (int tm = 0; tm < kTeams; ++tm) M = fmaxf(M, s_m[tm]);
    T* orow = out + (int64_t)row * hd;
    for (int d = threadIdx.x; d < hd; d += blockDim.x) {
        float num = 0.f, den = 0.f;
        for (int tm = 0; tm < kTeams; ++tm) {
            if (s_m[tm] == -INFINITY) continue;
            const float wt = __expf(s_m[tm] - M);
            num += wt * s_acc[tm][d];
            den += wt * s_l[tm];
        }
        orow[d] = from_f32<T>(num / den);
    }
}

// The compacted present of a sliding-window cache, 32-bit words over
// [B, KV, cap, hd]: row r < after = cache_end(p + S) holds position
// p + S - after + r (a cached row of src when before p, else a new row), rows from
// `after` on are zero (attention.rs:840-862). src is the past cache, or a copy of
// it when present is the same buffer (rows move towards the front).
__global__ __launch_bounds__(256) void gqa_sw_present_kernel(
    const uint32_t* __restrict__ src, const uint32_t* __restrict__ knew, uint32_t* __restrict__ dst,
    const int* __restrict__ seqlens, int S, int KV, int cap, int window, int row_words,
    int64_t total) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int w = (int)(i % row_words);
        const int64_t rr = i / row_words;
        const int r = (int)(rr % cap);
        const int64_t slab = rr / cap;
        const int b = (int)(slab / KV);
        const int64_t p = max((int64_t)seqlens[b] + 1 - S, (int64_t)0);
        const int gap = cap - window + 1;
        const int64_t after = sw_cache_end(p + S, cap, gap);
        uint32_t x = 0u;
        if (r < after) {
            const int64_t a = p + S - after + r;
            x = a < p ? src[(slab * cap + (a - p + sw_cache_end(p, cap, gap))) * row_words + w]
                      : knew[(slab * S + (a - p)) * row_words + w];
        }
        dst[i] = x;
    }
}

// grid (B*S*H), block 256 = 16 teams of 16 lanes; lane l of a team holds dims
// l, l+16, ..., l+16*(E-1) with E = hd / 16.
template <typename T>
__global__ __launch_bounds__(256) void gqa_ex_attn_kernel(
    const float* __restrict__ qf, const T* __restrict__ pk, const T* __restrict__ pv,
    const T* __restrict__ bias, int64_t bias_sb, int64_t bias_sh, int64_t bias_ss,
    T* __restrict__ out, int S, int H, int KV, int hd, int64_t pcap, int vp, float scale) {
    __shared__ float s_m[kTeams], s_l[kTeams];
    __shared__ float s_acc[kTeams][kMaxHead];
    const int row = blockIdx.x;  // (b*S + s)*H + h
    const int h = row % H;
    const int bs = row / H;
    const int b = bs / S, s = bs % S;
    const int G = H / KV;
    const int kh = h / G;
    const int team = threadIdx.x / kTeamLanes;
    const int lt = threadIdx.x % kTeamLanes;
    const int E = hd / kTeamLanes;
    const int nk = vp + s + 1;  // causal: keys [0, vp + s]
    const float* qrow = qf + (int64_t)row * hd;
    const T* kb = pk + ((int64_t)b * KV + kh) * pcap * hd;
    const T* vb = pv + ((int64_t)b * KV + kh) * pcap * hd;
    const T* brow = bias ? bias + b * bias_sb + h * bias_sh + s * bias_ss : nullptr;

    float qv[kMaxPerLane], acc[kMaxPerLane];
#pragma unroll
    for (int e = 0; e < kMaxPerLane; ++e) {
        qv[e] = e < E ? qrow[lt + kTeamLanes * e] : 0.f;
        acc[e] = 0.f;
    }
    float m = -INFINITY, l = 0.f;
    // Every lane runs the same trip count; a team whose key is past the end skips it.
    for (int base = 0; base < nk; base += kTeams) {
        const int j = base + team;
        const bool valid = j < nk;
        const T* kr = kb + (int64_t)(valid ? j : 0) * hd;
        float dot = 0.f;
#pragma unroll
        for (int e = 0; e < kMaxPerLane; ++e)
            if (e < E) dot += qv[e] * to_f32(kr[lt + kTeamLanes * e]);
        dot = group_sum<kTeamLanes>(dot);
        float sc = dot * scale + (brow && valid ? to_f32(brow[j]) : 0.f);
        if (!valid || sc == -INFINITY) continue;  // uniform over the team's 16 lanes
        const float mn = fmaxf(m, sc);
        const float corr = __expf(m - mn);  // m = -inf -> 0
        const float p = __expf(sc - mn);
        l = l * corr + p;
        const T* vr = vb + (int64_t)j * hd;
#pragma unroll
        for (int e = 0; e < kMaxPerLane; ++e)
            if (e < E) acc[e] = acc[e] * corr + p * to_f32(vr[lt + kTeamLanes * e]);
        m = mn;
    }
    if (lt == 0) {
        s_m[team] = m;
        s_l[team] = l;
    }
#pragma unroll
    for (int e = 0; e < kMaxPerLane; ++e)
        if (e < E) s_acc[team][lt + kTeamLanes * e] = acc[e];
    __syncthreads();
    float M = -INFINITY;
    for (int t = 0; t < kTeams; ++t) M = fmaxf(M, s_m[t]);
    T* orow = out + (int64_t)row * hd;
    for (int d = threadIdx.x; d < hd; d += blockDim.x) {
        float num = 0.f, den = 0.f;
        for (int t = 0; t < kTeams; ++t) {
            if (s_m[t] == -INFINITY) continue;
            const float wt = __expf(s_m[t] - M);
            num += wt * s_acc[t][d];
            den += wt * s_l[t];
        }
        orow[d] = from_f32<T>(num / den);  // every key masked: 0/0, as the softmax gives
    }
}

// fp32 without bias on the fp32 matrix cores (v_mfma_f32_32x32x2_f32: every product and sum
// in fp32, as in the kernel above). A workgroup takes 32 query rows (token, head of the
// group) of one KV head, and its 8 waves take every eighth tile of 32 keys, straight from
// memory: the rows of a tile are read once per workgroup, and the waves' states are merged
// through LDS at the end.
//   S^T = K Q^T    lane l: key (query) l & 31, step s: dims s and HD/2 + s for the lane
//                  halves, so a lane's share of a row is contiguous
//   O^T += V^T P^T step e: the lane halves' keys of accumulator e, P straight from the
//                  softmax's registers
// Bound: short prompts by the latency of a tile (two per wave at 512 keys), long ones by
// the fp32 matrix rate (64 cycles per instruction of 4096 operations). One workgroup per
// query row before: 512 tokens, 14 heads of 64 on 2: 114 -> 26 us; B 2, 300 tokens behind 2000,
// 32 heads of 128 on 8: 4400 -> 594 us; B 2, one token behind 2048: 445 -> 166 us. Errors
// against 64 bits 1.4e-7 -> 1.3e-7, 2.8e-7 -> 1.9e-7, 2.8e-7 -> 1.9e-7.
typedef float f32x16_t __attribute__((ext_vector_type(16)));
constexpr int kF32Rows = 32, kF32Keys = 32, kF32Waves = 8;
// S^T over pieces [I, I + N) of the head dims.
template <int I, int N>
__device__ __forceinline__ f32x16_t f32_dot_tree(const float4* k4, const float4* q4) {
    if constexpr (N == 1) {
        f32x16_t a;
#pragma unroll
        for (int e = 0; e < 16; ++e) a[e] = 0.f;
        a = __builtin_amdgcn_mfma_f32_32x32x2f32(k4[I].x, q4[I].x, a, 0, 0, 0);
        a = __builtin_amdgcn_mfma_f32_32x32x2f32(k4[I].y, q4[I].y, a, 0, 0, 0);
        a = __builtin_amdgcn_mfma_f32_32x32x2f32(k4[I].z, q4[I].z, a, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_32x32x2f32(k4[I].w, q4[I].w, a, 0, 0, 0);
    } else {
        const f32x16_t a = f32_dot_tree<I, N / 2>(k4, q4);
        const f32x16_t b = f32_dot_tree<I + N / 2, N - N / 2>(k4, q4);
        return a + b;
    }
}
template <int HD>
__global__ __launch_bounds__(64 * kF32Waves, 1) void gqa_f32_tile_kernel(
    const float* __restrict__ qf, const float* __restrict__ pk, const float* __restrict__ pv,
    float* __restrict__ out, int S, int H, int KV, int64_t pcap, int vp, float scale, int tiles) {
    constexpr int DT = HD / 32, HALF = HD / 2;
    __shared__ float s_o[kF32Waves][DT * 16 * 64];
    __shared__ float s_m[kF32Waves][32], s_l[kF32Waves][32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 31, hh = lane >> 5;
    const int G = H / KV, rows = S * G;
    // Tiles of later tokens, which walk more keys, first.
    const int tile = tiles - 1 - (int)blockIdx.x % tiles, bkv = (int)blockIdx.x / tiles;
    const int b = bkv / KV, kvh = bkv % KV;
    const int r0 = tile * kF32Rows, r = min(r0 + li, rows - 1);
    const int tok = r / G, head = kvh * G + r % G;
    const int nk = vp + min(r0 + kF32Rows - 1, rows - 1) / G + 1;  // causal bound of the tile
    const int seen_all = vp + r0 / G;  // keys up to here are visible to every row
    const int last = vp + tok;         // this row's last key
    const float* const kbase = pk + (int64_t)bkv * pcap * HD;
    const float* const vbase = pv + (int64_t)bkv * pcap * HD;

    float4 q4[HALF / 4];
    {
        const float* qrow = qf + (((int64_t)b * S + tok) * H + head) * HD + hh * HALF;
#pragma unroll
        for (int i = 0; i < HALF / 4; ++i) {
            q4[i] = *reinterpret_cast<const float4*>(qrow + 4 * i);
            if (scale < 0.f) q4[i] = make_float4(-q4[i].x, -q4[i].y, -q4[i].z, -q4[i].w);
        }
    }
    constexpr float kLog2e = 1.4426950408889634f;
    // Maxima are kept of the raw scores (a negative scale turns the sign of Q) and P is
    // exp2((s - m) * sc2): the difference is exact or nearly so where P is large, so that
    // no rounding of a large product reaches the exponent.
    const float sc2 = fabsf(scale) * kLog2e;
    float m = -INFINITY, l = 0.f;
    f32x16_t o[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[d][e] = 0.f;

    for (int kb = wave * kF32Keys; kb < nk; kb += kF32Waves * kF32Keys) {
        // Rows past the end read the last one; their keys are masked.
        const float* krow = kbase + (int64_t)min(kb + li, nk - 1) * HD + hh * HALF;
        float4 k4[HALF / 4];
#pragma unroll
        for (int i = 0; i < HALF / 4; ++i) k4[i] = *reinterpret_cast<const float4*>(krow + 4 * i);
        // The sum over the head dims as a tree over pieces of four steps: summed in one chain
        // the error was twice that of the kernel above (B 2, one token, 2048 keys, head 128:
        // 5.0e-7 relative to 64 bits against 2.8e-7).
        f32x16_t st = f32_dot_tree<0, HALF / 4>(k4, q4);
        // Accumulator e holds key 8 (e / 4) + 4 hh + e % 4 of query li.
        const bool part = kb + kF32Keys - 1 > seen_all;
        float mt = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int j = kb + 8 * (e / 4) + 4 * hh + (e & 3);
            st[e] = !part || j <= last ? st[e] : -INFINITY;
            mt = fmaxf(mt, st[e]);
        }
        const LanePair pm = swap32(mt);
        const float mn = fmaxf(m, fmaxf(pm.a, pm.b));
        const float corr = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - mn) * sc2);
        const float ref = mn == -INFINITY ? 0.f : mn;
        float lt = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            st[e] = __builtin_amdgcn_exp2f((st[e] - ref) * sc2);
            lt += st[e];
        }
        l = l * corr + lt;  // this lane's 16 of the tile's keys
        m = mn;
        const float* vcol = vbase + li;
        auto vrow = [&](int e) {
            return vcol + (int64_t)min(kb + 8 * (e / 4) + 4 * hh + (e & 3), nk - 1) * HD;
        };
        // A hidden key must not reach a row through 0 * infinity: where some keys are hidden
        // and some values are not finite, the products are taken one key at a time.
        bool odd = false;
        if (part) {
            float z = 0.f;
#pragma unroll
            for (int e = 0; e < 16; ++e)
#pragma unroll
                for (int d = 0; d < DT; ++d) z = fmaf(vrow(e)[d * 32], 0.f, z);
            odd = __any(z != 0.f);  // NaN
        }
        if (!odd) {
            // Each tile sums on its own, in two chains, before it joins O.
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                f32x16_t t0, t1;
#pragma unroll
                for (int e = 0; e < 16; ++e) t0[e] = t1[e] = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    t0 = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow(e)[d * 32], st[e], t0, 0, 0, 0);
                    t1 = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow(e + 8)[d * 32], st[e + 8], t1, 0,
                                                              0, 0);
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) o[d][e] = fmaf(o[d][e], corr, t0[e] + t1[e]);
            }
        } else {
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[d][e] *= corr;
#pragma unroll
            for (int e = 0; e < 16; ++e)
                for (int h2 = 0; h2 < 2; ++h2) {
                    const int j = kb + 8 * (e / 4) + 4 * h2 + (e & 3);
                    const float pj = __shfl(st[e], li + 32 * h2, 64);
                    const float* vr = vbase + (int64_t)min(j, nk - 1) * HD;
                    if (j > last) continue;
#pragma unroll
                    for (int d = 0; d < DT; ++d)
#pragma unroll
                        for (int i = 0; i < 16; ++i)
                            o[d][i] = fmaf(pj, vr[d * 32 + 8 * (i / 4) + 4 * hh + (i & 3)], o[d][i]);
                }
        }
    }
    const LanePair pl = swap32(l);
    l = pl.a + pl.b;
    if (hh == 0) {
        s_m[wave][li] = m;
        s_l[wave][li] = l;
    }
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) s_o[wave][(d * 16 + e) * 64 + lane] = o[d][e];
    __syncthreads();
    // Four consecutive dims of one row per thread and turn.
    for (int i = threadIdx.x; i < DT * 4 * 64; i += 64 * kF32Waves) {
        const int ln = i & 63, q = ln & 31, d = i / 256, e4 = (i >> 6) & 3;
        if (r0 + q >= rows) continue;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < kF32Waves; ++w) M = fmaxf(M, s_m[w][q]);
        float den = 0.f, num[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kF32Waves; ++w) {
            // A wave without a visible key has zeros, or NaN from NaN scores.
            const float f =
                s_m[w][q] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((s_m[w][q] - M) * sc2);
            den = fmaf(f, s_l[w][q], den);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                num[e] = fmaf(f, s_o[w][(d * 16 + 4 * e4 + e) * 64 + ln], num[e]);
        }
        const int tq = (r0 + q) / G, hq = kvh * G + (r0 + q) % G;
        float* dst = out + (((int64_t)b * S + tq) * H + hq) * HD + d * 32 + 8 * e4 + 4 * (ln >> 5);
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = num[e] / den;  // every key masked: 0/0
    }
}

// Whether the tiles finish an fp32 call before a workgroup per query row does (head 64, 96 or
// 128). Few keys or rows leave a tile's waves idle: 32 heads of 128 on 8, one token over 17
// keys, 15.0 us against 10.3 with a workgroup per row; 33 tokens 26.5 and 15.7; 32 sequences
// of one token over 91 keys, a KV head to each query head, 100 and 37; level at about 100
// keys, and 300 tokens 73 and 155. The estimates are in us, fitted to 7800 calls on MI355X
// (1-512 tokens, 1-32 sequences, up to 4500 keys, 8-32 heads); with the tiles favoured by
// less than a fifth the rows keep the call, and of those calls 6 were slower on the chosen
// kernel than a workgroup per row by more than 3 %, the worst 1.2 times.
bool f32_tiles_pay(int64_t B, int64_t S, int64_t H, int64_t KV, int hd, int64_t vp) {
    struct Cost {
        double row0, row_key, row, pair;          // a workgroup per row
        double tile0, round, round_key, tile_key;  // tiles
        int per_cu;                                // tiles that share a CU (LDS)
    };
    const Cost c = hd == 64   ? Cost{7.1, .07, .0022, 3.4e-5, 0., 11., .018, 1.6e-4, 2}
                   : hd == 96 ? Cost{7.7, .10, .0026, 4.7e-5, 3., 11.4, .052, 1.7e-4, 1}
                              : Cost{8.2, .13, .0029, 6.2e-5, 3.9, 12.5, .072, 2.0e-4, 1};
    const double n = (double)(vp + S), seen = (double)vp + 0.5 * (double)(S + 1);
    const double rows = (double)(B * S * H);
    const int64_t tiles = B * KV * ((S * (H / KV) + kF32Rows - 1) / kF32Rows);
    const int64_t slots = (int64_t)device_cu_count() * c.per_cu;
    const double rounds = (double)((tiles + slots - 1) / slots);
    double tile = c.tile0 + rounds * (c.round + c.round_key * n) + c.tile_key * tiles * seen;
    // Two or three waves with keys that are hidden to some rows, at heads of 96 and 128.
    if (hd > 64 && S > 1 && n > 32 && n <= 96) tile += 6.;
    return 1.2 * tile < c.row0 + c.row_key * n + c.row * rows + c.pair * rows * seen;
}

template <typename T>
int run_gqa_ex(const void* query, const void* key, const void* value, const void* past_key,
               const void* past_value, int64_t cap, int total, const void* cos_c,
               const void* sin_c, int half, int interleaved, const void* qw, const void* kw,
               float eps, const void* bias, int64_t sb, int64_t sh, int64_t ss, void* output,
               void* pk, void* pv, int B, int S, int H, int KV, int hd, float scale, void* ws,
               hipStream_t st) {
    int vp = total - S;
    bool shared;
    if (vp < 0 || vp > cap) {
        shared = false;
        vp = (int)cap;
    } else {
        shared = cap > vp;
    }
    const int64_t pcap = shared ? cap : cap + S;
    const bool packed = key == nullptr;
    const int64_t q_stride = packed ? (int64_t)(H + 2 * KV) * hd : (int64_t)H * hd;
    const int64_t kv_stride = packed ? q_stride : (int64_t)KV * hd;
    const T* q = static_cast<const T*>(query);
    const T* k = packed ? q + (int64_t)H * hd : static_cast<const T*>(key);
    const T* v = packed ? q + (int64_t)(H + KV) * hd : static_cast<const T*>(value);
    const float sc = scale != 0.f ? scale : 1.0f / sqrtf((float)hd);
    const bool aliased = (pk == past_key) && (pv == past_value);
    if (!aliased && cap > 0) {
        // Shared contract into a separate present: all cap rows; growing: the cap past rows.
        const int row_words = hd * (int)sizeof(T) / 4;
        const int64_t total_w = (int64_t)B * KV * cap * row_words;
        const int grid = (int)std::min<int64_t>((total_w + 255) / 256, 65536);
        hipLaunchKernelGGL(kv_rows_copy_kernel, dim3(grid), dim3(256), 0, st,
                           static_cast<const uint32_t*>(past_key), static_cast<uint32_t*>(pk), cap,
                           pcap, cap, row_words, total_w);
        hipLaunchKernelGGL(kv_rows_copy_kernel, dim3(grid), dim3(256), 0, st,
                           static_cast<const uint32_t*>(past_value), static_cast<uint32_t*>(pv),
                           cap, pcap, cap, row_words, total_w);
        if (int rc = check_launch("gqa_ex kv copy")) return rc;
    }
    float* qf = static_cast<float*>(ws);
    hipLaunchKernelGGL((gqa_ex_prep_kernel<T>), dim3(B * S, H + 2 * KV), dim3(64), 0, st, q, k, v,
                       q_stride, kv_stride, static_cast<const T*>(cos_c),
                       static_cast<const T*>(sin_c), half, interleaved, static_cast<const T*>(qw),
                       static_cast<const T*>(kw), eps, qf, static_cast<T*>(pk),
                       static_cast<T*>(pv), S, H, KV, hd, pcap, vp, nullptr, 0);
    if (int rc = check_launch("gqa_ex_prep")) return rc;
    if constexpr (std::is_same<T, float>::value) {
        // Row vectors of 16 bytes: ws and present are read so.
        const auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
        const int64_t tiles = ((int64_t)S * (H / KV) + kF32Rows - 1) / kF32Rows;
        const int64_t grid = (int64_t)B * KV * tiles;
        if (!bias && a16(ws) && a16(pk) && (hd == 64 || hd == 96 || hd == 128) &&
            grid <= 0x7fffffffLL && f32_tiles_pay(B, S, H, KV, hd, vp)) {
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * kF32Waves), 0, st, qf,
                                   static_cast<const float*>(pk), static_cast<const float*>(pv),
                                   static_cast<float*>(output), S, H, KV, pcap, vp, sc, (int)tiles);
                return check_launch("gqa_f32_tile");
            };
            if (hd == 64) return launch(gqa_f32_tile_kernel<64>);
            if (hd == 96) return launch(gqa_f32_tile_kernel<96>);
            return launch(gqa_f32_tile_kernel<128>);
        }
    }
    hipLaunchKernelGGL((gqa_ex_attn_kernel<T>), dim3(B * S * H), dim3(256), 0, st, qf,
                       static_cast<const T*>(pk), static_cast<const T*>(pv),
                       static_cast<const T*>(bias), sb, sh, ss, static_cast<T*>(output), S, H, KV,
                       hd, pcap, vp, sc);
    return check_launch("gqa_ex_attn");
}


// Sliding-window cache (attention.rs:725-880): prep (positions from seqlens_k, new
// rows to the workspace), attention over each query's window, then the compacted
// present. When present is the past buffer its rows move towards the front, so
// the past is copied aside first.
template <typename T>
int run_gqa_sliding(const void* query, const void* key, const void* value, const void* past_key,
                    const void* past_value, int cap, const int* seqlens, const void* cos_c,
                    const void* sin_c, int half, int max_pos, int interleaved, const void* qw,
                    const void* kw, float eps, int window, void* output, void* pk, void* pv,
                    int B, int S, int H, int KV, int hd, float scale, void* ws, hipStream_t st) {
    const bool packed = key == nullptr;
    const int64_t q_stride = packed ? (int64_t)(H + 2 * KV) * hd : (int64_t)H * hd;
    const int64_t kv_stride = packed ? q_stride : (int64_t)KV * hd;
    const T* q = static_cast<const T*>(query);
    const T* k = packed ? q + (int64_t)H * hd : static_cast<const T*>(key);
    const T* v = packed ? q + (int64_t)(H + KV) * hd : static_cast<const T*>(value);
    const float sc = scale != 0.f ? scale : 1.0f / sqrtf((float)hd);
    char* w = static_cast<char*>(ws);
    float* qf = reinterpret_cast<float*>(w);
    w += align256((size_t)B * S * H * hd * 4);
    const size_t new_bytes = align256((size_t)B * KV * S * hd * sizeof(T));
    T* knew = reinterpret_cast<T*>(w);
    T* vnew = reinterpret_cast<T*>(w + new_bytes);
    w += 2 * new_bytes;
    hipLaunchKernelGGL((gqa_ex_prep_kernel<T>), dim3(B * S, H + 2 * KV), dim3(64), 0, st, q, k, v,
                       q_stride, kv_stride, static_cast<const T*>(cos_c),
                       static_cast<const T*>(sin_c), half, interleaved, static_cast<const T*>(qw),
                       static_cast<const T*>(kw), eps, qf, knew, vnew, S, H, KV, hd, (int64_t)S, 0,
                       seqlens, max_pos);
    if (int rc = check_launch("gqa_sliding_prep")) return rc;
    hipLaunchKernelGGL((gqa_sw_attn_kernel<T>), dim3(B * S * H), dim3(256), 0, st, qf,
                       static_cast<const T*>(past_key), static_cast<const T*>(past_value), knew,
                       vnew, seqlens, static_cast<T*>(output), S, H, KV, hd, cap, window, sc);
    if (int rc = check_launch("gqa_sliding_attn")) return rc;
    const int row_words = hd * (int)sizeof(T) / 4;
    const int64_t total_w = (int64_t)B * KV * cap * row_words;
    if (total_w == 0) return ORTMI_OK;
    const int grid = (int)std::min<int64_t>((total_w + 255) / 256, 65536);
    const void* srcs[2] = {past_key, past_value};
    const T* news[2] = {knew, vnew};
    void* dsts[2] = {pk, pv};
    for (int i = 0; i < 2; ++i) {
        const uint32_t* src = static_cast<const uint32_t*>(srcs[i]);
        if (srcs[i] == dsts[i]) {  // in place: read the old rows from a copy
            uint32_t* copy = reinterpret_cast<uint32_t*>(w);
            hipLaunchKernelGGL(kv_rows_copy_kernel, dim3(grid), dim3(256), 0, st, src, copy,
                               (int64_t)cap, (int64_t)cap, (int64_t)cap, row_words, total_w);
            src = copy;
        }
        hipLaunchKernelGGL(gqa_sw_present_kernel, dim3(grid), dim3(256), 0, st, src,
                           reinterpret_cast<const uint32_t*>(news[i]),
                           static_cast<uint32_t*>(dsts[i]), seqlens, S, KV, cap, window,
                           row_words, total_w);
        if (int rc = check_launch("gqa_sliding_present")) return rc;
    }
    return ORTMI_OK;
}

}  // namespace
}  // namespace ortmi

using namespace ortmi;

extern "C" size_t ortmi_group_query_attention_ex_workspace_size(int64_t batch, int64_t seq_len,
                                                                int64_t num_heads,
                                                                int64_t head_size) {
    if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || head_size <= 0) return 0;
    return align256((size_t)batch * seq_len * num_heads * head_size * 4);
}

extern "C" int ortmi_group_query_attention_ex(
    const void* query, const void* key, const void* value, const void* past_key,
    const void* past_value, int64_t past_cap, int32_t total_sequence_length, const void* cos_cache,
    const void* sin_cache, int64_t rotary_half, int64_t max_pos, const void* q_norm_weight,
    const void* k_norm_weight, float qk_norm_epsilon, const void* attention_bias,
    int64_t bias_batch, int64_t bias_heads, int64_t bias_rows, int64_t bias_cols, void* output,
    void* present_key, void* present_value, int64_t batch, int64_t seq_len, int64_t num_heads,
    int64_t kv_num_heads, int64_t head_size, float scale, int32_t rotary_interleaved,
    int32_t dtype, void* workspace, size_t workspace_bytes, void* stream) {
    // Claim/op contract of rust/src/ops/attention.rs:1520-1745 and 556-952.
    ORTMI_REQUIRE(num_heads > 0 && kv_num_heads > 0 && num_heads % kv_num_heads == 0,
                  "GroupQueryAttention: num_heads must be a positive multiple of kv_num_heads");
    ORTMI_REQUIRE(head_size > 0 && head_size % 16 == 0 && head_size <= 256,
                  "GroupQueryAttention: head_size must be a multiple of 16 up to 256");
    ORTMI_REQUIRE(batch > 0 && seq_len > 0 && past_cap >= 0 && num_heads <= 65535 &&
                      batch * seq_len * num_heads <= 0x7fffffffLL,
                  "GroupQueryAttention: bad shape");
    ORTMI_REQUIRE(query && output && present_key && present_value,
                  "GroupQueryAttention: null tensor");
    ORTMI_REQUIRE((key == nullptr) == (value == nullptr),
                  "GroupQueryAttention: key and value must both be given or both be packed");
    ORTMI_REQUIRE(past_cap == 0 || (past_key && past_value), "GroupQueryAttention: null past");
    ORTMI_REQUIRE((q_norm_weight == nullptr) == (k_norm_weight == nullptr),
                  "GroupQueryAttention: q_norm_weight and k_norm_weight must be provided together");
    const bool rotary = cos_cache != nullptr;
    ORTMI_REQUIRE(rotary == (sin_cache != nullptr),
                  "GroupQueryAttention: cos_cache and sin_cache must both be given");
    int vp = total_sequence_length - (int)seq_len;
    if (vp < 0 || vp > past_cap) vp = (int)past_cap;
    if (rotary) {
        ORTMI_REQUIRE(rotary_half > 0 && 2 * rotary_half <= head_size,
                      "GroupQueryAttention: rotary dim exceeds head_size");
        ORTMI_REQUIRE(vp + seq_len <= max_pos,
                      "GroupQueryAttention: position exceeds the cos/sin cache");
    }
    int64_t sb = 0, sh = 0, ss = 0;
    if (attention_bias) {
        ORTMI_REQUIRE((bias_batch == 1 || bias_batch == batch) &&
                          (bias_heads == 1 || bias_heads == num_heads) && bias_rows >= seq_len &&
                          bias_cols >= vp + seq_len,
                      "GroupQueryAttention: attention_bias must be [batch or 1, num_heads or 1, "
                      ">= sequence_length, >= attended keys]");
        ss = bias_cols;
        sh = bias_heads > 1 ? bias_rows * bias_cols : 0;
        sb = bias_batch > 1 ? bias_heads * bias_rows * bias_cols : 0;
    }
    if (past_cap > 0 && (past_key == present_key) != (past_value == present_value))
        return fail(ORTMI_E_INVALID, "GroupQueryAttention: present_key/value alias mismatch");
    const bool shared_c = (total_sequence_length - seq_len >= 0) &&
                          (total_sequence_length - seq_len <= past_cap) &&
                          past_cap > total_sequence_length - seq_len;
    if (!shared_c && past_cap > 0)
        ORTMI_REQUIRE(past_key != present_key,
                      "GroupQueryAttention: growing contract cannot write in place");
    if (shared_c)
        ORTMI_REQUIRE(total_sequence_length <= past_cap,
                      "GroupQueryAttention: total_sequence_length exceeds the KV buffer capacity");
    const size_t need =
        ortmi_group_query_attention_ex_workspace_size(batch, seq_len, num_heads, head_size);
    if (!workspace || workspace_bytes < need)
        return fail(ORTMI_E_WORKSPACE, "GroupQueryAttention: workspace too small");
    hipStream_t st = as_stream(stream);
#define ORTMI_GQA_EX(T)                                                                          \
    return run_gqa_ex<T>(query, key, value, past_key, past_value, past_cap,                      \
                         total_sequence_length, cos_cache, sin_cache, (int)rotary_half,          \
                         rotary_interleaved, q_norm_weight, k_norm_weight, qk_norm_epsilon,      \
                         attention_bias, sb, sh, ss, output, present_key, present_value,         \
                         (int)batch, (int)seq_len, (int)num_heads, (int)kv_num_heads,            \
                         (int)head_size, scale, workspace, st)
    if (dtype == ORTMI_F32) ORTMI_GQA_EX(float);
    if (dtype == ORTMI_F16) ORTMI_GQA_EX(half_t);
    if (dtype == ORTMI_BF16) ORTMI_GQA_EX(uint16_t);
#undef ORTMI_GQA_EX
    return fail(ORTMI_E_INVALID, "GroupQueryAttention: dtype must be fp32, fp16 or bf16");
}

extern "C" size_t ortmi_group_query_attention_sliding_workspace_size(int64_t batch,
                                                                     int64_t seq_len,
                                                                     int64_t num_heads,
                                                                     int64_t kv_num_heads,
                                                                     int64_t head_size,
                                                                     int64_t past_cap) {
    if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || kv_num_heads <= 0 || head_size <= 0 ||
        past_cap < 0)
        return 0;
    // fp32 queries, new K/V rows and one past copy, sized for 4-byte elements.
    return align256((size_t)batch * seq_len * num_heads * head_size * 4) +
           2 * align256((size_t)batch * kv_num_heads * seq_len * head_size * 4) +
           align256((size_t)batch * kv_num_heads * past_cap * head_size * 4);
}

extern "C" int ortmi_group_query_attention_sliding(
    const void* query, const void* key, const void* value, const void* past_key,
    const void* past_value, int64_t past_cap, const int32_t* seqlens_k, const void* cos_cache,
    const void* sin_cache, int64_t rotary_half, int64_t max_pos, const void* q_norm_weight,
    const void* k_norm_weight, float qk_norm_epsilon, int64_t local_window_size, void* output,
    void* present_key, void* present_value, int64_t batch, int64_t seq_len, int64_t num_heads,
    int64_t kv_num_heads, int64_t head_size, float scale, int32_t rotary_interleaved,
    int32_t dtype, void* workspace, size_t workspace_bytes, void* stream) {
    // attention.rs:725-735 and the claim at 1552-1575.
    ORTMI_REQUIRE(num_heads > 0 && kv_num_heads > 0 && num_heads % kv_num_heads == 0,
                  "GroupQueryAttention: num_heads must be a positive multiple of kv_num_heads");
    ORTMI_REQUIRE(head_size > 0 && head_size % 16 == 0 && head_size <= 256,
                  "GroupQueryAttention: head_size must be a multiple of 16 up to 256");
    ORTMI_REQUIRE(batch > 0 && seq_len > 0 && num_heads <= 65535 && past_cap <= 0x7fffffffLL &&
                      batch * seq_len * num_heads <= 0x7fffffffLL,
                  "GroupQueryAttention: bad shape");
    ORTMI_REQUIRE(local_window_size > 0 && local_window_size <= past_cap,
                  "GroupQueryAttention: sliding cache requires 0 < local_window_size <= capacity");
    ORTMI_REQUIRE(query && output && present_key && present_value && past_key && past_value &&
                      seqlens_k,
                  "GroupQueryAttention: null tensor");
    ORTMI_REQUIRE((key == nullptr) == (value == nullptr),
                  "GroupQueryAttention: key and value must both be given or both be packed");
    ORTMI_REQUIRE((q_norm_weight == nullptr) == (k_norm_weight == nullptr),
                  "GroupQueryAttention: q_norm_weight and k_norm_weight must be provided together");
    const bool rotary = cos_cache != nullptr;
    ORTMI_REQUIRE(rotary == (sin_cache != nullptr),
                  "GroupQueryAttention: cos_cache and sin_cache must both be given");
    if (rotary)
        ORTMI_REQUIRE(rotary_half > 0 && 2 * rotary_half <= head_size && max_pos > 0,
                      "GroupQueryAttention: rotary dim exceeds head_size");
    if ((past_key == present_key) != (past_value == present_value))
        return fail(ORTMI_E_INVALID, "GroupQueryAttention: present_key/value alias mismatch");
    const size_t need = ortmi_group_query_attention_sliding_workspace_size(
        batch, seq_len, num_heads, kv_num_heads, head_size, past_cap);
    if (!workspace || workspace_bytes < need)
        return fail(ORTMI_E_WORKSPACE, "GroupQueryAttention: workspace too small");
    hipStream_t st = as_stream(stream);
#define ORTMI_GQA_SW(T)                                                                          \
    return run_gqa_sliding<T>(query, key, value, past_key, past_value, (int)past_cap, seqlens_k,  \
                              cos_cache, sin_cache, (int)rotary_half, (int)max_pos,              \
                              rotary_interleaved, q_norm_weight, k_norm_weight, qk_norm_epsilon, \
                              (int)local_window_size, output, present_key, present_value,        \
                              (int)batch, (int)seq_len, (int)num_heads, (int)kv_num_heads,       \
                              (int)head_size, scale, workspace, st)
    if (dtype == ORTMI_F32) ORTMI_GQA_SW(float);
    if (dtype == ORTMI_F16) ORTMI_GQA_SW(half_t);
    if (dtype == ORTMI_BF16) ORTMI_GQA_SW(uint16_t);
#undef ORTMI_GQA_SW
    return fail(ORTMI_E_INVALID, "GroupQueryAttention: dtype must be fp32, fp16 or bf16");
}
