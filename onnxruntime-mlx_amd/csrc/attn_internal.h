// The matrix-core tiles of GroupQueryAttention prompts (attn_tile.hip), called by the entry
// point in attention.hip.
#pragma once

#include <algorithm>

#include "common.h"

namespace ortmi {

// Query rows (token, head of the group) of one tile workgroup.
constexpr int kAttnRows = 128;

// Query rows of a dense call: head h of token t at q + t * tok_stride + h * hd, rotated
// as it is loaded by rows pos of cos/sin (half = hd / 2; null: taken as it is).
template <typename T>
struct QueryRows {
    const T* q;
    int64_t tok_stride;
    const T* cos;
    const T* sin;
    int interleaved;
};

// Dense prefill over present [B, KV, cap, hd]: queries at positions vp + s, keys
// [0, vp + s]. With nsplit > 1 the keys are cut in chunks of `chunk`; rows of more than
// one chunk leave partials [row][nsplit][hd + 2] and their split count (0: written).
// Queries 16-byte aligned; k and v too at hd 96, at any element at hd 64 and 128.
template <typename T>
int gqa_tile(const QueryRows<T>& q, const T* k, const T* v, int64_t cap, int B, int S, int H,
             int KV, int hd, int vp, float scale, T* out, int chunk, int nsplit, float* part,
             int* nsplit_row, hipStream_t st);

}  // namespace ortmi
