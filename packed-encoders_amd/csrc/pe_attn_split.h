// Split calls: few query rows against long key segments (requests that continue a cached prefix, from
// one decoded token to a short tail). A workgroup of the tiled kernels walks its tile's keys
// one after another, so such a call fills a fraction of the chip and lasts as long as its longest
// segment: 16 segments of up to 8,192 keys at 32:8 heads of 128 were 128 workgroups and 128 serial
// key tiles, the call 245 us for 327 MB. Split, a workgroup takes one chunk of the keys (grid y)
// and writes its unnormalised rows with their maximum and sum in fp32, and merge_kernel adds the
// chunks of a row: 89 us (3.7 TB/s). split_of (pe_attn_capi.hip) holds the rule and its figures.
//
// The tiled kernels take SPLIT as a template flag: same loads, products and softmax over the
// chunk, one query tile per work entry, partial rows instead of the epilogue. A row whose tile
// reads a single chunk gets the bits of the unsplit kernel (its weight is 1).
#pragma once

#include "pe_attn_stage.h"

namespace pe {

// The work entry and head group of a split call's workgroup. Those that read the same keys (the head
// groups of one kv head, over the `tiles` consecutive entries that a segment has on average) go to one
// XCD, eight workgroups apart, so that all but the first of them find the keys in that XCD's L2;
// dealt one by one to the XCDs, each fetched them again (split_deal, pe_attn_capi.hip).
__device__ __forceinline__ void split_item(const AttnParams &p, int &entry, int &hg) {
    const int x = blockIdx.x, members = p.share * p.tiles;
    if (members <= 1) {
        entry = x / p.hgroups;
        hg = x - entry * p.hgroups;
        return;
    }
    const int round = x / (8 * members), r = x - round * 8 * members;
    const int unit = round * 8 + (r & 7), member = r >> 3, kv_heads = p.hgroups / p.share;
    const int block = unit / kv_heads, tile = member / p.share;
    entry = block * p.tiles + tile;
    hg = (unit - block * kv_heads) * p.share + member - tile * p.share;
}

// Place of a row's partials: (chunk, query row, head).
__device__ __forceinline__ int64_t part_slot(const AttnParams &p, int chunk, int row, int qh) {
    return ((int64_t)chunk * p.total_q + row) * p.hq + qh;
}

// A wave's 32-row block in the 32x32 accumulator layout: lane (col, kg) holds dims
// 32 db + 8 jj + 4 kg + i of its row. `row` is the packed query row; rows past the segment or the
// call's tokens are not stored.
template <int DB>
__device__ __forceinline__ void store_part(const f32x16 (&o)[DB], float m, float l, int kg, const AttnParams &p, int row,
                                           int qh, bool live) {
    if (!live || row >= p.total_q) return;
    const int64_t slot = part_slot(p, blockIdx.y, row, qh);
    float *dst = p.part_o + slot * (32 * DB) + 4 * kg;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
            *reinterpret_cast<f32x4 *>(dst + 32 * db + 8 * jj) =
                f32x4{o[db][4 * jj], o[db][4 * jj + 1], o[db][4 * jj + 2], o[db][4 * jj + 3]};
    if (kg == 0) {
        p.part_ml[2 * slot] = m;
        p.part_ml[2 * slot + 1] = l;
    }
}

// A wave's 16-row block in the 16x16 accumulator layout: lane (c16, g4) holds dims 16 db + 4 g4 + i.
template <int DB>
__device__ __forceinline__ void store_part16(const f32x4 (&o)[DB], float m, float l, int g4, const AttnParams &p, int row,
                                             int qh, bool live) {
    if (!live || row >= p.total_q) return;
    const int64_t slot = part_slot(p, blockIdx.y, row, qh);
    float *dst = p.part_o + slot * (16 * DB) + 4 * g4;
#pragma unroll
    for (int db = 0; db < DB; ++db) *reinterpret_cast<f32x4 *>(dst + 16 * db) = o[db];
    if (g4 == 0) {
        p.part_ml[2 * slot] = m;
        p.part_ml[2 * slot + 1] = l;
    }
}

// Adds the chunks of 1024 / D rows of a work entry's query tile (bm rows) for one head: D / 4 lanes
// per row, four dims each. Chunks are read in order and weighed against the row's largest
// maximum, so the result does not depend on which workgroup finished first. Bound by latency: the
// loops are unrolled so that several chunks' loads are in flight, and each row group has a
// workgroup of its own.
template <int D, bool GATE, bool DIRECT>
__global__ __launch_bounds__(256) void merge_kernel(AttnParams p, int bm) {
    constexpr int LPR = D / 4, RPP = 256 / LPR;  // lanes per row, rows per pass
    const WorkItem wi = DIRECT ? find_work<true>(p, blockIdx.x, bm) : load_work(p, blockIdx.x);
    if (!wi.valid || wi.L > p.max_seqlen || wi.Lk > p.max_seqlen_k || wi.Lk < 0) return;
    const int first = wi.qt_first * bm, last = min(wi.L, first + bm);
    if (first >= last) return;
    const int off = wi.Lk - wi.L;
    const int klo = p.wl >= 0 ? max(0, first + off - p.wl) : 0;
    const int khi = p.wr >= 0 ? min(wi.Lk, last + off + p.wr) : wi.Lk;
    const int c0 = klo / p.chunk, c1 = khi > klo ? (khi + p.chunk - 1) / p.chunk : c0;
    const int r = first + blockIdx.z * RPP + threadIdx.x / LPR;
    const int row = wi.start + r;
    if (r >= last || row >= p.total_q) return;
    const int qh = blockIdx.y, dim = 4 * (threadIdx.x % LPR);
    const int64_t step = part_slot(p, 1, 0, 0), slot0 = part_slot(p, c0, row, qh);
    const float2 *ml = reinterpret_cast<const float2 *>(p.part_ml) + slot0;
    const float *part = p.part_o + slot0 * D + dim;
    const int n = c1 - c0;
    float m = kNegInf;
#pragma unroll 8
    for (int c = 0; c < n; ++c) m = fmaxf(m, ml[c * step].x);
    float l = 0.0f;
    f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
    for (int c = 0; c < n; ++c) {
        const float2 s = ml[c * step];
        const f32x4 x = *reinterpret_cast<const f32x4 *>(part + c * step * D);
        const float w = s.x == kNegInf ? 0.0f : exp2_fast(s.x - m);
        l = fmaf(s.y, w, l);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = fmaf(x[i], w, o[i]);
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    bf16x4 s = {};
    if constexpr (GATE)
        s = sigmoid4(*reinterpret_cast<const bf16x4 *>(p.g + (int64_t)row * p.g_st + (int64_t)qh * p.g_sh + dim));
    // gated: bf16(bf16(o) * bf16(sigmoid(g))), as every epilogue
    const bf16x4 y = round4<GATE>(o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv, s);
    *reinterpret_cast<bf16x4 *>(p.o + (int64_t)row * p.o_st + (int64_t)qh * p.o_sh + dim) = y;
}

}  // namespace pe
