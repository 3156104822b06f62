// Elementwise and row-wise passes of an encoder layer around its attention and products (gfx950):
// LayerNorm with the residual add folded in, and the GeGLU gate of the MLP. Both are bound by
// HBM: every tensor is read or written once, in 16-byte pieces, everything else stays in
// registers.
#pragma once

#include "pe_attn_device.h"

namespace pe {

// ----------------------------------------------------------------------------- LayerNorm

struct NormParams {
    const __bf16 *x;    // [rows, cols], contiguous
    const __bf16 *res;  // the residual added first, or NULL
    const __bf16 *w;    // [cols]
    __bf16 *sum;        // bf16(x + res) (written), only with a residual
    __bf16 *out;        // LayerNorm(x + res) * w (written)
    int64_t rows;
    int32_t cols;  // a multiple of 8
    float inv_cols;
    float eps;
};

// Sum over the wave's 64 lanes, the same bits on every lane: rotations within 16 lanes (DPP row_ror
// by 8, 4, 2, 1), then the 16- and 32-lane swaps.
__device__ __forceinline__ float wave_sum(float x) {
    auto ror = [](float v, auto n) {
        return __builtin_bit_cast(
            float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + decltype(n)::value, 0xf, 0xf, true));
    };
    x += ror(x, std::integral_constant<int, 8>{});
    x += ror(x, std::integral_constant<int, 4>{});
    x += ror(x, std::integral_constant<int, 2>{});
    x += ror(x, std::integral_constant<int, 1>{});
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto s16 = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    x = __builtin_bit_cast(float, (unsigned)s16[0]) + __builtin_bit_cast(float, (unsigned)s16[1]);
    const unsigned w = __builtin_bit_cast(unsigned, x);
    const auto s32 = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return __builtin_bit_cast(float, (unsigned)s32[0]) + __builtin_bit_cast(float, (unsigned)s32[1]);
}

// One wave per row, NC 16-byte pieces per lane (piece c * 64 + lane), so a row's statistics never
// leave the wave: no LDS, no barrier, and the mean and the squared deviations are taken from the
// row held in registers. Statistics in fp32 over the bf16 values the row holds (the sum is rounded
// to bf16 first, as the residual stream is stored). The mean adds x / cols, so that no finite row
// overflows it. With the residual at 32,438 x 768: 31.4 us for 199 MB (6.3 TB/s), against 53.3 +
// 24.3 us for torch's add and LayerNorm, which move the sum twice more.
template <int NC, bool ADD>
__global__ __launch_bounds__(256) void layer_norm_kernel(NormParams p) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + uniform(threadIdx.x >> 6);
    if (row >= p.rows) return;
    const int64_t base = row * p.cols;
    const int pieces = p.cols >> 3;
    bf16x8 v[NC], r[ADD ? NC : 1], w[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = c * 64 + lane;
        v[c] = i < pieces ? ld_g16(p.x + base + 8 * i) : bf16x8{};
        if constexpr (ADD) r[c] = i < pieces ? ld_g16(p.res + base + 8 * i) : bf16x8{};
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = c * 64 + lane;
        w[c] = i < pieces ? ld_g16(p.w + 8 * i) : bf16x8{};
    }
    float mean = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if constexpr (ADD) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[c][j] = (__bf16)((float)v[c][j] + (float)r[c][j]);
            const int i = c * 64 + lane;
            if (i < pieces) *reinterpret_cast<bf16x8 *>(p.sum + base + 8 * i) = v[c];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) mean = fmaf((float)v[c][j], p.inv_cols, mean);
    }
    mean = wave_sum(mean);
    float var = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        float part = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float d = (float)v[c][j] - mean;
            part = fmaf(d, d, part);
        }
        var += c * 64 + lane < pieces ? part : 0.0f;
    }
    var = wave_sum(var) * p.inv_cols;
    const float rstd = rsqrtf(var + p.eps);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = c * 64 + lane;
        bf16x8 y;
#pragma unroll
        for (int j = 0; j < 8; ++j) y[j] = (__bf16)(((float)v[c][j] - mean) * rstd * (float)w[c][j]);
        if (i < pieces) *reinterpret_cast<bf16x8 *>(p.out + base + 8 * i) = y;
    }
}

// ----------------------------------------------------------------------------- GeGLU

struct GegluParams {
    const __bf16 *proj;  // [rows, 2 * width], contiguous: (input, gate)
    __bf16 *out;         // [rows, width] (written)
    int64_t pieces;      // rows * width / 8
    int32_t per_row;     // width / 8
};

// gelu(x) = x * Phi(x), Phi the normal distribution function, written through its lower tail
// Phi(-a) = t * 2^(Q(t) - a^2 log2(e) / 2), t = 1 / (1 + 0.22 a), a = |x|: the Gaussian factor is
// taken out exactly and the rest is smooth in t, so one polynomial serves every a. Q is a degree-7
// Chebyshev fit, on [0, 15], of log2(erfcx(a / sqrt 2) / 2) - log2(t); the fit's relative error is
// 3.4e-7, also far out in the negative tail, where 1 + erf(x) loses its digits. Past 15 the power
// of two underflows long before the polynomial matters. 18 VALU instructions and two transcendentals
// per value, against about three times that for erff: with erff the pass is bound by the VALU, not
// by memory.
__device__ __forceinline__ float gelu(float x) {
    const float a = __builtin_fabsf(x);
    const float t = __builtin_amdgcn_rcpf(fmaf(0.22f, a, 1.0f));
    float q = 0.601593779f;
    q = fmaf(q, t, -2.31846865f);
    q = fmaf(q, t, 3.11951201f);
    q = fmaf(q, t, -2.07529329f);
    q = fmaf(q, t, 1.29951664f);
    q = fmaf(q, t, 0.409144346f);
    q = fmaf(q, t, 1.47609864f);
    q = fmaf(q, t, -3.51210317f);
    const float tail = t * exp2_fast(fmaf(x * x, -0.5f * kLog2e, q));
    return x * (x < 0.0f ? tail : 1.0f - tail);
}

// One thread per 16-byte output piece: gelu(input) * gate in fp32, rounded once. At 32,438 x 1,152:
// 39.4 us for 224 MB (5.7 TB/s), against 70.6 + 38.9 us for torch's gelu and product, which also
// write and read the rounded gelu.
__global__ __launch_bounds__(256) void geglu_kernel(GegluParams p) {
    const int64_t first = (int64_t)blockIdx.x * 256;  // the workgroup's first piece
    const int64_t row0 = first / p.per_row;
    const unsigned at = (unsigned)(first - row0 * p.per_row) + threadIdx.x;
    if (first + threadIdx.x >= p.pieces) return;
    const unsigned down = at / (unsigned)p.per_row;
    const int64_t row = row0 + down;
    const int64_t col = 8 * (int64_t)(at - down * (unsigned)p.per_row), width = 8 * (int64_t)p.per_row;
    const __bf16 *src = p.proj + row * 2 * width + col;
    const bf16x8 x = ld_g16(src), g = ld_g16(src + width);
    bf16x8 y;
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = (__bf16)(gelu((float)x[j]) * (float)g[j]);
    *reinterpret_cast<bf16x8 *>(p.out + row * width + col) = y;
}

}  // namespace pe
