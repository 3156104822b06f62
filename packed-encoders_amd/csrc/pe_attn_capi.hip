// C ABI of libpe_attn.so (declared in include/pe_attn.h): argument checks, host-side sizing
// and the launches of the plan, short, tiled and RoPE kernels on the caller's stream.
//
// Nothing here reads device memory, synchronises or allocates, so every entry point can be
// captured into a HIP graph. No exception crosses the ABI; failures are status codes.
#include "../../include/pe_attn.h"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <mutex>

#include "pe_attn_band64.h"
#include "pe_attn_device.h"
#include "pe_attn_global64.h"
#include "pe_attn_plan.h"
#include "pe_attn_short.h"
#include "pe_attn_tiled.h"
#include "pe_attn_tiled_wide16.h"
#include "pe_dense.h"
#include "pe_rope.h"

namespace pe {
// Workspace of pe_varlen_attn_fwd_noalloc: one copy per GPU, in device memory for the life of
// the process. In host code `scratch` names a host-side stand-in, never the device array: the
// array is reached only through the address hipGetSymbolAddress returns for the current
// device, kept per device (static_scratch below).
__device__ __align__(256) unsigned char scratch[PE_ATTN_STATIC_SCRATCH_BYTES];
}  // namespace pe

namespace {

using pe::AttnParams;

constexpr int kMaxDevices = 64;
std::mutex scratch_lock;
void *scratch_ptr[kMaxDevices];

// The current device's address of pe::scratch, looked up once per device.
int static_scratch(void **ptr) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return PE_ATTN_ELAUNCH;
    std::lock_guard<std::mutex> guard(scratch_lock);
    if (!scratch_ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(pe::scratch)) != hipSuccess || !p) return PE_ATTN_ELAUNCH;
        scratch_ptr[dev] = p;
    }
    *ptr = scratch_ptr[dev];
    return PE_ATTN_OK;
}

// gfx950 routing boundary for batches longer than the short kernel's largest key capacity,
// per head dim, fitted to the short-vs-tiled sweep (bench.py --dispatch-sweep): 64 for head_dim
// 64, 32 for head_dim 128. Batches whose longest segment fits that capacity run every segment
// in the short kernel.
constexpr int kShortCapacity = 128;
constexpr int default_boundary(int head_dim) { return head_dim == 64 ? 64 : 32; }
constexpr int kMaxStrip = 64;         // query tiles per tiled-kernel workgroup, at most

int gcd_int(int a, int b) {
    while (b) {
        const int t = a % b;
        a = b;
        b = t;
    }
    return a;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Structural checks shared by every entry point; pointers and strides only when a launch
// will read them (workspace sizing needs sizes alone).
int check_args(const pe_attn_args *a, bool need_pointers = true) {
    if (!a || a->struct_size != sizeof(pe_attn_args)) return PE_ATTN_EINVAL;
    if (a->dtype != PE_ATTN_DTYPE_BF16) return PE_ATTN_EUNSUPPORTED;
    if (a->n_seq < 0 || a->total_tokens < 0 || a->max_seqlen < 0) return PE_ATTN_EINVAL;
    if (a->n_heads_q < 1 || a->n_heads_kv < 1 || a->n_heads_q % a->n_heads_kv) return PE_ATTN_EINVAL;
    if (a->head_dim != 64 && a->head_dim != 128 && a->head_dim != 256) return PE_ATTN_EUNSUPPORTED;
    if (!(a->softmax_scale > 0.0f) || a->softmax_scale != a->softmax_scale) return PE_ATTN_EINVAL;
    if (a->window_left < -1 || a->window_right < -1) return PE_ATTN_EINVAL;
    if (a->causal != 0 && a->causal != 1) return PE_ATTN_EINVAL;
    if (a->short_max < -1 || a->short_max > 128) return PE_ATTN_EINVAL;
    if (a->strip < 0 || a->strip > kMaxStrip) return PE_ATTN_EINVAL;
    if (a->band_kernel < 0 || a->band_kernel > 2) return PE_ATTN_EINVAL;
    if (a->min_seqlen < 0 || a->min_seqlen > a->max_seqlen) return PE_ATTN_EINVAL;
    if (a->cu_seqlens_k && (a->total_tokens_k < 0 || a->max_seqlen_k < 0)) return PE_ATTN_EINVAL;
    if (a->rope_cos || a->rope_sin) {
        if (!a->rope_cos || !a->rope_sin || a->rope_table_rows < 1 || a->rope_table_stride < a->head_dim ||
            (a->rope_table_stride & 7) || !aligned16(a->rope_cos) || !aligned16(a->rope_sin))
            return PE_ATTN_EINVAL;
        // The fused prologue lives in the short kernel (prepare() also needs every segment short),
        // which reads the tables through a buffer resource with 32-bit offsets.
        if (a->head_dim > 128 || a->cu_seqlens_k) return PE_ATTN_EUNSUPPORTED;
        if ((int64_t)a->rope_table_rows * a->rope_table_stride * 2 >= (int64_t)1 << 31) return PE_ATTN_EUNSUPPORTED;
    }
    if (!need_pointers || a->n_seq == 0 || a->total_tokens == 0) return PE_ATTN_OK;
    if (!a->q || !a->k || !a->v || !a->o || !a->cu_seqlens) return PE_ATTN_EINVAL;
    const void *ptrs[4] = {a->q, a->k, a->v, a->o};
    for (const void *p : ptrs)
        if (!aligned16(p)) return PE_ATTN_EINVAL;
    const int64_t strides[8] = {a->q_stride_token, a->q_stride_head, a->k_stride_token, a->k_stride_head,
                                a->v_stride_token, a->v_stride_head, a->o_stride_token, a->o_stride_head};
    for (int64_t s : strides)
        if (s < 0 || (s & 7)) return PE_ATTN_EINVAL;
    if (a->gate) {
        if (!aligned16(a->gate) || a->gate_stride_token < 0 || a->gate_stride_head < 0 ||
            (a->gate_stride_token & 7) || (a->gate_stride_head & 7))
            return PE_ATTN_EINVAL;
    }
    // Kernels address a segment through 32-bit buffer offsets bounded by its last row: rows
    // must not overlap (token stride >= head_dim) and a segment must span < 2 GiB per tensor.
    const int64_t kv_rows = a->cu_seqlens_k ? a->total_tokens_k : a->total_tokens;
    const int64_t kv_max = a->cu_seqlens_k ? a->max_seqlen_k : a->max_seqlen;
    const int64_t token_strides[5] = {a->q_stride_token, a->k_stride_token, a->v_stride_token, a->o_stride_token,
                                      a->gate ? a->gate_stride_token : a->head_dim};
    for (int i = 0; i < 5; ++i) {
        const int64_t s = token_strides[i];
        const bool kv = i == 1 || i == 2;
        if ((kv ? kv_rows : a->total_tokens) > 1 && s < a->head_dim) return PE_ATTN_EINVAL;
        if ((kv ? kv_max : (int64_t)a->max_seqlen) * s * 2 + 2 * a->head_dim >= (int64_t)1 << 31)
            return PE_ATTN_EUNSUPPORTED;
    }
    return PE_ATTN_OK;
}

int routing_boundary(const pe_attn_args *a) {
    if (a->head_dim > 128) return 0;  // the short kernel covers head_dim <= 128
    if (a->short_max >= 0) return a->short_max;
    const int32_t longest = a->cu_seqlens_k && a->max_seqlen_k > a->max_seqlen ? a->max_seqlen_k : a->max_seqlen;
    return longest > 0 && longest <= kShortCapacity ? longest : default_boundary(a->head_dim);
}

// The boundary a call routes by: 0 (every segment to the tiled kernels) when the caller's
// lower bound on the lengths leaves no segment short, which spares the short pass's launch.
int effective_short_max(const pe_attn_args *a) {
    const int sm = routing_boundary(a);
    return a->min_seqlen > sm ? 0 : sm;
}

int heads_per_tile(const pe_attn_args *a) { return gcd_int(a->n_heads_q / a->n_heads_kv, 4); }

// Upper bound on (segment, strip) entries the plan can emit, from host-known sizes only:
// a segment of L > short_max tokens has ceil(L / bm) query tiles in ceil(tiles / strip) strips.
int64_t tile_capacity(const pe_attn_args *a, int short_max, int bm, int strip) {
    const int32_t max_k = a->cu_seqlens_k ? a->max_seqlen_k : a->max_seqlen;
    if (a->n_seq == 0 || a->total_tokens == 0 || (a->max_seqlen <= short_max && max_k <= short_max)) return 0;
    const int64_t n = a->n_seq, t = a->total_tokens;
    // With separate key segments a segment of few queries can still be long (its keys): every
    // segment may then reach the tiled kernel.
    const int64_t n_long = short_max > 0 && !a->cu_seqlens_k ? (t / (short_max + 1) < n ? t / (short_max + 1) : n) : n;
    const int64_t tiles_per_seg = (a->max_seqlen + bm - 1) / bm;
    const int64_t by_shape = n * ((tiles_per_seg + strip - 1) / strip);
    const int64_t tiles_by_tokens = (t + n_long * (bm - 1)) / bm;
    const int64_t by_tokens = (tiles_by_tokens + n_long * (strip - 1)) / strip;
    return by_shape < by_tokens ? by_shape : by_tokens;
}

// Query tiles (128 rows x heads) of a call, from host-known sizes.
int64_t query_tiles(const pe_attn_args *a) { return (int64_t)a->total_tokens / 128 * a->n_heads_q; }

// Whether a call's long segments run the streaming band kernel (band64_attn_kernel) rather than
// the tiled kernel: its window shape, one query head per kv head group, shared key segments,
// and the caller's band_kernel choice; by default a call of at least kBandMinTiles query tiles.
// Both thresholds are fitted to a sweep of C2-like document mixes and equal-length batches
// (12 heads, +-64; attention_dispatch.fit_band_rule): the tiled kernel's short-lived
// workgroups (three per CU) win every call below about 13K tiles, the band kernel's strips
// (two workgroups per CU, each key block staged once) win large document mixes by 1-6% from
// about 24K tiles, at strip 8; the thresholds sit halfway (geometric) between those points.
constexpr int64_t kBandMinTiles = 17667;
constexpr int64_t kBandStrip8Tiles = 17667;
bool uses_band64(const pe_attn_args *a) {
    const int wr = a->causal ? 0 : a->window_right;
    const bool shape = a->head_dim == 64 && !a->cu_seqlens_k && heads_per_tile(a) == 1 &&
                       pe::band64_window(a->window_left, wr);
    if (!shape || a->band_kernel == 2) return false;
    return a->band_kernel == 1 || query_tiles(a) >= kBandMinTiles;
}

// Query tiles per tiled-kernel workgroup: the caller's choice, else the gfx950 default. The
// band kernel streams its key blocks along a strip: 8 tiles from kBandStrip8Tiles on, 4 on the
// smaller calls that force it (band_kernel = 1).
int effective_strip(const pe_attn_args *a) {
    if (a->strip > 0) return a->strip;
    if (!uses_band64(a)) return 1;
    return query_tiles(a) >= kBandStrip8Tiles ? 8 : 4;
}

AttnParams make_params(const pe_attn_args *a, int short_max) {
    AttnParams p;
    std::memset(&p, 0, sizeof(p));
    p.q = static_cast<const __bf16 *>(a->q);
    p.k = static_cast<const __bf16 *>(a->k);
    p.v = static_cast<const __bf16 *>(a->v);
    p.g = static_cast<const __bf16 *>(a->gate);
    p.o = static_cast<__bf16 *>(a->o);
    p.cu = a->cu_seqlens;
    p.cuk = a->cu_seqlens_k ? a->cu_seqlens_k : a->cu_seqlens;
    p.q_st = a->q_stride_token;
    p.q_sh = a->q_stride_head;
    p.k_st = a->k_stride_token;
    p.k_sh = a->k_stride_head;
    p.v_st = a->v_stride_token;
    p.v_sh = a->v_stride_head;
    p.o_st = a->o_stride_token;
    p.o_sh = a->o_stride_head;
    p.g_st = a->gate_stride_token;
    p.g_sh = a->gate_stride_head;
    p.n_seq = a->n_seq;
    p.hq = a->n_heads_q;
    p.group = a->n_heads_q / a->n_heads_kv;
    p.wl = a->window_left;
    p.wr = a->window_right;
    if (a->causal) p.wr = 0;  // causal = no key to the right of the query
    p.short_max = short_max;
    p.max_seqlen = a->max_seqlen;
    p.max_seqlen_k = a->cu_seqlens_k ? a->max_seqlen_k : a->max_seqlen;
    p.strip = effective_strip(a);
    p.band = uses_band64(a) ? 1 : 0;
    p.c = a->softmax_scale * pe::kLog2e;
    p.rcos = static_cast<const __bf16 *>(a->rope_cos);
    p.rsin = static_cast<const __bf16 *>(a->rope_sin);
    p.rst = a->rope_table_stride;
    p.rrows = a->rope_table_rows;
    return p;
}

template <int D, int SK, int HPW, bool GATE>
int launch_short_t(const AttnParams &p, hipStream_t stream) {
    dim3 grid(p.n_seq, (p.hq + HPW - 1) / HPW);
    if (p.rcos)
        hipLaunchKernelGGL((pe::short_attn_kernel<D, SK, HPW, GATE, true>), grid, dim3(256), 0, stream, p);
    else
        hipLaunchKernelGGL((pe::short_attn_kernel<D, SK, HPW, GATE, false>), grid, dim3(256), 0, stream, p);
    return hipGetLastError() == hipSuccess ? PE_ATTN_OK : PE_ATTN_ELAUNCH;
}

// Compute units of an MI355X.
constexpr int64_t kCUs = 256;

// Static short-kernel choice (pe_attn_short_config): key capacity SK (32/64/128) and heads per
// workgroup, sized so the workgroup's K and V^T stay within ~75 KB of LDS (two workgroups per CU).
// short_launch_shape refines it for a call.
void short_shape(int max_len, int d, int *sk, int *hpw) {
    *sk = max_len <= 32 ? 32 : (max_len <= 64 ? 64 : 128);
    if (d == 64)
        *hpw = *sk == 128 ? 2 : 4;
    else
        *hpw = *sk == 32 ? 4 : (*sk == 64 ? 2 : 1);
}

// hpw never exceeds the shape's default (short_shape), the most heads whose K and V fit LDS (and for
// a capacity of 96, which short_launch_shape takes, that of 128).
template <int D, int SK, bool GATE>
int launch_short_h(const AttnParams &p, int hpw, hipStream_t stream) {
    constexpr int kMax = (D == 64 ? 4 : 2) * 64 / SK;  // short_shape's hpw (4, 4, 2, 2 / 4, 2, 1, 1)
    if constexpr (kMax >= 4)
        if (hpw == 4) return launch_short_t<D, SK, 4, GATE>(p, stream);
    if constexpr (kMax >= 2)
        if (hpw == 2) return launch_short_t<D, SK, 2, GATE>(p, stream);
    return launch_short_t<D, SK, 1, GATE>(p, stream);
}

template <int D, bool GATE>
int launch_short_d(const AttnParams &p, int sk, int hpw, hipStream_t stream) {
    if (sk == 32) return launch_short_h<D, 32, GATE>(p, hpw, stream);
    if (sk == 64) return launch_short_h<D, 64, GATE>(p, hpw, stream);
    if (sk == 96) return launch_short_h<D, 96, GATE>(p, hpw, stream);
    return launch_short_h<D, 128, GATE>(p, hpw, stream);
}

// Heads per short-kernel workgroup for a call: the shape's default, halved while the call
// would give fewer than eight workgroups per CU (a small batch: more, smaller workgroups, which
// fit more per CU and hide each other's load latency). Measured on gfx950: C3's 512 query
// segments (1,536 four-head workgroups, three rounds of two per CU) run their short pass 12 %
// faster with two heads per workgroup and 1 % slower with one; a 4,096-segment query batch
// keeps four heads (two: 1 % slower, one: 10 % slower); C1's 32 segments run one head each.
int short_heads(int hpw, int64_t n_seq, int hq) {
    while (hpw > 1 && n_seq * ((hq + hpw - 1) / hpw) < 8 * kCUs) hpw /= 2;
    return hpw;
}

// The shape a call launches: short_shape's, with two refinements that buy workgroups per CU.
//  * Segments of at most 96 tokens take a capacity of 96 instead of 128: 48 instead of 64 KB for two
//    heads of 64, three workgroups instead of two. 1,223 x U{12..92}: 100 -> 89 us (fused RoPE, where
//    the tables made it one workgroup of 96 KB, 200 -> 121 us); 1,000 x U{4..96} at 8 x 128:
//    101 -> 90 us.
//  * With fused RoPE a workgroup also holds its keys' table rows, so from capacity 64 on it takes
//    half the heads: 4,096 x U{16..64}: 48 KB, three per CU, against 80 KB, two, 250 -> 235 us;
//    2,048 x U{64..128}: 64 KB against 96 KB, 473 -> 322 us; 1,024 x U{8..64} at 8 x 128:
//    116 -> 101 us. At capacity 32 the default stays (two heads instead of four: 93 -> 111 us).
void short_launch_shape(int max_len, int d, bool rope, int64_t n_seq, int hq, int *sk, int *hpw) {
    short_shape(max_len, d, sk, hpw);
    if (*sk == 128 && max_len <= 96) *sk = 96;
    if (rope && *sk >= 64 && *hpw > 1) *hpw /= 2;
    *hpw = short_heads(*hpw, n_seq, hq);
}

int launch_short(const AttnParams &p, int d, bool gate, int short_max, hipStream_t stream) {
    int sk, hpw;
    short_launch_shape(short_max, d, p.rcos != nullptr, p.n_seq, p.hq, &sk, &hpw);
    if (d == 64) return gate ? launch_short_d<64, true>(p, sk, hpw, stream) : launch_short_d<64, false>(p, sk, hpw, stream);
    if (d == 128) return gate ? launch_short_d<128, true>(p, sk, hpw, stream) : launch_short_d<128, false>(p, sk, hpw, stream);
    return PE_ATTN_EUNSUPPORTED;
}

// head_dim 256 runs wide16_attn_kernel with kWide16Waves waves of 16 query rows per workgroup:
// four waves (one per SIMD) and a 64 KB ring, so two workgroups share a CU and run out of
// step (one's softmax and epilogue under the other's MFMAs); eight waves with a 128 KB ring,
// one workgroup per CU, measured 6% slower on C5.
constexpr int kWide16Waves = 4;

// Key tile and LDS ring depth per head dim: 48 KB (head_dim 64: three workgroups per CU, two
// tiles in flight each), 64 KB (head_dim 128 and 256: two workgroups per CU).
template <int D>
struct TiledShape {
    static constexpr int BN = D >= 256 ? 32 : 64;
    static constexpr int NS = D == 64 ? 3 : (D == 256 ? (kWide16Waves == 8 ? 4 : 2) : 2);
};

// Query rows per tiled-kernel tile for g query heads per workgroup (the plan's tile height).
// Global head_dim 64 calls run global64_attn_kernel, whose waves hold 64 query rows.
bool global64(const pe_attn_args *a) {
    return a->head_dim == 64 && a->window_left < 0 && a->window_right < 0 && !a->causal;
}

int tile_rows(const pe_attn_args *a, int g) {
    if (a->head_dim == 256) return 16 * kWide16Waves / g;
    return (global64(a) ? 64 : 32) * (4 / g);
}

template <int D, int G, bool GATE, bool WIN>
int launch_tiled_t(AttnParams p, int64_t cap, hipStream_t stream) {
    constexpr int BN = TiledShape<D>::BN, NS = TiledShape<D>::NS;
    p.hgroups = p.hq / G;
    // Banded head_dim 64 launches deal work to the 8 XCDs in runs (tiled_attn_kernel): whole
    // rounds of runs, the surplus workgroups exiting at once.
    // head_dim 128 / 256 launches deal every call that way, in runs of the workgroups an XCD
    // holds at once.
    const int64_t run = D == 64    ? 8LL * pe::kXcdRun * p.hgroups
                        : D == 256 ? 8LL * pe::wide16_run<kWide16Waves, NS>(p.hgroups)
                                   : 8LL * pe::wide_run(p.hgroups);
    const int64_t blocks = (D > 64 || WIN) ? (cap * p.hgroups + run - 1) / run * run : cap * p.hgroups;
    if (blocks <= 0) return PE_ATTN_OK;
    if (blocks > 0x7fffffffLL) return PE_ATTN_EUNSUPPORTED;
    if constexpr (D == 64 && !WIN)
        hipLaunchKernelGGL((pe::global64_attn_kernel<G, GATE>), dim3((unsigned)blocks), dim3(256), 0, stream, p);
    else if constexpr (D == 64 && G == 1)
        if (p.band)
            hipLaunchKernelGGL((pe::band64_attn_kernel<GATE>), dim3((unsigned)blocks), dim3(256), 0, stream, p);
        else
            hipLaunchKernelGGL((pe::tiled_attn_kernel<D, G, BN, NS, GATE, WIN>), dim3((unsigned)blocks), dim3(256), 0,
                               stream, p);
    else if constexpr (D == 64)
        hipLaunchKernelGGL((pe::tiled_attn_kernel<D, G, BN, NS, GATE, WIN>), dim3((unsigned)blocks), dim3(256), 0,
                           stream, p);
    else if constexpr (D == 256)
        hipLaunchKernelGGL((pe::wide16_attn_kernel<D, kWide16Waves, G, NS, GATE, WIN>), dim3((unsigned)blocks),
                           dim3(64 * kWide16Waves), 0, stream, p);
    else
        hipLaunchKernelGGL((pe::wide_attn_kernel<D, G, BN, NS, GATE, WIN>), dim3((unsigned)blocks), dim3(256), 0,
                           stream, p);
    return hipGetLastError() == hipSuccess ? PE_ATTN_OK : PE_ATTN_ELAUNCH;
}

template <int D, bool GATE, bool WIN>
int launch_tiled_g(const AttnParams &p, int g, int64_t cap, hipStream_t stream) {
    if (g == 4) return launch_tiled_t<D, 4, GATE, WIN>(p, cap, stream);
    if (g == 2) return launch_tiled_t<D, 2, GATE, WIN>(p, cap, stream);
    return launch_tiled_t<D, 1, GATE, WIN>(p, cap, stream);
}

template <int D>
int launch_tiled_d(const AttnParams &p, int g, bool gate, int64_t cap, hipStream_t stream) {
    const bool win = p.wl >= 0 || p.wr >= 0;
    if (gate) return win ? launch_tiled_g<D, true, true>(p, g, cap, stream) : launch_tiled_g<D, true, false>(p, g, cap, stream);
    return win ? launch_tiled_g<D, false, true>(p, g, cap, stream) : launch_tiled_g<D, false, false>(p, g, cap, stream);
}

// How a split launch deals its workgroups to the XCDs (split_item): sets p.share and p.tiles, returns
// the workgroups per chunk. Fewer than eight sets of keys are dealt one by one: each chunk then has its
// XCDs to itself. Unsplit / dealt one by one / so, us, causal: 32 x U{1400..2500} keys, one row, 12:4 x 256
// (three head groups a kv head) 90 / 121 / 63; 64 x the same, 12:2 x 128 (three) 68 / 75 / 59; 62 x
// U{500..8000}, 64-row tails (four tiles), 8:2 x 256, 330 / 385 / 281.
int64_t split_deal(AttnParams &p, int g, int64_t cap) {
    p.share = p.group / g;
    p.tiles = (int)((2 * cap + p.n_seq) / (2 * (int64_t)p.n_seq));
    if (p.tiles < 1) p.tiles = 1;
    const int64_t units = (cap + p.tiles - 1) / p.tiles * (p.hgroups / p.share), members = (int64_t)p.share * p.tiles;
    if (members == 1 || units < 8) {
        p.share = p.tiles = 1;
        return cap * p.hgroups;
    }
    return (units + 7) / 8 * 8 * members;
}

// Split launches (pe_attn_split.h): one workgroup per work entry, head group and key chunk, then the
// merge of every entry's rows.
template <int D, int G, bool DIRECT>
int launch_split_t(AttnParams p, int bm, int64_t cap, int chunks, hipStream_t stream) {
    constexpr int BN = TiledShape<D>::BN, NS = TiledShape<D>::NS;
    p.hgroups = p.hq / G;
    // Workgroup i runs on XCD i % 8: one workgroup past a multiple of 8 per chunk spreads a segment's
    // chunks over the XCDs, which hold unequal shares of the keys otherwise.
    const int64_t items = split_deal(p, G, cap);
    const dim3 grid((unsigned)(items + (9 - items % 8) % 8), chunks);
    if constexpr (D == 64)
        hipLaunchKernelGGL((pe::tiled_attn_kernel<D, G, BN, NS, false, true, true, DIRECT>), grid, dim3(256), 0, stream, p);
    else if constexpr (D == 128)
        hipLaunchKernelGGL((pe::wide_attn_kernel<D, G, BN, NS, false, true, true, DIRECT>), grid, dim3(256), 0, stream, p);
    else
        hipLaunchKernelGGL((pe::wide16_attn_kernel<D, kWide16Waves, G, NS, false, true, true, DIRECT>), grid,
                           dim3(64 * kWide16Waves), 0, stream, p);
    if (hipGetLastError() != hipSuccess) return PE_ATTN_ELAUNCH;
    // rows of the longest tile the call can hold, in groups of 1024 / D
    const int rows = p.max_seqlen < bm ? p.max_seqlen : bm;
    const dim3 merge((unsigned)cap, p.hq, (rows * D + 1023) / 1024);
    if (p.g)
        hipLaunchKernelGGL((pe::merge_kernel<D, true, DIRECT>), merge, dim3(256), 0, stream, p, bm);
    else
        hipLaunchKernelGGL((pe::merge_kernel<D, false, DIRECT>), merge, dim3(256), 0, stream, p, bm);
    return hipGetLastError() == hipSuccess ? PE_ATTN_OK : PE_ATTN_ELAUNCH;
}

// Small split calls (chunks under kSplitDirectChunk keys: the chip is not full) take their work items
// without a plan, which is 4 to 5 us of 20 to 50: 1 x 8,192 keys 24.6 -> 19.2 us, 24 x U{600..2000}
// 47 -> 41. Larger ones gain more from the plan's order, longest segments first: 16 x U{512..8192}
// 91 us planned, 100 in batch order.
constexpr int kSplitDirectChunk = 1024;
bool split_direct(const AttnParams &p) { return p.n_seq <= pe::kDirectSegments && p.chunk < kSplitDirectChunk; }

template <int D, int G>
int launch_split_g(const AttnParams &p, int bm, int64_t cap, int chunks, hipStream_t stream) {
    return split_direct(p) ? launch_split_t<D, G, true>(p, bm, cap, chunks, stream)
                           : launch_split_t<D, G, false>(p, bm, cap, chunks, stream);
}

template <int D>
int launch_split_d(const AttnParams &p, int g, int bm, int64_t cap, int chunks, hipStream_t stream) {
    if (g == 4) return launch_split_g<D, 4>(p, bm, cap, chunks, stream);
    if (g == 2) return launch_split_g<D, 2>(p, bm, cap, chunks, stream);
    return launch_split_g<D, 1>(p, bm, cap, chunks, stream);
}

// Whether a call runs without a plan: a narrow two-sided window (full tiles cost about the same in any
// order; at +-600 that no longer holds and the longest-first plan is as good) in the tiled kernel,
// over at most kDirectSegments segments. The plan kernel takes 5 to 9 us of such a call, finding a
// tile from cu_seqlens about what reading its work entry takes. Calls with and without the plan, us, both
// in one build, 12 heads, +-64: 64 documents of median 400 tokens (30,894 in all) 54.0 -> 47.5, 8 documents
// 21.4 -> 13.2, 1 x 3,000 21.1 -> 12.7, 256 x median 300 143.4 -> 136.5; 64 documents causal with 256 keys
// to the left 60.7 -> 53.7. 16 x 8,192 at 16 heads (16,384 tiles x heads) 240.0 -> 246.7, so the largest
// calls keep it. The staged entry points do too: layers share their plan.
constexpr int kDirectWindow = 256;
constexpr int64_t kDirectMaxTiles = 12288;
bool plans_itself(const pe_attn_args *a) {
    const int wr = a->causal ? 0 : a->window_right;
    return a->head_dim == 64 && a->window_left >= 0 && wr >= 0 && !a->cu_seqlens_k && a->strip <= 1 &&
           (int64_t)a->window_left + wr <= kDirectWindow && a->n_seq <= pe::kDirectSegments &&
           query_tiles(a) <= kDirectMaxTiles && !uses_band64(a);
}

template <int G>
int launch_direct_g(AttnParams p, bool gate, int64_t cap, hipStream_t stream) {
    constexpr int BN = TiledShape<64>::BN, NS = TiledShape<64>::NS;
    p.hgroups = p.hq / G;
    const int64_t run = 8LL * pe::kXcdRun * p.hgroups, blocks = (cap * p.hgroups + run - 1) / run * run;
    if (blocks > 0x7fffffffLL) return PE_ATTN_EUNSUPPORTED;
    const dim3 grid((unsigned)blocks), block(256);
    if (gate)
        hipLaunchKernelGGL((pe::tiled_attn_kernel<64, G, BN, NS, true, true, false, true>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((pe::tiled_attn_kernel<64, G, BN, NS, false, true, false, true>), grid, block, 0, stream, p);
    return hipGetLastError() == hipSuccess ? PE_ATTN_OK : PE_ATTN_ELAUNCH;
}

int launch_direct(const AttnParams &p, int g, bool gate, int64_t cap, hipStream_t stream) {
    if (g == 4) return launch_direct_g<4>(p, gate, cap, stream);
    if (g == 2) return launch_direct_g<2>(p, gate, cap, stream);
    return launch_direct_g<1>(p, gate, cap, stream);
}

int launch_tiled(const AttnParams &p, int d, int g, bool gate, int64_t cap, hipStream_t stream) {
    if (d == 64) return launch_tiled_d<64>(p, g, gate, cap, stream);
    if (d == 128) return launch_tiled_d<128>(p, g, gate, cap, stream);
    if (d == 256) return launch_tiled_d<256>(p, g, gate, cap, stream);
    return PE_ATTN_EUNSUPPORTED;
}

constexpr size_t kWorkspaceHeader = 256;  // the entry counts live here, list follows aligned

// Workspace layout: [0, 256) header (int32 entries written, int32 entries needed), then the
// list of (segment, first query tile, query start, query rows) int4 entries.
struct Plan {
    int sm, g, bm, strip;
    int64_t cap;
};

int prepare(const pe_attn_args *a, Plan *plan) {
    int rc = check_args(a);
    if (rc) return rc;
    plan->sm = effective_short_max(a);
    // RoPE tables: the fused prologue is the short kernel's, so no segment may reach a tiled one.
    if (a->rope_cos && (plan->sm == 0 || a->max_seqlen > plan->sm)) return PE_ATTN_EUNSUPPORTED;
    plan->g = heads_per_tile(a);
    plan->bm = tile_rows(a, plan->g);
    plan->strip = effective_strip(a);
    plan->cap = tile_capacity(a, plan->sm, plan->bm, plan->strip);
    if (plan->cap > 0x7fffffffLL) return PE_ATTN_EUNSUPPORTED;
    return PE_ATTN_OK;
}

size_t list_bytes(int64_t cap) { return cap > 0 ? kWorkspaceHeader + (size_t)cap * sizeof(int4) : 0; }

int64_t capacity_of(const pe_attn_args *a) {
    return tile_capacity(a, effective_short_max(a), tile_rows(a, heads_per_tile(a)), effective_strip(a));
}

// A split of a call's key segments (pe_attn_split.h): the keys of a chunk, the most chunks a
// segment has, and the bytes of their partial rows behind the list. No split: chunks 1, bytes 0.
struct Split {
    int chunk, chunks;
    size_t offset, bytes;
};

// Splits calls with key segments of their own that would leave the chip waiting for a few long
// walks, from host-known sizes. The chunk is the smallest (256 to 1,536 keys, in whole key tiles)
// at which the call's workgroups still fit the chip at once: smaller chunks add partial rows and
// rounds of short-lived workgroups, larger ones leave it idle. A call of more than two unsplit
// workgroups per CU stays unsplit (62 x U{478..3374} at 12:12 x 64, 744 workgroups: 85 us, split 94),
// as does one whose longest walk is at most 1,536 keys or barely more than a
// chunk (the merge and the partial rows cost about 10 us), or that split_pays tells so. Measured, us, unsplit / chunk 256 /
// 512 / 768 / 1,024 / 1,536, causal, by segments x keys, tails, heads x head_dim (the rule's choice):
// (with the short pass and a plan; both are spared below)
//   1 x 8,192, 1 row, 32:8 x 128                207 / 25 / 28 / 34 / 38 / 53        (256)
//   4 x 4,096, 16 rows, 32:8 x 128              114 / 32 / 32 / 38 / 41 / 52        (320)
//   16 x U{512..8192}, U{1..32}, 32:8 x 128     259 / 127 / 105 / 99 / 105 / 93     (1,408)
//   64 x U{512..4096}, U{1..32}, 32:8 x 128     168 / 225 / 190 / 187 / 178 / 166   (unsplit)
//   24 x U{600..2000}, U{1..16}, 32:8 x 128     76 / 56 / 51 / 46 / 45 / 55         (640)
//   64 x U{512..8192}, U{1..16}, 8:2 x 256      381 / 160 / 141 / 135 / 147 / 130   (1,280)
//   16 x U{512..8192}, U{1..32}, 12:12 x 64     138 / 70 / 67 / 67 / 69 / 68        (1,408)
constexpr int64_t kSplitMinChunk = 256, kSplitMaxChunk = 1536;
constexpr size_t kSplitMaxBytes = (size_t)256 << 20;

// A bound on the keys of one segment: max_seqlen_k or, where that is a capacity far above the lengths,
// all the keys of the call. 16 x 1,000 keys, one row each, 32:8 x 128, max_seqlen_k 131,072: 342 chunks
// of 384 keys for every segment took 97.6 us, 32 of 512 take 26.0, unsplit it is 42.7.
int32_t longest_keys(const pe_attn_args *a) {
    return a->max_seqlen_k < a->total_tokens_k ? a->max_seqlen_k : a->total_tokens_k;
}

// Whether the split call is the faster one, by estimates (us) fitted to 3,200 calls timed both ways
// (five head counts, 5 to 500 workgroups, 1 to 8 query tiles per segment, seven length distributions). The
// unsplit call lasts as long as its longest walk (17, 30 or 40 ns a key by head_dim), but no less than
// the keys take from memory (5.5 TB/s where they exceed the caches). The split call spreads all walks
// over the chip (27, 30 or 52 ns a key with every slot taken) or streams the keys, and adds 6 us and
// the partial rows, written and read back at 2.9 TB/s. Without the rule every call of up to two workgroups
// per CU was split and 390 of the 3,200 got slower, unsplit / split: 62 x 4,000 keys, 16-row tails, 32:8 x
// 128 181 / 247; 62 x 8,000, 128-row tails, 8:8 x 128 371 / 521. With it four do, by 5 % at most; one-row
// tails at such sizes stay split: 64 x 4,096 keys, 32:8 x 128, 215 / 202. Two margins, each from 1,700 more
// calls of which up to 30 got slower by 3 to 18 % without them:
//  * A bound may be far above the longest segment. From three quarters of two workgroups per CU on, one
//    past twice the mean counts as 1.4 times the mean (82 x U{1400..2500} keys, 96-row tails, 8:1 x 64
//    under 16,384 59 / 69; 256 x U{100..300}, one row, 8:2 x 256 under 4,096 28 / 33). A call that does have
//    such a segment then stays unsplit (240 x 100 keys and one of 4,096, 8:2 x 256, 148 / 47).
//  * Chunks do not begin where windows do, so a windowed call has to gain a quarter (25 x U{500..8000}
//    keys, 1,700 to the left, 96-row tails, 8:2 x 64 40 / 46).
bool split_pays(const pe_attn_args *a, int64_t reach, int64_t longest, int64_t keys, int64_t chunk, int64_t groups,
                int64_t slots) {
    const double walk = a->head_dim == 64 ? 0.017 : a->head_dim == 128 ? 0.030 : 0.040;
    const double busy = a->head_dim == 64 ? 0.027 : a->head_dim == 128 ? 0.030 : 0.052;
    const double mean = (double)(keys < reach ? keys : reach);
    const double walked = 2 * groups >= 3 * kCUs && reach > 2 * mean ? 1.4 * mean : (double)reach;
    const double stream = mean * a->n_seq * a->n_heads_kv * a->head_dim * 4e-6;  // MB of keys and values
    const double rows = (mean / chunk + 0.5) * a->total_tokens * a->n_heads_q;   // a row's chunks, on average
    const double partial = rows * (a->head_dim + 2) * 4e-6;                      // MB
    const double unsplit = walked * walk > stream / 5.5 ? walked * walk : stream / 5.5;
    const double spread = mean * groups / slots * busy > stream / 6.0 ? mean * groups / slots * busy : stream / 6.0;
    return 6.0 + spread + 0.7 * partial < (reach < longest ? 0.75 : 1.0) * unsplit;
}

Split split_of(const pe_attn_args *a, int g, int bm, int64_t cap) {
    Split s = {0, 1, 0, 0};
    if (!a->cu_seqlens_k || cap == 0 || a->strip > 1 || a->total_tokens == 0 || global64(a)) return s;
    // the most keys a query tile reads
    const int wr = a->causal ? 0 : a->window_right;
    const int64_t longest = longest_keys(a);
    int64_t reach = longest;
    if (a->window_left >= 0 && wr >= 0 && (int64_t)bm + a->window_left + wr < reach) reach = (int64_t)bm + a->window_left + wr;
    const int64_t slots = a->head_dim == 64 ? 3 * kCUs : 2 * kCUs;  // resident workgroups
    const int64_t groups = cap * (a->n_heads_q / g);
    if (reach <= kSplitMaxChunk || groups > 2 * kCUs) return s;
    // A segment's chunks are its keys over the chunk and half a chunk more, on average; an eighth of
    // the chip is left for uneven lengths (a few workgroups too many cost a whole round).
    const int64_t keys = (int64_t)a->total_tokens_k / a->n_seq + 1, room = slots * 7 / 4 - groups;
    int64_t chunk = (2 * groups * keys + room - 1) / room;
    // Every work entry launches a workgroup for each chunk the longest segment can have, and those past
    // a segment's keys exit at once: eight rounds of the resident workgroups in all, at most. It matters
    // where the bound is far above the lengths, us unsplit / chunk 256 / this rule, one row each,
    // max_seqlen_k 8,192, head_dim 128: 32 x 300 keys, 32:8 heads, 26.6 / 30.6 (16 rounds) / 21.6;
    // 200 x 200 keys, 8:2 heads, 27.1 / 34.0 (25) / 25.1. Four rounds cost 16 x 1,000 keys 26 -> 34.
    const int64_t within = longest * groups / (8 * slots);
    if (chunk < within) chunk = within;
    chunk = chunk < kSplitMinChunk ? kSplitMinChunk : chunk > kSplitMaxChunk ? kSplitMaxChunk : (chunk + 63) / 64 * 64;
    if (2 * reach < 3 * chunk) return s;
    const int chunks = (int)((longest + chunk - 1) / chunk);
    if (!split_pays(a, reach, longest, keys, chunk, groups, slots)) return s;
    const size_t rows = (size_t)chunks * a->total_tokens * a->n_heads_q;
    if (chunks > 65535 || a->n_heads_q > 65535 || rows > kSplitMaxBytes / (4 * (a->head_dim + 2))) return s;
    s.chunk = (int)chunk;
    s.chunks = chunks;
    s.offset = (list_bytes(cap) + 255) / 256 * 256;
    s.bytes = rows * 4 * (a->head_dim + 2);
    return s;
}

int check_workspace(const Plan &plan, const void *workspace, size_t bytes) {
    if (plan.cap > 0 && (!workspace || !aligned16(workspace) || bytes < list_bytes(plan.cap)))
        return PE_ATTN_EWORKSPACE;
    return PE_ATTN_OK;
}

AttnParams planned_params(const pe_attn_args *a, const Plan &plan, const void *workspace) {
    AttnParams p = make_params(a, plan.sm);
    p.work_count = static_cast<const int32_t *>(workspace);
    p.work = reinterpret_cast<const int4 *>(static_cast<const char *>(workspace) + kWorkspaceHeader);
    p.work_cap = (int)plan.cap;
    return p;
}

template <int D>
int launch_rope(const pe::RopeParams &p, hipStream_t stream) {
    const int64_t threads = (int64_t)p.n_rows * 2 * p.heads * (D / 16);
    const int64_t blocks = (threads + 255) / 256;
    if (blocks > 0x7fffffffLL) return PE_ATTN_EUNSUPPORTED;
    hipLaunchKernelGGL(pe::rope_qkv_kernel<D>, dim3((unsigned)blocks), dim3(256), 0, stream, p);
    return hipGetLastError() == hipSuccess ? PE_ATTN_OK : PE_ATTN_ELAUNCH;
}

template <bool ADD>
int launch_norm(const pe::NormParams &p, hipStream_t stream) {
    const int64_t blocks = (p.rows + 3) / 4;
    if (blocks > 0x7fffffffLL) return PE_ATTN_EUNSUPPORTED;
    const dim3 grid((unsigned)blocks), block(256);
    const int pieces = (p.cols / 8 + 63) / 64;  // 16-byte pieces per lane
    if (pieces <= 1)
        hipLaunchKernelGGL((pe::layer_norm_kernel<1, ADD>), grid, block, 0, stream, p);
    else if (pieces <= 2)
        hipLaunchKernelGGL((pe::layer_norm_kernel<2, ADD>), grid, block, 0, stream, p);
    else if (pieces <= 4)
        hipLaunchKernelGGL((pe::layer_norm_kernel<4, ADD>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((pe::layer_norm_kernel<8, ADD>), grid, block, 0, stream, p);
    return hipGetLastError() == hipSuccess ? PE_ATTN_OK : PE_ATTN_ELAUNCH;
}

// The boundary a split call routes by. By default its short segments take the split kernel as well,
// which serves any length: that spares the short pass, 4.7 us of a 92 us call that has none of them.
int split_short_max(const pe_attn_args *a) { return a->short_max < 0 ? 0 : a->short_max; }

// A call split into key chunks.
int launch_split(const pe_attn_args *call, const Split &split, void *workspace, size_t workspace_bytes,
                 hipStream_t stream) {
    pe_attn_args a = *call;
    a.short_max = split_short_max(&a);
    a.max_seqlen_k = longest_keys(&a);  // what the partial rows are sized for: a longer segment is skipped
    Plan plan;
    int rc = prepare(&a, &plan);
    if (rc) return rc;
    AttnParams p = planned_params(&a, plan, workspace);
    p.part_o = reinterpret_cast<float *>(static_cast<char *>(workspace) + split.offset);
    p.part_ml = p.part_o + split.bytes / 4 / (a.head_dim + 2) * a.head_dim;
    p.chunk = split.chunk;
    p.total_q = a.total_tokens;
    if ((rc = pe_attn_short_fwd(&a, stream))) return rc;
    if (!split_direct(p) && (rc = pe_attn_plan(&a, workspace, workspace_bytes, stream))) return rc;
    if (a.head_dim == 64) return launch_split_d<64>(p, plan.g, plan.bm, plan.cap, split.chunks, stream);
    if (a.head_dim == 128) return launch_split_d<128>(p, plan.g, plan.bm, plan.cap, split.chunks, stream);
    return launch_split_d<256>(p, plan.g, plan.bm, plan.cap, split.chunks, stream);
}

}  // namespace

extern "C" {

int pe_attn_abi_version(void) { return PE_ATTN_ABI_VERSION; }

const char *pe_attn_strerror(int status) {
    switch (status) {
        case PE_ATTN_OK: return "ok";
        case PE_ATTN_EINVAL: return "invalid argument";
        case PE_ATTN_EUNSUPPORTED: return "unsupported configuration";
        case PE_ATTN_EWORKSPACE: return "workspace missing or too small";
        case PE_ATTN_ELAUNCH: return "kernel launch failed";
        case PE_ATTN_ESCRATCH: return "needs more than the static scratch (PE_ATTN_STATIC_SCRATCH_BYTES)";
        default: return "unknown status";
    }
}

int pe_attn_workspace_size(const pe_attn_args *a, size_t *bytes) {
    if (!bytes) return PE_ATTN_EINVAL;
    const int rc = check_args(a, false);
    if (rc) return rc;
    const int64_t cap = capacity_of(a);
    const int g = heads_per_tile(a);
    const Split split = split_of(a, g, tile_rows(a, g), cap);
    *bytes = split.bytes ? split.offset + split.bytes : list_bytes(cap);
    return PE_ATTN_OK;
}

int pe_attn_plan_size(const pe_attn_args *a, size_t *bytes) {
    if (!bytes) return PE_ATTN_EINVAL;
    const int rc = check_args(a, false);
    if (rc) return rc;
    *bytes = list_bytes(capacity_of(a));
    return PE_ATTN_OK;
}

int pe_attn_key_chunks(const pe_attn_args *a) {
    const int rc = check_args(a, false);
    if (rc) return rc;
    const int g = heads_per_tile(a);
    return split_of(a, g, tile_rows(a, g), capacity_of(a)).chunks;
}

int pe_attn_plan(const pe_attn_args *a, void *workspace, size_t workspace_bytes, hipStream_t stream) {
    Plan plan;
    int rc = prepare(a, &plan);
    if (rc) return rc;
    if (plan.cap == 0) return PE_ATTN_OK;
    rc = check_workspace(plan, workspace, workspace_bytes);
    if (rc) return rc;
    int32_t *count = static_cast<int32_t *>(workspace);
    int4 *work = reinterpret_cast<int4 *>(static_cast<char *>(workspace) + kWorkspaceHeader);
    const int wr = a->causal ? 0 : a->window_right;
    hipLaunchKernelGGL(pe::plan_kernel, dim3(1), dim3(1024), 0, stream, a->cu_seqlens,
                       a->cu_seqlens_k ? a->cu_seqlens_k : a->cu_seqlens, a->n_seq, plan.sm, a->max_seqlen,
                       a->cu_seqlens_k ? a->max_seqlen_k : a->max_seqlen, plan.bm, plan.strip, a->window_left, wr,
                       a->head_dim > 64 ? 1 : 0, work, count, (int)plan.cap);
    return hipGetLastError() == hipSuccess ? PE_ATTN_OK : PE_ATTN_ELAUNCH;
}

int pe_attn_short_fwd(const pe_attn_args *a, hipStream_t stream) {
    Plan plan;
    const int rc = prepare(a, &plan);
    if (rc) return rc;
    if (plan.sm == 0 || a->n_seq == 0 || a->total_tokens == 0) return PE_ATTN_OK;
    const AttnParams p = make_params(a, plan.sm);
    return launch_short(p, a->head_dim, a->gate != nullptr, plan.sm, stream);
}

int pe_attn_tiled_fwd(const pe_attn_args *a, const void *workspace, size_t workspace_bytes, hipStream_t stream) {
    Plan plan;
    int rc = prepare(a, &plan);
    if (rc) return rc;
    if (plan.cap == 0) return PE_ATTN_OK;
    rc = check_workspace(plan, workspace, workspace_bytes);
    if (rc) return rc;
    const AttnParams p = planned_params(a, plan, workspace);
    return launch_tiled(p, a->head_dim, plan.g, a->gate != nullptr, plan.cap, stream);
}

int pe_varlen_attn_fwd(const pe_attn_args *a, void *workspace, size_t workspace_bytes, hipStream_t stream) {
    Plan plan;
    int rc = prepare(a, &plan);
    if (rc) return rc;
    rc = check_workspace(plan, workspace, workspace_bytes);
    if (rc) return rc;
    // Split where the workspace holds the partial rows; one sized for the list alone runs unsplit.
    const Split split = split_of(a, plan.g, plan.bm, plan.cap);
    if (split.bytes && workspace_bytes >= split.offset + split.bytes)
        return launch_split(a, split, workspace, workspace_bytes, stream);
    if ((rc = pe_attn_short_fwd(a, stream))) return rc;
    if (plan.cap > 0 && plans_itself(a))
        return launch_direct(make_params(a, plan.sm), plan.g, a->gate != nullptr, plan.cap, stream);
    if ((rc = pe_attn_plan(a, workspace, workspace_bytes, stream))) return rc;
    return pe_attn_tiled_fwd(a, workspace, workspace_bytes, stream);
}

int pe_varlen_attn_fwd_noalloc(const pe_attn_args *a, hipStream_t stream) {
    size_t need = 0;
    int rc = pe_attn_workspace_size(a, &need);
    if (rc) return rc;
    // Where the partial rows of a split do not fit, the list alone: the call then runs unsplit.
    if (need > PE_ATTN_STATIC_SCRATCH_BYTES && (rc = pe_attn_plan_size(a, &need))) return rc;
    if (need > PE_ATTN_STATIC_SCRATCH_BYTES) return PE_ATTN_ESCRATCH;
    void *ws = nullptr;
    if (need > 0 && (rc = static_scratch(&ws))) return rc;
    // Nothing in the workspace needs clearing: the plan writes the entry counts before the
    // tiled kernel reads them, and entries only up to that count.
    return pe_varlen_attn_fwd(a, ws, need, stream);
}

int pe_packed_short_attn_fwd(const pe_attn_args *a, hipStream_t stream) {
    int rc = check_args(a, false);
    if (rc) return rc;
    const int32_t smax = a->cu_seqlens_k && a->max_seqlen_k > a->max_seqlen ? a->max_seqlen_k : a->max_seqlen;
    if (smax <= 0 || smax > 128) return PE_ATTN_EUNSUPPORTED;
    if (a->head_dim > 128) return PE_ATTN_EUNSUPPORTED;
    rc = check_args(a);
    if (rc) return rc;
    if (a->n_seq == 0 || a->total_tokens == 0) return PE_ATTN_OK;
    AttnParams p = make_params(a, smax);
    return launch_short(p, a->head_dim, a->gate != nullptr, smax, stream);
}

int pe_attn_short_config(int32_t max_seqlen, int32_t head_dim, int32_t out[4]) {
    if (!out || max_seqlen <= 0 || max_seqlen > 128 || (head_dim != 64 && head_dim != 128)) return PE_ATTN_EINVAL;
    int sk, hpw;
    short_shape(max_seqlen, head_dim, &sk, &hpw);
    out[0] = 32;
    out[1] = sk;
    out[2] = hpw;
    out[3] = 4;
    return PE_ATTN_OK;
}

int pe_attn_kernels(const pe_attn_args *a, int32_t out[6]) {
    int rc = check_args(a, false);
    if (rc) return rc;
    if (!out) return PE_ATTN_EINVAL;
    pe_attn_args routed = *a;
    if (pe_attn_key_chunks(a) > 1) routed.short_max = split_short_max(a);
    const int sm = effective_short_max(&routed);
    int sk = 0, heads = 0;
    if (sm > 0) short_launch_shape(sm, a->head_dim, a->rope_cos != nullptr, a->n_seq, a->n_heads_q, &sk, &heads);
    const int g = heads_per_tile(a);
    const int32_t max_k = a->cu_seqlens_k ? a->max_seqlen_k : a->max_seqlen;
    const bool tiled = a->n_seq > 0 && a->total_tokens > 0 && (a->max_seqlen > sm || max_k > sm);
    int kernel = PE_ATTN_KERNEL_NONE;
    if (tiled) {
        if (a->head_dim == 256) kernel = PE_ATTN_KERNEL_WIDE16;
        else if (a->head_dim == 128) kernel = PE_ATTN_KERNEL_WIDE;
        else if (global64(a)) kernel = PE_ATTN_KERNEL_GLOBAL64;
        else kernel = uses_band64(a) ? PE_ATTN_KERNEL_BAND64 : PE_ATTN_KERNEL_TILED;
    }
    out[0] = sk;
    out[1] = kernel;
    out[2] = tiled ? effective_strip(a) : 0;
    out[3] = tiled ? tile_rows(a, g) : 0;
    const int64_t groups = heads ? (int64_t)a->n_seq * ((a->n_heads_q + heads - 1) / heads) : 0;
    out[4] = heads;
    out[5] = (int32_t)(groups < 0x7fffffff ? groups : 0x7fffffff);
    return PE_ATTN_OK;
}

int pe_rope_qkv_fwd(const pe_rope_args *a, hipStream_t stream) {
    if (!a || a->struct_size != sizeof(pe_rope_args)) return PE_ATTN_EINVAL;
    if (a->dtype != PE_ATTN_DTYPE_BF16) return PE_ATTN_EUNSUPPORTED;
    if (a->head_dim != 64 && a->head_dim != 128 && a->head_dim != 256) return PE_ATTN_EUNSUPPORTED;
    if (a->n_rows < 0 || a->n_heads < 1 || a->table_rows < 1) return PE_ATTN_EINVAL;
    if (a->n_rows == 0) return PE_ATTN_OK;
    if (!a->qkv || !a->cos || !a->sin || !a->q_out || !a->k_out) return PE_ATTN_EINVAL;
    const void *ptrs[5] = {a->qkv, a->cos, a->sin, a->q_out, a->k_out};
    for (const void *p : ptrs)
        if (!aligned16(p)) return PE_ATTN_EINVAL;
    const int64_t width = 3LL * a->n_heads * a->head_dim;
    if (a->qkv_stride_row < width || (a->qkv_stride_row & 7)) return PE_ATTN_EINVAL;
    if (a->table_stride_row < a->head_dim || (a->table_stride_row & 7)) return PE_ATTN_EINVAL;
    pe::RopeParams p;
    p.qkv = static_cast<const __bf16 *>(a->qkv);
    p.cos = static_cast<const __bf16 *>(a->cos);
    p.sin = static_cast<const __bf16 *>(a->sin);
    p.q_out = static_cast<__bf16 *>(a->q_out);
    p.k_out = static_cast<__bf16 *>(a->k_out);
    p.qkv_st = a->qkv_stride_row;
    p.table_st = a->table_stride_row;
    p.table_rows = a->table_rows;
    p.n_rows = a->n_rows;
    p.heads = a->n_heads;
    if (a->head_dim == 64) return launch_rope<64>(p, stream);
    if (a->head_dim == 128) return launch_rope<128>(p, stream);
    return launch_rope<256>(p, stream);
}

int pe_rope_gather_fwd(const int64_t *positions, int64_t max_positions, float theta, int64_t rows, int32_t head_dim,
                       void *cos, void *sin, hipStream_t stream) {
    if (rows < 0 || max_positions < 0 || !(theta > 0.0f)) return PE_ATTN_EINVAL;
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) return PE_ATTN_EUNSUPPORTED;
    if (rows == 0) return PE_ATTN_OK;
    if (!positions || !cos || !sin || !aligned16(cos) || !aligned16(sin)) return PE_ATTN_EINVAL;
    if (rows > INT64_MAX / 16) return PE_ATTN_EINVAL;
    const int64_t threads = rows * (head_dim / 16), blocks = threads / 256 + (threads % 256 != 0);
    if (blocks > 0x7fffffffLL) return PE_ATTN_EUNSUPPORTED;
    const pe::RopeRowsParams p = {positions, static_cast<__bf16 *>(cos), static_cast<__bf16 *>(sin), rows, max_positions,
                                  theta};
    const dim3 grid((unsigned)blocks), block(256);
    if (head_dim == 64)
        hipLaunchKernelGGL(pe::rope_rows_kernel<64>, grid, block, 0, stream, p);
    else if (head_dim == 128)
        hipLaunchKernelGGL(pe::rope_rows_kernel<128>, grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL(pe::rope_rows_kernel<256>, grid, block, 0, stream, p);
    return hipGetLastError() == hipSuccess ? PE_ATTN_OK : PE_ATTN_ELAUNCH;
}

int pe_layer_norm_fwd(const void *x, const void *residual, const void *weight, void *sum, void *out, int64_t rows,
                      int32_t cols, float eps, hipStream_t stream) {
    if (rows < 0 || cols < 1) return PE_ATTN_EINVAL;
    if ((cols & 7) || cols > PE_LAYER_NORM_MAX_COLS) return PE_ATTN_EUNSUPPORTED;
    if (rows == 0) return PE_ATTN_OK;
    if (!x || !weight || !out || (residual != nullptr) != (sum != nullptr)) return PE_ATTN_EINVAL;
    const void *ptrs[5] = {x, residual, weight, sum, out};
    for (const void *p : ptrs)
        if (!aligned16(p)) return PE_ATTN_EINVAL;
    pe::NormParams p;
    p.x = static_cast<const __bf16 *>(x);
    p.res = static_cast<const __bf16 *>(residual);
    p.w = static_cast<const __bf16 *>(weight);
    p.sum = static_cast<__bf16 *>(sum);
    p.out = static_cast<__bf16 *>(out);
    p.rows = rows;
    p.cols = cols;
    p.inv_cols = 1.0f / (float)cols;
    p.eps = eps;
    return residual ? launch_norm<true>(p, stream) : launch_norm<false>(p, stream);
}

int pe_geglu_fwd(const void *proj, void *out, int64_t rows, int32_t width, hipStream_t stream) {
    if (rows < 0 || width < 1) return PE_ATTN_EINVAL;
    if (width & 7) return PE_ATTN_EUNSUPPORTED;
    if (rows == 0) return PE_ATTN_OK;
    if (!proj || !out || !aligned16(proj) || !aligned16(out)) return PE_ATTN_EINVAL;
    pe::GegluParams p;
    p.proj = static_cast<const __bf16 *>(proj);
    p.out = static_cast<__bf16 *>(out);
    p.per_row = width / 8;
    if (rows > INT64_MAX / p.per_row) return PE_ATTN_EINVAL;
    p.pieces = rows * p.per_row;
    const int64_t blocks = p.pieces / 256 + (p.pieces % 256 != 0);
    if (blocks > 0x7fffffffLL) return PE_ATTN_EUNSUPPORTED;
    hipLaunchKernelGGL(pe::geglu_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, p);
    return hipGetLastError() == hipSuccess ? PE_ATTN_OK : PE_ATTN_ELAUNCH;
}

}  // extern "C"
