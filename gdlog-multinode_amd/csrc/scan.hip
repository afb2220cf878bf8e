// scan.hip -- device-wide exclusive scans and stream compaction (unique,
// filter).  Tiles of 4096 items: 256 threads, each wave owns 1024 consecutive
// items processed in 16 rounds of 64 lanes, so every round's loads and the
// compacted stores are contiguous across the wave.
#include "gdl_internal.hpp"

namespace gdl {

constexpr int TB = 256;
constexpr int TI = 16;
constexpr int TILE = TB * TI;
constexpr int WSPAN = 64 * TI;

__device__ __forceinline__ u64 tile_item(u64 base, int w, int r, int lane) {
    return base + (u64)w * WSPAN + (u64)r * 64 + lane;
}

__device__ __forceinline__ u64 wave_bcast_last(u64 v) { return __shfl(v, 63, 64); }

// Sum of a tile -> block_sums[blockIdx.x]
__global__ __launch_bounds__(TB) void k_scan_reduce(const u32 *in, u64 n, u64 *block_sums) {
    __shared__ u64 s_w[TB / 64 + 1];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const u64 base = (u64)blockIdx.x * TILE;
    u64 acc = 0;
#pragma unroll
    for (int r = 0; r < TI; ++r) {
        u64 i = tile_item(base, w, r, lane);
        if (i < n) acc += (u64)in[i];
    }
    u64 tot;
    block_exclusive_scan<TB>(acc, s_w, &tot);
    if (t == 0) block_sums[blockIdx.x] = tot;
}

// Exclusive scan in place by one block; v[n] = total, also stored to
// *total_out.  Each thread scans 4 consecutive elements per round of 4 * BLOCK.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_scan_top(u64 *v, u64 n, u64 *total_out) {
    __shared__ u64 s_w[BLOCK / 64 + 1];
    const int t = threadIdx.x;
    u64 carry = 0;
    for (u64 b = 0; b < n; b += 4 * BLOCK) {
        const u64 i0 = b + 4 * (u64)t;
        u64 x[4];
        u64 sum = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x[j] = i0 + j < n ? v[i0 + j] : 0;
            sum += x[j];
        }
        u64 tot;
        u64 ex = carry + block_exclusive_scan<BLOCK>(sum, s_w, &tot);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (i0 + j < n) v[i0 + j] = ex;
            ex += x[j];
        }
        carry += tot;
    }
    if (t == 0) {
        v[n] = carry;
        *total_out = carry;
    }
}

// Exclusive scan of a tile with the block offset from block_sums.
__global__ __launch_bounds__(TB) void k_scan_down(const u32 *in, u64 n, const u64 *block_sums,
                                                  u64 *out) {
    __shared__ u64 s_w[TB / 64 + 1];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const u64 base = (u64)blockIdx.x * TILE;
    u64 ex[TI];
    u64 carry = 0;
#pragma unroll
    for (int r = 0; r < TI; ++r) {
        u64 i = tile_item(base, w, r, lane);
        u64 v = i < n ? (u64)in[i] : 0;
        u64 inc = wave_inclusive_scan(v);
        ex[r] = carry + inc - v;
        carry += wave_bcast_last(inc);
    }
    if (lane == 0) s_w[w] = carry;
    __syncthreads();
    u64 woff = 0;
    for (int k = 0; k < w; ++k) woff += s_w[k];
    const u64 off = block_sums[blockIdx.x] + woff;
#pragma unroll
    for (int r = 0; r < TI; ++r) {
        u64 i = tile_item(base, w, r, lane);
        if (i < n) out[i] = off + ex[r];
    }
}

// ---- compaction: mode 0 = unique (adjacent-different), 1 = predicate filter
// (flag(i, k, prev): key k at i, after key prev where the flag asks for it)
struct UniqueFlag {
    static constexpr bool kPrev = true;
    __device__ __forceinline__ bool operator()(u64 i, u64 k, u64 prev) const {
        return i == 0 || prev != k;
    }
};
struct PredFlag {
    static constexpr bool kPrev = false;
    int op, lhs, rhs;
    __device__ __forceinline__ bool operator()(u64, u64 k, u64) const {
        return eval_pred(k, op, lhs, rhs);
    }
};
// keeps in[i] where flags[i] != 0
struct ByteFlag {
    static constexpr bool kPrev = false;
    const uint8_t *flags;
    __device__ __forceinline__ bool operator()(u64 i, u64, u64) const {
        return flags[i] != 0;
    }
};

// First index in [lo, hi) of sorted keys whose prefix (key >> shift) is >= p.
__device__ __forceinline__ u64 prefix_lower_bound(const u64 *keys, u64 lo, u64 hi, u64 p,
                                                  int shift) {
    while (lo < hi) {
        const u64 mid = lo + ((hi - lo) >> 1);
        if ((keys[mid] >> shift) < p) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// std::set_difference(b, a) under the order of the prefix key >> shift, over
// arrays sorted by key (hence by prefix): of the m elements of b sharing a
// prefix that n elements of a have, the first min(m, n) are dropped and the
// rest kept, in order.
struct PrefixDiffFlag {
    static constexpr bool kPrev = false;
    const u64 *b;
    const u64 *a;
    u64 na;
    int shift;
    __device__ __forceinline__ bool operator()(u64 i, u64 k, u64) const {
        const u64 p = k >> shift;
        const u64 first_b = prefix_lower_bound(b, 0, i, p, shift);
        const u64 lo = prefix_lower_bound(a, 0, na, p, shift);
        const u64 n = prefix_lower_bound(a, lo, na, p + 1, shift) - lo;
        return i - first_b >= n;
    }
};

// Writes the kept keys of a tile after those of the tiles before it
// (tile_before), the total to *n_out: one read of the keys in one launch.
// 41M sorted keys, 31M distinct: 0.146 ms, 3.9 TB/s (a count launch, a scan and
// a write launch took 0.078 + 0.008 + 0.131); CSPA's small ones 7.2 us instead
// of 7.1 + 3 + 6.
template <int B, typename F>
__global__ __launch_bounds__(B) void k_compact(const u64 *in, u64 n, F flag, TileLook look,
                                               u64 *out, u64 *n_out) {
    __shared__ u32 s_w[B / 64];
    __shared__ u64 s_before;
    __shared__ u32 s_tile;
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const u32 tile = tile_ticket(look, &s_tile);
    const u64 base = (u64)tile * (B * TI);
    u64 keys[TI];
    u32 bits = 0;  // flag of round r in bit r
    u32 kept = 0;
#pragma unroll
    for (int r = 0; r < TI; ++r) {
        const u64 i = tile_item(base, w, r, lane);
        keys[r] = i < n ? in[i] : 0;
    }
    u64 last = 0;  // the key before a round's first
    if constexpr (F::kPrev) {
        const u64 first = tile_item(base, w, 0, 0);
        if (first > 0 && first < n) last = in[first - 1];
    }
#pragma unroll
    for (int r = 0; r < TI; ++r) {
        const u64 i = tile_item(base, w, r, lane);
        u64 prev = 0;
        if constexpr (F::kPrev) {
            prev = wave_shift_up(keys[r], last);
            last = wave_last(keys[r]);
        }
        const bool f = i < n && flag(i, keys[r], prev);
        bits |= (u32)f << r;
        kept += (u32)__popcll(__ballot(f));
    }
    if (lane == 0) s_w[w] = kept;
    __syncthreads();
    if (t < 64) {
        u64 all = lane < B / 64 ? s_w[lane] : 0;
        for (int d = 32; d >= 1; d >>= 1) all += __shfl_xor(all, d, 64);
        const u64 before = tile_before(look, tile, all);
        if (t == 0) {
            s_before = before;
            if (tile == gridDim.x - 1) *n_out = before + all;
        }
    }
    __syncthreads();
    u64 off = s_before;
    for (int k = 0; k < w; ++k) off += s_w[k];
    const u64 lt = lane_mask_lt();
#pragma unroll
    for (int r = 0; r < TI; ++r) {
        const bool f = (bits >> r) & 1;
        const u64 bal = __ballot(f);
        // (past the caches where the output is larger than they are)
        if (f) {
            u64 *to = &out[off + __popcll(bal & lt)];
            if constexpr (B == 1024) __builtin_nontemporal_store(keys[r], to);
            else *to = keys[r];
        }
        off += __popcll(bal);
    }
}

// Exclusive scan of u32 values to u64 in one launch (ScanTile).
template <int B>
__global__ __launch_bounds__(B) void k_scan_one(const u32 *in, u64 n, TileLook look, u64 *out,
                                                u64 *total) {
    using Tile = ScanTile<B>;
    __shared__ Tile s;
    const u64 base = (u64)tile_ticket(look, &s.tile) * Tile::kTile;
#pragma unroll
    for (int r = 0; r < Tile::kPer; ++r) {
        const u32 x = r * B + threadIdx.x;
        s.in[Tile::pad(x)] = base + x < n ? in[base + x] : 0;
    }
    __syncthreads();
    s.scan(look, base, n, out, total);
}

// ----------------------------------------------------------------- host side

static gdl_status scan_three(gdl_ctx *ctx, const u32 *d_in, u64 n, u64 *d_out, u64 *total_host) {
    if (n == 0) {
        GDL_HIP(ctx, hipMemsetAsync(d_out, 0, sizeof(u64), ctx->stream));
        if (total_host) {
            GDL_HIP(ctx, hipStreamSynchronize(ctx->stream));
            *total_host = 0;
        }
        return GDL_OK;
    }
    const u64 nb = (n + TILE - 1) / TILE;
    Scratch scr(ctx);
    u64 *bs;
    GDL_TRY(scr.get(nb + 1, &bs));
    {
        KTimer kt(ctx, K_SCAN_REDUCE, 4.0 * n);
        hipLaunchKernelGGL(k_scan_reduce, dim3((unsigned)nb), dim3(TB), 0, ctx->stream, d_in, n,
                           bs);
        GDL_TRY(check_launch(ctx, "k_scan_reduce"));
    }
    {
        KTimer kt(ctx, K_SCAN_TOP, 16.0 * nb);
        hipLaunchKernelGGL(k_scan_top<1024>, dim3(1), dim3(1024), 0, ctx->stream, bs, nb,
                           d_out + n);
        GDL_TRY(check_launch(ctx, "k_scan_top"));
    }
    {
        KTimer kt(ctx, K_SCAN_DOWN, 12.0 * n);
        hipLaunchKernelGGL(k_scan_down, dim3((unsigned)nb), dim3(TB), 0, ctx->stream, d_in, n, bs,
                           d_out);
        GDL_TRY(check_launch(ctx, "k_scan_down"));
    }
    if (total_host) GDL_TRY(read_u64(ctx, d_out + n, total_host));
    return GDL_OK;
}

gdl_status exclusive_scan_u32_to_u64(gdl_ctx *ctx, const u32 *d_in, u64 n, u64 *d_out,
                                     u64 *total_host) {
    // One launch where that is exact: the scans of a program's joins (most of
    // them below 4096 values) are bound by launches, and CSPA's 102 at 500 ids
    // take 6.4 us each, where three launches took 6.0 + 3.0 + 7.8.
    // (A recorded graph takes the three: they keep nothing in the context.)
    if (n == 0 || n > kScanOnePass || records_graph(ctx))
        return scan_three(ctx, d_in, n, d_out, total_host);
    // (tiles of 8192 values from 2^18 on, a quarter of the tickets: 2M values
    // 12 us, in tiles of 2048 24 us)
    const bool big = n >= 1ull << 18;
    const u64 tile = (big ? 1024 : TB) * 8, nt = (n + tile - 1) / tile;
    Scratch scr(ctx);
    TileLook look;
    GDL_TRY(tile_look(ctx, nt, &scr, &look));
    {
        KTimer kt(ctx, K_SCAN_ONE, 12.0 * n);
        auto launch = [&](auto kern, int block) {
            hipLaunchKernelGGL(kern, dim3((unsigned)nt), dim3(block), 0, ctx->stream, d_in, n,
                               look, d_out, total_host ? result_words(ctx) : nullptr);
        };
        if (big) launch(k_scan_one<1024>, 1024);
        else launch(k_scan_one<TB>, TB);
        GDL_TRY(check_launch(ctx, "k_scan_one"));
    }
    return total_host ? read_result(ctx, total_host) : GDL_OK;
}

template <typename F>
static gdl_status compact_impl(gdl_ctx *ctx, const u64 *d_in, u64 n, F flag, u64 *d_out,
                               u64 *n_out) {
    if (n == 0) {
        *n_out = 0;
        return GDL_OK;
    }
    // tiles of 16384 keys from 2^20 on: tickets come at 11 ns each, 41M keys
    // in tiles of 4096 are 10,000 of them; smaller tiles below, for more CUs
    const bool big = n >= 1ull << 20;
    const u64 tile = (big ? 1024 : TB) * TI, nt = (n + tile - 1) / tile;
    Scratch scr(ctx);
    TileLook look;
    GDL_TRY(tile_look(ctx, nt, &scr, &look));
    {
        KTimer kt(ctx, K_COMPACT, 8.0 * n);  // and the kept keys' writes, below
        auto launch = [&](auto kern, int block) {
            hipLaunchKernelGGL(kern, dim3((unsigned)nt), dim3(block), 0, ctx->stream, d_in, n,
                               flag, look, d_out, result_words(ctx));
        };
        if (big) launch(k_compact<1024, F>, 1024);
        else launch(k_compact<TB, F>, TB);
        GDL_TRY(check_launch(ctx, "k_compact"));
    }
    GDL_TRY(read_result(ctx, n_out));
    ctx->stats[K_COMPACT].alg_bytes += 8.0 * (double)*n_out;
    return GDL_OK;
}

gdl_status unique_keys(gdl_ctx *ctx, const u64 *d_in, u64 n, u64 *d_out, u64 *n_out) {
    return compact_impl(ctx, d_in, n, UniqueFlag{}, d_out, n_out);
}

gdl_status compact_flags(gdl_ctx *ctx, const u64 *d_in, const uint8_t *flags, u64 n, u64 *d_out,
                         u64 *n_out) {
    return compact_impl(ctx, d_in, n, ByteFlag{flags}, d_out, n_out);
}

gdl_status filter_keys(gdl_ctx *ctx, const u64 *d_in, u64 n, gdl_pred pred, u64 *d_out,
                       u64 *n_out) {
    return compact_impl(ctx, d_in, n, PredFlag{pred.op, pred.lhs, pred.rhs}, d_out, n_out);
}

}  // namespace gdl

using namespace gdl;

extern "C" {

gdl_status gdl_unique_u64(gdl_ctx *ctx, const uint64_t *d_sorted, uint64_t n, uint64_t *d_out,
                          uint64_t *n_out) {
    if (!ctx || !n_out || (n && (!d_sorted || !d_out))) return GDL_ERR_INVALID_ARG;
    return unique_keys(ctx, d_sorted, n, d_out, n_out);
}

gdl_status gdl_filter_u64(gdl_ctx *ctx, const uint64_t *d_in, uint64_t n, gdl_pred pred,
                          uint64_t *d_out, uint64_t *n_out) {
    if (!ctx || !n_out || (n && (!d_in || !d_out))) return GDL_ERR_INVALID_ARG;
    if (!valid_pred(pred, 2)) return fail(ctx, GDL_ERR_INVALID_ARG, "gdl_filter_u64: bad predicate");
    return filter_keys(ctx, d_in, n, pred, d_out, n_out);
}

gdl_status gdl_compact_flags_u64(gdl_ctx *ctx, const uint64_t *d_in, const uint8_t *d_flags,
                                 uint64_t n, uint64_t *d_out, uint64_t *n_out) {
    if (!ctx || !n_out || (n && (!d_in || !d_flags || !d_out))) return GDL_ERR_INVALID_ARG;
    return compact_flags(ctx, d_in, d_flags, n, d_out, n_out);
}

gdl_status gdl_set_difference_prefix_u64(gdl_ctx *ctx, const uint64_t *d_b, uint64_t nb,
                                         const uint64_t *d_a, uint64_t na, int shift,
                                         uint64_t *d_out, uint64_t *n_out) {
    if (!ctx || !n_out || (nb && (!d_b || !d_out)) || (na && !d_a)) return GDL_ERR_INVALID_ARG;
    if (shift < 0 || shift > 63)
        return fail(ctx, GDL_ERR_INVALID_ARG, "gdl_set_difference_prefix_u64: shift 0..63");
    return compact_impl(ctx, d_b, nb, PrefixDiffFlag{d_b, d_a, na, shift}, d_out, n_out);
}

gdl_status gdl_join_scan(gdl_ctx *ctx, const uint32_t *d_counts, uint64_t n, uint64_t *d_offsets,
                         uint64_t *total) {
    if (!ctx || !d_offsets || (n && !d_counts)) return GDL_ERR_INVALID_ARG;
    u64 tot = 0;
    GDL_TRY(exclusive_scan_u32_to_u64(ctx, d_counts, n, d_offsets, &tot));
    if (total) *total = tot;
    return GDL_OK;
}

}  // extern "C"
