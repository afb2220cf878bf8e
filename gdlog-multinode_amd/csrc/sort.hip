// sort.hip -- LSD radix sort of u64 tuple keys for gfx950.
//
// The key (c0 << 32) | c1 is first compressed order-preservingly to
// (c0 << lo_bits) | c1 (lo_bits = bit length bound of c1), so the number of
// digit passes is ceil((hi_bits + lo_bits) / r) instead of 64 / r, for the
// context's radix width r (4..8 bits, default 8; digits narrower than 8 bits
// leave the upper histogram rows empty).  With r = 8, 9-bit digits (512
// bins, two per thread) are used where they save a pass: 36-bit keys (two
// 18-bit ids) sort in 4 passes instead of 5.
//
// Over n > 4096 keys: one read of the keys counts the digits of every pass
// (k_rs_hist); then one launch per pass (k_rs_pass) reads and writes them
// once, a tile learning where its digits go from the tiles before it.
// Arrays of at most 4096 keys are sorted by one launch that runs every pass in
// LDS.
#include "gdl_internal.hpp"

namespace gdl {

constexpr int RS_B = 256;           // threads per block
constexpr int RS_I = 16;            // keys per thread
constexpr int RS_TILE = RS_B * RS_I; // 4096
constexpr int RS_WSPAN = 64 * RS_I;  // keys per wave
constexpr int RADIX = 256;          // 8-bit digits (the one-block sort)

__device__ __forceinline__ u64 compress_key(u64 k, int lo_bits) {
    return ((k >> 32) << lo_bits) | (k & 0xffffffffull);
}
__device__ __forceinline__ u64 expand_key(u64 k, int lo_bits) {
    return ((k >> lo_bits) << 32) | (k & ((1ull << lo_bits) - 1ull));
}
// A pass's digit: `pass` packs the shift (bits 0..7) and the digit width
// (bits 8..11, 4..8 bits; the tuned radix width).
__device__ __forceinline__ u32 digit_of(u64 k, int pass) {
    return (u32)(k >> (pass & 0xff)) & ((1u << (pass >> 8)) - 1u);
}
__host__ __device__ __forceinline__ int pass_code(int shift, int bits) {
    return shift | (bits << 8);
}

__device__ __forceinline__ u64 tile_pos(int w, int r, int lane) {
    return (u64)w * RS_WSPAN + (u64)r * 64 + lane;
}

// Lanes of this wave that hold the same RB-bit digit (among `valid` lanes).
template <int RB>
__device__ __forceinline__ u64 match_digit(u32 d, bool valid) {
    const u64 live = __ballot(valid);
    u32 lo = (u32)live, hi = (u32)(live >> 32);
#pragma unroll
    for (int b = 0; b < RB; ++b) {
        // all ones where this lane's bit is set: a peer's bit equals it
        const u32 m = (u32)((int)(d << (31 - b)) >> 31);
        const u64 bal = __ballot(m != 0);
        lo &= ~((u32)bal ^ m);
        hi &= ~((u32)(bal >> 32) ^ m);
    }
    const u64 peers = ((u64)hi << 32) | lo;
    return peers;
}

// Ranks the 16 keys a thread holds (wave-contiguous layout) within the tile,
// for digits of up to RB bits (2^RB bins, 2^RB / 256 per thread): on return
// s_hist[w][d] = exclusive offset of wave w's keys of digit d inside the
// tile's digit-d run, s_start[d] = start of digit d's run in the tile, and
// rank[r] = rank of key r among its wave's keys of the same digit.
template <int RB>
__device__ __forceinline__ void rank_tile(const u64 *keys, const bool *valid, u32 *rank, int shift,
                                          u32 (*s_hist)[1 << RB], u32 *s_start, u64 *s_scan) {
    constexpr int R = 1 << RB, DPT = R / RS_B;
    const int t = threadIdx.x, w = t >> 6;
    const u64 lt = lane_mask_lt();
    for (int x = t; x < 4 * R; x += RS_B) (&s_hist[0][0])[x] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_I; ++r) {
        const u32 d = digit_of(keys[r], shift);
        const u64 peers = match_digit<RB>(d, valid[r]);
        const u32 before = s_hist[w][d];
        const u32 within = (u32)__popcll(peers & lt);
        __builtin_amdgcn_wave_barrier();
        if (valid[r] && within == 0) s_hist[w][d] = before + (u32)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        rank[r] = before + within;
    }
    __syncthreads();
    // thread t owns digits t * DPT .. t * DPT + DPT - 1 (consecutive)
    u32 c[DPT][4];
    u32 sum = 0;
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
        const int d = t * DPT + j;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            c[j][v] = s_hist[v][d];
            sum += c[j][v];
        }
    }
    u64 tot;
    u32 start = (u32)block_exclusive_scan<RS_B>((u64)sum, s_scan, &tot);
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
        const int d = t * DPT + j;
        s_start[d] = start;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            s_hist[v][d] = start;
            start += c[j][v];
        }
    }
    __syncthreads();
}

// ---- multi-tile passes ----------------------------------------------------
// Two alternating arrays of running digit counts, one word per tile and digit:
// 2 bits of state (1 = the tile's own count, 2 = the count up to and with the
// tile) and the value, in one store.
template <typename S>
struct DigitState {
    static constexpr int kShift = 8 * sizeof(S) - 2;
    static __device__ __forceinline__ void put(S *p, u32 state, u64 v) {
        __hip_atomic_store(p, (S)(((S)state << kShift) | (S)v), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    // Keys of this digit in the tiles before `tile` (> 0); row: the digit's
    // word of tile 0, rows R words apart.  Reads 4 predecessors at a time, and
    // waits only for tiles whose block runs and publishes its own count
    // without waiting (tiles are handed out in the order blocks start).
    template <int R>
    static __device__ __forceinline__ u64 before(const S *row, u32 tile) {
        constexpr int W = 4;
        u64 sum = 0;
        for (long long j = (long long)tile - 1; j >= 0;) {
            S w[W];
#pragma unroll
            for (int k = 0; k < W; ++k)
                w[k] = j - k >= 0 ? __hip_atomic_load(row + (j - k) * R, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT)
                                  : (S)2 << kShift;
            int used = 0;
            bool open = true, done = false;
#pragma unroll
            for (int k = 0; k < W; ++k) {
                const u32 state = (u32)(w[k] >> kShift);
                open = open && !done && state != 0;
                if (open) {
                    sum += (u64)(w[k] & (((S)1 << kShift) - 1));
                    ++used;
                    done = state == 2;
                }
            }
            if (done) break;
            if (used == 0) __builtin_amdgcn_s_sleep(1);
            j -= used;
        }
        return sum;
    }
};

// The counts of a sort in a recorded graph (a kernel, not a memset node).
__global__ __launch_bounds__(256) void k_rs_clear(u32 *hist) {
    const u32 i = blockIdx.x * 256 + threadIdx.x;
    if (i < kSortWords) hist[i] = 0;
}

// Digit counts of every pass in one read of the keys: hist[p << RB | digit]
// (zero before), LDS counters per block, two copies by wave parity.  A wave
// whose keys all have one digit (the high digits of sorted or clustered keys)
// adds it once.  Also clears the passes' first array of digit states.  Four
// 9-bit digits of 41M keys: 0.100 ms, 3.3 TB/s.
constexpr int RH_B = 1024;
template <int RB>
__global__ __launch_bounds__(RH_B) void k_rs_hist(const u64 *in, u64 n, int lo_bits, int xf,
                                                  int dbits, int passes, u32 *hist, u32 *state,
                                                  u64 state_words) {
    constexpr int BINS = kSortCounts;  // passes << RB is at most this
    __shared__ u32 s_h[2][BINS];
    const int t = threadIdx.x, copy = (t >> 6) & 1;
    const u64 g = (u64)blockIdx.x * RH_B + t, stride = (u64)gridDim.x * RH_B;
    for (u64 i = g; i < state_words; i += stride) state[i] = 0;
    const int bins = passes << RB;
    for (int x = t; x < bins; x += RH_B) s_h[0][x] = s_h[1][x] = 0;
    __syncthreads();
    auto count = [&](u64 k) {
        if (xf) k = compress_key(k, lo_bits);
        for (int p = 0; p < passes; ++p) {
            const u32 d = digit_of(k, pass_code(p * dbits, dbits));
            const u32 one = __builtin_amdgcn_readfirstlane(d);
            const u64 here = __ballot(true), others = __ballot(d != one);
            if (others)
                atomicAdd(&s_h[copy][(p << RB) | d], 1u);
            else if ((t & 63) == __ffsll((unsigned long long)here) - 1)
                atomicAdd(&s_h[copy][(p << RB) | d], (u32)__popcll(here));
        }
    };
    u64 i = g;
    for (; i + 3 * stride < n; i += 4 * stride) {
        const u64 k0 = in[i], k1 = in[i + stride], k2 = in[i + 2 * stride], k3 = in[i + 3 * stride];
        count(k0);
        count(k1);
        count(k2);
        count(k3);
    }
    for (; i < n; i += stride) count(in[i]);
    __syncthreads();
    for (int x = t; x < bins; x += RH_B) {
        const u32 c = s_h[0][x] + s_h[1][x];
        if (c) atomicAdd(&hist[x], c);
    }
}

// One pass: a block takes a tile of B x I keys, ranks them (wave64 ballot
// match per 64 keys, running LDS counts per wave), publishes the tile's digit
// counts, places the keys in digit order in LDS, learns the counts of the
// tiles before (DigitState::before), and stores the keys run by run, so
// consecutive lanes store consecutive addresses.  The keys are read and
// written once.  The first pass clears the counts of the sort before (`clear`)
// for the next.  41M keys: 0.198 ms a pass, 3.3 TB/s (a count launch, a scan
// over tiles and a scatter launch took 0.120 + 0.022 + 0.250); 100,000 keys:
// 7.9 us (7.4 + 3.4 + 11).  x_flags: 1 compress on reading, 2 expand on writing.
template <int RB, int B, int I, typename S>
__global__ __launch_bounds__(B) void k_rs_pass(const u64 *in, u64 *out, u64 n, int pass,
                                               int lo_bits, int x_flags, const u32 *hist, S *state,
                                               S *state_next, u32 *ticket, u32 *clear,
                                               u32 *err) {
    constexpr int R = 1 << RB, NW = B / 64, TILE = B * I;
    constexpr int DPT = R > B ? R / B : 1;  // digits a thread owns (threads past R / DPT: none)
    constexpr int WORDS = TILE > NW * R / 2 ? TILE : NW * R / 2;
    __shared__ u64 s_keys[WORDS];  // first the waves' digit counts, then the tile's keys
    __shared__ u32 s_dst[R];       // a digit's destination minus its start in the tile
    __shared__ u64 s_scan[NW + 1];
    __shared__ u32 s_tile;
    u32 *s_hist = (u32 *)s_keys;
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const u64 lt = lane_mask_lt();
    if (t == 0) s_tile = atomicAdd(ticket, 1u);
    for (int x = t; x < NW * R; x += B) s_hist[x] = 0;
    __syncthreads();
    const u32 tile = s_tile;
    const u64 base = (u64)tile * TILE;
    const u32 tile_n = n - base < (u64)TILE ? (u32)(n - base) : (u32)TILE;
    u64 keys[I];
    u32 pos[I];
#pragma unroll
    for (int r = 0; r < I; ++r) {
        const u32 x = (u32)w * (64 * I) + (u32)r * 64 + lane;
        keys[r] = x < tile_n ? in[base + x] : 0;
    }
    for (int d = t; d < R; d += B) state_next[(u64)tile * R + d] = 0;
    if (clear && tile == 0)
        for (u32 x = t; x < kSortWords; x += B) clear[x] = 0;
    u32 *wh = s_hist + w * R;
#pragma unroll
    for (int r = 0; r < I; ++r) {
        const bool valid = (u32)w * (64 * I) + (u32)r * 64 + lane < tile_n;
        if (x_flags & 1) keys[r] = compress_key(keys[r], lo_bits);
        const u32 d = digit_of(keys[r], pass);
        const u64 peers = match_digit<RB>(d, valid);
        const u32 before = wh[d];
        const u32 within = (u32)__popcll(peers & lt);
        __builtin_amdgcn_wave_barrier();
        if (valid && within == 0) wh[d] = before + (u32)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        pos[r] = before + within;
    }
    __syncthreads();
    // thread t owns digits t * DPT ..: tile count (published at once), start in
    // the tile, start in the output
    u32 sum[DPT];
    u64 both = 0;  // output counts in the high half, tile counts in the low
    const bool owner = t * DPT < R;
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
        const int d = t * DPT + j;
        sum[j] = 0;
        if (!owner) continue;
        for (int v = 0; v < NW; ++v) sum[j] += s_hist[v * R + d];
        DigitState<S>::put(state + (u64)tile * R + d, tile ? 1 : 2, sum[j]);
        both += ((u64)hist[d] << 32) | sum[j];
    }
    u64 all;
    u64 at = block_exclusive_scan<B>(both, s_scan, &all);
    u32 to[DPT];
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
        const int d = t * DPT + j;
        if (!owner) continue;
        u32 start = (u32)at;
        to[j] = (u32)(at >> 32) - start;
        at += ((u64)hist[d] << 32) | sum[j];
        for (int v = 0; v < NW; ++v) {
            const u32 c = s_hist[v * R + d];
            s_hist[v * R + d] = start;
            start += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < I; ++r) pos[r] += wh[digit_of(keys[r], pass)];
    __syncthreads();  // the counts make room for the keys
#pragma unroll
    for (int r = 0; r < I; ++r)
        if ((u32)w * (64 * I) + (u32)r * 64 + lane < tile_n && pos[r] < (u32)TILE)
            s_keys[pos[r]] = keys[r];
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
        const int d = t * DPT + j;
        if (!owner) continue;
        if (tile) {
            const u64 b = DigitState<S>::template before<R>(state + d, tile);
            DigitState<S>::put(state + (u64)tile * R + d, 2, b + sum[j]);
            to[j] += (u32)b;
        }
        s_dst[d] = to[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < I; ++j) {
        const u32 p = (u32)j * B + t;
        if (p < tile_n) {
            u64 k = s_keys[p];
            const u32 dst = s_dst[digit_of(k, pass)] + p;
            if (x_flags & 2) k = expand_key(k, lo_bits);
            if (dst < n) out[dst] = k;
            else atomicOr(err, 2u);  // inconsistent digit counts: never write out of bounds
        }
    }
}

// Whole sort of n <= 4096 keys in one block: every pass runs in LDS.
// With UNIQUE, adjacent duplicates are dropped and the count is stored to
// *n_out.
template <bool XF, bool UNIQUE>
__global__ __launch_bounds__(RS_B) void k_rs_oneblock(const u64 *in, u64 *out, u32 n, int passes,
                                                      int lo_bits, u64 *n_out) {
    __shared__ u64 s_keys[RS_TILE];
    __shared__ u32 s_hist[4][RADIX];
    __shared__ u32 s_start[RADIX];
    __shared__ u64 s_scan[RS_B / 64 + 1];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    u64 keys[RS_I];
    bool valid[RS_I];
    u32 rank[RS_I];
#pragma unroll
    for (int r = 0; r < RS_I; ++r) {
        const u64 p = tile_pos(w, r, lane);
        valid[r] = p < n;
        u64 k = valid[r] ? in[p] : 0;
        if (XF) k = compress_key(k, lo_bits);
        keys[r] = k;
    }
    // passes packs the pass count (bits 0..7) and the digit width (8..11)
    const int n_pass = passes & 0xff, dbits = passes >> 8;
    for (int pass = 0; pass < n_pass; ++pass) {
        const int shift = pass_code(pass * dbits, dbits);
        rank_tile<8>(keys, valid, rank, shift, s_hist, s_start, s_scan);
#pragma unroll
        for (int r = 0; r < RS_I; ++r)
            if (valid[r]) {
                const u32 pos = s_hist[w][digit_of(keys[r], shift)] + rank[r];
                if (pos < (u32)RS_TILE) s_keys[pos] = keys[r];
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < RS_I; ++r)
            if (valid[r]) keys[r] = s_keys[tile_pos(w, r, lane)];
        __syncthreads();
    }
    if (!UNIQUE) {
#pragma unroll
        for (int r = 0; r < RS_I; ++r) {
            if (valid[r]) out[tile_pos(w, r, lane)] = XF ? expand_key(keys[r], lo_bits) : keys[r];
        }
        return;
    }
    // keys[r] sits at tile position tile_pos(w, r, lane); s_keys holds the
    // sorted tile when passes > 0, otherwise reload it.
    if (n_pass == 0) {
#pragma unroll
        for (int r = 0; r < RS_I; ++r)
            if (valid[r]) s_keys[tile_pos(w, r, lane)] = keys[r];
        __syncthreads();
    }
    const u64 lt = lane_mask_lt();
    u64 carry = 0;
    u32 bits = 0;
#pragma unroll
    for (int r = 0; r < RS_I; ++r) {
        const u64 p = tile_pos(w, r, lane);
        const bool f = valid[r] && (p == 0 || s_keys[p - 1] != keys[r]);
        bits |= (u32)f << r;
        carry += __popcll(__ballot(f));
    }
    if (lane == 0) s_scan[w] = carry;
    __syncthreads();
    u64 off = 0;
    for (int k = 0; k < w; ++k) off += s_scan[k];
#pragma unroll
    for (int r = 0; r < RS_I; ++r) {
        const bool f = (bits >> r) & 1u;
        const u64 bal = __ballot(f);
        if (f) out[off + __popcll(bal & lt)] = XF ? expand_key(keys[r], lo_bits) : keys[r];
        off += __popcll(bal);
    }
    if (t == RS_B - 1) *n_out = off;  // wave 3's running offset ends at the total
}

// The OR of each column over all keys (their bit lengths), to result[0] and
// result[1] by the last block.
__global__ __launch_bounds__(256) void k_key_bits(const u64 *in, u64 n, CtxWords *words,
                                                  u64 *result) {
    __shared__ u64 s_or[4];
    u64 both = 0;
    for (u64 i = (u64)blockIdx.x * 256 + threadIdx.x; i < n; i += (u64)gridDim.x * 256)
        both |= in[i];
    for (int d = 32; d >= 1; d >>= 1) both |= __shfl_xor(both, d, 64);
    if ((threadIdx.x & 63) == 0) s_or[threadIdx.x >> 6] = both;
    __syncthreads();
    if (threadIdx.x) return;
    for (int w = 1; w < 4; ++w) both |= s_or[w];
    atomicOr(&words->bits[0], (unsigned long long)(both >> 32));
    atomicOr(&words->bits[1], (unsigned long long)(both & 0xffffffffull));
    if (!last_block(&words->bits[2])) return;
    result[0] = atomicExch(&words->bits[0], 0ull);
    result[1] = atomicExch(&words->bits[1], 0ull);
    atomicExch(&words->bits[2], 0ull);
}

static int bit_length(u64 v) { return v ? 64 - __builtin_clzll(v) : 0; }

static gdl_status measure_bits(gdl_ctx *ctx, const u64 *d_in, u64 n, int *hi_bits, int *lo_bits) {
    // (two blocks a CU for large arrays: three atomics each, on one line)
    const unsigned grid = (unsigned)std::min<u64>(grid_for(n, 256 * 8), 512);
    {
        KTimer kt(ctx, K_KEY_BITS, 8.0 * n);
        hipLaunchKernelGGL(k_key_bits, dim3(grid), dim3(256), 0, ctx->stream, d_in, n, ctx->words,
                           result_words(ctx));
        GDL_TRY(check_launch(ctx, "k_key_bits"));
    }
    u64 h[2];
    GDL_TRY(read_result(ctx, h, 2));
    *hi_bits = bit_length(h[0]);
    *lo_bits = bit_length(h[1]);
    return GDL_OK;
}

// The multi-tile LSD passes over n > 4096 keys with digits of dbits <= RB
// bits (2^RB histogram bins); the last pass lands in d_out.
template <int RB, int B, int I, typename S>
static gdl_status tile_passes_of(gdl_ctx *ctx, const u64 *d_in, u64 n, int lo_bits, bool xf,
                                 int dbits, int passes, u64 *d_out) {
    constexpr int R = 1 << RB;
    const u32 nb = (u32)((n + B * I - 1) / (B * I));
    Scratch scr(ctx);
    S *state;
    u64 *tmp = nullptr;
    if (passes > 1) GDL_TRY(scr.get(n, &tmp));
    GDL_TRY(scr.get(2 * (u64)R * nb, &state));  // last: larger tiles need less
    // A recorded sort replays with the set it was recorded with, whatever sorts
    // ran in between: recorded sorts share one that no other sort uses, and each
    // clears it itself (they follow each other on the stream: their scratch is
    // one block of the pool, too).
    const bool recorded = records_graph(ctx);
    u32 *hist = ctx->words->sort[2], *other = nullptr;
    if (recorded) {
        hipLaunchKernelGGL(k_rs_clear, dim3((kSortWords + 255) / 256), dim3(256), 0, ctx->stream,
                           hist);
        GDL_TRY(check_launch(ctx, "k_rs_clear"));
    } else {
        if (ctx->sort_dirty)
            GDL_HIP(ctx,
                    hipMemsetAsync(ctx->words->sort, 0, sizeof(ctx->words->sort), ctx->stream));
        ctx->sort_dirty = true;  // until every launch has been made
        hist = ctx->words->sort[ctx->sort_set];
        other = ctx->words->sort[ctx->sort_set ^ 1];
    }
    {
        KTimer kt(ctx, K_RS_HIST, 8.0 * n);
        const u64 cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
        hipLaunchKernelGGL(k_rs_hist<RB>, dim3(std::min<u64>(grid_for(n, 8 * RH_B), cus)),
                           dim3(RH_B), 0, ctx->stream, d_in, n, lo_bits, (int)xf, dbits, passes,
                           hist, (u32 *)state, (u64)R * nb * (sizeof(S) / sizeof(u32)));
        GDL_TRY(check_launch(ctx, "k_rs_hist"));
    }
    const u64 *src = d_in;
    for (int p = 0; p < passes; ++p) {
        u64 *dst = ((passes - 1 - p) % 2 == 0) ? d_out : tmp;
        const int x_flags = xf ? (p == 0 ? 1 : 0) | (p == passes - 1 ? 2 : 0) : 0;
        KTimer kt(ctx, K_RS_PASS, 16.0 * n);
        hipLaunchKernelGGL((k_rs_pass<RB, B, I, S>), dim3(nb), dim3(B), 0, ctx->stream, src, dst,
                           n, pass_code(p * dbits, dbits), lo_bits, x_flags, hist + (size_t)p * R,
                           state + (u64)(p & 1) * R * nb, state + (u64)(~p & 1) * R * nb,
                           hist + kSortCounts + p, p ? nullptr : other, ctx->d_err);
        GDL_TRY(check_launch(ctx, "k_rs_pass"));
        src = dst;
    }
    if (recorded) return GDL_OK;
    ctx->sort_set ^= 1;
    ctx->sort_dirty = false;
    return GDL_OK;
}

template <int RB>
static gdl_status tile_passes(gdl_ctx *ctx, const u64 *d_in, u64 n, int lo_bits, bool xf,
                              int dbits, int passes, u64 *d_out) {
    // Tiles: 2048 keys up to 2^18 (more CUs at work), 4096 up to 2^20, 8192
    // above (longer runs per digit in the stores, fewer tickets); few keys a
    // thread, so a wave's serial ranking is short.  Measured, us for 4 passes:
    // 100,000 keys 40 (256 threads x 8: 43), 1M 70 (512 x 8: 72), 2.5M 101 (4096
    // keys a tile: 117), 41M 895 (512 x 16: 928).  A digit's running count fits
    // 30 bits below 2^30 keys; from there the words are of 64 bits, and tiles of
    // 16384 keys halve their number (2^30 keys 23.9 ms, in tiles of 8192 30.5).
    // Smaller tiles need more memory for their words: where it does not hold
    // them, tiles of 8192 keys are taken.
    gdl_status st = GDL_ERR_OUT_OF_MEMORY;
    if (n <= 1ull << 18)
        st = tile_passes_of<RB, 512, 4, u32>(ctx, d_in, n, lo_bits, xf, dbits, passes, d_out);
    else if (n <= 1ull << 20)
        st = tile_passes_of<RB, 1024, 4, u32>(ctx, d_in, n, lo_bits, xf, dbits, passes, d_out);
    if (st != GDL_ERR_OUT_OF_MEMORY) return st;
    if (n < 1ull << 30)
        return tile_passes_of<RB, 1024, 8, u32>(ctx, d_in, n, lo_bits, xf, dbits, passes, d_out);
    return tile_passes_of<RB, 1024, 16, u64>(ctx, d_in, n, lo_bits, xf, dbits, passes, d_out);
}

// Shared driver of sort and sort+unique.  For n <= 4096 with `unique`,
// *n_unique receives the unique count (the caller then skips unique_keys).
static gdl_status sort_driver(gdl_ctx *ctx, const u64 *d_in, u64 n, int hi_bits, int lo_bits,
                              u64 *d_out, bool unique, u64 *n_unique, bool *uniqued) {
    *uniqued = false;
    if (n == 0) return GDL_OK;
    if (n >= 0xffffffffull) return fail(ctx, GDL_ERR_OVERFLOW, "sort: more than 2^32-1 keys");
    if (hi_bits < 0 || lo_bits < 0) GDL_TRY(measure_bits(ctx, d_in, n, &hi_bits, &lo_bits));
    if (hi_bits > 32 || lo_bits > 32)
        return fail(ctx, GDL_ERR_INVALID_ARG, "sort: key bit bounds above 32");
    const bool xf = lo_bits < 32;
    const int total_bits = hi_bits + (xf ? lo_bits : 32);
    const int dbits = ctx->tune.radix_bits;  // 4..8
    const int passes = (total_bits + dbits - 1) / dbits;
    const int pcode = passes | (dbits << 8);

    if (n <= (u64)RS_TILE) {
        KTimer kt(ctx, K_RS_ONEBLOCK, 16.0 * n);
        u64 *cnt = nullptr;
        Scratch scr(ctx);
        if (unique) GDL_TRY(scr.get(1, &cnt));
        if (xf) {
            if (unique)
                hipLaunchKernelGGL((k_rs_oneblock<true, true>), dim3(1), dim3(RS_B), 0, ctx->stream,
                                   d_in, d_out, (u32)n, pcode, lo_bits, cnt);
            else
                hipLaunchKernelGGL((k_rs_oneblock<true, false>), dim3(1), dim3(RS_B), 0,
                                   ctx->stream, d_in, d_out, (u32)n, pcode, lo_bits, cnt);
        } else {
            if (unique)
                hipLaunchKernelGGL((k_rs_oneblock<false, true>), dim3(1), dim3(RS_B), 0,
                                   ctx->stream, d_in, d_out, (u32)n, pcode, lo_bits, cnt);
            else
                hipLaunchKernelGGL((k_rs_oneblock<false, false>), dim3(1), dim3(RS_B), 0,
                                   ctx->stream, d_in, d_out, (u32)n, pcode, lo_bits, cnt);
        }
        GDL_TRY(check_launch(ctx, "k_rs_oneblock"));
        if (unique) {
            GDL_TRY(read_u64(ctx, cnt, n_unique));
            *uniqued = true;
        }
        return GDL_OK;
    }

    if (passes == 0) {  // every key equal
        GDL_HIP(ctx, hipMemcpyAsync(d_out, d_in, n * sizeof(u64), hipMemcpyDeviceToDevice,
                                    ctx->stream));
        return GDL_OK;
    }
    // nine-bit digits where they save a pass (36-bit keys: 4 passes, not 5;
    // 18-bit keys: 2, not 3)
    if (dbits == 8 && (total_bits + 8) / 9 < passes)
        return tile_passes<9>(ctx, d_in, n, lo_bits, xf, 9, (total_bits + 8) / 9, d_out);
    return tile_passes<8>(ctx, d_in, n, lo_bits, xf, dbits, passes, d_out);
}

gdl_status sort_keys(gdl_ctx *ctx, const u64 *d_in, u64 n, int hi_bits, int lo_bits, u64 *d_out) {
    u64 dummy;
    bool uniqued;
    return sort_driver(ctx, d_in, n, hi_bits, lo_bits, d_out, false, &dummy, &uniqued);
}

gdl_status sort_unique_keys(gdl_ctx *ctx, const u64 *d_in, u64 n, int hi_bits, int lo_bits,
                            u64 *d_out, u64 *n_out) {
    if (n == 0) {
        *n_out = 0;
        return GDL_OK;
    }
    bool uniqued = false;
    if (n <= (u64)RS_TILE)
        return sort_driver(ctx, d_in, n, hi_bits, lo_bits, d_out, true, n_out, &uniqued);
    Scratch scr(ctx);
    u64 *tmp;
    GDL_TRY(scr.get(n, &tmp));
    GDL_TRY(sort_driver(ctx, d_in, n, hi_bits, lo_bits, tmp, false, n_out, &uniqued));
    return unique_keys(ctx, tmp, n, d_out, n_out);
}

}  // namespace gdl

using namespace gdl;

extern "C" {

gdl_status gdl_sort_u64(gdl_ctx *ctx, const uint64_t *d_in, uint64_t n, int hi_bits, int lo_bits,
                        uint64_t *d_out) {
    if (!ctx || (n && (!d_in || !d_out))) return GDL_ERR_INVALID_ARG;
    if (n && d_in == d_out) return fail(ctx, GDL_ERR_INVALID_ARG, "gdl_sort_u64: d_in == d_out");
    return sort_keys(ctx, d_in, n, hi_bits, lo_bits, d_out);
}

gdl_status gdl_key_bits(gdl_ctx *ctx, const uint64_t *d_keys, uint64_t n, int *hi_bits,
                        int *lo_bits) {
    if (!ctx || !hi_bits || !lo_bits || (n && !d_keys)) return GDL_ERR_INVALID_ARG;
    if (n == 0) {
        *hi_bits = *lo_bits = 0;
        return GDL_OK;
    }
    return measure_bits(ctx, d_keys, n, hi_bits, lo_bits);
}

gdl_status gdl_sort_unique_u64(gdl_ctx *ctx, const uint64_t *d_in, uint64_t n, int hi_bits,
                               int lo_bits, uint64_t *d_out, uint64_t *n_out) {
    if (!ctx || !n_out || (n && (!d_in || !d_out))) return GDL_ERR_INVALID_ARG;
    if (n && d_in == d_out)
        return fail(ctx, GDL_ERR_INVALID_ARG, "gdl_sort_unique_u64: d_in == d_out");
    return sort_unique_keys(ctx, d_in, n, hi_bits, lo_bits, d_out, n_out);
}

}  // extern "C"
