// merge.hip -- merge path over two sorted duplicate-free key arrays
// A (full) and B (newt) with A-first tie order.  One pass yields
//   U = A u B   (flush_delta's merge, newt accumulation) and
//   D = B \ A   (the set difference of the semi-naive step).
// A B-key is a duplicate exactly when the A-key consumed just before it is
// equal (equal keys are adjacent in merge order and A goes first).
//
// One launch: a block takes a tile of keys of the merged sequence, finds where
// its B-keys go among its A-keys, counts the duplicates, learns how many the
// tiles before hold (tile_before), and writes its part of U and D.
#include "gdl_internal.hpp"

namespace gdl {

constexpr int MG_I = 8;  // keys per thread

// Number of A-keys among the first `diag` keys of the merge (A first on ties),
// by a whole wave: 64 probes a round (5 rounds for 41M keys, where a thread's
// binary search is 26 dependent loads).
__device__ __forceinline__ u64 merge_path(const u64 *A, u64 na, const u64 *B, u64 nb, u64 diag) {
    const int lane = threadIdx.x & 63;
    u64 lo = diag > nb ? diag - nb : 0;
    u64 hi = diag < na ? diag : na;
    while (lo < hi) {
        const u64 step = (hi - lo + 63) / 64;
        const u64 m = lo + (u64)lane * step;
        const u64 past = ~__ballot(m < hi && A[m] <= B[diag - 1 - m]);
        const int f = past ? __ffsll((unsigned long long)past) - 1 : 64;
        if (f == 0) break;  // A[lo] comes after the diagonal
        const u64 next = lo + (u64)f * step;
        lo += (u64)(f - 1) * step + 1;
        if (next < hi) hi = next;
    }
    return lo;
}

// The exclusive prefix sums of the population counts of N words, by one whole
// wave; returns the total.
template <int N>
__device__ __forceinline__ u32 scan_words(const u64 *words, u32 *before) {
    constexpr int PER = N > 64 ? N / 64 : 1;
    const int lane = threadIdx.x & 63;
    u32 c[PER], sum = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = lane * PER + j;
        c[j] = i < N ? (u32)__popcll(words[i]) : 0;
        sum += c[j];
    }
    u32 x = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const u32 y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    u32 at = x - sum;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = lane * PER + j;
        if (i < N) before[i] = at;
        at += c[j];
    }
    return __shfl(x, 63, 64);
}

// U (may be null) gets A u B, D (may be null) B \ A; *dups the duplicates'
// number, so |U| = na + nb - *dups and |D| = nb - *dups.  Each B-key finds its
// place among the tile's A-keys by a search in LDS and marks it in a bit
// array; the output at w of the tile is then the B-key after as many B-keys as
// are marked before w, or the A-key after the rest.  Consecutive lanes write
// consecutive outputs.  41M + 2M keys: 0.235 ms, 2.9 TB/s (a count and a write
// launch, each merging a thread's 8 keys one by one, took 0.245 + 0.309 ms).
template <int MG_B>
__global__ __launch_bounds__(MG_B) void k_merge(const u64 *A, u64 na, const u64 *B, u64 nb,
                                                u64 *U, u64 *D, TileLook look, u64 *dups,
                                                u32 *err) {
    constexpr int MG_TILE = MG_B * MG_I, MG_W = MG_TILE / 64;
    __shared__ u64 s[MG_TILE];
    __shared__ u64 s_is_b[MG_W], s_dup[MG_W];
    __shared__ u32 s_nb[MG_W], s_nd[MG_W];  // marks in the words before
    __shared__ u64 s_split[2], s_before;
    __shared__ u32 s_tile;
    const int t = threadIdx.x, lane = t & 63;
    const u32 tile = tile_ticket(look, &s_tile);
    const u64 d0 = (u64)tile * MG_TILE, tot = na + nb;
    const u64 d1 = d0 + MG_TILE < tot ? d0 + MG_TILE : tot;
    if (t < 128) {
        const u64 i = merge_path(A, na, B, nb, t < 64 ? d0 : d1);
        if (lane == 0) s_split[t >> 6] = i;
    }
    if (t < MG_W) s_is_b[t] = s_dup[t] = 0;
    __syncthreads();
    const u64 i0 = s_split[0], j0 = d0 - i0;
    // sorted inputs give i0 <= i1 <= i0 + (d1 - d0); anything else is treated
    // as an empty tile so no LDS or global index leaves its buffer
    u32 la = 0, lb = 0;
    if (s_split[1] < i0 || s_split[1] - i0 > d1 - d0) {
        if (t == 0) atomicOr(err, 4u);
    } else {
        la = (u32)(s_split[1] - i0);
        lb = (u32)(d1 - d0) - la;
    }
#pragma unroll
    for (int r = 0; r < MG_I; ++r) {
        const u32 x = r * MG_B + t;
        if (x < la + lb) s[x] = x < la ? A[i0 + x] : B[j0 + (x - la)];
    }
    const bool has_prev = i0 > 0;
    const u64 prev = has_prev ? A[i0 - 1] : 0;
    __syncthreads();
    u32 place[MG_I];  // of this thread's B-keys; bit 31: a duplicate
#pragma unroll
    for (int r = 0; r < MG_I; ++r) {
        const u32 x = r * MG_B + t;
        if (x >= lb) continue;
        const u64 v = s[la + x];
        u32 lo = 0, hi = la;  // A-keys <= v
        while (lo < hi) {
            const u32 mid = (lo + hi) >> 1;
            if (s[mid] <= v) lo = mid + 1;
            else hi = mid;
        }
        const bool dup = lo ? s[lo - 1] == v : has_prev && prev == v;
        const u32 w = lo + x;
        atomicOr((unsigned long long *)&s_is_b[w >> 6], 1ull << (w & 63));
        if (dup) atomicOr((unsigned long long *)&s_dup[w >> 6], 1ull << (w & 63));
        place[r] = w | (dup ? 1u << 31 : 0u);
    }
    __syncthreads();
    if (t < 64) {
        const u64 mine = scan_words<MG_W>(s_dup, s_nd);
        const u64 before = tile_before(look, tile, mine);
        if (t == 0) {
            s_before = before;
            if (tile == gridDim.x - 1) *dups = before + mine;
        }
    } else if (t < 128) {
        scan_words<MG_W>(s_is_b, s_nb);
    }
    __syncthreads();
    const u64 before = s_before;
    if (U) {
        const u64 lt = lane_mask_lt();
#pragma unroll
        for (int r = 0; r < MG_I; ++r) {
            const u32 w = r * MG_B + t;
            if (w >= la + lb) continue;
            const u64 is_b = s_is_b[w >> 6], dup = s_dup[w >> 6];
            const u32 nb_at = s_nb[w >> 6] + (u32)__popcll(is_b & lt);
            const u32 nd_at = s_nd[w >> 6] + (u32)__popcll(dup & lt);
            const u64 at = d0 + w - nd_at - before;
            if (!((dup >> lane) & 1ull) && at < tot)
                __builtin_nontemporal_store(((is_b >> lane) & 1ull) ? s[la + nb_at] : s[w - nb_at],
                                            &U[at]);
        }
    }
    if (D) {
#pragma unroll
        for (int r = 0; r < MG_I; ++r) {
            const u32 x = r * MG_B + t;
            if (x >= lb || (place[r] >> 31)) continue;
            const u32 w = place[r];
            const u32 nd_at =
                s_nd[w >> 6] + (u32)__popcll(s_dup[w >> 6] & ((1ull << (w & 63)) - 1ull));
            const u64 at = j0 + x - nd_at - before;
            if (at < nb) D[at] = s[la + x];  // (always, if the inputs are sorted)
        }
    }
}

static gdl_status merge_impl(gdl_ctx *ctx, const u64 *A, u64 na, const u64 *B, u64 nb, u64 *U,
                             u64 *n_u, u64 *D, u64 *n_d) {
    const u64 tot = na + nb;
    if (tot == 0) {
        if (n_u) *n_u = 0;
        if (n_d) *n_d = 0;
        return GDL_OK;
    }
    // Tickets come at 11 ns each (atomics on one word), so 41M + 2M keys in
    // tiles of 2048 took 395 us, 240 of them in 21,000 tickets; in tiles of
    // 8192 keys it takes 235 us.  Below 2^19 keys the smaller tiles spread over
    // more CUs.
    const bool big = tot >= 1ull << 19;
    const u64 tile = (big ? 1024 : 256) * MG_I, nt = (tot + tile - 1) / tile;
    if (nt > 0x7fffffffull) return fail(ctx, GDL_ERR_OVERFLOW, "merge: too many tiles");
    Scratch scr(ctx);
    TileLook look;
    GDL_TRY(tile_look(ctx, nt, &scr, &look));
    {
        // algorithmic bytes: read A and B here; the U / D writes are added
        // below once their sizes are known
        KTimer kt(ctx, K_MERGE, 8.0 * tot);
        auto launch = [&](auto kern, int block) {
            hipLaunchKernelGGL(kern, dim3((unsigned)nt), dim3(block), 0, ctx->stream, A, na, B, nb,
                               U, D, look, result_words(ctx), ctx->d_err);
        };
        if (big) launch(k_merge<1024>, 1024);
        else launch(k_merge<256>, 256);
        GDL_TRY(check_launch(ctx, "k_merge"));
    }
    u64 dups = 0;
    GDL_TRY(read_result(ctx, &dups));
    ctx->stats[K_MERGE].alg_bytes += (U ? 8.0 * (tot - dups) : 0.0) + (D ? 8.0 * (nb - dups) : 0.0);
    if (n_u) *n_u = tot - dups;
    if (n_d) *n_d = nb - dups;
    return GDL_OK;
}

}  // namespace gdl

using namespace gdl;

extern "C" {

gdl_status gdl_merge_union_u64(gdl_ctx *ctx, const uint64_t *d_a, uint64_t na, const uint64_t *d_b,
                               uint64_t nb, uint64_t *d_out, uint64_t *n_out) {
    if (!ctx || !n_out || (na && !d_a) || (nb && !d_b) || ((na + nb) && !d_out))
        return GDL_ERR_INVALID_ARG;
    return merge_impl(ctx, d_a, na, d_b, nb, d_out, n_out, nullptr, nullptr);
}

gdl_status gdl_set_difference_u64(gdl_ctx *ctx, const uint64_t *d_b, uint64_t nb,
                                  const uint64_t *d_a, uint64_t na, uint64_t *d_out,
                                  uint64_t *n_out) {
    if (!ctx || !n_out || (na && !d_a) || (nb && !d_b) || (nb && !d_out))
        return GDL_ERR_INVALID_ARG;
    if (nb == 0) {
        *n_out = 0;
        return GDL_OK;
    }
    return merge_impl(ctx, d_a, na, d_b, nb, nullptr, nullptr, d_out, n_out);
}

gdl_status gdl_merge_diff_u64(gdl_ctx *ctx, const uint64_t *d_full, uint64_t nf,
                              const uint64_t *d_newt, uint64_t nn, uint64_t *d_full_out,
                              uint64_t *n_full_out, uint64_t *d_delta, uint64_t *n_delta) {
    if (!ctx || !n_delta || (nf && !d_full) || (nn && (!d_newt || !d_delta)))
        return GDL_ERR_INVALID_ARG;
    if (d_full_out && !n_full_out) return GDL_ERR_INVALID_ARG;
    return merge_impl(ctx, d_full, nf, d_newt, nn, d_full_out, n_full_out, d_delta, n_delta);
}

}  // extern "C"
