// join.hip -- prefix hash index, hash join (count, scan, materialize),
// projection.
//
// Index: open addressing with linear probing over the distinct join prefixes
// of a sorted key array; each slot maps a prefix to its run [begin,
// begin + count).  Slot = 16 bytes, probed with one 128-bit load.  The run
// length is stored saturated at 2^24 - 1 and recomputed by galloping search
// in a probe that finds it so.
//
// Materialize is load-balanced: blocks take tiles of 2048 consecutive outputs
// and find the outer tuples that own them in LDS (JoinTile).
#include "gdl_internal.hpp"

namespace gdl {

constexpr int JB = 256;
constexpr int JM_I = 8;
constexpr int JM_TILE = JB * JM_I;  // outputs of a block's tile

// First index >= from whose prefix differs from p (keys sorted, keys[from - 1]
// has prefix p; n when the run lasts to the end), found by the whole wave: the
// next 64 keys, then 64 probes at doubling distances, then 64-way narrowing.
__device__ __forceinline__ u64 wave_run_end(const u64 *keys, u64 n, u64 from, u64 p, int shift) {
    const int lane = threadIdx.x & 63;
    auto first_out = [&](bool in) {  // the first lane outside the run, 64 if none
        const u64 out = ~__ballot(in);
        return out ? __ffsll((unsigned long long)out) - 1 : 64;
    };
    auto same = [&](u64 i, u64 end) { return i < end && (keys[i] >> shift) == p; };
    int f = first_out(same(from + lane, n));
    if (f < 64) return from + f < n ? from + f : n;
    f = first_out(lane < 40 && same(from + (64ull << lane) - 1, n));
    u64 lo = f ? from + (64ull << (f - 1)) - 1 : from + 63;  // in the run
    u64 hi = from + (64ull << f) - 1;                         // past it
    if (hi > n) hi = n;
    while (hi - lo > 1) {
        const u64 step = (hi - lo + 63) / 64;
        f = first_out(same(lo + (u64)(lane + 1) * step, hi));
        const u64 next = lo + (u64)(f + 1) * step;
        lo += (u64)f * step;
        if (next < hi) hi = next;
    }
    return hi;
}

// emit(i, prefix, end) on the lane of every run [i, end) that starts in the
// wave's span of 64 R consecutive keys from `base`; returns the number of
// them.  One streaming read of the keys: run starts are ballots, a run ends at
// the next set bit, and only the span's last run looks past the span.  (A
// galloping search from every run start, a serial chain of dependent loads
// for a few lanes of each wave, took 1.76 ms to count 41M keys in 262k runs
// and 0.58 ms to build the direct-mapped index; this takes 0.12 and 0.08 ms,
// 2.7 and 4.0 TB/s.)
template <int R, typename F>
__device__ __forceinline__ u32 span_runs(const u64 *keys, u64 n, int shift, u64 base, F emit) {
    const int lane = threadIdx.x & 63;
    u64 p[R], heads[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const u64 i = base + (u64)r * 64 + lane;
        p[r] = i < n ? keys[i] >> shift : 0;
    }
    u64 before = base > 0 ? keys[base - 1] >> shift : 0;
    u32 count = 0;
    u64 last = 0;  // prefix of the span's last key
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const u64 i = base + (u64)r * 64 + lane;
        const u64 up = wave_shift_up(p[r], before);  // in every lane
        const bool head = i < n && (i == 0 || up != p[r]);
        heads[r] = __ballot(head);
        count += (u32)__popcll(heads[r]);
        last = before = wave_last(p[r]);
    }
    if (count == 0) return 0;
    const u64 end = base + 64ull * R;
    u64 next = end < n ? wave_run_end(keys, n, end, last, shift) : n;  // uniform
#pragma unroll
    for (int r = R - 1; r >= 0; --r) {
        const u64 at = base + (u64)r * 64;
        if ((heads[r] >> lane) & 1ull) {
            const u64 later = lane < 63 ? heads[r] >> (lane + 1) : 0;
            emit(at + lane, p[r], later ? at + lane + __ffsll((unsigned long long)later) : next);
        }
        if (heads[r]) next = at + __ffsll((unsigned long long)heads[r]) - 1;
    }
    return count;
}

// Spans of 1024 keys a wave (R = 16) for large arrays; of 256 below 2^22 keys,
// where the longer ones leave CUs without a wave: count and build of 2M keys 48
// us with short spans and 54 with long, of 4M 60 and 63, of 4.2M 61-63 and
// 60-64, of 8M 73-75 and 76-79, of 16M 119 and 102.  The hash build takes 256
// and 64: its lanes insert one run after another, a chain of atomics that
// grows with the span (1M keys in 400k runs: 37 us with 64 or 256).
constexpr u64 kLongSpan = 1ull << 22;

// result[0] = distinct prefixes, result[1] = the longest run, result[2] = the
// largest prefix (the last key's: keys are sorted), by the last block.  One
// block of 16 waves per CU: the atomics all go to the same two words, ~12 ns
// each (1024 blocks of 4 waves spent 25 us on them).
constexpr int IC_B = 1024;
template <int R>
__global__ __launch_bounds__(IC_B) void k_idx_count(const u64 *keys, u64 n, int shift,
                                                    CtxWords *words, u64 *result) {
    __shared__ u64 s_sum[IC_B / 64], s_max[IC_B / 64];
    u64 acc = 0, mx = 0;
    const u64 span = 64ull * R;
    for (u64 b = ((u64)blockIdx.x * (IC_B / 64) + (threadIdx.x >> 6)) * span; b < n;
         b += (u64)gridDim.x * (IC_B / 64) * span)
        acc += span_runs<R>(keys, n, shift, b, [&](u64 i, u64, u64 end) {
            mx = end - i > mx ? end - i : mx;
        });
    for (int d = 32; d >= 1; d >>= 1) {
        const u64 o = __shfl_xor(mx, d, 64);
        mx = o > mx ? o : mx;
    }
    if ((threadIdx.x & 63) == 0) {
        s_sum[threadIdx.x >> 6] = acc;
        s_max[threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        u64 a = 0, m = 0;
        for (int w = 0; w < IC_B / 64; ++w) {
            a += s_sum[w];
            m = s_max[w] > m ? s_max[w] : m;
        }
        if (a) atomicAdd(&words->idx[0], (unsigned long long)a);
        if (m) atomicMax(&words->idx[1], (unsigned long long)m);
        if (last_block(&words->idx[2])) {
            result[0] = atomicExch(&words->idx[0], 0ull);
            result[1] = atomicExch(&words->idx[1], 0ull);
            result[2] = keys[n - 1] >> shift;
            atomicExch(&words->idx[2], 0ull);
        }
    }
}

__device__ __forceinline__ u64 run_word(u64 i, u64 end) {
    const u64 cnt = end - i;
    return (i << kCountBits) | (cnt < kCountSat ? cnt : kCountSat);
}

template <int R>
__global__ __launch_bounds__(JB) void k_idx_build(const u64 *keys, u64 n, int shift,
                                                  IdxSlot *slots, u64 n_slots, u32 *err) {
    const u64 nbk = n_slots / kBucket, span = 64ull * R;
    for (u64 first = ((u64)blockIdx.x * (JB / 64) + (threadIdx.x >> 6)) * span; first < n;
         first += (u64)gridDim.x * (JB / 64) * span)
        span_runs<R>(keys, n, shift, first, [&](u64 i, u64 p, u64 end) {
            const u64 val = run_word(i, end);
            u64 b = mulhi64(mix64(p), nbk);
            bool placed = false;
            for (u64 step = 0; step < nbk && !placed; ++step) {
                for (u64 j = 0; j < kBucket; ++j) {
                    IdxSlot *e = slots + b * kBucket + j;
                    if (e->val != 0) continue;
                    const unsigned long long old =
                        atomicCAS((unsigned long long *)&e->val, 0ull, (unsigned long long)val);
                    if (old == 0ull) {
                        e->key = p;
                        placed = true;
                        break;
                    }
                }
                if (++b == nbk) b = 0;
            }
            if (!placed) atomicOr(err, 1u);
        });
}

// Direct-mapped index: the run word of each prefix (run starts only).
template <int R>
__global__ __launch_bounds__(JB) void k_idx_build_dense(const u64 *keys, u64 n, int shift,
                                                        u64 *words, u64 range) {
    const u64 span = 64ull * R;
    for (u64 b = ((u64)blockIdx.x * (JB / 64) + (threadIdx.x >> 6)) * span; b < n;
         b += (u64)gridDim.x * (JB / 64) * span)
        span_runs<R>(keys, n, shift, b, [&](u64 i, u64 p, u64 end) {
            if (p < range) words[p] = run_word(i, end);
        });
}

__device__ __forceinline__ bool lookup_run(const IdxSlot *slots, u64 n_slots, const u64 *keys,
                                           u64 n, int shift, u64 p, u64 *begin, u64 *count) {
    if (!idx_probe(slots, n_slots, p, begin, count)) return false;
    if (*begin >= n) return false;  // an index never points past its array
    if (*count == kCountSat) *count = run_end(keys, n, *begin, p, shift) - *begin;
    if (*count > n - *begin) *count = n - *begin;
    return true;
}

__global__ __launch_bounds__(JB) void k_idx_lookup(const IdxSlot *slots, u64 n_slots,
                                                   const u64 *keys, u64 n, int shift,
                                                   const u64 *q, u64 nq, u64 *begin, u32 *count) {
    for (u64 i = (u64)blockIdx.x * JB + threadIdx.x; i < nq; i += (u64)gridDim.x * JB) {
        u64 b = 0, c = 0;
        if (!lookup_run(slots, n_slots, keys, n, shift, q[i], &b, &c)) c = 0;
        begin[i] = b;
        count[i] = (u32)c;
    }
}

__global__ __launch_bounds__(JB) void k_join_count(const IdxSlot *slots, u64 n_slots,
                                                   const u64 *inner, u64 n_inner, int shift,
                                                   const u64 *outer, u64 n_outer, u32 *counts,
                                                   u64 *begins) {
    for (u64 i = (u64)blockIdx.x * JB + threadIdx.x; i < n_outer; i += (u64)gridDim.x * JB) {
        const u64 p = outer[i] >> shift;
        u64 b = 0, c = 0;
        if (!lookup_run(slots, n_slots, inner, n_inner, shift, p, &b, &c)) c = 0;
        counts[i] = (u32)c;
        begins[i] = b;
    }
}

// The outer tuples' run starts and the exclusive scan of their run lengths in
// one launch (a count launch and a scan are 3.2 + 5.7 us for CSPA's joins, most
// of them below 4096 outer tuples).
template <int B>
__global__ __launch_bounds__(B) void k_join_offsets(const IdxSlot *slots, u64 n_slots,
                                                    const u64 *inner, u64 n_inner, int shift,
                                                    const u64 *outer, u64 n_outer, TileLook look,
                                                    u64 *begins, u64 *offsets, u64 *total) {
    using Tile = ScanTile<B>;
    __shared__ Tile s;
    const u64 base = (u64)tile_ticket(look, &s.tile) * Tile::kTile;
#pragma unroll
    for (int r = 0; r < Tile::kPer; ++r) {
        const u32 x = r * B + threadIdx.x;
        const u64 i = base + x;
        u64 b = 0, c = 0;
        if (i < n_outer) {
            if (!lookup_run(slots, n_slots, inner, n_inner, shift, outer[i] >> shift, &b, &c))
                b = c = 0;
            begins[i] = b;
        }
        s.in[Tile::pad(x)] = (u32)c;
    }
    __syncthreads();
    s.scan(look, base, n_outer, offsets, total);
}

// ---- outputs numbered by the exclusive scan of the run lengths -------------
// A block takes tiles of JB * I consecutive outputs.  The outer tuples whose
// runs meet the tile are compacted in LDS and their first outputs marked in a
// bit array, so the owner of output w is a population count away, and
// consecutive lanes take consecutive outputs: inner reads and stores are
// coalesced whatever the run lengths.  (Each thread used to find its 8
// consecutive outputs' owner by a binary search over all offsets, ~21
// dependent loads at 2M outer tuples, and stored through LDS.)
template <int I>
struct JoinTile {
    static constexpr int kTile = JB * I, kWords = kTile / 64;
    u64 src[kTile];    // owner's begin - its first output: inner index = src + output
    u64 key[kTile];    // owner's outer key
    u64 mark[kWords];  // bit w: an owner's outputs start at w (bit 0 always)
    u32 base[kWords];  // marks in the words before
    u64 lo;            // an outer tuple at or before the tile's first owner
};

// jt.lo = the last outer tuple o with offsets[o] <= t0, by wave 0 (64-way
// search: 4 rounds of loads at 2M outer tuples).  Every thread calls it.
template <int I>
__device__ __forceinline__ void join_tile_seek(JoinTile<I> &jt, const u64 *offsets, u64 n_outer,
                                               u64 t0) {
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        u64 lo = 0, hi = n_outer;  // offsets[lo] <= t0, offsets[hi] > t0
        while (hi - lo > 1) {
            const u64 step = (hi - lo + 63) / 64;
            const u64 i = lo + (u64)(lane + 1) * step;
            const u64 past = ~__ballot(i < hi && offsets[i] <= t0);
            const int f = past ? __ffsll((unsigned long long)past) - 1 : 64;
            const u64 next = lo + (u64)(f + 1) * step;
            lo += (u64)f * step;
            if (next < hi) hi = next;
        }
        if (lane == 0) jt.lo = lo;
    }
    __syncthreads();
}

// The last outer tuple o of [lo, lo + len) with offsets[o] <= p, when lo's is.
__device__ __forceinline__ u64 last_at_most(const u64 *offsets, u64 lo, u64 len, u64 p) {
    while (len > 1) {
        const u64 half = len >> 1;
        if (offsets[lo + half] <= p) lo += half;
        len -= half;
    }
    return lo;
}

// The owners of the outputs [t0, t1) where most outer tuples have none (a walk
// over all of a tile's, by one block, took 5.6 ms at 1,544 outputs of 2M): every
// output is marked, its slot its own number.  A thread searches for the owner
// of the first of its I consecutive outputs, and at the end of a run for the
// next owner at doubling distances.  Every thread of a block calls it; ends
// with a barrier.
template <int I>
__device__ __forceinline__ void join_tile_search(JoinTile<I> &jt, const u64 *outer, u64 n_outer,
                                                 const u64 *offsets, const u64 *begins, u64 t0,
                                                 u64 t1) {
    const int t = threadIdx.x;
    const u64 p0 = t0 + (u64)t * I;
    if (p0 < t1) {
        u64 o = last_at_most(offsets, 0, n_outer, p0);
        u64 end = offsets[o + 1], src = begins[o] - offsets[o], key = outer[o];
#pragma unroll 1
        for (int r = 0; r < I && p0 + r < t1; ++r) {
            const u64 p = p0 + r;
            if (p >= end) {
                u64 step = 1;
                ++o;
                while (o + step < n_outer && offsets[o + step] <= p) {
                    o += step;
                    step *= 2;
                }
                o = last_at_most(offsets, o, step < n_outer - o ? step : n_outer - o, p);
                end = offsets[o + 1];
                src = begins[o] - offsets[o];
                key = outer[o];
            }
            jt.src[t * I + r] = src;
            jt.key[t * I + r] = key;
        }
    }
    if (t < JoinTile<I>::kWords) {
        jt.mark[t] = ~0ull;
        jt.base[t] = 64 * t;
    }
    __syncthreads();
}

// The owners of the outputs [t0, t1), at most a tile; jt.lo from
// join_tile_seek or from the tile before.  Every thread of a block of JB calls
// it; ends with a barrier.  jt.lo moves on to the last owner.
template <int I>
__device__ __forceinline__ void join_tile_owners(JoinTile<I> &jt, const u64 *outer, u64 n_outer,
                                                 const u64 *offsets, const u64 *begins, u64 t0,
                                                 u64 t1) {
    constexpr int W = JoinTile<I>::kWords;
    const int t = threadIdx.x;
    const u64 lo = jt.lo;
    if (t < W) jt.mark[t] = 0;
    __syncthreads();
    // nearly always one outer tuple a thread: its values stay in registers
    u64 b = 0, e = 0, begin = 0, key = 0;
    const bool first = lo + t < n_outer;
    if (first) {
        b = offsets[lo + t];
        e = offsets[lo + t + 1];
        begin = begins[lo + t];
        key = outer[lo + t];
    }
    auto mark = [&](u64 b, u64 e) {
        if (b < t1 && e > b && e > t0) {
            const u32 w = (u32)((b > t0 ? b : t0) - t0);
            atomicOr((unsigned long long *)&jt.mark[w >> 6], 1ull << (w & 63));
        }
    };
    if (first) mark(b, e);
    for (u64 o = lo + t + JB; o < n_outer && offsets[o] < t1; o += JB)
        mark(offsets[o], offsets[o + 1]);
    __syncthreads();
    if (t < 64) {
        u32 c = t < W ? (u32)__popcll(jt.mark[t]) : 0, x = c;
        for (int d = 1; d < 64; d <<= 1) {
            const u32 y = __shfl_up(x, d, 64);
            if (t >= d) x += y;
        }
        if (t < W) jt.base[t] = x - c;
    }
    __syncthreads();
    auto place = [&](u64 o, u64 b, u64 e, u64 begin, u64 key) {
        if (b < t1 && e > b && e > t0) {
            const u32 w = (u32)((b > t0 ? b : t0) - t0);
            const u32 at = jt.base[w >> 6] +
                           (u32)__popcll(jt.mark[w >> 6] & ((1ull << (w & 63)) - 1ull));
            jt.src[at] = begin - b;
            jt.key[at] = key;
            if (e >= t1) jt.lo = o;  // the owner of the last output
        }
    };
    if (first) place(lo + t, b, e, begin, key);
    for (u64 o = lo + t + JB; o < n_outer && offsets[o] < t1; o += JB)
        place(o, offsets[o], offsets[o + 1], begins[o], outer[o]);
    __syncthreads();
}

// Slot in jt.src / jt.key of the owner of the tile's output w, where the wave's
// lanes hold w = 64 x + lane.
template <int I>
__device__ __forceinline__ u32 join_tile_owner(const JoinTile<I> &jt, u32 w) {
    const u64 le = (2ull << (w & 63)) - 1ull;  // all ones for bit 63
    return jt.base[w >> 6] + (u32)__popcll(jt.mark[w >> 6] & le) - 1;
}

// offsets: n_outer + 1 entries (offsets[n_outer] == total).  A block takes
// `per` consecutive tiles and looks for its first owner once.  Bound by the
// stores and the runs' reads: 313M outputs of 2M outer tuples over 41M inner
// keys took 1.81 ms with a binary search per thread, take 1.22 ms, and 1.15 ms
// with nontemporal stores, which leave the caches to the inner keys (5 GB read
// and written at 4.4 TB/s; a large copy reaches 4.8).
template <int I, bool SPARSE>
__global__ __launch_bounds__(JB) void k_join_materialize(const u64 *inner, const u64 *outer,
                                                         u64 n_outer, const u64 *offsets,
                                                         const u64 *begins, u64 total, u32 per,
                                                         int arity, int s0, int s1, u64 *out) {
    constexpr int TILE = JoinTile<I>::kTile;
    __shared__ JoinTile<I> jt;
    u64 t0 = (u64)blockIdx.x * per * TILE;
    if constexpr (!SPARSE) join_tile_seek(jt, offsets, n_outer, t0);
    for (u32 k = 0; k < per && t0 < total; ++k, t0 += TILE) {
        const u64 t1 = t0 + TILE < total ? t0 + TILE : total;
        if constexpr (SPARSE)
            join_tile_search(jt, outer, n_outer, offsets, begins, t0, t1);
        else
            join_tile_owners(jt, outer, n_outer, offsets, begins, t0, t1);
        u64 ik[I], ok[I];
#pragma unroll
        for (int r = 0; r < I; ++r) {
            const u32 w = r * JB + threadIdx.x;
            if (t0 + w < t1) {
                const u32 at = join_tile_owner(jt, w);
                ik[r] = inner[jt.src[at] + (t0 + w)];
                ok[r] = jt.key[at];
            }
        }
#pragma unroll
        for (int r = 0; r < I; ++r) {
            const u32 w = r * JB + threadIdx.x;
            if (t0 + w < t1)
                __builtin_nontemporal_store(apply_map(ik[r], ok[r], arity, s0, s1), &out[t0 + w]);
        }
        __syncthreads();  // the next tile overwrites the owners
    }
}

// Join fused with insert-if-absent into a hash set.  Each wave takes 64
// outer tuples, probes their runs, and flattens the (outer, run position)
// pairs with a wave prefix sum, so every lane handles one produced tuple per
// round whatever the run lengths (a hub run is spread over the wave).  New
// keys are staged per wave in LDS and flushed with one atomic per kStage keys
// (the cursor).
constexpr u32 kStage = 256;
constexpr u64 kHubRun = 32;  // longer inner runs may use the load-balanced variant

// How a fused join's blocks hand over their counts: one atomic on the cursor
// word gives a block its place in the output and tells it whether it is the
// last (atomics on one word take 11 ns each, and the blocks all end at about
// the same time), which then has all of them.
enum EndMode {
    END_WORDS,   // cursor: new keys (50 bits), blocks (14); produced counts in a word per block
    END_PACKED,  // cursor: new keys (27 bits), produced tuples (27), blocks (10)
};
constexpr u32 kPackedBits = 27, kPackedBlocks = 1023;
template <int END>
struct EndCursor {
    static constexpr int kNewBits = END == END_PACKED ? kPackedBits : kDoneBit;
    static constexpr int kBlocksAt = END == END_PACKED ? 2 * kPackedBits : kDoneBit;
    static constexpr u64 kNew = (1ull << kNewBits) - 1;
};

// Writes stay below out_cap; a cursor past it tells the host the caller's
// output bound was wrong.
template <int END>
__device__ __forceinline__ void flush_stage(const u64 *stage, u32 n, u64 *out, u64 out_cap,
                                            unsigned long long *cursor, u64 base, int lane) {
    unsigned long long pos = 0;
    if (lane == 0)
        pos = base + (atomicAdd(cursor, (unsigned long long)n) & EndCursor<END>::kNew);
    pos = __shfl(pos, 0, 64);
    for (u32 x = lane; x < n; x += 64)
        if (pos + x < out_cap) out[pos + x] = stage[x];
}

// What the last block learns.
struct EndCounts {
    u64 fresh, produced;  // END_WORDS: produced is still in the blocks' words
};

// End of a fused-join block: what the waves still stage goes out at the place
// that the cursor gives, and the block's counts are handed over (EndMode).
// END_WORDS: the produced count is at the device's coherence point before the
// cursor says that the block is done (an agent-scope store that has been waited
// for).  Returns whether this block is the last.  Every thread calls it.
template <int B, int END>
__device__ __forceinline__ bool block_final_flush(u64 (*s_stage)[kStage], u32 staged,
                                                  u64 produced, u64 *out, u64 out_cap,
                                                  unsigned long long *cursor, u64 base,
                                                  unsigned long long *produced_to,
                                                  EndCounts *counts) {
    using C = EndCursor<END>;
    __shared__ u32 s_cnt[B / 64];
    __shared__ u64 s_prod[B / 64];
    __shared__ u64 s_base, s_all;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int d = 32; d >= 1; d >>= 1) produced += __shfl_xor(produced, d, 64);
    if (lane == 0) {
        s_cnt[w] = staged;
        s_prod[w] = produced;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        u64 tot = 0, prod = 0;
        for (int v = 0; v < B / 64; ++v) {
            tot += s_cnt[v];
            prod += s_prod[v];
        }
        u64 add = (1ull << C::kBlocksAt) | tot;
        if constexpr (END == END_WORDS) {
            __hip_atomic_store(&produced_to[blockIdx.x], (unsigned long long)prod,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            order_memory();
        } else {
            add += prod << kPackedBits;
        }
        const u64 old = atomicAdd(cursor, (unsigned long long)add);
        s_base = base + (old & C::kNew);
        s_all = old + add;
    }
    __syncthreads();
    u64 off = s_base;
    for (int v = 0; v < w; ++v) off += s_cnt[v];
    const u64 *stage = s_stage[w];
    for (u32 x = lane; x < staged; x += 64)
        if (off + x < out_cap) out[off + x] = stage[x];
    const u64 all = s_all;
    counts->fresh = all & C::kNew;
    counts->produced = (all >> kPackedBits) & EndCursor<END_PACKED>::kNew;
    return (all >> C::kBlocksAt) == gridDim.x;
}

// The sum of the blocks' produced words (END_WORDS), by the last block.
template <int B>
__device__ __forceinline__ u64 sum_produced(const unsigned long long *produced) {
    __shared__ u64 s_sum[B / 64];
    u64 sum = 0;
    for (u32 i = threadIdx.x; i < gridDim.x; i += B)
        sum += __hip_atomic_load(&produced[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 64);
    if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = sum;
    __syncthreads();
    sum = 0;
    for (int v = 0; v < B / 64; ++v) sum += s_sum[v];
    return sum;
}

// The last block of a fused join: new keys, produced tuples and whether a key
// was outside the id bound to the host; the context's words back to zero.
template <int B>
__device__ __forceinline__ void publish_join(CtxWords *words, u64 fresh, u64 *result) {
    const u64 produced = sum_produced<B>(words->produced);
    if (threadIdx.x) return;
    result[0] = fresh;
    result[1] = produced;
    result[2] = atomicExch(&words->outside, 0ull);
    atomicExch(&words->cursor, 0ull);
}

// Target of a fused join's inserts: one hash set, or one set per fixpoint
// instance of a batch, chosen by the key's top bits (key >> seg_shift).
struct HsSel {
    u64 *slots;
    u64 mask;
    const gdl_hs_seg *segs;
    u32 n_segs;
    int seg_shift;
    // > 0: the caller sized the set and the output by this id bound; a
    // produced key with an id at or above 2^dom_bits is not inserted and
    // sets *outside
    int dom_bits;
};

// The set a key belongs to (slots == nullptr: a segment with no set).
template <bool SEG>
__device__ __forceinline__ gdl_hs_seg sel_set(const HsSel &h, const gdl_hs_seg *s_segs, u64 key) {
    if constexpr (SEG) {
        const u64 s = key >> h.seg_shift;
        if (s >= h.n_segs) return gdl_hs_seg{nullptr, 0};
        return s_segs[s];
    } else {
        (void)s_segs;
        return gdl_hs_seg{h.slots, h.mask};
    }
}

template <bool SEG>
__device__ __forceinline__ void load_segs(const HsSel &h, gdl_hs_seg *s_segs) {
    if constexpr (SEG) {
        for (u32 i = threadIdx.x; i < h.n_segs; i += blockDim.x) s_segs[i] = h.segs[i];
        __syncthreads();
    } else {
        (void)h;
        (void)s_segs;
    }
}

// Inserts the live keys (bit r of `live`: keys[r]) and returns which were new.
// The home-slot CASes (bitmap: a plain load, since a set bit proves
// membership, then the ORs) of all of them are in flight together; keys that
// met another key at home are then probed for one per lane and round, so a
// wave takes as many probe rounds as its unluckiest lane has collisions, not
// one for every r that collided somewhere.
template <int N, bool SEG>
__device__ __forceinline__ u32 insert_keys(const HsSel &sel, const gdl_hs_seg *s_segs,
                                           const u64 *keys, u32 live, unsigned long long *outside) {
    unsigned long long old[N];
    u32 bm = 0;     // keys that went to a bitmap set (old: the bit before)
    u32 probe = 0;  // keys that need the full probe
    u32 fresh = 0;
#pragma unroll
    for (int r = 0; r < N; ++r) {
        old[r] = 0;
        if (!((live >> r) & 1u)) continue;
        const gdl_hs_seg hs = sel_set<SEG>(sel, s_segs, keys[r]);
        if (sel.dom_bits && !bm_in_domain(keys[r], sel.dom_bits)) {
            atomicOr(outside, 1ull);
            order_memory();  // before this block is done
            live &= ~(1u << r);
        } else if (!hs.slots) {
            live &= ~(1u << r);
        } else if (hs.mask & kHsBitmap) {
            const int kb = (int)(hs.mask & 63);
            if (bm_in_domain(keys[r], kb)) {
                const u64 b = bm_bit(keys[r], kb);
                old[r] = ((const u64 *)hs.slots)[b >> 6] & (1ull << (b & 63));
                bm |= 1u << r;
            } else {
                probe |= 1u << r;  // flags the set
            }
        } else if (keys[r] != kHsEmpty) {
            old[r] = atomicCAS((unsigned long long *)((u64 *)hs.slots + (mix64(keys[r]) & hs.mask)),
                               (unsigned long long)kHsEmpty, (unsigned long long)keys[r]);
        } else {
            probe |= 1u << r;
        }
    }
#pragma unroll
    for (int r = 0; r < N; ++r) {
        if (((bm >> r) & 1u) && old[r] == 0) {
            const gdl_hs_seg hs = sel_set<SEG>(sel, s_segs, keys[r]);
            const u64 b = bm_bit(keys[r], (int)(hs.mask & 63));
            const u64 m = 1ull << (b & 63);
            old[r] = atomicOr((unsigned long long *)((u64 *)hs.slots + (b >> 6)),
                              (unsigned long long)m) & m;
        }
    }
#pragma unroll
    for (int r = 0; r < N; ++r) {
        const u32 bit = 1u << r;
        if (!(live & bit) || (probe & bit)) continue;
        if (bm & bit) fresh |= old[r] == 0 ? bit : 0u;
        else if (old[r] == (unsigned long long)kHsEmpty) fresh |= bit;
        else if (old[r] != (unsigned long long)keys[r]) probe |= bit;
    }
    while (probe) {
        const u32 bit = probe & (0u - probe);
        u64 k = keys[0];
#pragma unroll
        for (int r = 1; r < N; ++r) k = (bit >> r) & 1u ? keys[r] : k;
        const gdl_hs_seg hs = sel_set<SEG>(sel, s_segs, k);
        const bool is_new =
            (hs.mask & kHsBitmap) || k == kHsEmpty
                ? hs_insert_key((u64 *)hs.slots, hs.mask, k)
                : hs_probe_from((u64 *)hs.slots, hs.mask, k, (mix64(k) + 1) & hs.mask);
        if (is_new) fresh |= bit;
        probe &= ~bit;
    }
    return fresh;
}

// One block's share of a fused join + insert (the blocks of the grid stride
// over the outer tuples): new keys go to out from base + *cursor on.  END,
// produced_to, counts and the result as in block_final_flush; *outside flags a
// key outside the id bound.
template <int B, bool SEG, int END>
__device__ __forceinline__ bool join_insert_blocks(
    const IdxSlot *slots, u64 n_slots, const u64 *inner, u64 n_inner, int shift, const u64 *outer,
    u64 n_outer, int arity, int s0, int s1, int pop, int plhs, int prhs, HsSel sel, u64 *out,
    u64 out_cap, unsigned long long *cursor, u64 out_base, unsigned long long *produced_to,
    unsigned long long *outside, EndCounts *counts) {
    __shared__ u64 s_excl[B], s_b[B], s_ok[B];
    __shared__ u64 s_stage[B / 64][kStage];
    __shared__ gdl_hs_seg s_segs[SEG ? kMaxSegs : 1];
    load_segs<SEG>(sel, s_segs);
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const u64 lt = lane_mask_lt();
    const u64 *wx = s_excl + w * 64;
    u64 *stage = s_stage[w];
    u32 staged = 0;  // wave-uniform
    u64 produced = 0;
    for (u64 base = (u64)blockIdx.x * B; base < n_outer; base += (u64)gridDim.x * B) {
        const u64 i = base + threadIdx.x;
        u64 b = 0, c = 0, ok = 0;
        if (i < n_outer) {
            ok = outer[i];
            if (!lookup_run(slots, n_slots, inner, n_inner, shift, ok >> shift, &b, &c)) c = 0;
        }
        const u64 incl = wave_inclusive_scan(c);
        const u64 total = __shfl(incl, 63, 64);
        s_excl[threadIdx.x] = incl - c;
        s_b[threadIdx.x] = b;
        s_ok[threadIdx.x] = ok;
        wave_sync_lds();
        // (two rounds together, to overlap their chains, were slower: 23.8
        // against 18.0 us for a body of the 200k-node tree)
        for (u64 q = 0; q < total; q += 64) {
            const u64 t = q + lane;
            u64 key = 0;
            u32 live = 0;
            if (t < total) {
                // the last lane whose run starts at or before t owns position t
                int lo = 0, hi = 63;
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (wx[mid] <= t) lo = mid;
                    else hi = mid - 1;
                }
                const u64 j = t - wx[lo];
                key = apply_map(inner[s_b[w * 64 + lo] + j], s_ok[w * 64 + lo], arity, s0, s1);
                live = eval_pred(key, pop, plhs, prhs);
            }
            produced += live;
            const bool fresh = insert_keys<1, SEG>(sel, s_segs, &key, live, outside);
            const u64 bal = __ballot(fresh);
            const u32 cnt = (u32)__popcll(bal);
            if (staged + cnt > kStage) {
                wave_sync_lds();
                flush_stage<END>(stage, staged, out, out_cap, cursor, out_base, lane);
                staged = 0;
                wave_sync_lds();
            }
            if (fresh) stage[staged + __popcll(bal & lt)] = key;
            staged += cnt;
        }
        wave_sync_lds();  // s_excl / s_b / s_ok are rewritten next round
    }
    return block_final_flush<B, END>(s_stage, staged, produced, out, out_cap, cursor, out_base,
                                     produced_to, counts);
}

template <int B, bool SEG>
__global__ __launch_bounds__(B) void k_join_insert(
    const IdxSlot *slots, u64 n_slots, const u64 *inner, u64 n_inner, int shift, const u64 *outer,
    u64 n_outer, int arity, int s0, int s1, int pop, int plhs, int prhs, HsSel sel, u64 *out,
    u64 out_cap, u64 out_base, CtxWords *words, u64 *result) {
    EndCounts c;
    if (join_insert_blocks<B, SEG, END_WORDS>(slots, n_slots, inner, n_inner, shift, outer,
                                              n_outer, arity, s0, s1, pop, plhs, prhs, sel, out,
                                              out_cap, &words->cursor, out_base, words->produced,
                                              &words->outside, &c))
        publish_join<B>(words, c.fresh, result);
}

// State of a stream-ordered linear fixpoint (gdl_fixpoint_linear) in device
// memory.
struct LinState {
    unsigned long long cursor;    // the running body's counts (EndMode)
    u64 delta_begin, delta_end;   // the body's delta: log[delta_begin, delta_end)
    u64 size;                     // hash set members
    u64 hs_limit;                 // members the set may reach (a fraction of its capacity)
    u64 log_cap;                  // log capacity, keys
    u64 max_run;                  // longest inner run: new tuples <= |delta| x max_run
    u64 delta_limit;              // a larger delta ends the chunk (the grid was sized smaller)
    u32 stop;                     // 0 run, 1 fixpoint, 2 grow first, 3 body limit, 4 overflow
    u32 body;                     // bodies finished in this call
    u32 max_bodies;
    u32 pad_;
};
enum : u32 { kLinRun = 0, kLinFixpoint = 1, kLinGrow = 2, kLinLimit = 3, kLinOverflow = 4 };

// End of a body (thread 0 of the last block to finish): record its counts,
// move the delta window to the nd tuples it appended from d1 on, and decide
// whether the next enqueued body runs.  The plain stores reach the next body
// at its launch.
__device__ void linear_epilogue(LinState *st, u64 *counts, u64 d1, u64 nd, u64 produced) {
    const u64 end = d1 + nd;
    const u32 b = st->body;
    counts[2 * b] = nd;
    counts[2 * b + 1] = produced;
    const u64 size = st->size + nd;
    st->size = size;
    st->delta_begin = d1;
    st->delta_end = end;
    st->cursor = 0;
    st->body = b + 1;
    u32 stop = kLinRun;
    if (end > st->log_cap) stop = kLinOverflow;
    else if (nd == 0) stop = kLinFixpoint;
    else if (b + 1 >= st->max_bodies || nd > st->delta_limit) stop = kLinLimit;
    else if (size + nd * st->max_run > st->hs_limit || end + nd * st->max_run > st->log_cap)
        stop = kLinGrow;
    st->stop = stop;
}

// One body of out := out U map(inner x delta) with FULL = hash set + append
// log: the delta is the log's last segment, new tuples are appended after it.
// A stop code set by an earlier body makes it return at once.  produced: a
// word per block (END_WORDS).
template <int B, int END>
__global__ __launch_bounds__(B) void k_linear_body(const IdxSlot *slots, u64 n_slots,
                                                   const u64 *inner, u64 n_inner, int shift,
                                                   int arity, int s0, int s1, int pop, int plhs,
                                                   int prhs, u64 *hs_slots, u64 hs_mask, u64 *log,
                                                   LinState *st, unsigned long long *produced,
                                                   u64 *counts) {
    if (st->stop != kLinRun) return;  // the same for every block
    const u64 d0 = st->delta_begin, d1 = st->delta_end;
    EndCounts c;
    if (!join_insert_blocks<B, false, END>(
            slots, n_slots, inner, n_inner, shift, log + d0, d1 - d0, arity, s0, s1, pop, plhs,
            prhs, HsSel{hs_slots, hs_mask, nullptr, 0, 0, 0}, log, st->log_cap, &st->cursor, d1,
            produced, nullptr, &c))
        return;
    // the last block: every other one's counts are at the coherence point
    if constexpr (END == END_WORDS) c.produced = sum_produced<B>(produced);
    if (threadIdx.x == 0) linear_epilogue(st, counts, d1, c.fresh, c.produced);
}

// Load-balanced variant for inner relations with long runs: outputs are
// numbered by the exclusive scan of run lengths (offsets), a block takes `per`
// consecutive tiles of JM_TILE outputs (JoinTile), each thread JM_I of a
// tile's, and the home-slot CASes of all of them go out back to back before
// collisions are resolved.  (With a binary search over the offsets per thread
// and a walk along them, CSPA's 22 joins at 500 ids took 96 us on average;
// 32 now.)
template <bool SEG>
__global__ __launch_bounds__(JB) void k_join_insert_lb(
    const u64 *inner, const u64 *outer, u64 n_outer, const u64 *offsets, const u64 *begins,
    u64 total, u32 per, int arity, int s0, int s1, int pop, int plhs, int prhs, HsSel sel,
    u64 *out, u64 out_cap, u64 out_base, CtxWords *words, u64 *result) {
    __shared__ JoinTile<JM_I> jt;
    __shared__ u64 s_stage[JB / 64][kStage];
    __shared__ gdl_hs_seg s_segs[SEG ? kMaxSegs : 1];
    load_segs<SEG>(sel, s_segs);
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const u64 lt = lane_mask_lt();
    u64 *stage = s_stage[w];
    u32 staged = 0;
    u64 produced = 0;
    u64 tile0 = (u64)blockIdx.x * per * JM_TILE;
    join_tile_seek(jt, offsets, n_outer, tile0);
    for (u32 k = 0; k < per && tile0 < total; ++k, tile0 += JM_TILE) {
        const u64 tile1 = tile0 + JM_TILE < total ? tile0 + JM_TILE : total;
        join_tile_owners(jt, outer, n_outer, offsets, begins, tile0, tile1);
        u64 keys[JM_I];
        u32 live = 0;  // bit r: output r exists and passes the predicate
#pragma unroll
        for (int r = 0; r < JM_I; ++r) {
            const u32 x = r * JB + threadIdx.x;
            keys[r] = 0;
            if (tile0 + x < tile1) {
                const u32 at = join_tile_owner(jt, x);
                keys[r] = apply_map(inner[jt.src[at] + (tile0 + x)], jt.key[at], arity, s0, s1);
                if (eval_pred(keys[r], pop, plhs, prhs)) live |= 1u << r;
            }
        }
        __syncthreads();  // the next tile overwrites the owners
        produced += __popc(live);
        const u32 fresh = insert_keys<JM_I, SEG>(sel, s_segs, keys, live, &words->outside);
#pragma unroll
        for (int r = 0; r < JM_I; ++r) {
            const bool f = (fresh >> r) & 1u;
            const u64 bal = __ballot(f);
            const u32 cnt = (u32)__popcll(bal);
            if (staged + cnt > kStage) {
                wave_sync_lds();
                flush_stage<END_WORDS>(stage, staged, out, out_cap, &words->cursor, out_base, lane);
                staged = 0;
                wave_sync_lds();
            }
            if (f) stage[staged + __popcll(bal & lt)] = keys[r];
            staged += cnt;
        }
    }
    EndCounts c;
    if (block_final_flush<JB, END_WORDS>(s_stage, staged, produced, out, out_cap, &words->cursor,
                                         out_base, words->produced, &c))
        publish_join<JB>(words, c.fresh, result);
}

__global__ __launch_bounds__(JB) void k_project(const u64 *in, u64 n, int arity, int s0, int s1,
                                                u64 *out) {
    for (u64 i = (u64)blockIdx.x * JB + threadIdx.x; i < n; i += (u64)gridDim.x * JB) {
        const u64 k = in[i];
        out[i] = apply_map(k, k, arity, s0, s1);
    }
}

static unsigned stride_grid(gdl_ctx *ctx, u64 n) {
    const u64 cap = grid_cap(ctx);
    u64 g = (n + JB - 1) / JB;
    if (g > cap) g = cap;
    return (unsigned)(g ? g : 1);
}

// Consecutive tiles a block takes: one until every CU has its four blocks
// (LDS allows no more), then up to eight, which spread the search for a
// block's first owner over them.
static u32 tiles_per_block(const gdl_ctx *ctx, u64 tiles) {
    const u64 cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    return (u32)std::max<u64>(1, std::min<u64>(8, tiles / (cus * 4)));
}

static bool valid_map(const gdl_colmap &m, bool join) {
    if (m.arity < 1 || m.arity > 2) return false;
    const int maxsrc = join ? 3 : 1;
    for (int c = 0; c < m.arity; ++c)
        if (m.src[c] < 0 || m.src[c] > maxsrc) return false;
    return true;
}

gdl_status index_build(gdl_ctx *ctx, const u64 *keys, u64 n, int prefix_cols, gdl_index *out) {
    out->slots = nullptr;
    out->n_slots = 0;
    out->n_distinct = 0;
    out->prefix_cols = prefix_cols;
    out->max_run = 0;
    out->dense = 0;
    if (n == 0) return GDL_OK;
    const int shift = prefix_cols >= 2 ? 0 : 32;
    u64 distinct = 0, max_run = 0, max_prefix = 0;
    {
        KTimer kt(ctx, K_IDX_COUNT, 8.0 * n);
        const u64 cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
        if (n >= kLongSpan)
            hipLaunchKernelGGL(k_idx_count<16>, dim3(std::min<u64>(grid_for(n, IC_B * 16), cus)),
                               dim3(IC_B), 0, ctx->stream, keys, n, shift, ctx->words,
                               result_words(ctx));
        else
            hipLaunchKernelGGL(k_idx_count<4>, dim3(std::min<u64>(grid_for(n, IC_B * 4), cus)),
                               dim3(IC_B), 0, ctx->stream, keys, n, shift, ctx->words,
                               result_words(ctx));
        GDL_TRY(check_launch(ctx, "k_idx_count"));
        u64 h[3];
        GDL_TRY(read_result(ctx, h, 3));
        distinct = h[0];
        max_run = h[1];
        max_prefix = h[2];
    }
    out->n_distinct = distinct;
    out->max_run = max_run;
    // one column of ids that are dense enough: a direct-mapped array of run
    // words no larger than the hash index (or at most 1 MB)
    const u64 hash_slots = (u64)((double)distinct / (double)ctx->cfg.load_factor) + 1;
    if (prefix_cols == 1 && max_prefix < std::max<u64>(2 * hash_slots, 1ull << 17)) {
        const u64 range = max_prefix + 1;
        void *p = nullptr;
        std::string err;
        gdl_status st = ctx->alloc->alloc(range * sizeof(u64), &p, &err);
        if (st != GDL_OK) return fail(ctx, st, err);
        GDL_HIP(ctx, hipMemsetAsync(p, 0, range * sizeof(u64), ctx->stream));
        KTimer kt(ctx, K_IDX_BUILD, 8.0 * n + 8.0 * (double)distinct);
        if (n >= kLongSpan)
            hipLaunchKernelGGL(k_idx_build_dense<16>, dim3(stride_grid(ctx, n / 16)), dim3(JB), 0,
                               ctx->stream, keys, n, shift, (u64 *)p, range);
        else
            hipLaunchKernelGGL(k_idx_build_dense<4>, dim3(stride_grid(ctx, n / 4)), dim3(JB), 0,
                               ctx->stream, keys, n, shift, (u64 *)p, range);
        GDL_TRY(check_launch(ctx, "k_idx_build_dense"));
        out->slots = p;
        out->n_slots = range;
        out->dense = 1;
        return GDL_OK;
    }
    u64 n_slots = (u64)((double)distinct / (double)ctx->cfg.load_factor) + 1;
    if (n_slots <= distinct) n_slots = distinct + 1;
    n_slots = (n_slots + kBucket - 1) / kBucket * kBucket;  // whole buckets
    void *p = nullptr;
    std::string err;
    gdl_status st = ctx->alloc->alloc(n_slots * sizeof(IdxSlot), &p, &err);
    if (st != GDL_OK) return fail(ctx, st, err);
    GDL_HIP(ctx, hipMemsetAsync(p, 0, n_slots * sizeof(IdxSlot), ctx->stream));
    {
        KTimer kt(ctx, K_IDX_BUILD, 8.0 * n + 16.0 * (double)distinct);
        if (n >= kLongSpan)
            hipLaunchKernelGGL(k_idx_build<4>, dim3(stride_grid(ctx, n / 4)), dim3(JB), 0,
                               ctx->stream, keys, n, shift, (IdxSlot *)p, n_slots, ctx->d_err);
        else
            hipLaunchKernelGGL(k_idx_build<1>, dim3(stride_grid(ctx, n)), dim3(JB), 0,
                               ctx->stream, keys, n, shift, (IdxSlot *)p, n_slots, ctx->d_err);
        GDL_TRY(check_launch(ctx, "k_idx_build"));
    }
    out->slots = p;
    out->n_slots = n_slots;
    out->n_distinct = distinct;
    out->max_run = max_run;
    return GDL_OK;
}

gdl_status join_count(gdl_ctx *ctx, const u64 *inner, u64 n_inner, const gdl_index *idx,
                      const u64 *outer, u64 n_outer, u32 *counts, u64 *begins) {
    if (n_outer == 0) return GDL_OK;
    const int shift = idx->prefix_cols >= 2 ? 0 : 32;
    if (n_inner == 0 || idx->n_slots == 0) {
        GDL_HIP(ctx, hipMemsetAsync(counts, 0, n_outer * sizeof(u32), ctx->stream));
        GDL_HIP(ctx, hipMemsetAsync(begins, 0, n_outer * sizeof(u64), ctx->stream));
        return GDL_OK;
    }
    KTimer kt(ctx, K_JOIN_COUNT, 8.0 * n_outer + 16.0 * n_outer + 12.0 * n_outer);
    hipLaunchKernelGGL(k_join_count, dim3(stride_grid(ctx, n_outer)), dim3(JB), 0, ctx->stream,
                       (const IdxSlot *)idx->slots, idx_arg(idx), inner, n_inner, shift, outer,
                       n_outer, counts, begins);
    return check_launch(ctx, "k_join_count");
}

gdl_status join_offsets(gdl_ctx *ctx, const u64 *inner, u64 n_inner, const gdl_index *idx,
                        const u64 *outer, u64 n_outer, u64 *begins, u64 *offsets, u64 *total) {
    if (n_outer == 0 || n_inner == 0 || idx->n_slots == 0 || n_outer > kScanOnePass) {
        Scratch scr(ctx);
        u32 *counts;
        GDL_TRY(scr.get(n_outer, &counts));
        GDL_TRY(join_count(ctx, inner, n_inner, idx, outer, n_outer, counts, begins));
        return exclusive_scan_u32_to_u64(ctx, counts, n_outer, offsets, total);
    }
    // tiles of 8192 outer tuples from 2^18 on (fewer tickets), of 2048 below
    const int shift = idx->prefix_cols >= 2 ? 0 : 32;
    const bool big = n_outer >= 1ull << 18;
    const u64 tile = (big ? 1024 : JB) * 8, nt = (n_outer + tile - 1) / tile;
    Scratch scr(ctx);
    TileLook look;
    GDL_TRY(tile_look(ctx, nt, &scr, &look));
    {
        KTimer kt(ctx, K_JOIN_COUNT, 8.0 * n_outer + 16.0 * n_outer + 16.0 * n_outer);
        auto launch = [&](auto kern, int block) {
            hipLaunchKernelGGL(kern, dim3((unsigned)nt), dim3(block), 0, ctx->stream,
                               (const IdxSlot *)idx->slots, idx_arg(idx), inner, n_inner, shift,
                               outer, n_outer, look, begins, offsets, result_words(ctx));
        };
        if (big) launch(k_join_offsets<1024>, 1024);
        else launch(k_join_offsets<JB>, JB);
        GDL_TRY(check_launch(ctx, "k_join_offsets"));
    }
    return read_result(ctx, total);
}

gdl_status join_materialize(gdl_ctx *ctx, const u64 *inner, const u64 *outer, u64 n_outer,
                            const u64 *offsets, const u64 *begins, u64 total, gdl_colmap map,
                            u64 *out) {
    if (total == 0) return GDL_OK;
    if ((total + JM_TILE - 1) / JM_TILE > 0x7fffffffull)
        return fail(ctx, GDL_ERR_OVERFLOW, "join: output too large");
    KTimer kt(ctx, K_JOIN_MAT, 16.0 * total);
    // Fewer outputs than outer tuples: owners by search, one tile a block, in
    // as few outputs a thread as leave the chip full (a search is a chain of
    // ~21 loads).  2M outer tuples, us by walk | I = 1 | 2 | 8, and before the
    // walk (a search for every 8 outputs, then one tuple after the other):
    //   16,000 outputs in runs of 8   532 |  8 |  8 | 10, before 10
    //   20,000 in runs of 1           641 |  8 | 12 | 52, before 882
    //   320,000 in runs of 8           56 | 12 | 12 | 12, before 12
    //   800,000 in runs of 8           38 | 28 | 16 | 16, before 17
    //   1.6M in runs of 8              28 | 51 | 31 | 21, before 26
    // and where the rule changes over, by walk | I = 2 | 4 | 8:
    //   2M in runs of 1                32 | 37 | 45 | 65, before 80
    //   2M in runs of 40               26 | 24 | 17 | 18, before 20
    // I = 2 also for a few outputs of many tuples: 4M of 20M in runs of 1
    // 245 us, I = 4 448, before 370; in runs of 40 49, 34, 34.
    const bool sparse = total < n_outer;
    auto launch = [&](auto kern, u64 tile) {
        const u64 nt = (total + tile - 1) / tile;
        const u32 per = sparse ? 1 : tiles_per_block(ctx, nt);
        hipLaunchKernelGGL(kern, dim3(grid_for(nt, per)), dim3(JB), 0, ctx->stream, inner, outer,
                           n_outer, offsets, begins, total, per, map.arity, map.src[0],
                           map.arity == 2 ? map.src[1] : 0, out);
    };
    if (!sparse) launch(k_join_materialize<JM_I, false>, JM_TILE);
    else if (total <= 1ull << 18) launch(k_join_materialize<1, true>, JB);
    else if (total <= 1ull << 20 || total < n_outer / 4) launch(k_join_materialize<2, true>, 2 * JB);
    else launch(k_join_materialize<4, true>, 4 * JB);
    return check_launch(ctx, "k_join_materialize");
}

}  // namespace gdl

using namespace gdl;

extern "C" {

gdl_status gdl_index_build(gdl_ctx *ctx, const uint64_t *d_sorted, uint64_t n, int prefix_cols,
                           gdl_index *out) {
    if (!ctx || !out || (n && !d_sorted) || prefix_cols < 1 || prefix_cols > 2)
        return GDL_ERR_INVALID_ARG;
    return index_build(ctx, d_sorted, n, prefix_cols, out);
}

gdl_status gdl_index_free(gdl_ctx *ctx, gdl_index *idx) {
    if (!ctx || !idx) return GDL_ERR_INVALID_ARG;
    if (idx->slots) {
        std::string err;
        gdl_status st = ctx->alloc->free(idx->slots, &err);
        if (st != GDL_OK) return fail(ctx, st, err);
    }
    idx->slots = nullptr;
    idx->n_slots = 0;
    idx->n_distinct = 0;
    idx->dense = 0;
    return GDL_OK;
}

gdl_status gdl_index_lookup(gdl_ctx *ctx, const gdl_index *idx, const uint64_t *d_sorted,
                            uint64_t n_sorted, const uint64_t *d_prefixes, uint64_t n,
                            uint64_t *d_begin, uint32_t *d_count) {
    if (!ctx || !idx || (n && (!d_prefixes || !d_begin || !d_count))) return GDL_ERR_INVALID_ARG;
    if (n == 0) return GDL_OK;
    if (idx->n_slots == 0) {
        GDL_HIP(ctx, hipMemsetAsync(d_count, 0, n * sizeof(u32), ctx->stream));
        GDL_HIP(ctx, hipMemsetAsync(d_begin, 0, n * sizeof(u64), ctx->stream));
        return GDL_OK;
    }
    const int shift = idx->prefix_cols >= 2 ? 0 : 32;
    KTimer kt(ctx, K_IDX_LOOKUP, 28.0 * n);
    hipLaunchKernelGGL(k_idx_lookup, dim3(stride_grid(ctx, n)), dim3(JB), 0, ctx->stream,
                       (const IdxSlot *)idx->slots, idx_arg(idx), d_sorted, n_sorted, shift,
                       d_prefixes, n, d_begin, d_count);
    return check_launch(ctx, "k_idx_lookup");
}

gdl_status gdl_join_count(gdl_ctx *ctx, const uint64_t *d_inner, uint64_t n_inner,
                          const gdl_index *inner_idx, const uint64_t *d_outer, uint64_t n_outer,
                          uint32_t *d_counts, uint64_t *d_begins) {
    if (!ctx || !inner_idx || (n_outer && (!d_outer || !d_counts || !d_begins)) ||
        (n_inner && !d_inner))
        return GDL_ERR_INVALID_ARG;
    return join_count(ctx, d_inner, n_inner, inner_idx, d_outer, n_outer, d_counts, d_begins);
}

gdl_status gdl_join_materialize(gdl_ctx *ctx, const uint64_t *d_inner, const uint64_t *d_outer,
                                uint64_t n_outer, const uint64_t *d_offsets,
                                const uint64_t *d_begins, uint64_t total, gdl_colmap map,
                                uint64_t *d_out) {
    if (!ctx || (total && (!d_inner || !d_outer || !d_offsets || !d_begins || !d_out)))
        return GDL_ERR_INVALID_ARG;
    if (!valid_map(map, true)) return fail(ctx, GDL_ERR_INVALID_ARG, "bad join column map");
    return join_materialize(ctx, d_inner, d_outer, n_outer, d_offsets, d_begins, total, map, d_out);
}

gdl_status gdl_join(gdl_ctx *ctx, const uint64_t *d_inner, uint64_t n_inner,
                    const gdl_index *inner_idx, const uint64_t *d_outer, uint64_t n_outer,
                    gdl_colmap map, gdl_pred pred, uint64_t **d_out, uint64_t *n_out) {
    if (!ctx || !inner_idx || !d_out || !n_out || (n_outer && !d_outer) || (n_inner && !d_inner))
        return GDL_ERR_INVALID_ARG;
    if (!valid_map(map, true)) return fail(ctx, GDL_ERR_INVALID_ARG, "bad join column map");
    if (!valid_pred(pred, map.arity))
        return fail(ctx, GDL_ERR_INVALID_ARG, "bad join predicate");
    *d_out = nullptr;
    *n_out = 0;
    if (n_outer == 0 || n_inner == 0) return GDL_OK;
    Scratch scr(ctx);
    u64 *begins, *offsets;
    GDL_TRY(scr.get(n_outer, &begins));
    GDL_TRY(scr.get(n_outer + 1, &offsets));
    u64 total = 0;
    GDL_TRY(join_offsets(ctx, d_inner, n_inner, inner_idx, d_outer, n_outer, begins, offsets,
                         &total));
    if (total == 0) return GDL_OK;
    void *buf = nullptr;
    std::string err;
    gdl_status st = ctx->alloc->alloc(total * sizeof(u64), &buf, &err);
    if (st != GDL_OK) return fail(ctx, st, err);
    u64 *res = (u64 *)buf;
    st = join_materialize(ctx, d_inner, d_outer, n_outer, offsets, begins, total, map, res);
    if (st != GDL_OK) {
        ctx->alloc->free(buf, nullptr);
        return st;
    }
    if (pred.op != GDL_PRED_NONE) {
        void *fbuf = nullptr;
        st = ctx->alloc->alloc(total * sizeof(u64), &fbuf, &err);
        if (st != GDL_OK) {
            ctx->alloc->free(buf, nullptr);
            return fail(ctx, st, err);
        }
        u64 kept = 0;
        st = filter_keys(ctx, res, total, pred, (u64 *)fbuf, &kept);
        ctx->alloc->free(buf, nullptr);
        if (st != GDL_OK) {
            ctx->alloc->free(fbuf, nullptr);
            return st;
        }
        *d_out = (u64 *)fbuf;
        *n_out = kept;
        return GDL_OK;
    }
    *d_out = res;
    *n_out = total;
    return GDL_OK;
}

}  // extern "C"

// Fused join + insert.  SEG = false: into one set `hs`, growing it and the
// output (*d_new, *new_cap) to the bound.  SEG = true: into the per-instance
// sets of `sel`, which the caller has sized, and into the caller's output of
// *new_cap keys (a fixed buffer; an overrun is reported, never written).
template <bool SEG>
static gdl_status join_insert_impl(gdl_ctx *ctx, const u64 *d_inner, u64 n_inner,
                                   const gdl_index *inner_idx, const u64 *d_outer, u64 n_outer,
                                   gdl_colmap map, gdl_pred pred, gdl_hashset *hs, HsSel sel,
                                   u64 **d_new, u64 *new_cap, u64 *n_new, u64 *n_raw) {
    *n_raw = 0;
    if (n_outer == 0 || n_inner == 0 || inner_idx->n_slots == 0) return GDL_OK;
    const int shift = inner_idx->prefix_cols >= 2 ? 0 : 32;
    // upper bound of produced tuples: |outer| x longest inner run, or an
    // exact count when that bound is loose
    const u64 mr = inner_idx->max_run ? inner_idx->max_run : n_inner;
    u64 bound = (n_outer > ~0ull / mr) ? ~0ull : n_outer * mr;
    const u64 loose_limit = std::max<u64>(1ull << 24, 4 * n_outer);
    const u64 cap_blocks = std::min<u64>(grid_cap(ctx), kMaxEndBlocks);
    const int fb = (int)ctx->tune.join_block;  // block of the flattened kernel
    // the count sizes the output set and buffer; with per-instance sets (SEG)
    // the caller has sized both already (the output capacity is checked after
    // the kernel), so only the load-balanced kernel below counts, for its
    // offsets
    // (and a join that would run on bit matrices if its bound were its count)
    bool counted = !SEG && bound > loose_limit;
    if constexpr (!SEG)
        counted = counted || dense_join_pays(ctx, hs, map, pred, inner_idx->prefix_cols, n_inner,
                                             n_outer, bound);
    Scratch lb(ctx);
    u64 *begins = nullptr, *offsets = nullptr;
    if (counted) {
        GDL_TRY(lb.get(n_outer, &begins));
        GDL_TRY(lb.get(n_outer + 1, &offsets));
        GDL_TRY(join_offsets(ctx, d_inner, n_inner, inner_idx, d_outer, n_outer, begins, offsets,
                             &bound));
    }
    if (bound == 0) return GDL_OK;
    if constexpr (!SEG) {
        // many tuples per new one over a small id domain: bit matrices
        gdl_status ds = GDL_OK;
        if (counted && dense_join_insert(ctx, d_inner, n_inner, d_outer, n_outer, map, pred,
                                         inner_idx->prefix_cols, hs, bound, d_new, new_cap,
                                         n_new, n_raw, &ds))
            return ds;
    }
    // The wave-flattened kernel is balanced inside a wave but not across
    // waves: a wave whose 64 outer tuples hit a hub walks the whole hub run,
    // one step (64 outputs) per hub tuple.  Number the outputs and spread
    // them over the grid instead when that is long against the expected
    // steps per wave.
    const u64 waves = std::min<u64>((n_outer + fb - 1) / fb, cap_blocks) * (fb / 64);
    const u64 avg_run = std::max<u64>(1, n_inner / std::max<u64>(1, inner_idx->n_distinct));
    const u64 est_total = counted ? bound : n_outer * avg_run;
    // (or when there are too few waves for the work: each would walk many
    // 64-output steps, each a chain of dependent loads)
    const bool balanced =
        mr > kHubRun && (mr * 16 > est_total / waves || est_total / (waves * 64) > 32);
    if (ctx->cfg.verbose)
        fprintf(stderr,
                "gdl: join_insert outer %llu inner %llu max_run %llu produced %s%llu set %s%d -> %s\n",
                (unsigned long long)n_outer, (unsigned long long)n_inner, (unsigned long long)mr,
                counted ? "" : "<= ", (unsigned long long)bound,
                hs && hs->key_bits ? "bitmap " : "hash ", hs ? (int)hs->key_bits : 0,
                balanced ? "balanced" : "wave-flattened");
    if (balanced && !counted) {
        GDL_TRY(lb.get(n_outer, &begins));
        GDL_TRY(lb.get(n_outer + 1, &offsets));
        GDL_TRY(join_offsets(ctx, d_inner, n_inner, inner_idx, d_outer, n_outer, begins, offsets,
                             &bound));
        if (bound == 0) return GDL_OK;
    }
    if constexpr (!SEG) {
        // new members are distinct keys of the id domain the set does not
        // hold yet: at most the domain's free keys, however many tuples the
        // join produces
        u64 room = ~0ull;
        if (hs->key_bits) {
            room = hs->capacity - std::min(hs->capacity, hs->size);
        } else if (ctx->id_bits > 0 && ctx->id_bits < 32) {
            const u64 dom = 1ull << (2 * ctx->id_bits);
            room = dom - std::min(dom, hs->size);
            sel.dom_bits = ctx->id_bits;  // the kernel checks every key against it
        }
        const u64 new_bound = std::min(bound, room);
        // size for up to 2 |outer| new members at the load factor; the bound
        // only has to fit
        GDL_TRY(hashset_reserve2(ctx, hs, std::max<u64>(2 * n_outer, 1024), new_bound));
        sel.slots = (u64 *)hs->slots;
        sel.mask = hs_arg(hs);
        if (*n_new + new_bound > *new_cap || !*d_new) {
            const u64 cap = *n_new + new_bound + (*n_new + new_bound) / 4 + 1024;
            void *p = nullptr;
            std::string err;
            gdl_status st = ctx->alloc->alloc(cap * sizeof(u64), &p, &err);
            if (st != GDL_OK) return fail(ctx, st, err);
            if (*n_new)
                GDL_HIP(ctx, hipMemcpyAsync(p, *d_new, *n_new * sizeof(u64),
                                            hipMemcpyDeviceToDevice, ctx->stream));
            if (*d_new) ctx->alloc->free(*d_new, nullptr);
            *d_new = (u64 *)p;
            *new_cap = cap;
        }
    }
    if (balanced) {
        KTimer kt(ctx, K_JOIN_INSERT, 24.0 * n_outer);
        const u64 nt = (bound + JM_TILE - 1) / JM_TILE;
        const u32 per = (u32)((nt + cap_blocks - 1) / cap_blocks);
        hipLaunchKernelGGL(k_join_insert_lb<SEG>, dim3(grid_for(nt, per)), dim3(JB), 0,
                           ctx->stream, d_inner, d_outer, n_outer, offsets, begins, bound, per,
                           map.arity, map.src[0],
                           map.arity == 2 ? map.src[1] : 0, pred.op, pred.lhs, pred.rhs, sel,
                           *d_new, *new_cap, (u64)*n_new, ctx->words, result_words(ctx));
        GDL_TRY(check_launch(ctx, "k_join_insert_lb"));
    } else {
        KTimer kt(ctx, K_JOIN_INSERT, 8.0 * n_outer + 64.0 * n_outer);
        const unsigned g = (unsigned)std::max<u64>(1, std::min<u64>((n_outer + fb - 1) / fb,
                                                                    cap_blocks));
        auto launch = [&](auto kern, int block) {
            hipLaunchKernelGGL(kern, dim3(g), dim3(block), 0, ctx->stream,
                               (const IdxSlot *)inner_idx->slots, idx_arg(inner_idx), d_inner,
                               n_inner, shift, d_outer, n_outer, map.arity, map.src[0],
                               map.arity == 2 ? map.src[1] : 0, pred.op, pred.lhs, pred.rhs, sel,
                               *d_new, *new_cap, (u64)*n_new, ctx->words, result_words(ctx));
        };
        switch (fb) {
            case 64: launch(k_join_insert<64, SEG>, 64); break;
            case 128: launch(k_join_insert<128, SEG>, 128); break;
            case 512: launch(k_join_insert<512, SEG>, 512); break;
            default: launch(k_join_insert<256, SEG>, 256); break;
        }
        GDL_TRY(check_launch(ctx, "k_join_insert"));
    }
    u64 h[3];
    GDL_TRY(read_result(ctx, h, 3));
    h[0] += *n_new;  // the output's end
    if (h[2])
        return fail(ctx, GDL_ERR_OVERFLOW,
                    "fused join: a produced key has an id at or above 2^" +
                        std::to_string(sel.dom_bits) + ", the context's id bound (gdl_set_id_bits)");
    if (h[0] > *new_cap)
        return fail(ctx, GDL_ERR_OVERFLOW, "fused join: new tuples exceed the output capacity (" +
                                               std::to_string(h[0]) + " > " +
                                               std::to_string(*new_cap) + ")");
    const u64 added = h[0] - *n_new;
    // inner run reads + hash probes per produced tuple, new keys written
    ctx->stats[K_JOIN_INSERT].alg_bytes += 16.0 * h[1] + 8.0 * added;
    if constexpr (!SEG) hs->size += added;
    *n_new = h[0];
    *n_raw = h[1];
    return GDL_OK;
}

extern "C" {

gdl_status gdl_join_insert(gdl_ctx *ctx, const uint64_t *d_inner, uint64_t n_inner,
                           const gdl_index *inner_idx, const uint64_t *d_outer, uint64_t n_outer,
                           gdl_colmap map, gdl_pred pred, gdl_hashset *hs, uint64_t **d_new,
                           uint64_t *new_cap, uint64_t *n_new, uint64_t *n_raw) {
    if (!ctx || !inner_idx || !hs || !d_new || !new_cap || !n_new || !n_raw ||
        (n_outer && !d_outer) || (n_inner && !d_inner))
        return GDL_ERR_INVALID_ARG;
    if (!valid_map(map, true)) return fail(ctx, GDL_ERR_INVALID_ARG, "bad join column map");
    if (!valid_pred(pred, map.arity))
        return fail(ctx, GDL_ERR_INVALID_ARG, "bad join predicate");
    return join_insert_impl<false>(ctx, d_inner, n_inner, inner_idx, d_outer, n_outer, map, pred,
                                   hs, HsSel{nullptr, 0, nullptr, 0, 0}, d_new, new_cap, n_new,
                                   n_raw);
}

gdl_status gdl_join_insert_seg(gdl_ctx *ctx, const uint64_t *d_inner, uint64_t n_inner,
                               const gdl_index *inner_idx, const uint64_t *d_outer,
                               uint64_t n_outer, gdl_colmap map, gdl_pred pred,
                               const gdl_hs_seg *d_segs, uint32_t n_segs, int seg_shift,
                               uint64_t *d_out, uint64_t out_cap, uint64_t *n_out,
                               uint64_t *n_raw) {
    if (!ctx || !inner_idx || !d_segs || !n_out || !n_raw || (n_outer && !d_outer) ||
        (n_inner && !d_inner) || (out_cap && !d_out))
        return GDL_ERR_INVALID_ARG;
    if (n_segs == 0 || n_segs > kMaxSegs || seg_shift < 1 || seg_shift > 63)
        return fail(ctx, GDL_ERR_INVALID_ARG, "segmented join insert: 1..256 sets, shift 1..63");
    if (!valid_map(map, true)) return fail(ctx, GDL_ERR_INVALID_ARG, "bad join column map");
    if (!valid_pred(pred, map.arity))
        return fail(ctx, GDL_ERR_INVALID_ARG, "bad join predicate");
    *n_out = 0;
    u64 *out = d_out;
    u64 cap = out_cap;
    return join_insert_impl<true>(ctx, d_inner, n_inner, inner_idx, d_outer, n_outer, map, pred,
                                  nullptr, HsSel{nullptr, 0, d_segs, n_segs, seg_shift}, &out,
                                  &cap, n_out, n_raw);
}

gdl_status gdl_fixpoint_linear(gdl_ctx *ctx, const uint64_t *d_inner, uint64_t n_inner,
                               const gdl_index *inner_idx, gdl_colmap map, gdl_pred pred,
                               gdl_hashset *hs, uint64_t **d_log, uint64_t *log_cap,
                               uint64_t *delta_begin, uint64_t *delta_end, int max_bodies,
                               uint64_t *h_new, uint64_t *h_raw, int *bodies) {
    if (!ctx || !inner_idx || !hs || !d_log || !log_cap || !delta_begin || !delta_end ||
        !h_new || !h_raw || !bodies || (n_inner && !d_inner) || *delta_begin > *delta_end ||
        (*delta_end && !*d_log) || *delta_end > *log_cap)
        return GDL_ERR_INVALID_ARG;
    if (!valid_map(map, true)) return fail(ctx, GDL_ERR_INVALID_ARG, "bad join column map");
    if (!valid_pred(pred, map.arity))
        return fail(ctx, GDL_ERR_INVALID_ARG, "bad join predicate");
    *bodies = 0;
    if (max_bodies <= 0) return GDL_OK;
    if (n_inner == 0 || inner_idx->n_slots == 0 || *delta_end == *delta_begin) {
        h_new[0] = h_raw[0] = 0;  // one body, nothing produced: the fixpoint
        *delta_begin = *delta_end;
        *bodies = 1;
        return GDL_OK;
    }
    // at most 128 bodies per host wait (on the 200k-node tree 128 beat 32 by
    // 2.5 %; 64 did not; a chunk that stops early leaves no-op launches)
    constexpr int kChunk = 128;
    // a body is bound by its launch and the latency of each tuple's chain of
    // dependent accesses (~0.6 us a load): of the 21 us of a body of 190k outer
    // tuples the launch takes 4, the key 5, the insert 8 (what its atomics take
    // at their rate, 25e9 a second at random places whatever their scope; 4 of
    // the 17 us of the tree's average body), the end of its blocks 1.4.  So
    // every outer tuple gets its own lane (more chains in flight).  Blocks of 512
    // (each ends with an atomic on the shared cursor, 11 ns one after another,
    // but also waits for its slowest wave): 17.1 us a body on the 200k-node tree,
    // 18.0 with 256 and 18.4 with 1024; of 256 up to 2^16 outer tuples (50,000
    // nodes: 9.4 against 10.3 us)
    const int shift = inner_idx->prefix_cols >= 2 ? 0 : 32;
    const u64 mr = std::max<u64>(inner_idx->max_run, 1);
    Scratch scr(ctx);
    u64 *st_words, *counts;
    GDL_TRY(scr.get((sizeof(LinState) + 7) / 8, &st_words));
    GDL_TRY(scr.get(2 * kChunk, &counts));
    LinState *st = (LinState *)st_words;
    u64 d0 = *delta_begin, d1 = *delta_end;
    // TC's map over a bitmap FULL: bodies whose delta is dense run on bit
    // matrices (dense.hip); the delta size where they start
    const bool tc_map = map.arity == 2 && map.src[0] == GDL_COL_INNER1 &&
                        map.src[1] == GDL_COL_OUTER1 && pred.op == GDL_PRED_NONE &&
                        inner_idx->prefix_cols == 1;
    const gdl_dense_rule rule{GDL_DENSE_TC, d_inner, n_inner, nullptr, 0, 0, 0};
    u64 dense_at = tc_map ? dense_threshold_for(ctx, hs, GDL_DENSE_TC, n_inner, 0) : ~0ull;
    int done = 0, ramp = 4;
    while (done < max_bodies) {
        const u64 nd = d1 - d0;
        if (nd >= dense_at) {
            int nb = 0;
            u64 end = d1;
            GDL_TRY(dense_run(ctx, &rule, hs, *d_log + d0, nd, d_log, log_cap, &end,
                              max_bodies - done, h_new + done, h_raw + done, &nb));
            if (nb > 0) {
                done += nb;
                const u64 last = h_new[done - 1];
                d0 = end - last;
                d1 = end;
                if (last == 0) break;  // the fixpoint
                continue;
            }
            dense_at = ~0ull;  // declined (ids beyond the set's domain): tuple bodies only
        }
        const u64 worst = nd > (~0ull >> 20) / mr ? (~0ull >> 20) : nd * mr;
        // the set: the next chunk's bodies (about |delta| each) at the load
        // factor and the worst body at 0.9; when it has to grow, it grows to
        // room for 4x its size more (each growth is a rehash of every member,
        // so a set that keeps growing is rehashed every ~5x, not every 2x);
        // the log: the worst body after the delta, grown 2x at a time (each
        // growth copies it)
        const u64 next = std::max<u64>(nd, 1024) * (u64)std::min(ramp, kChunk);
        GDL_TRY(hashset_reserve2(ctx, hs, next, std::max(worst, next), 0.0,
                                 std::max<u64>(next, 4 * hs->size)));
        u64 need_log = d1 + std::max<u64>(worst, 4096);
        if (*log_cap < need_log) {
            need_log = std::max<u64>(need_log, 2 * *log_cap);  // geometric
            void *p = nullptr;
            std::string err;
            gdl_status s = ctx->alloc->alloc(need_log * sizeof(u64), &p, &err);
            if (s != GDL_OK) return fail(ctx, s, err);
            if (d1)
                GDL_HIP(ctx, hipMemcpyAsync(p, *d_log, d1 * sizeof(u64), hipMemcpyDeviceToDevice,
                                            ctx->stream));
            if (*d_log) ctx->alloc->free(*d_log, nullptr);
            *d_log = (u64 *)p;
            *log_cap = need_log;
        }
        // as many bodies of this delta's size as the log holds: a body that
        // finds it full stops the chunk, and the launches after it return at
        // once but still cost a launch each (50,000-node tree: 4.07 ms so,
        // 4.34 ms without).  The log is not grown for them: a run that fits
        // its memory needs no room beyond the next body's.
        const u64 fit = (*log_cap - d1 - worst) / nd + 1;
        const int k = (int)std::min<u64>(fit, (u64)std::min({ramp, kChunk, max_bodies - done}));
        LinState h{};
        h.cursor = 0;
        h.delta_begin = d0;
        h.delta_end = d1;
        h.size = hs->size;
        h.hs_limit = hs->key_bits ? ~0ull : (u64)(kHsHardLoad * (double)hs->capacity);
        h.log_cap = *log_cap;
        h.max_run = mr;
        h.max_bodies = (u32)k;
        // a grid for this delta (one outer tuple per thread); a body whose
        // delta outgrows it 8x ends the chunk, so the next chunk is launched
        // wider
        // the counts of a body packed in one word while they fit it: produced
        // tuples (and so new ones) below 2^27, at most 1023 blocks
        const u64 packed_limit = ((1ull << kPackedBits) - 1) / mr;
        const u64 LB = nd <= std::min<u64>(1u << 16, packed_limit) ? 256 : 512;
        const u64 want = (nd + LB - 1) / LB;
        const u64 most = std::min<u64>(grid_cap(ctx), kMaxEndBlocks);
        const unsigned g = (unsigned)std::min<u64>(most, std::max<u64>(want, 16));
        h.delta_limit = g >= most ? ~0ull : (u64)g * LB * 8;
        // a delta that turns dense ends the chunk too (bit-matrix bodies next)
        if (dense_at != ~0ull) h.delta_limit = std::min<u64>(h.delta_limit, dense_at - 1);
        const bool packed = g <= kPackedBlocks && nd <= packed_limit;
        if (packed) h.delta_limit = std::min<u64>(h.delta_limit, packed_limit);
        Staging stg(ctx);
        GDL_TRY(stg.up(st, &h, sizeof(h)));
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(g), dim3((unsigned)LB), 0, ctx->stream,
                               (const IdxSlot *)inner_idx->slots, idx_arg(inner_idx), d_inner,
                               n_inner, shift, map.arity, map.src[0],
                               map.arity == 2 ? map.src[1] : 0, pred.op, pred.lhs, pred.rhs,
                               (u64 *)hs->slots, hs_arg(hs), *d_log, st, ctx->words->produced,
                               counts);
        };
        for (int i = 0; i < k; ++i) {
            KTimer kt(ctx, K_LINEAR, 0.0);
            if (!packed) launch(k_linear_body<512, END_WORDS>);
            else if (LB == 512) launch(k_linear_body<512, END_PACKED>);
            else launch(k_linear_body<256, END_PACKED>);
            GDL_TRY(check_launch(ctx, "k_linear_body"));
        }
        LinState r{};
        u64 c[2 * kChunk];
        u32 dev_err = 0;
        GDL_TRY(stg.later(&r, st, sizeof(r)));
        GDL_TRY(stg.later(c, counts, sizeof(c)));
        GDL_TRY(stg.later(&dev_err, ctx->d_err, sizeof(u32)));
        GDL_TRY(stg.land());  // one wait for the state, the counts and the error word
        GDL_TRY(device_error_status(ctx, dev_err));
        if (r.stop == kLinOverflow)
            return fail(ctx, GDL_ERR_OVERFLOW, "linear fixpoint: a body outgrew its log bound");
        u64 outer_n = nd;
        for (u32 b = 0; b < r.body && done < max_bodies; ++b, ++done) {
            h_new[done] = c[2 * b];
            h_raw[done] = c[2 * b + 1];
            // probe + outer read per outer tuple, inner read + hash probe per
            // produced tuple, the new keys written
            ctx->stats[K_LINEAR].alg_bytes += 72.0 * outer_n + 16.0 * c[2 * b + 1] + 8.0 * c[2 * b];
            outer_n = c[2 * b];
        }
        hs->size = r.size;
        d0 = r.delta_begin;
        d1 = r.delta_end;
        if (r.stop == kLinFixpoint || r.body == 0) break;
        // chunks double while every enqueued body runs (a stopped chunk's
        // remaining launches return at once, but still cost a launch)
        ramp = (int)r.body == k ? std::min(2 * ramp, kChunk) : std::max(4, (int)r.body);
    }
    *bodies = done;
    *delta_begin = d0;
    *delta_end = d1;
    return GDL_OK;
}

gdl_status gdl_project_u64(gdl_ctx *ctx, const uint64_t *d_in, uint64_t n, gdl_colmap map,
                           uint64_t *d_out) {
    if (!ctx || (n && (!d_in || !d_out))) return GDL_ERR_INVALID_ARG;
    if (!valid_map(map, false)) return fail(ctx, GDL_ERR_INVALID_ARG, "bad copy column map");
    if (n == 0) return GDL_OK;
    KTimer kt(ctx, K_PROJECT, 16.0 * n);
    hipLaunchKernelGGL(k_project, dim3(stride_grid(ctx, n)), dim3(JB), 0, ctx->stream, d_in, n,
                       map.arity, map.src[0], map.arity == 2 ? map.src[1] : 0, d_out);
    return check_launch(ctx, "k_project");
}

}  // extern "C"
