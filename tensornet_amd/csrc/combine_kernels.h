// The step TensorFlow runs around the pull / push ops of a slot: the combiner of
// tf.nn.embedding_lookup_sparse on the pulled rows (forward) and the reduction of
// its gradient to one row per distinct sign (backward), which the reference
// receives ready-made as the `grads` input of SparseTablePush
// (tensornet/layers/embedding_features.py:278-280, core/kernels/sparse_table_ops.cc:336-352).
//
//   forward   out[b, :] = (sum over the lookups i of example b, in order, of var[mapped[i], :]) / d(n_b)
//             d(n) = 1 (sum), n (mean), sqrt(n) (sqrtn); an example without lookups gives zeros
//   backward  g[u, :]   = sum over the lookups i of distinct sign u of dout[b(i), :] * (1 / d(n_b(i)))
//
// Both are deterministic.  The forward sums run in occurrence order, and so do the backward
// sums of the signs with few lookups; a sign with ORDER_MID (64) lookups or more in a slot is
// summed by a workgroup, whose thread groups take every so many of its lookups and whose
// partial sums are added in group order (k_reduce_pooled).  (On the path of few launches a sign
// with more than POOL_PIECE (32) lookups is summed in pieces of as many, k_small_pool.)  The
// backward pass gets the lookups of every distinct sign side by side, in position order, from a
// counting sort per slot followed by an ordering of every sign's lookups by position
// (k_place_lookups, k_order_segments).
#ifndef TN_COMBINE_KERNELS_H_
#define TN_COMBINE_KERNELS_H_

#include "sparse_kernels.h"

namespace tn {

enum { COMBINE_SUM = 0, COMBINE_MEAN = 1, COMBINE_SQRTN = 2 };
constexpr int COMBINE_WINDOW = 8;  // lookups of an example / of a distinct sign read ahead with independent loads

// In these kernels a SlotDesc carries: values = mapped ids (forward) / signs (backward),
// mapped = example index of every lookup, grads = rows to read (variable / pooled gradient),
// var = rows to write (forward: out[batch, dim]), rows = rows of `grads`, len = lookups.
__device__ __forceinline__ const int64_t* example_of(const SlotDesc& d) { return d.mapped; }

__device__ __forceinline__ float combine_divisor(uint32_t n, int combiner) {
    if (combiner == COMBINE_SUM || n == 0) return 1.f;
    return combiner == COMBINE_MEAN ? (float)n : sqrtf((float)n);
}

// How many of the sorted ids ex[0 .. n) lie below `x`, by a workgroup of 256 threads: every round looks at 256 places
// of what is left, so 65 536 ids take two round trips (a binary search: sixteen).  A function of the array and x alone:
// whatever the order of the ids, two workgroups that ask for the same x get the same answer.  sh: 5 words of LDS.
__device__ __forceinline__ uint32_t ids_below(const int64_t* __restrict__ ex, uint32_t n, int64_t x, uint32_t* sh) {
    uint32_t lo = 0, len = n;  // the answer lies in [lo, lo + len]
    while (len > 0) {
        const uint32_t step = (len + 255) / 256;
        const uint32_t at = threadIdx.x * step;
        const bool below = at < len && ex[lo + at] < x;
        const uint32_t c = block_sum_256(below ? 1u : 0u, sh);  // places below x: the first c of them, if the ids are sorted
        if (step == 1) return lo + c;
        if (c == 0) return lo;
        lo += (c - 1) * step + 1;
        len = min(step - 1, n - lo);
    }
    return lo;
}

// Forward: a workgroup takes `per` examples of a slot (items of a call are numbered slot by slot): it finds their
// lookups, which are consecutive, and every group of LPG lanes sums the rows of an example's lookups in order, divides,
// and writes the output row (zeros for an example without lookups).  One pass: a kernel that first worked out where the
// lookups of every example start cost a launch and a pass over the ids of its own (27 us at 5 M lookups).
//
// The example ids are checked on the way: the workgroups' shares of a slot's lookups follow each other without a gap
// whatever the ids are (each ends where ids_below puts the start of the next, the first starts at 0, the last ends at
// the slot's end), so every lookup is looked at by one workgroup, which wants it to lie among its examples and not
// before its predecessor.
//
// The variable rows of a slot are read again and again: every die of the chip takes a contiguous share of the items, so
// that a slot's rows (1.3 MB at 20 k distinct signs of 16 elements) are in the L2 of the die that wants them.  By the
// counters they are: 4.9 M lookups read 225 MB from memory where every row and id once are 206, 62 % of the requests to L2
// hit; 121 us, 2.7 TB/s, the wavefronts wait 61 % of their cycles.
template <int LPG, bool ANY>
__global__ __launch_bounds__(256) void k_combine_fwd(const SlotDesc* __restrict__ descs, uint32_t items, uint32_t per_slot,
                                                     uint32_t per, int dim, int64_t batch, int combiner, DevStatus* status) {
    extern __shared__ uint32_t range[];  // [per] first lookup of an example, [per] the lookup after its last
    __shared__ uint32_t sh[5];
    const int sub = threadIdx.x % LPG;
    const DieShare share(items);
    uint32_t err = 0;
    for (uint32_t item = share.first; item < share.end; item += share.step) {
        const uint32_t sl = item / per_slot;
        const int64_t b0 = (int64_t)(item - sl * per_slot) * per;
        const uint32_t nb = (uint32_t)min((int64_t)per, batch - b0);
        const SlotDesc d = descs[sl];
        const int64_t* __restrict__ ex = example_of(d);
        for (uint32_t i = threadIdx.x; i < 2 * per; i += 256) range[i] = 0;
        const uint32_t lo = b0 == 0 ? 0u : ids_below(ex, d.len, b0, sh);
        const uint32_t hi = b0 + nb >= batch ? d.len : ids_below(ex, d.len, b0 + nb, sh);
        __syncthreads();
        if (hi < lo) err |= DEV_ERR_GRAD_ROWS;
        for (uint32_t i = lo + threadIdx.x; i < hi; i += 256) {
            const int64_t x = ex[i], prev = i > 0 ? ex[i - 1] : -1, next = i + 1 < d.len ? ex[i + 1] : batch;
            if (x < b0 || x >= b0 + nb || prev > x) {
                err |= DEV_ERR_GRAD_ROWS;
                continue;
            }
            if (prev != x || i == lo) range[x - b0] = i;
            if (next != x || i + 1 == hi) range[per + (x - b0)] = i + 1;
        }
        __syncthreads();
        const int64_t* __restrict__ ids = d.values;
        const float* __restrict__ rows = d.grads;
        for (uint32_t e = threadIdx.x / LPG; e < nb; e += 256 / LPG) {
            const uint32_t from = range[e], to = max(range[per + e], from);
            const float div = combine_divisor(to - from, combiner);
            float* o = d.var + (b0 + e) * dim;
            for (int c0 = 0; c0 < dim; c0 += 4 * LPG) {  // (rows of more than 128 elements: once more for the next ones)
                float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
                // windows of COMBINE_WINDOW lookups: ids first, then their rows, all loads independent; the additions
                // run in lookup order
                for (uint32_t j0 = from; j0 < to; j0 += COMBINE_WINDOW) {
                    int64_t wid[COMBINE_WINDOW];
                    float4 wr[COMBINE_WINDOW];
#pragma unroll
                    for (int q = 0; q < COMBINE_WINDOW; q++) wid[q] = j0 + q < to ? ids[j0 + q] : -1;
#pragma unroll
                    for (int q = 0; q < COMBINE_WINDOW; q++) {
                        const bool ok = wid[q] >= 0 && wid[q] < d.rows;
                        if (j0 + q < to && !ok) err |= DEV_ERR_VAR_CAPACITY;
                        wr[q] = ok ? row_part<ANY>(rows + wid[q] * dim + c0, sub, dim - c0) : make_float4(0.f, 0.f, 0.f, 0.f);
                    }
#pragma unroll
                    for (int q = 0; q < COMBINE_WINDOW; q++) {
                        if (j0 + q >= to) break;
                        acc.x += wr[q].x;
                        acc.y += wr[q].y;
                        acc.z += wr[q].z;
                        acc.w += wr[q].w;
                    }
                }
                put_row_part<ANY>(o + c0, sub, dim - c0, make_float4(acc.x / div, acc.y / div, acc.z / div, acc.w / div));
            }
        }
        __syncthreads();
    }
    if (err) atomicOr(&status->err, err);
}

// Behind the last kernel of a call: its error flags to the host, in one word with the number of the call, for which the
// host polls (a wait on the stream returns about ten microseconds later).  The flags are taken and set to zero for the
// next call, which may come on another stream as soon as the word is out, by one atomic.
__global__ void k_report(DevStatus* status, uint64_t* host_word, uint32_t seq) {
    if (threadIdx.x != 0) return;
    const uint32_t err = __hip_atomic_exchange(&status->err, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long w = (unsigned long long)err | ((unsigned long long)seq << 32);
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(host_word), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Backward, step 1: the value of every lookup: its example in the high word, the number of
// lookups of that example in the low word -- all the reduction needs to know about the lookup, so
// that it reads them in the order of the distinct signs instead of chasing positions.
//
// 16 bytes move per lookup; what bounded it were chains of loads (a thread found the slot of a lookup by bisection, then
// its descriptor, then its id, and the first lookup of an example walked to its last one and wrote all their values).
// A wavefront now takes KEY_ITEMS runs of 64 lookups, their loads in flight together, and reads the extents of its
// examples off a ballot of the places where the id changes; an example that goes on beyond the run is followed there by
// the whole wavefront.  4.9 M lookups: 60 -> 35 us.
constexpr int KEY_ITEMS = 4;
constexpr uint32_t KEY_TILE = 256 * KEY_ITEMS;

__global__ __launch_bounds__(256) void k_lookup_keys(const SlotDesc* __restrict__ descs,
                                                     const uint32_t* __restrict__ lbase, int N, uint32_t L,
                                                     int64_t batch, uint64_t* __restrict__ vals, DevStatus* status,
                                                     uint32_t* long_count) {
    __shared__ uint32_t lb[MAX_SLOTS + 1];
    load_lbase(lb, lbase, N);
    // [1], [2]: entries of the lists of k_place_lookups
    if (blockIdx.x == 0 && threadIdx.x < 3) long_count[threadIdx.x] = 0;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t ntiles = (L + KEY_TILE - 1) / KEY_TILE;
    for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const uint32_t g0 = tile * KEY_TILE, g1 = min(L, g0 + KEY_TILE) - 1;
        const int s0 = find_slot(lb, N, g0);
        const bool one_slot = g1 < lb[s0 + 1];  // the usual case: the tile lies inside one slot
        int sl[KEY_ITEMS];
        int64_t b[KEY_ITEMS], prev[KEY_ITEMS];
#pragma unroll
        for (int j = 0; j < KEY_ITEMS; j++) {
            const uint32_t gi = g0 + (wave * KEY_ITEMS + j) * 64 + lane;
            sl[j] = s0;
            b[j] = prev[j] = -1;
            if (gi <= g1) {
                if (!one_slot) sl[j] = find_slot(lb, N, gi);
                const int64_t* ex = example_of(descs[sl[j]]);
                const uint32_t i = gi - lb[sl[j]];
                b[j] = ex[i];
                if (i > 0) prev[j] = ex[i - 1];
            }
        }
#pragma unroll
        for (int j = 0; j < KEY_ITEMS; j++) {
            const uint32_t base = g0 + (wave * KEY_ITEMS + j) * 64, gi = base + lane;
            const bool active = gi <= g1;
            if (active && (b[j] < 0 || b[j] >= batch || prev[j] > b[j])) {
                atomicOr(&status->err, DEV_ERR_GRAD_ROWS);
                status->abort = 1;  // nothing downstream may run
            }
            // where an example starts (the first lookup of a slot does: prev is -1 there; and what lies behind the last one)
            const unsigned long long heads = __ballot(!active || b[j] != prev[j]);
            uint32_t back = 0, ahead = 0;  // lookups of the first / last example of the run before / behind it
            if (!(heads & 1ull)) {
                const int64_t x = __shfl(b[j], 0);
                const int s = __shfl(sl[j], 0);
                const int64_t* ex = example_of(descs[s]);
                for (uint32_t i = base - lb[s];; i -= 64) {  // lookups [0, i) of the slot are left
                    const unsigned long long other = __ballot(lane >= i || ex[i - 1 - lane] != x);
                    if (other) {
                        back += (uint32_t)__ffsll((long long)other) - 1;
                        break;
                    }
                    back += 64;
                }
            }
            if (base + 63 <= g1) {
                const int64_t x = __shfl(b[j], 63);
                const int s = __shfl(sl[j], 63);
                const int64_t* ex = example_of(descs[s]);
                const uint32_t len = lb[s + 1] - lb[s];
                for (uint32_t i = base + 64 - lb[s];; i += 64) {
                    const unsigned long long other = __ballot(i + lane >= len || ex[i + lane] != x);
                    if (other) {
                        ahead += (uint32_t)__ffsll((long long)other) - 1;
                        break;
                    }
                    ahead += 64;
                }
            }
            if (active) {
                const unsigned long long below = heads & (~0ull >> (63 - lane)), above = heads & ~(~0ull >> (63 - lane));
                const uint32_t to_start = below ? lane - (63 - (uint32_t)__clzll((long long)below)) : lane + back;
                const uint32_t to_end = above ? (uint32_t)__ffsll((long long)above) - 1 - lane : 64 - lane + ahead;
                vals[gi] = ((uint64_t)b[j] << 32) | (uint64_t)(to_start + to_end);
            }
        }
    }
}

// Step 2: the values of the lookups of every distinct index side by side, in position order:
// svals[seg_off[u] .. seg_off[u + 1]).
//   k_place_lookups  a few workgroups per slot (the distinct indices of a slot's lookups fill a window of their
//                    own, ascending with the slots): counts the lookups of every index in an LDS array, scans
//                    the counts into seg_off, and puts the position of every lookup into its index's segment -- in
//                    the order the atomics arrive; indices with ORDER_MID lookups or more are listed for the kernels
//                    below
//   rank_short       a lookup of a short segment finds its place by counting the positions of its segment below its own
//   rank_mid         a sorting network in LDS, one workgroup per segment of ORDER_MID .. ORDER_HUGE - 1 lookups
//   order_huge       the few longer segments: a bitmap of their positions in LDS, one workgroup each
//                    (the three are workgroups of one launch, k_order_segments)
// A slot with more distinct signs than the LDS array holds (lds_cap) keeps its counters in `gcur`.
constexpr int PLACE_THREADS = 1024;
constexpr int PLACE_ITEMS = 8;
constexpr uint32_t ORDER_MID = 64;
constexpr uint32_t ORDER_HUGE = 1024;

// `parts` workgroups per slot: each of them streams all lookups of the slot (they come out of L2 after the first)
// and takes those whose distinct index lies in its share of the slot's window of distinct indices.  The lookups of the
// indices below its share, which it counts on the way, come before its own.
//
// What bounds it is the chain of each of its few workgroups (two passes over the slot's lookups with an LDS atomic each, the
// scan between them): the wavefronts wait 85 % of their cycles while 79 MB are read and 49 written (39 and 28 would do), 1.0
// TB/s.  Only the position is stored, 4 bytes per lookup, and not the index and the value with it (12 bytes): a die has
// the windows of a dozen slots in its L2 at a time (2.5 MB at 49 k lookups a slot; 7.5 MB with the value, more than its
// L2), and lines that are written out half filled are read and written again.
// 4.9 M lookups in 100 slots: 168 us before, 135 with one workgroup per slot and 125 with two.
__global__ __launch_bounds__(PLACE_THREADS) void k_place_lookups(
    const uint32_t* __restrict__ lbase, const uint32_t* __restrict__ ubase, int N, uint32_t L,
    const uint32_t* __restrict__ u_of_gi, uint32_t* __restrict__ tpos, uint32_t* __restrict__ seg_off,
    uint32_t* __restrict__ gcur, uint32_t lds_cap, uint32_t* __restrict__ mid_list, uint32_t* __restrict__ huge_list,
    uint32_t* counts, const DevStatus* status, uint32_t parts) {
    extern __shared__ uint32_t lcur[];
    __shared__ uint32_t red[PLACE_THREADS / 64];
    __shared__ uint32_t carry_sh;
    if (status->abort) return;
    const int sl = blockIdx.x / parts;
    const uint32_t part = blockIdx.x % parts;
    const uint32_t l0 = lbase[sl], len = lbase[sl + 1] - l0;
    const uint32_t ub = ubase[sl], us = ubase[sl + 1] - ub;
    if (sl == N - 1 && part == 0 && threadIdx.x == 0) seg_off[ubase[N]] = L;
    if (len == 0) return;
    // my share of the slot's distinct indices (relative to ub)
    const uint32_t r0 = (uint32_t)((uint64_t)us * part / parts), r1 = (uint32_t)((uint64_t)us * (part + 1) / parts);
    const uint32_t mine = r1 - r0;
    if (mine == 0) return;
    uint32_t* const cur = mine <= lds_cap ? lcur : gcur + ub + r0;
    const uint32_t* const keys = u_of_gi + l0;
    for (uint32_t i = threadIdx.x; i < mine; i += PLACE_THREADS) cur[i] = 0;
    __syncthreads();
    // (eight lookups per thread at a time, their loads in flight together)
    uint32_t below = 0;  // lookups of the indices before my share
    for (uint32_t i0 = threadIdx.x; i0 < len; i0 += PLACE_THREADS * PLACE_ITEMS) {
        uint32_t k[PLACE_ITEMS];
#pragma unroll
        for (int j = 0; j < PLACE_ITEMS; j++) {
            const uint32_t i = i0 + j * PLACE_THREADS;
            k[j] = i < len ? (keys[i] & ~FIRST_BIT) - ub : 0xFFFFFFFFu;
        }
#pragma unroll
        for (int j = 0; j < PLACE_ITEMS; j++) {
            if (k[j] < r0)
                below++;
            else if (k[j] < r1)
                atomicAdd(&cur[k[j] - r0], 1u);
        }
    }
    {
        uint32_t total;
        block_excl_scan<uint32_t, PLACE_THREADS / 64>(below, red, &total);
        if (threadIdx.x == 0) carry_sh = l0 + total;  // the lookups of the slots before, and of the shares before, come first
    }
    __syncthreads();
    for (uint32_t i0 = 0; i0 < mine; i0 += PLACE_THREADS) {
        const uint32_t i = i0 + threadIdx.x;
        const uint32_t cnt = i < mine ? ld_relaxed(cur + i) : 0u;  // (counted by atomics: not through the L1 cache)
        uint32_t total;
        const uint32_t at = carry_sh + block_excl_scan<uint32_t, PLACE_THREADS / 64>(cnt, red, &total);
        if (i < mine) {
            cur[i] = at;
            seg_off[ub + r0 + i] = at;
            if (cnt >= ORDER_HUGE)
                huge_list[atomicAdd(&counts[2], 1u)] = ub + r0 + i;
            else if (cnt >= ORDER_MID)
                mid_list[atomicAdd(&counts[1], 1u)] = ub + r0 + i;
        }
        __syncthreads();
        if (threadIdx.x == 0) carry_sh += total;
        __syncthreads();
    }
    for (uint32_t i0 = threadIdx.x; i0 < len; i0 += PLACE_THREADS * PLACE_ITEMS) {
        uint32_t k[PLACE_ITEMS];
#pragma unroll
        for (int j = 0; j < PLACE_ITEMS; j++) {
            const uint32_t i = i0 + j * PLACE_THREADS;
            k[j] = i < len ? (keys[i] & ~FIRST_BIT) - ub : 0xFFFFFFFFu;
        }
#pragma unroll
        for (int j = 0; j < PLACE_ITEMS; j++)
            if (k[j] >= r0 && k[j] < r1) tpos[atomicAdd(&cur[k[j] - r0], 1u)] = l0 + i0 + j * PLACE_THREADS;
    }
}

// The lookups in the order of their segments: the runs of a die (DieRuns) keep to one slot, whose distinct indices and
// values, read by position, are then more often in its L2.  4.9 M lookups: 78 -> 62 us.  Bound by the reads by
// position: with the longer segments beside it 340 MB come from memory where 87 would do (56 % of the L2's requests hit),
// 4.4 TB/s, about what random granules reach.
constexpr uint32_t RANK_RUN = 128;

__device__ __forceinline__ void rank_short(uint32_t L, const uint32_t* __restrict__ u_of_gi,
                                           const uint64_t* __restrict__ vals, const uint32_t* __restrict__ tpos,
                                           const uint32_t* __restrict__ seg_off, uint64_t* __restrict__ svals, uint32_t block,
                                           uint32_t blocks) {
    for (DieRuns r((L + 255) / 256, RANK_RUN, block, blocks); r.more(); r.next()) {
        const uint32_t t = r.item() * 256 + threadIdx.x;
        if (t >= L) continue;
        const uint32_t gi = tpos[t];
        const uint32_t u = u_of_gi[gi] & ~FIRST_BIT;
        const uint64_t v = vals[gi];
        const uint32_t lo = seg_off[u], hi = seg_off[u + 1];
        if (hi - lo >= ORDER_MID) continue;
        uint32_t rank = 0;
        for (uint32_t j = lo; j < hi; j++) rank += tpos[j] < gi ? 1u : 0u;
        svals[lo + rank] = v;
    }
}

// seg: ORDER_HUGE words of LDS
__device__ __forceinline__ void rank_mid(const uint32_t* __restrict__ mid_list, uint32_t n_mid,
                                         const uint32_t* __restrict__ seg_off, const uint64_t* __restrict__ vals,
                                         const uint32_t* __restrict__ tpos, uint64_t* __restrict__ svals, uint32_t* seg,
                                         uint32_t block, uint32_t blocks) {
    for (uint32_t k = block; k < n_mid; k += blocks) {
        const uint32_t u = mid_list[k];
        const uint32_t lo = seg_off[u], n = seg_off[u + 1] - lo;  // ORDER_MID <= n < ORDER_HUGE
        uint32_t p2 = ORDER_MID;
        while (p2 < n) p2 <<= 1;
        // bitonic sorting network over the segment padded with the largest value to a power of two
        for (uint32_t i = threadIdx.x; i < p2; i += 256) seg[i] = i < n ? tpos[lo + i] : 0xFFFFFFFFu;
        __syncthreads();
        for (uint32_t size = 2; size <= p2; size <<= 1) {
            for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                for (uint32_t t = threadIdx.x; t < p2 / 2; t += 256) {
                    const uint32_t a = 2 * t - (t & (stride - 1));  // lower element of the t-th pair
                    const uint32_t b = a + stride;
                    const bool up = (a & size) == 0;
                    const uint32_t x = seg[a], y = seg[b];
                    if ((x > y) == up) {
                        seg[a] = y;
                        seg[b] = x;
                    }
                }
                __syncthreads();
            }
        }
        for (uint32_t i = threadIdx.x; i < n; i += 256) svals[lo + i] = vals[seg[i]];
        __syncthreads();
    }
}

// A segment of many lookups is ordered by a bitmap of their positions in the slot, HUGE_WINDOW of these at a time (the
// place of a lookup: bits set below its own).  The bitmap of a slot of 49 k lookups with its prefix sums takes 9 KB of LDS,
// so a CU holds eight workgroups; counters per example, as this had before, took 64 KB at 16384 examples, or memory.
// Beside rank_mid (72 -> 42 us), 4.9 M lookups: 57 -> 34 us.
constexpr uint32_t HUGE_WINDOW = 1u << 17;
inline size_t order_huge_room(size_t max_len) { return (std::min<size_t>(max_len, HUGE_WINDOW) + 63) / 64; }

// bits: [room] words of LDS, then [room] numbers of set bits before the word
__device__ __forceinline__ void order_huge(const uint32_t* __restrict__ huge_list, uint32_t n_huge,
                                           const uint32_t* __restrict__ lbase, const uint32_t* __restrict__ ubase, int N,
                                           const uint32_t* __restrict__ seg_off, const uint64_t* __restrict__ vals,
                                           const uint32_t* __restrict__ tpos, uint64_t* __restrict__ svals,
                                           unsigned long long* bits, uint32_t room, uint32_t* red, uint32_t block,
                                           uint32_t blocks) {
    uint32_t* const before = reinterpret_cast<uint32_t*>(bits + room);
    for (uint32_t k = block; k < n_huge; k += blocks) {
        const uint32_t u = huge_list[k];
        const uint32_t lo = seg_off[u], hi = seg_off[u + 1];
        const int sl = find_slot(ubase, N, u);
        const uint32_t l0 = lbase[sl], len = lbase[sl + 1] - l0;
        uint32_t done = 0;  // lookups of the windows before
        for (uint32_t w0 = 0; w0 < len; w0 += HUGE_WINDOW) {
            const uint32_t span = min(len - w0, HUGE_WINDOW), words = (span + 63) / 64;  // (words <= room)
            for (uint32_t i = threadIdx.x; i < words; i += 256) bits[i] = 0;
            __syncthreads();
            for (uint32_t j = lo + threadIdx.x; j < hi; j += 256) {
                const uint32_t p = tpos[j] - l0 - w0;  // (a position before the window: beyond it)
                if (p < span) atomicOr(&bits[p >> 6], 1ull << (p & 63));
            }
            __syncthreads();
            for (uint32_t i0 = 0; i0 < words; i0 += 256) {
                const uint32_t i = i0 + threadIdx.x;
                uint32_t total;
                const uint32_t x = block_excl_scan_256<uint32_t>(i < words ? (uint32_t)__popcll(bits[i]) : 0u, red, &total);
                if (i < words) before[i] = done + x;
                done += total;
                __syncthreads();
            }
            for (uint32_t j = lo + threadIdx.x; j < hi; j += 256) {
                const uint32_t gi = tpos[j], p = gi - l0 - w0;
                if (p < span) svals[lo + before[p >> 6] + (uint32_t)__popcll(bits[p >> 6] & ((1ull << (p & 63)) - 1ull))] = vals[gi];
            }
            __syncthreads();
        }
    }
}

// The three side by side in one launch, the longest segments first: each has segments of its own, and waits for chains.
// 860 k lookups: three launches 34 us, this one 21; 4.9 M: 86, as the three took on three streams, without the events
// between these.
constexpr uint32_t ORDER_HUGE_GRID = 1024, ORDER_MID_GRID = 2048;  // workgroups at most, which take their segments in turn
inline size_t order_lds(size_t room) { return std::max<size_t>(room * 12, ORDER_HUGE * sizeof(uint32_t)); }

__global__ __launch_bounds__(256) void k_order_segments(uint32_t L, const uint32_t* __restrict__ lbase,
                                                        const uint32_t* __restrict__ ubase, int N,
                                                        const uint32_t* __restrict__ u_of_gi,
                                                        const uint32_t* __restrict__ mid_list,
                                                        const uint32_t* __restrict__ huge_list, const uint32_t* counts,
                                                        const uint32_t* __restrict__ seg_off,
                                                        const uint64_t* __restrict__ vals, const uint32_t* __restrict__ tpos,
                                                        uint64_t* __restrict__ svals, uint32_t room, uint32_t huge_blocks,
                                                        uint32_t mid_blocks, const DevStatus* status) {
    extern __shared__ unsigned long long order_sh[];
    __shared__ uint32_t red[4];
    if (status->abort) return;
    const uint32_t b = blockIdx.x, long_blocks = huge_blocks + mid_blocks;
    if (b < huge_blocks)
        order_huge(huge_list, counts[2], lbase, ubase, N, seg_off, vals, tpos, svals, order_sh, room, red, b, huge_blocks);
    else if (b < long_blocks)
        rank_mid(mid_list, counts[1], seg_off, vals, tpos, svals, reinterpret_cast<uint32_t*>(order_sh), b - huge_blocks,
                 mid_blocks);
    else
        rank_short(L, u_of_gi, vals, tpos, seg_off, svals, b - long_blocks, gridDim.x - long_blocks);
}

// The sum of the shares of lookups from, from + step, ... below `to` of one distinct sign, in this order: every lookup
// has its example's pooled row times 1 / d(lookups of the example); four elements of a row, part c of them.  The
// values of a window first, then their rows, all loads of a kind independent.
template <bool ANY>
__device__ __forceinline__ float4 sum_shares(const float* __restrict__ pooled, const uint64_t* __restrict__ svals, uint32_t from,
                                             uint32_t to, uint32_t step, int dim, int c, int combiner) {
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (uint32_t j0 = from; j0 < to; j0 += COMBINE_WINDOW * step) {
        uint64_t v[COMBINE_WINDOW];
        float4 g[COMBINE_WINDOW];
#pragma unroll
        for (int q = 0; q < COMBINE_WINDOW; q++) v[q] = j0 + q * step < to ? svals[j0 + q * step] : 0ull;
#pragma unroll
        for (int q = 0; q < COMBINE_WINDOW; q++)
            g[q] = j0 + q * step < to ? row_part<ANY>(pooled + (v[q] >> 32) * (uint64_t)dim, c, dim)
                                      : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int q = 0; q < COMBINE_WINDOW; q++) {
            if (j0 + q * step >= to) break;
            const float scale = combiner == COMBINE_SUM ? 1.f : 1.f / combine_divisor((uint32_t)v[q], combiner);
            acc.x += g[q].x * scale;
            acc.y += g[q].y * scale;
            acc.z += g[q].z * scale;
            acc.w += g[q].w * scale;
        }
    }
    return acc;
}

// Step 3: a group of `chunks` threads per distinct index, four elements of the row each (whatever its length and
// alignment), sums its lookups' shares of the pooled gradient rows, in position order.  A distinct index with long_min
// lookups or more (a frequent sign) is left out: k_place_lookups has listed those, one workgroup each sums them
// (reduce_long).
//
// Bound by the rows it reads again and again: the pooled rows of a slot (1 MB at 16384 examples of 16 elements) are more
// often in the L2 of a die that works on one slot at a time, so the distinct indices go to the dies in runs of REDUCE_RUN
// workgroups (DieRuns; a grid-stride loop had every die read the rows of six slots).  4.9 M lookups of 16 elements:
// 172 -> 138 us, the frequent signs beside it 120 -> 93 us.  By the counters of both together 30 % of the L2's requests hit:
// 426 MB are read where each row and value once are 152, with what is written 3.8 TB/s.
constexpr uint32_t REDUCE_RUN = 256;

template <bool ANY>
__device__ __forceinline__ void reduce_short(const SlotDesc* __restrict__ descs, const uint32_t* __restrict__ ubase, int N,
                                             int dim, int combiner, const DevStatus* status,
                                             const uint32_t* __restrict__ seg_off, const uint64_t* __restrict__ svals,
                                             float* __restrict__ flat, uint32_t long_min, uint32_t* ub, uint32_t block,
                                             uint32_t blocks) {
    load_lbase(ub, ubase, N);
    const uint32_t chunks = (uint32_t)(dim + 3) / 4;
    const uint64_t total = (uint64_t)status->n_unique * chunks;
    for (DieRuns r((uint32_t)((total + 255) / 256), REDUCE_RUN, block, blocks); r.more(); r.next()) {
        const uint64_t t = (uint64_t)r.item() * 256 + threadIdx.x;
        if (t >= total) continue;
        const uint32_t u = (uint32_t)(t / chunks);
        const int c = (int)(t - (uint64_t)u * chunks);
        const uint32_t lo = seg_off[u], hi = seg_off[u + 1];
        if (hi - lo >= long_min) continue;
        const float* pooled = descs[find_slot(ub, N, u)].grads;  // the slot whose window of distinct indices holds u
        put_row_part<ANY>(flat + (uint64_t)u * dim, c, dim, sum_shares<ANY>(pooled, svals, lo, hi, 1, dim, c, combiner));
    }
}

// One workgroup per frequent distinct index: its 256 / chunks thread groups each sum every
// (256 / chunks)-th lookup in position order, then the partial sums are added in group order.
// The order of the additions is fixed, so the result does not vary from run to run.
template <bool ANY>
__device__ __forceinline__ void reduce_long(const SlotDesc* __restrict__ descs, const uint32_t* __restrict__ ubase, int N,
                                            int dim, int combiner, const uint32_t* __restrict__ seg_off,
                                            const uint64_t* __restrict__ svals, float* __restrict__ flat,
                                            const uint32_t* __restrict__ mid_list, const uint32_t* __restrict__ huge_list,
                                            const uint32_t* counts, float4* part, uint32_t block, uint32_t blocks) {
    const int chunks = (dim + 3) / 4;
    const int groups = 256 / chunks;
    const int q = threadIdx.x / chunks, c = threadIdx.x - q * chunks;
    // the frequent ones: the two lists k_place_lookups left (ORDER_MID lookups or more)
    const uint32_t n_mid = counts[1], n_long = n_mid + counts[2];
    for (uint32_t k = n_long - 1 - block; k < n_long; k -= blocks) {  // (the longest, which are listed last, first; ends by wrapping)
        const uint32_t u = k < n_mid ? mid_list[k] : huge_list[k - n_mid];
        const uint32_t lo = seg_off[u], hi = seg_off[u + 1];
        const float* pooled = descs[find_slot(ubase, N, u)].grads;
        if (q < groups) part[threadIdx.x] = sum_shares<ANY>(pooled, svals, lo + q, hi, groups, dim, c, combiner);
        __syncthreads();
        if (q == 0) {
            float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
            for (int g = 0; g < groups; g++) {
                const float4 p = part[g * chunks + c];
                sum.x += p.x;
                sum.y += p.y;
                sum.z += p.z;
                sum.w += p.w;
            }
            put_row_part<ANY>(flat + (uint64_t)u * dim, c, dim, sum);
        }
        __syncthreads();
    }
}

// Both side by side in one launch, the frequent signs first.  860 k lookups of 16 elements: 53 us in two launches, 46 in
// this one; 4.9 M: 140, as on two streams.
template <bool ANY>
__global__ __launch_bounds__(256) void k_reduce_pooled(const SlotDesc* __restrict__ descs,
                                                       const uint32_t* __restrict__ ubase, int N, int dim, int combiner,
                                                       const DevStatus* status, const uint32_t* __restrict__ seg_off,
                                                       const uint64_t* __restrict__ svals, float* __restrict__ flat,
                                                       uint32_t long_min, const uint32_t* __restrict__ mid_list,
                                                       const uint32_t* __restrict__ huge_list, const uint32_t* counts,
                                                       uint32_t long_blocks) {
    __shared__ union {
        uint32_t ub[MAX_SLOTS + 1];
        float4 part[256];
    } sh;
    if (status->abort) return;
    if (blockIdx.x < long_blocks)
        reduce_long<ANY>(descs, ubase, N, dim, combiner, seg_off, svals, flat, mid_list, huge_list, counts, sh.part, blockIdx.x,
                         long_blocks);
    else
        reduce_short<ANY>(descs, ubase, N, dim, combiner, status, seg_off, svals, flat, long_min, sh.ub,
                          blockIdx.x - long_blocks, gridDim.x - long_blocks);
}

}  // namespace tn

#endif  // TN_COMBINE_KERNELS_H_
