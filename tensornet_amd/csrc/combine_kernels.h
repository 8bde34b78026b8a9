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
// Both are deterministic.  The forward sums run in occurrence order.  So do the backward sums, but cut up: a workgroup's
// lookups, in the order of their signs, every POOL_PIECE (16) places (8, 4 of a few lookups); what a sign has in several pieces is added in order,
// what it has in several rounds of a workgroup round by round, what a frequent one has in several workgroups by halves
// (k_reduce_pooled, on the path of few launches k_small_pool; add_shares).
#ifndef TN_COMBINE_KERNELS_H_
#define TN_COMBINE_KERNELS_H_

#include "lookup_range.h"
#include "pool_items.h"

#include <algorithm>

namespace tn {

enum { COMBINE_SUM = 0, COMBINE_MEAN = 1, COMBINE_SQRTN = 2 };
constexpr int COMBINE_WINDOW = 8;  // lookups of an example read ahead with independent loads

// In these kernels a SlotDesc carries: values = mapped ids (forward) / signs (backward),
// mapped = example index of every lookup, grads = rows to read (variable / pooled gradient),
// var = rows to write (forward: out[batch, dim]), rows = rows of `grads`, len = lookups.
__device__ __forceinline__ Global<const int64_t> example_of(const SlotDesc& d) { return as_global((const int64_t*)d.mapped); }

__device__ __forceinline__ float combine_divisor(uint32_t n, int combiner) {
    if (combiner == COMBINE_SUM || n == 0) return 1.f;
    return combiner == COMBINE_MEAN ? (float)n : sqrtf((float)n);
}

// How many of the sorted ids ex[0 .. n) lie below x0 and how many below x1, by a workgroup of 256 threads: every round looks at
// 256 places of what is left, so 65 536 ids take two round trips (a binary search: sixteen).  Either is a function of the array
// and its x alone: whatever the order of the ids, two workgroups that ask for the same x get the same answer.  sh: 5 words of LDS.
__device__ __forceinline__ uint2 ids_below(Global<const int64_t> ex, uint32_t n, int64_t x0, int64_t x1, uint32_t* sh) {
    uint32_t lo[2] = {0, 0}, len[2] = {n, n};  // the answers lie in [lo, lo + len]
    const int64_t x[2] = {x0, x1};
    while (len[0] | len[1]) {
        uint32_t step[2], below = 0;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            step[k] = (len[k] + 255) / 256;
            const uint32_t at = threadIdx.x * step[k];
            if (at < len[k] && ex[lo[k] + at] < x[k]) below += 1u << (16 * k);
        }
        const uint32_t both = block_sum_256(below, sh);  // places below x: the first c of them, if the ids are sorted
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint32_t c = both >> (16 * k) & 0xFFFFu;
            if (len[k] == 0) continue;
            if (step[k] == 1) {
                lo[k] += c;
                len[k] = 0;
            } else if (c == 0) {
                len[k] = 0;
            } else {
                lo[k] += (c - 1) * step[k] + 1;
                len[k] = min(step[k] - 1, n - lo[k]);
            }
        }
    }
    return make_uint2(lo[0], lo[1]);
}

// Forward: a workgroup takes `per` examples of a slot (items of a call are numbered slot by slot): it finds their
// lookups, which are consecutive, and every group of LPG lanes sums the rows of an example's lookups in order, divides,
// and writes the output row (zeros for an example without lookups).  One pass: a kernel that first worked out where the
// lookups of every example start cost a launch and a pass over the ids of its own (27 us at 5 M lookups).
//
// The example ids are checked on the way: the workgroups' shares of a slot's lookups follow each other without a gap
// whatever the ids are (each ends where ids_below puts the start of the next, the first starts at 0, the last ends at
// the slot's end), so every lookup is looked at by one workgroup, which wants it to lie among its examples and not
// before its predecessor; what is summed lies among the lookups it looked at even where it refused some (lookup_range: a position
// ahead of them would be an index in front of `row`).  The same pass checks the mapped ids and leaves them in LDS where they fit (COMBINE_IDS): read where
// they are used, by every lane of a group, they were a round trip in front of every example's rows.  Rows of 16, 4.9 M lookups
// 121 -> 100 us, 860 k 29 -> 21, 20 k (104 workgroups) 7.9 -> 7.1.
//
// The variable rows of a slot are read again and again: every die of the chip takes a contiguous share of the items, so
// that a slot's rows (1.3 MB at 20 k distinct signs of 16 elements) are in the L2 of the die that wants them.  The 4.9 M lookups
// read 225 MB and write 105 in the 100 us, 3.3 TB/s.
struct NoDescs {};
__device__ __forceinline__ const SlotDesc& desc_of(const ArgDescs& a, const SlotDesc*, uint32_t sl) { return a.slot[sl]; }
__device__ __forceinline__ const SlotDesc& desc_of(const NoDescs&, const SlotDesc* __restrict__ d, uint32_t sl) { return d[sl]; }
constexpr uint32_t COMBINE_IDS = 2048;
constexpr uint32_t COMBINE_AHEAD = 2;  // lookups of a thread in flight while they are checked
template <int LPG, bool ANY, typename Descs>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ANY ? 6 : 7, 8))) void k_combine_fwd(Descs by_value, const SlotDesc* __restrict__ descs, uint32_t items, uint32_t per_slot,
                                                     uint32_t per, int dim, int64_t batch, int combiner, DevStatus* status) {
    extern __shared__ uint32_t range[];  // [per] first lookup of an example, [per] the lookup after its last
    __shared__ uint32_t row[COMBINE_IDS];
    __shared__ uint32_t sh[5];
    const int sub = threadIdx.x % LPG;
    const DieShare share(items);
    uint32_t err = 0;
    for (uint32_t item = share.first; item < share.end; item += share.step) {
        const uint32_t sl = item / per_slot;
        const int64_t b0 = (int64_t)(item - sl * per_slot) * per;
        const uint32_t nb = (uint32_t)min((int64_t)per, batch - b0);
        const SlotDesc d = desc_of(by_value, descs, sl);
        const Global<const int64_t> ex = example_of(d);
        const Global<const int64_t> ids = as_global(d.values);
        for (uint32_t i = threadIdx.x; i < 2 * per; i += 256) range[i] = 0;
        uint32_t lo = 0, hi = d.len;
        if (b0 > 0 || b0 + nb < batch) {
            const uint2 bound = ids_below(ex, d.len, b0, b0 + nb, sh);
            if (b0 > 0) lo = bound.x;
            if (b0 + nb < batch) hi = bound.y;
        }
        const bool narrow = d.rows < (int64_t)NO_ROW, kept = narrow && hi - lo <= COMBINE_IDS;
        __syncthreads();
        if (hi < lo) err |= DEV_ERR_GRAD_ROWS;
        for (uint32_t i0 = lo + threadIdx.x; i0 < hi; i0 += 256 * COMBINE_AHEAD) {
            int64_t x[COMBINE_AHEAD], prev[COMBINE_AHEAD], next[COMBINE_AHEAD], id[COMBINE_AHEAD];
#pragma unroll
            for (uint32_t q = 0; q < COMBINE_AHEAD; q++) {
                const uint32_t i = i0 + 256 * q;
                if (i >= hi) continue;
                x[q] = ex[i];
                prev[q] = i > 0 ? ex[i - 1] : -1;
                next[q] = i + 1 < d.len ? ex[i + 1] : batch;
                id[q] = kept ? ids[i] : 0;
            }
#pragma unroll
            for (uint32_t q = 0; q < COMBINE_AHEAD; q++) {
                const uint32_t i = i0 + 256 * q;
                if (i >= hi) continue;
                if (kept) {
                    const bool ok = id[q] >= 0 && id[q] < d.rows;
                    row[i - lo] = ok ? (uint32_t)id[q] : NO_ROW;
                    if (!ok) err |= DEV_ERR_VAR_CAPACITY;
                }
                if (x[q] < b0 || x[q] >= b0 + nb || prev[q] > x[q]) {
                    err |= DEV_ERR_GRAD_ROWS;
                    continue;
                }
                if (prev[q] != x[q] || i == lo) range[x[q] - b0] = i;
                if (next[q] != x[q] || i + 1 == hi) range[per + (x[q] - b0)] = i + 1;
            }
        }
        __syncthreads();
        const float* __restrict__ rows = d.grads;
        for (uint32_t e = threadIdx.x / LPG; e < nb; e += 256 / LPG) {
            const LookupRange mine = lookup_range(range[e], range[per + e], lo);
            const uint32_t from = mine.from, to = mine.to;
            const float div = combine_divisor(to - from, combiner);
            float* o = d.var + (b0 + e) * dim;
            for (int c0 = 0; c0 < dim; c0 += 4 * LPG) {  // (rows of more than 128 elements: once more for the next ones)
                float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
                // windows of COMBINE_WINDOW lookups, their rows' loads independent; the additions run in lookup order
                for (uint32_t j0 = from; j0 < to; j0 += COMBINE_WINDOW) {
                    uint32_t r[COMBINE_WINDOW];
                    float4 wr[COMBINE_WINDOW];
                    if (kept) {
#pragma unroll
                        for (uint32_t q = 0; q < COMBINE_WINDOW; q++) r[q] = j0 + q < to ? row[j0 + q - lo] : NO_ROW;
                    } else if (narrow) {
#pragma unroll
                        for (uint32_t q = 0; q < COMBINE_WINDOW; q++) {
                            const int64_t id = j0 + q < to ? ids[j0 + q] : -1;
                            const bool ok = id >= 0 && id < d.rows;
                            if (j0 + q < to && !ok) err |= DEV_ERR_VAR_CAPACITY;
                            r[q] = ok ? (uint32_t)id : NO_ROW;
                        }
                    } else {  // (a variable of four billion rows)
#pragma unroll 1
                        for (uint32_t j = j0; j < min(j0 + COMBINE_WINDOW, to); j++) {
                            const int64_t id = ids[j];
                            if (id < 0 || id >= d.rows) {
                                err |= DEV_ERR_VAR_CAPACITY;
                                continue;
                            }
                            const float4 v = row_part<ANY>(rows + id * dim + c0, sub, dim - c0);
                            acc = make_float4(acc.x + v.x, acc.y + v.y, acc.z + v.z, acc.w + v.w);
                        }
                        continue;
                    }
#pragma unroll
                    for (uint32_t q = 0; q < COMBINE_WINDOW; q++)
                        wr[q] = r[q] != NO_ROW ? row_part<ANY>(rows + (uint64_t)r[q] * dim + c0, sub, dim - c0)
                                               : make_float4(0.f, 0.f, 0.f, 0.f);
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
static __global__ void k_report(DevStatus* status, uint64_t* host_word, uint32_t seq) {
    if (threadIdx.x != 0) return;
    const uint32_t err = __hip_atomic_exchange(&status->err, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long w = (unsigned long long)err | ((unsigned long long)seq << 32);
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(host_word), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr uint32_t KEY_ITEMS = 8;
constexpr uint32_t KEY_WAVES = 4;
constexpr uint32_t POOL_TILE = 64 * KEY_WAVES * KEY_ITEMS;
constexpr uint32_t POOL_PARTS = 2048;  // of a slot at most
// 49 k lookups a slot: 31 parts (1600) 148 us, 28 (1800) 144, 48 (1024) 144 and the shares 12 for 9; of 4 k: 3 parts 33, 4 parts
// (1024, 1360) 34 to 36.  (Powers of two only, three workgroups to a CU: 4 parts 44, of 211 slots one and a tenth of a round.)
constexpr uint32_t POOL_FILL = 1600;
constexpr uint32_t POOL_SPREAD = 64;
// (4 M rows of 16: one at a time 167 us, two 164, four 163, eight 162)
constexpr uint32_t POOL_ROWS_LOG2 = 2, POOL_ROWS = 1u << POOL_ROWS_LOG2;
constexpr uint32_t POOL_EXTRA = 64;
constexpr uint32_t POOL_SHARES = POOL_SPREAD + POOL_EXTRA;
// Slots of more than POOL_SPREAD_FROM lookups have spread signs.  Shorter ones of several parts have extra ones only, and
// only if the pull has found a heavy sign in the batch (DevStatus::heavy), or did not look for one: it is up to three further
// rounds there, and finding it and adding up the shares are two launches.
constexpr uint32_t POOL_SPREAD_FROM = 6403;

// How a slot's lookups are shared out to the backward pass's workgroups: in tiles of POOL_TILE for step 1, for step 2 in
// as many parts as POOL_FILL lookups each on average ask for.  The distinct indices of the slot ascend with the signs' first occurrences, so
// that the frequent signs come early.  The lookups of the first `spread` indices of a slot with many parts are dealt to these
// run by run (64 lookups), and every part leaves a share of those signs' sums (k_reduce_pooled_shares adds them up): a sign
// with 8 % of a slot's lookups would be three rounds of one part, and the last workgroup's.  So are those of up to POOL_EXTRA
// further ones with half as many lookups as a part or more (k_pool_frequent).  The other indices are
// dealt to the parts in turn, POOL_ROWS at a time (whose rows share a line or two).  Tiles and parts of a call are numbered through the slots so that a slot's first is known from the
// lookups before it; some numbers are nobody's.
struct PoolShare {
    uint32_t parts_max;  // of the longest slot
    uint32_t extra_from; // slots of more lookups may have extra spread signs
    PoolShare(uint32_t max_len, bool heavy) : parts_max(parts(max_len)), extra_from(heavy ? POOL_FILL : POOL_SPREAD_FROM) {}
    static __host__ __device__ uint32_t parts(uint32_t len) {
        const uint32_t n = (len + POOL_FILL - 1) / POOL_FILL;
        return n < 1 ? 1u : n < POOL_PARTS ? n : POOL_PARTS;
    }
    __host__ __device__ bool spreads(uint32_t len) const { return len > extra_from; }  // has extra ones, maybe
    static __host__ __device__ uint32_t spread(uint32_t len) { return len > POOL_SPREAD_FROM ? POOL_SPREAD : 0u; }
    static __host__ __device__ uint32_t first_tile(uint32_t slot, uint32_t lookups_before) {
        return lookups_before / POOL_TILE + slot;
    }
    static __host__ __device__ uint32_t first_part(uint32_t slot, uint32_t lookups_before) {
        return lookups_before / POOL_FILL + slot;
    }
};
// Turns: x = q * parts + part, without a division.
struct PoolTurn {
    uint32_t parts, magic;
    __device__ __forceinline__ explicit PoolTurn(uint32_t n) : parts(n), magic(n > 1 ? 0xFFFFFFFFu / n + 1u : 0u) {}
    __device__ __forceinline__ uint32_t turn(uint32_t x) const {
        if (parts == 1) return x;
        const uint32_t q = __umulhi(x, magic);  // x / parts, or one more
        return q * parts > x ? q - 1u : q;
    }
    __device__ __forceinline__ uint32_t part(uint32_t x) const { return x - turn(x) * parts; }
    // an index that is not spread: whose it is, which of its part's, and back (less the part's own first one)
    __device__ __forceinline__ uint32_t part_of(uint32_t index) const { return part(index >> POOL_ROWS_LOG2); }
    __device__ __forceinline__ uint32_t key_of(uint32_t index) const {
        return (turn(index >> POOL_ROWS_LOG2) << POOL_ROWS_LOG2) | (index & (POOL_ROWS - 1u));
    }
    __device__ __forceinline__ uint32_t index_of(uint32_t key) const {
        return ((key >> POOL_ROWS_LOG2) * parts << POOL_ROWS_LOG2) | (key & (POOL_ROWS - 1u));
    }
};

// Which signs of a slot that has spread ones are frequent although they come late -- behind the first distinct ones, or where
// the lookups are grouped: `extra`, per slot the number of them, then their indices.  Left to one part such a sign is a chain
// of rounds: 100 slots of 49 k lookups, 80 % of them a sign that comes 101st, k_reduce_pooled 632 us, so 155; a step of one
// slot of a million 9.2 ms, so 0.27.  The counts of a sample decide: 128 runs of sixteen lookups (in a short slot fewer) at
// places that are even but for a jitter (positions with a period would all look alike).  A workgroup per slot, a chain of one
// round trip and LDS: 6.7 us for 100 slots of 49 k.  What is chosen depends on the lookups alone, not on the order of atomics.
constexpr uint32_t FREQUENT_RUN = 16, FREQUENT_SAMPLES = 2048, FREQUENT_TABLE = 4096;
constexpr uint32_t FREQUENT_LEAST = 8;  // of the sample, however long the slot: fewer are chance
constexpr uint32_t FREQUENT_LISTED = FREQUENT_SAMPLES / FREQUENT_LEAST;
static __global__ __launch_bounds__(POOL_THREADS) void k_pool_frequent(const uint32_t* __restrict__ lbase,
                                                                       const uint32_t* __restrict__ ubase,
                                                                       const uint32_t* __restrict__ u_of_gi, PoolShare share,
                                                                       uint32_t* __restrict__ extra) {
    __shared__ uint32_t index[FREQUENT_TABLE], count[FREQUENT_TABLE];
    __shared__ uint32_t listed[FREQUENT_LISTED], times[FREQUENT_LISTED], n_listed;
    const uint32_t sl = blockIdx.x, tid = threadIdx.x, l0 = lbase[sl], len = lbase[sl + 1] - l0, ub = ubase[sl];
    uint32_t* const out = extra + sl * (POOL_EXTRA + 1);
    const uint32_t spread = share.spread(len);
    if (!share.spreads(len)) {
        if (tid == 0) out[0] = 0;
        return;
    }
    constexpr uint32_t PER = FREQUENT_SAMPLES / POOL_THREADS;
    const uint32_t runs = min(FREQUENT_SAMPLES / FREQUENT_RUN, len / (2 * FREQUENT_RUN));  // (several parts: len is POOL_FILL and more)
    uint32_t x[PER];
#pragma unroll
    for (uint32_t j = 0; j < PER; j++) {
        const uint32_t r = (j * POOL_THREADS + tid) / FREQUENT_RUN;
        x[j] = NO_ROW;
        if (r >= runs) continue;
        const uint32_t from = (uint32_t)((uint64_t)len * r / runs), room = (uint32_t)((uint64_t)len * (r + 1) / runs) - from;
        const uint32_t jitter = (uint32_t)(((uint64_t)((r + 1) * 2654435761u) * (room - FREQUENT_RUN + 1)) >> 32);
        x[j] = (u_of_gi[l0 + from + jitter + tid % FREQUENT_RUN] & ~FIRST_BIT) - ub;  // (room: two runs' at least)
    }
    for (uint32_t i = tid; i < FREQUENT_TABLE; i += POOL_THREADS) {
        index[i] = NO_ROW;
        count[i] = 0;
    }
    if (tid == 0) n_listed = 0;
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < PER; j++) {
        if (x[j] < spread || x[j] == NO_ROW) continue;
        for (uint32_t h = (x[j] * 2654435761u) / (uint32_t)(0x100000000ull / FREQUENT_TABLE);; h = (h + 1) % FREQUENT_TABLE) {
            const uint32_t old = atomicCAS(&index[h], NO_ROW, x[j]);
            if (old != NO_ROW && old != x[j]) continue;  // (half of the entries stay free)
            atomicAdd(&count[h], 1u);
            break;
        }
    }
    __syncthreads();
    const uint32_t least = max(FREQUENT_LEAST, (uint32_t)((uint64_t)runs * FREQUENT_RUN * (POOL_FILL / 2) / len));
    for (uint32_t i = tid; i < FREQUENT_TABLE; i += POOL_THREADS) {
        if (count[i] < least) continue;
        const uint32_t k = atomicAdd(&n_listed, 1u);
        listed[k] = index[i];
        times[k] = count[i];
    }
    __syncthreads();
    const uint32_t n = n_listed;
    if (tid == 0) out[0] = min(n, POOL_EXTRA);
    if (tid >= n) return;
    uint32_t rank = 0;  // the most frequent first, of those alike the one that comes first
    for (uint32_t i = 0; i < n; i++)
        rank += times[i] > times[tid] || (times[i] == times[tid] && listed[i] < listed[tid]) ? 1u : 0u;
    if (rank < POOL_EXTRA) out[1 + rank] = listed[tid];
}
static_assert(FREQUENT_LISTED <= POOL_THREADS && FREQUENT_SAMPLES % POOL_THREADS == 0 && 2 * FREQUENT_SAMPLES <= FREQUENT_TABLE, "");

// Backward, step 1.  A tile of POOL_TILE lookups of a slot leaves an item for every lookup -- example, sign, lookups of the
// example --, the items of a part side by side in the order of their positions, and where the parts start among them.
//
// 20 bytes move per lookup (4.9 M: 34 us, 2.9 TB/s).  A wavefront takes KEY_ITEMS runs of 64 lookups and the ids of the 64 lookups on
// either side, their loads in flight together, and reads the extents of its examples off ballots of the places where the id changes;
// an example that goes on beyond those is followed there by the whole wavefront.  (Every run's ends followed through memory, a
// round trip each, sixteen one after the other: 4.9 M 48 us, 860 k of 211 slots 15.7 and now 11.9.)  Places in a part come from ballots over the bits of the part's number (as in
// k_table_part): no atomics whose order of arrival would show.
// An item: x the example, y bits 0-10 its lookups (POOL_COUNT_MANY: as many or more), 11 the sign's first lookup, 12-31 the
// key: of the first `spread` distinct indices these themselves, of the extra ones spread + their place among them, of the
// others which of their part's they are behind those.
constexpr uint32_t POOL_COUNT_MANY = 0x7FF;
constexpr uint32_t POOL_FIRST = 0x800;
constexpr uint32_t POOL_KEY_SHIFT = 12;

inline size_t pool_tile_lds(uint32_t parts) { return (size_t)KEY_WAVES * parts * sizeof(uint32_t); }

static __global__ __launch_bounds__(256) void k_lookup_keys(const SlotDesc* __restrict__ descs, const uint32_t* __restrict__ lbase,
                                                     const uint32_t* __restrict__ ubase, uint32_t N,
                                                     const uint32_t* __restrict__ u_of_gi, int64_t batch,
                                                     uint2* __restrict__ pool, uint16_t* __restrict__ poff, PoolShare share,
                                                     const uint32_t* __restrict__ extra, DevStatus* status,
                                                     HostWord compared, uint32_t* host_err) {
    extern __shared__ uint32_t cnt[];  // [parts][KEY_WAVES]
    __shared__ uint32_t more[POOL_EXTRA];
    __shared__ uint32_t wsum[KEY_WAVES];
    __shared__ uint32_t slot;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    compared.tell();
    if (tid == 0) slot = N;
    __syncthreads();
    for (uint32_t s = tid; s < N; s += 256) {
        const uint32_t a = lbase[s], b = lbase[s + 1], t = blockIdx.x - share.first_tile(s, a);  // (wraps before the slot)
        if (t < (b - a + POOL_TILE - 1) / POOL_TILE) slot = s;
    }
    __syncthreads();
    if (slot == N) return;
    const uint32_t sl = slot, l0 = lbase[sl], len = lbase[sl + 1] - l0;
    const uint32_t t0 = (blockIdx.x - share.first_tile(sl, l0)) * POOL_TILE;
    const uint32_t ub = ubase[sl], parts = share.parts(len), spread = share.spread(len);
    const PoolTurn turn(parts);
    const uint32_t bits = parts > 1 ? 32 - (uint32_t)__clz((int)(parts - 1)) : 0u;  // of a part's number
    const uint32_t extras = share.spreads(len) ? extra[sl * (POOL_EXTRA + 1)] : 0u, spread_all = spread + extras;
    const Global<const int64_t> ex = example_of(descs[sl]);
    // the wavefront's lookups, and the 64 on either side of them (places outside the slot: another lookup's, not looked at)
    const uint32_t w0 = t0 + wave * KEY_ITEMS * 64;
    int64_t id[KEY_ITEMS];
    uint32_t u[KEY_ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < KEY_ITEMS; j++) id[j] = ex[min(w0 + j * 64 + lane, len - 1)];
    const int64_t id_before = ex[min(w0 > lane ? w0 - 1 - lane : 0u, len - 1)];
    const int64_t id_behind = ex[min(w0 + KEY_ITEMS * 64 + lane, len - 1)];
#pragma unroll
    for (uint32_t j = 0; j < KEY_ITEMS; j++) u[j] = u_of_gi[l0 + min(w0 + j * 64 + lane, len - 1)];
    for (uint32_t i = tid; i < parts * KEY_WAVES; i += 256) cnt[i] = 0;
    if (tid < extras) more[tid] = extra[sl * (POOL_EXTRA + 1) + 1 + tid];
    __syncthreads();
    // numbered through: the spread indices first, then the others
    if (extras == 0) {
#pragma unroll
        for (uint32_t j = 0; j < KEY_ITEMS; j++) u[j] -= ub;
    } else {
        uint32_t to[KEY_ITEMS];
#pragma unroll
        for (uint32_t j = 0; j < KEY_ITEMS; j++) {
            const uint32_t index = (u[j] & ~FIRST_BIT) - ub;
            to[j] = index < spread ? index : index + extras;
        }
        for (uint32_t e = 0; e < extras; e++) {
            const uint32_t x = more[e] + extras;
#pragma unroll
            for (uint32_t j = 0; j < KEY_ITEMS; j++) to[j] = to[j] == x ? ~(spread + e) : to[j];
        }
#pragma unroll
        for (uint32_t j = 0; j < KEY_ITEMS; j++) u[j] = (u[j] & FIRST_BIT) | ((int)to[j] < 0 ? ~to[j] : to[j]);
    }
    // Example ids in 32 bits from here on: those that do not fit are refused (batch is 2^32 at most).  Where an example starts
    // (the first lookup of a slot does, and what lies behind the last one):
    uint32_t b[KEY_ITEMS];
    unsigned long long heads[KEY_ITEMS];
    bool bad = false;
    uint32_t last = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)id_before);  // of the run before
#pragma unroll
    for (uint32_t j = 0; j < KEY_ITEMS; j++) {
        const uint32_t i = w0 + j * 64 + lane;
        const bool active = i < len;
        b[j] = (uint32_t)id[j];
        uint32_t prev = (uint32_t)__shfl_up((int)b[j], 1);
        if (lane == 0) prev = last;
        last = (uint32_t)__builtin_amdgcn_readlane((int)b[j], 63);
        bad |= active && ((uint64_t)id[j] >= (uint64_t)batch || (i > 0 && prev > b[j]));
        heads[j] = __ballot(!active || i == 0 || b[j] != prev);
    }
    // lookups of a run's last example behind it: as far as the next run's ids go, from the last one on through memory
    uint32_t ahead[KEY_ITEMS];
    ahead[KEY_ITEMS - 1] = 0;
    if (w0 + KEY_ITEMS * 64 < len) {
        unsigned long long other = __ballot(w0 + KEY_ITEMS * 64 + lane >= len || (uint32_t)id_behind != last);
        for (uint32_t e = w0 + KEY_ITEMS * 64; !other; other = __ballot(e + lane >= len || (uint32_t)ex[min(e + lane, len - 1)] != last)) {
            ahead[KEY_ITEMS - 1] += 64;
            e += 64;
        }
        ahead[KEY_ITEMS - 1] += (uint32_t)__ffsll((long long)other) - 1;
    }
#pragma unroll
    for (uint32_t j = KEY_ITEMS - 1; j > 0; j--) ahead[j - 1] = heads[j] ? (uint32_t)__ffsll((long long)heads[j]) - 1 : 64 + ahead[j];
    uint32_t back = 0;  // ... of its first example ahead of it
    if (!(heads[0] & 1ull)) {
        const uint32_t x = (uint32_t)__builtin_amdgcn_readfirstlane((int)b[0]);
        unsigned long long other = __ballot(lane >= w0 || (uint32_t)id_before != x);
        for (uint32_t e = w0; !other; other = __ballot(lane >= e || (uint32_t)ex[e > lane ? e - 1 - lane : 0u] != x)) {  // lookups [0, e) are left
            back += 64;
            e -= 64;
        }
        back += (uint32_t)__ffsll((long long)other) - 1;
    }
    uint32_t count[KEY_ITEMS], at[KEY_ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < KEY_ITEMS; j++) {
        const uint32_t i = w0 + j * 64 + lane;
        const bool active = i < len;
        const unsigned long long below = heads[j] & (~0ull >> (63 - lane)), above = heads[j] & ~(~0ull >> (63 - lane));
        const uint32_t to_start = below ? lane - (63 - (uint32_t)__clzll((long long)below)) : lane + back;
        const uint32_t to_end = above ? (uint32_t)__ffsll((long long)above) - 1 - lane : 64 - lane + ahead[j];
        count[j] = min(to_start + to_end, POOL_COUNT_MANY);
        // the next run's first example, if that is not its own first
        if (j + 1 < KEY_ITEMS && !(heads[j + 1 < KEY_ITEMS ? j + 1 : j] & 1ull)) back = heads[j] ? 1 + (uint32_t)__clzll((long long)heads[j]) : 64 + back;
        // its place among the tile's lookups of its part: behind those of earlier runs and lanes
        const uint32_t index = u[j] & ~FIRST_BIT;
        const uint32_t part = index < spread_all ? turn.part(i >> 6) : turn.part_of(index - spread_all);
        const uint32_t k = part * KEY_WAVES + wave;
        unsigned long long same = __ballot(active);
        for (uint32_t q = 0; q < bits; q++) {
            const unsigned long long m = __ballot((part >> q) & 1u);
            same &= ((part >> q) & 1u) ? m : ~m;
        }
        at[j] = 0;
        if (active) at[j] = cnt[k] + (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
        wave_sync();
        if (active && (uint32_t)__ffsll((long long)same) - 1 == lane) cnt[k] += (uint32_t)__popcll(same);
        wave_sync();
    }
    if (bad) {
        atomicOr(&status->err, DEV_ERR_GRAD_ROWS);
        if (host_err) *host_err = DEV_ERR_GRAD_ROWS;
        status->abort = 1;  // nothing downstream may run
    }
    __syncthreads();
    const uint32_t total = parts * KEY_WAVES, each = (total + 255) / 256;
    uint32_t sum = 0;
    for (uint32_t q = 0; q < each; q++) sum += tid * each + q < total ? cnt[tid * each + q] : 0u;
    uint32_t x = block_excl_scan_256<uint32_t>(sum, wsum, nullptr);
    uint16_t* off = poff + (size_t)blockIdx.x * (share.parts_max + 1);
    for (uint32_t q = 0; q < each; q++) {
        const uint32_t k = tid * each + q;
        if (k >= total) break;
        const uint32_t c = cnt[k];
        cnt[k] = x;
        if (k % KEY_WAVES == 0) off[k / KEY_WAVES] = (uint16_t)x;
        x += c;
    }
    if (tid == 0) off[parts] = (uint16_t)min(POOL_TILE, len - t0);
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < KEY_ITEMS; j++) {
        const uint32_t i = w0 + j * 64 + lane, index = u[j] & ~FIRST_BIT;
        if (i >= len) continue;
        const uint32_t part = index < spread_all ? turn.part(i >> 6) : turn.part_of(index - spread_all);
        const uint32_t key = index < spread_all ? index : spread_all + turn.key_of(index - spread_all);
        pool[l0 + t0 + cnt[part * KEY_WAVES + wave] + at[j]] =
            make_uint2(b[j], count[j] | (u[j] & FIRST_BIT ? POOL_FIRST : 0u) | (key << POOL_KEY_SHIFT));
    }
}

// The lookups of example x in a slot's sorted ids.
__device__ __forceinline__ uint32_t lookups_of(Global<const int64_t> ex, uint32_t n, int64_t x) {
    uint32_t bound[2];
    for (int k = 0; k < 2; k++) {  // the first id >= x, then > x
        uint32_t lo = 0, len = n;
        while (len > 0) {
            const uint32_t half = len / 2;
            if (ex[lo + half] < x + k) {
                lo += half + 1;
                len -= half + 1;
            } else {
                len = half;
            }
        }
        bound[k] = lo;
    }
    return bound[1] - bound[0];
}

// Step 2: the gradient of every distinct sign, a workgroup per part of a slot: the part's items, tile after tile,
// POOL_ITEMS_MAX at a time, sorted and summed in LDS (pool_items).  What a further round has of a sign is added to what the
// round before left; the round that meets a sign's first lookup writes its row.  The sums of the signs that are spread over
// the parts go to the part's own rows of `shares`, `has` tells which there are.  The order of all additions is fixed.
//
// What bounds it is a workgroup's chain (slot, tiles, items; sort; rows; shares), so it wants
// as many workgroups on a CU as there is room for, four.  4.9 M lookups in 100 slots, rows of 16: 148 us, of which the list of a
// part's items takes 39, the sort 35, the sums 50 and writing the rows 20 (each left out in turn), and 134 to 139 since the sort's turns
// follow the items (pool_items); 860 k in 211 slots: 34.
// (A counting sort of the lookups through memory, an ordering pass and a reduction by sign, k_lookup_keys' work included: 390
// for 205 and 103 for 48.)
static_assert(POOL_SPREAD == 64 && POOL_EXTRA <= POOL_SPREAD, "k_reduce_pooled_shares");
template <int LPG, bool ANY>
__global__ __launch_bounds__(POOL_THREADS) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_reduce_pooled(const SlotDesc* __restrict__ descs,
                                                                const uint32_t* __restrict__ lbase,
                                                                const uint32_t* __restrict__ ubase, uint32_t N,
                                                                const uint2* __restrict__ pool,
                                                                const uint16_t* __restrict__ poff, int dim, int D, int combiner,
                                                                const DevStatus* status, float* __restrict__ flat,
                                                                PoolShare share, const uint32_t* __restrict__ extra,
                                                                float* __restrict__ shares, uint64_t* __restrict__ has) {
    __shared__ PoolLds lds;
    __shared__ uint32_t slot;
    __shared__ unsigned long long have[POOL_SHARES / 64], had[POOL_SHARES / 64];  // spread signs with a sum so far, before the round
    // the workgroups of a slot, which read the same rows, on one die (DieShare, an item per workgroup)
    const uint32_t item = blockIdx.x % XCDS * (gridDim.x / XCDS) + blockIdx.x / XCDS;  // (the grid is a multiple of XCDS)
    if (status->abort | status->mismatch) return;
    const uint32_t tid = threadIdx.x;
    if (tid == 0) slot = N;
    if (tid < POOL_SHARES / 64) have[tid] = had[tid] = 0;
    __syncthreads();
    for (uint32_t s = tid; s < N; s += POOL_THREADS) {
        const uint32_t a = lbase[s], b = lbase[s + 1], q = item - share.first_part(s, a);  // (wraps before the slot)
        if (b > a && q < share.parts(b - a)) slot = s;
    }
    __syncthreads();
    if (slot == N) return;
    const uint32_t sl = slot, l0 = lbase[sl], len = lbase[sl + 1] - l0, ub = ubase[sl], us = ubase[sl + 1] - ub;
    const PoolTurn turn(share.parts(len));
    const uint32_t part = item - share.first_part(sl, l0), tile0 = share.first_tile(sl, l0);
    const uint32_t spread = share.spread(len), spread_all = spread + (share.spreads(len) ? extra[sl * (POOL_EXTRA + 1)] : 0u);
    if (!spread_all && part << POOL_ROWS_LOG2 >= us) return;
    const uint32_t rest = ub + spread + (part << POOL_ROWS_LOG2);  // the part's first row of an index that is not spread
    const uint32_t top = us > spread ? spread_all + turn.key_of(us - 1 - spread) + POOL_ROWS : us - 1, bits = top ? 32 - (uint32_t)__clz((int)top) : 0u;
    const float* pooled = descs[sl].grads;
    const Global<const int64_t> ex = example_of(descs[sl]);
    const uint32_t mine = (len + POOL_TILE - 1) / POOL_TILE;
    uint32_t* const before = lds.list;                   // [POOL_THREADS + 1]: items of my part in the tiles before
    uint32_t* const start = before + POOL_THREADS + 1;   // [POOL_THREADS]: where they are in a tile
    for (uint32_t g0 = 0; g0 < mine; g0 += POOL_THREADS) {  // tiles, as many at a time as there are threads
        uint32_t total = 1;
        for (uint32_t done = 0; done < total; done += POOL_ITEMS_MAX) {
            {  // (again in a further round: the sums of the one before took the list's place)
                uint32_t c = 0, lo = 0;
                if (g0 + tid < mine) {
                    const uint16_t* off = poff + (size_t)(tile0 + g0 + tid) * (share.parts_max + 1) + part;
                    lo = off[0];
                    c = off[1] - lo;
                }
                const uint32_t x = block_excl_scan<uint32_t, POOL_WAVES>(c, lds.wsum, &total);
                before[tid] = x;
                start[tid] = (g0 + tid) * POOL_TILE + lo;
                if (tid == 0) before[POOL_THREADS] = total;
            }
            __syncthreads();
            const uint32_t n = min(POOL_ITEMS_MAX, total - done);  // (total < done: a part without items here, no round)
#pragma unroll
            for (uint32_t j = 0; j < POOL_ITEMS; j++) {
                const uint32_t i = j * POOL_THREADS + tid;
                if (i < n && done < total) {
                    const uint32_t t = (uint32_t)find_slot(before, (int)min(mine - g0, (uint32_t)POOL_THREADS), done + i);
                    const uint2 v = pool[l0 + start[t] + (done + i - before[t])];
                    uint32_t count = v.y & POOL_COUNT_MANY;
                    if (combiner != COMBINE_SUM && count == POOL_COUNT_MANY) count = lookups_of(ex, len, (int64_t)v.x);
                    const float scale = pool_scale((float)count, combiner);
                    lds.key[i] = v.y >> POOL_KEY_SHIFT;
                    lds.example[i] = v.x;
                    lds.scale[i] = v.y & POOL_FIRST ? scale : -scale;
                }
            }
            if (done < total)
                pool_items<LPG, ANY>(lds, n, bits, pooled, dim, D, [&](uint32_t key, bool first, bool& add) {
                    if (key < spread_all) {
                        add = ((had[key / 64] >> (key % 64)) & 1ull) != 0;
                        atomicOr(&have[key / 64], 1ull << (key % 64));
                        return shares + ((uint64_t)item * POOL_SHARES + key) * dim;
                    }
                    add = !first;
                    return flat + (uint64_t)(rest + turn.index_of(key - spread_all)) * dim;
                });
            else
                __syncthreads();
            if (spread_all) {
                if (tid < POOL_SHARES / 64) had[tid] = have[tid];
                __syncthreads();
            }
        }
    }
    if (spread_all && tid < POOL_SHARES / 64) has[(uint64_t)item * (POOL_SHARES / 64) + tid] = have[tid];
}

// The sums of the spread signs, a wavefront per sign.
template <int LPG, bool ANY>
__global__ __launch_bounds__(256) void k_reduce_pooled_shares(const uint32_t* __restrict__ lbase,
                                                              const uint32_t* __restrict__ ubase, int dim, int D,
                                                              const DevStatus* status, const float* __restrict__ shares,
                                                              const uint64_t* __restrict__ has, float* __restrict__ flat,
                                                              PoolShare share, const uint32_t* __restrict__ extra) {
    if (status->abort | status->mismatch) return;
    constexpr uint32_t PER = 256 / 64;
    const uint32_t sl = blockIdx.x / (POOL_SPREAD / PER), key0 = blockIdx.x % (POOL_SPREAD / PER) * PER + threadIdx.x / 64;
    const uint32_t l0 = lbase[sl], len = lbase[sl + 1] - l0, ub = ubase[sl], us = ubase[sl + 1] - ub;
    const uint32_t p0 = share.first_part(sl, l0);
    if (len == 0 || !share.spreads(len)) return;
    const uint32_t* const more = extra + sl * (POOL_EXTRA + 1);
    const uint32_t spread = share.spread(len), spread_all = spread + more[0];
    for (uint32_t key = key0; key < spread_all; key += POOL_SPREAD) {  // (the same for a whole wavefront)
        const uint32_t index = key < spread ? key : more[1 + key - spread];
        if (index >= us) return;
        add_shares<LPG, ANY>(
            share.parts(len), D,
            [&](uint32_t q) { return ((has[(uint64_t)(p0 + q) * (POOL_SHARES / 64) + key / 64] >> (key % 64)) & 1ull) != 0; },
            [&](uint32_t q) { return shares + ((uint64_t)(p0 + q) * POOL_SHARES + key) * dim; },
            flat + (uint64_t)(ub + index) * dim);
    }
}

}  // namespace tn

#endif  // TN_COMBINE_KERNELS_H_
