// Pull and push of a small batch (slots of a few thousand lookups at most) in few launches.  A batch of a few
// thousand lookups spends its time in dependent launches (2 to 3 us each, whatever the kernel does) and in the round
// trips inside them, so here
//
//   pull  k_small_slots          per slot and share of its signs: first occurrences in LDS (sparse_table_ops.cc:115-137),
//                                lookup-or-insert of every distinct sign (sparse_table.cc:52-66), its record filed by
//                                bucket; every workgroup reports to the host, which returns when it has them all
//         k_small_group_finish   ranks of the first occurrences -> mapped ids, rows into the variables
//                                (sparse_table_ops.cc:244-265); beside it, per bucket: the groups of equal signs over all
//                                slots, their records in slot order
//   push  k_small_verify         comparison with the plan's signs, click sums; beside it the ranks into the records
//         k_small_pool           (pooled gradients) the gradient of every distinct sign from those of its examples; with
//                                heavy signs k_small_pool_shares, which adds up what a slot's workgroups have of them
//         k_small_apply          per bucket: every sign's records in order (tells the host that the comparison is complete)
//
// Workgroups of one launch never wait for each other, and none needs another's results: what needs them runs in the
// next launch.  The host waits for the first launch of a pull and the first of a push only; the launches behind those
// run while it prepares the next call.
#ifndef TN_SMALL_BATCH_H_
#define TN_SMALL_BATCH_H_

#include "pool_items.h"
#include "remap_lds.h"

#include <algorithm>

namespace tn {

constexpr int SMALL_SLOT_MAX = 8192;         // lookups of a slot at most
constexpr int SMALL_SLOT_SHORT = 4096;       // ... that a workgroup of SMALL_THREADS holds in registers
constexpr int SMALL_SLOT_BITS = 13;          // a position in a slot, its rank, its occurrences fit in 13, 13 and 14 bits
constexpr int SMALL_SLOTS = 512;             // slots at most (the LDS of small_emit_bucket: 300 slots of 2912 lookups, 512 of 576)
constexpr int SMALL_PARTS_MAX = 16;          // workgroups of k_small_slots per slot at most
constexpr int SMALL_SEGMENTS = 256;          // ... and for all slots together where a slot has more than one
constexpr int SMALL_WORKGROUPS = SMALL_SLOTS > SMALL_SEGMENTS ? SMALL_SLOTS : SMALL_SEGMENTS;  // of k_small_slots at most
constexpr int SMALL_PART_LOOKUPS = 128;      // lookups of a slot per workgroup aimed at
constexpr int SMALL_BUCKET_RECORDS = 64;     // records per bucket aimed at (if every lookup were distinct)
constexpr int SMALL_BUCKETS_MAX = 2048;
// Larger batches: as many buckets as the chip holds workgroups of k_small_apply at once, four on a CU, then one for so many
// lookups.  (Two thousand of 64 lookups each are two rounds of workgroups and twice the heads, scans and slots to go through.)
// Push and pull, sum of the kernels, us, up to 2048 buckets of 64 lookups and so: 26 slots of 4096, Adam rows of 16 43.0 and 40.2
// (768 of them 41.7); AdaGrad rows of 16 80 of 2000 54.0 and 50.2, 40 of 4000 50.8 and 48.1, 12 of 8000 46.6 and 44.5; rows of 64 80
// of 2000 74.5 and 71.4; 30 of 8000, Adam rows of 16 55.9 and 53.2 (one for 256 52.0); 47 of 6400, rows of 8 + 2 65.5 and 63.2 (65.8);
// 40 of 8192, rows of 64, one for 160 183.2, 192 189.  Not a few more than the chip holds: 1032 instead of 1020, 20 slots of 6500, rows
// of 64, k_small_apply 30.2 and 28.3.
// Rows of more than 32 elements: only as few as leave a CU as many workgroups of k_small_pull_rest, most of which copy rows then
// (small_rest_held).  With five to a CU instead of eight: 24 slots of 8192, AdaGrad rows of 64 22.7 us and 18.3, 20 of 8192 under Adam
// 19.8 and 17.0; shorter rows gain more by fewer buckets.
// Batches whose signs are nearly all in most slots lose: 10 000 ids in 20 slots of 8192, Adam rows of 1 44.7 and 47.0, the signs with
// many records having half as many wavefronts.
constexpr size_t SMALL_BUCKETS_FEW = 1024;
constexpr size_t small_bucket_lookups(int dim) { return dim > 32 ? 160 : 192; }
constexpr int SMALL_THREADS = 512;           // k_small_slots; twice as many for slots of more than SMALL_SLOT_SHORT lookups
constexpr int SMALL_ITEMS = SMALL_SLOT_SHORT / SMALL_THREADS;
constexpr int SMALL_WORDS = SMALL_SLOT_MAX / 64;  // 64-lookup words of a slot
constexpr uint32_t SMALL_HEAVY_MAX = SMALL_SLOT_MAX / HEAVY_LOOKUPS;  // heavy signs of a slot at most
constexpr uint32_t SMALL_NONE = 0xFFFFu;     // no position
constexpr int SMALL_NEW = 512;               // rows a workgroup of k_small_slots lists to fill them with all its threads
constexpr int FINISH_THREADS = 256;          // k_small_group_finish
constexpr int SMALL_TILE = 1024;             // lookups per workgroup of k_small_verify
static_assert(SMALL_SLOT_MAX <= (1 << SMALL_SLOT_BITS) && SMALL_SLOT_MAX == 2 * SMALL_SLOT_SHORT, "positions fit");

// How a small batch is laid out: worked out by the pull, kept with its plan.
struct SmallShape {
    int N;
    uint32_t L, max_len;
    uint32_t parts;    // workgroups of k_small_slots per slot, each with a share of the signs (by hash range)
    uint32_t nbp;      // buckets per part: parts * nbp buckets in all, a bucket's signs all lie in one part
    uint32_t words;    // 64-lookup words of the longest slot
    uint32_t cap;      // room of a bucket, in records
    __host__ __device__ uint32_t buckets() const { return parts * nbp; }
};

// The plan of a small batch.  Lookups are numbered through the slots (gi); a distinct sign of a slot is known by its
// first lookup.
struct SmallPlan {
    SlotDesc* descs;       // the slots' tensors (pull)
    SlotDesc* push_descs;  // ... (push)
    uint64_t* vals_copy;   // sign of every lookup
    uint16_t* first_of;    // position in its slot of the first lookup with the same sign
    uint32_t* row_at;      // first lookups: table row of the sign
    uint16_t* rank_at;     // first lookups: rank among the slot's first lookups
    int32_t* click_at;     // first lookups: sum of the labels (a push adds them, the updates take them back to zero)
    uint64_t* bits;        // [slot][part][words]: first lookups found by the part's workgroup
    uint2* recs;           // records {row, position | occurrences << 13} of slot s, part p from parts * lbase(s) + p * len(s) on, by bucket
    uint16_t* boff;        // [slot][part][nbp + 1]: where the buckets start in them
    uint4* head;           // per bucket {signs with one record, with a few, with many, records of the latter two}
    uint2* group;          // per bucket, `cap` each: {row, first record | records << 16}; those with many records from the end on
    uint4* member;         // per bucket, `cap` each: records {gi, rank | slot << 16, occurrences, 0}, those of a sign in slot
                           // order (the rank comes in with a push, k_small_verify)
    uint16_t* heavy;       // [slot][part][SMALL_HEAVY_MAX]: first lookups of the heavy signs (HEAVY_LOOKUPS), then SMALL_NONE
    uint32_t* bad;         // != 0: a bucket did not fit, a push has to analyse the batch itself
};

__device__ __forceinline__ void host_store(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// What a workgroup of k_small_slots tells the host, in one word: its distinct signs, the rows it inserted, whether the
// table is full, whether it has a heavy sign, and the number of the call, which says that the word is this call's.
constexpr int SMALL_REPORT_BITS = 14;
__host__ __device__ inline uint64_t small_report(uint32_t n_first, uint32_t n_new, bool full, bool heavy, uint32_t seq) {
    return (uint64_t)n_first | ((uint64_t)n_new << SMALL_REPORT_BITS) | ((uint64_t)(full ? 1 : 0) << (2 * SMALL_REPORT_BITS)) |
           ((uint64_t)(heavy ? 2 : 0) << (2 * SMALL_REPORT_BITS)) | ((uint64_t)seq << 32);
}

// Entries of the LDS table of k_small_slots: room for a slot of distinct signs that all fall into one part, and two
// per lookup expected.
inline uint32_t small_entries(uint32_t max_len, uint32_t parts) {
    const uint32_t expected = 2 * ((max_len + parts - 1) / parts) + 64;
    return expected > max_len + 64 ? expected : max_len + 64;
}
inline size_t small_slots_lds(uint32_t entries, uint32_t max_len, uint32_t nbp) {
    // keys and words (entry `entries`: the sign EMPTY_KEY), bucket counters, list of the entries in use
    return ((size_t)entries + 1) * 12 + (size_t)(nbp + 1) * 4 + align_up((size_t)max_len * 2, 8);
}

// First launch of a small pull: `parts` workgroups per slot.  Each of them reads all signs of the slot and keeps those
// of its hash range: the shares of a slot need nothing of each other (workgroups that each worked out the whole slot
// and then took a share of the probes repeated the slot's remap up to eight times).  What bounds it is a chain of
// round trips -- descriptor, signs, probe, second probe -- and a CU's rate of random 64-byte reads (0.2 per ns), hence
// many workgroups with about a hundred signs each.
// The descriptor of slot `sl` for the whole workgroup, into LDS, and with `keep` into the plan, for the launches after this one:
// what is to be done before and after the workgroup clears its LDS, while a descriptor in the host's buffer is on its way.
struct DescFetch {
    uint32_t word = 0;
    __device__ __forceinline__ void start(const ArgDescs&, int) {}
    __device__ __forceinline__ void start(const HostDescs& d, int sl) {
        if (threadIdx.x < sizeof(SlotDesc) / 4) word = reinterpret_cast<const uint32_t*>(d.slot + sl)[threadIdx.x];
    }
    __device__ __forceinline__ void finish(const ArgDescs& d, int sl, SlotDesc& sd, SlotDesc* keep) const {
        if (threadIdx.x != 0) return;
        sd = d.slot[sl];
        if (keep) *keep = d.slot[sl];
    }
    __device__ __forceinline__ void finish(const HostDescs&, int, SlotDesc& sd, SlotDesc* keep) const {
        if (threadIdx.x >= sizeof(SlotDesc) / 4) return;
        reinterpret_cast<uint32_t*>(&sd)[threadIdx.x] = word;
        if (keep) reinterpret_cast<uint32_t*>(keep)[threadIdx.x] = word;
    }
};

template <int THREADS, typename Descs>
__device__ __forceinline__ void small_slots(const SmallShape& b, const SmallPlan& p, const Descs& descs, uint32_t entries,
                                            const Store& s, const OptDev& o, uint64_t seed, DevStatus* status,
                                            uint64_t* host_words, uint32_t seq) {
    extern __shared__ unsigned long long smem64[];
    unsigned long long* keys = smem64;
    uint32_t* word = reinterpret_cast<uint32_t*>(keys + entries + 1);  // bits 16-31 smallest position, 0-15 occurrences
    uint32_t* hist = word + entries + 1;                              // [nbp + 1]
    uint16_t* used = reinterpret_cast<uint16_t*>(hist + b.nbp + 1);   // [max_len]: the entries in use
    __shared__ SlotDesc sd;
    __shared__ unsigned long long bits[SMALL_WORDS];
    __shared__ uint32_t wsum[THREADS / 64];
    __shared__ uint32_t sh_first, sh_new, sh_full, sh_heavy;
    __shared__ uint16_t heavy[SMALL_HEAVY_MAX];
    __shared__ uint32_t new_row[SMALL_NEW];
    __shared__ uint16_t new_ent[SMALL_NEW];
    const int sl = blockIdx.x / b.parts;
    const uint32_t part = blockIdx.x % b.parts;
    const uint32_t tid = threadIdx.x;
    DescFetch fetch;
    fetch.start(descs, sl);
    for (uint32_t i = tid; i <= entries; i += THREADS) {
        keys[i] = EMPTY_KEY;
        word[i] = 0xFFFF0000u;
    }
    for (uint32_t i = tid; i <= b.nbp; i += THREADS) hist[i] = 0;
    for (uint32_t i = tid; i < SMALL_WORDS; i += THREADS) bits[i] = 0;
    if (tid == 0) sh_first = sh_new = sh_full = sh_heavy = 0;
    if (tid < SMALL_HEAVY_MAX) heavy[tid] = SMALL_NONE;
    if (blockIdx.x == 0) {
        if (tid < sizeof(DevStatus) / 4) reinterpret_cast<uint32_t*>(status)[tid] = 0;
        if (tid == 0) *p.bad = 0;
    }
    fetch.finish(descs, sl, sd, part == 0 ? p.descs + sl : nullptr);
    __syncthreads();
    const Global<const int64_t> values = as_global(sd.values);
    const uint32_t len = sd.len, lbase = sd.lbase;
    uint64_t sg[SMALL_ITEMS];
#pragma unroll
    for (int j = 0; j < SMALL_ITEMS; j++) {
        const uint32_t pos = j * THREADS + tid;
        sg[j] = pos < len ? (uint64_t)values[pos] : 0;
    }
    // the lookups of my share: entry of the sign, smallest position
    uint32_t ent[SMALL_ITEMS];
#pragma unroll
    for (int j = 0; j < SMALL_ITEMS; j++) {
        const uint32_t pos = j * THREADS + tid;
        ent[j] = 0xFFFFFFFFu;
        if (pos >= len) continue;
        if (part == 0) p.vals_copy[lbase + pos] = sg[j];
        const uint64_t h = mix64(sg[j]);
        if (scale32((uint32_t)(h >> 32), b.parts) != part) continue;
        uint32_t e = entries;
        if (sg[j] != EMPTY_KEY) {
            e = scale32((uint32_t)h, entries);
            for (;;) {  // more entries than lookups: a free one exists
                unsigned long long old = keys[e];
                if (old == EMPTY_KEY) old = atomicCAS(&keys[e], (unsigned long long)EMPTY_KEY, sg[j]);
                if (old == EMPTY_KEY || old == sg[j]) break;
                e = e + 1 == entries ? 0 : e + 1;
            }
        }
        atomicMin(&word[e], pos << 16);
        ent[j] = e;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < SMALL_ITEMS; j++) {
        if (ent[j] == 0xFFFFFFFFu) continue;
        const uint32_t pos = j * THREADS + tid;
        const uint32_t f = atomicAdd(&word[ent[j]], 1u) >> 16;
        p.first_of[lbase + pos] = (uint16_t)f;
        if (f == pos) {
            atomicOr(&bits[pos >> 6], 1ull << (pos & 63));
            used[atomicAdd(&sh_first, 1u)] = (uint16_t)ent[j];
        }
    }
    __syncthreads();
    // A thread per distinct sign (a slot that is all one part's may have more of them than the workgroup has threads):
    // lookup-or-insert in the table (optimizer_kernel.h:299-308), place in its bucket.  The rows it inserts are listed
    // and filled by all threads: one lane of a wavefront drawing the normal deviates of a row would hold up the others.
    const uint32_t n_first = sh_first;
    uint32_t row[SMALL_ITEMS], place[SMALL_ITEMS], bk[SMALL_ITEMS];
#pragma unroll
    for (int r = 0; r < SMALL_ITEMS; r++) {
        const uint32_t i = r * THREADS + tid;
        row[r] = NO_ROW;
        place[r] = bk[r] = 0;
        if (i < n_first) {
            const uint32_t e = used[i];
            const uint64_t sign = (uint64_t)keys[e];
            const uint32_t w = word[e];
            if ((w & 0xFFFFu) >= HEAVY_LOOKUPS) heavy[atomicAdd(&sh_heavy, 1u)] = (uint16_t)(w >> 16);
            bool is_new = false;
            row[r] = probe_slot<true>(s, sign, is_new);
            if (is_new) {
                const uint32_t k = atomicAdd(&sh_new, 1u);
                if (k < (uint32_t)SMALL_NEW) {
                    new_row[k] = row[r];
                    new_ent[k] = (uint16_t)e;
                } else {
                    init_row(s, o, seed, sign, row[r]);
                }
            }
            if (row[r] == NO_ROW) sh_full = 1;
            bk[r] = scale32((uint32_t)(mix64(sign) >> 32), b.buckets()) - part * b.nbp;
            place[r] = atomicAdd(&hist[bk[r]], 1u);
        }
    }
    __syncthreads();
    if (tid == 0) {
        __hip_atomic_store(reinterpret_cast<unsigned long long*>(host_words + blockIdx.x),
                           (unsigned long long)small_report(n_first, sh_new, sh_full != 0, sh_heavy != 0, seq), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
        if (sh_new) atomicAdd(s.count, (unsigned long long)sh_new);
    }
    // where the buckets start among the part's records
    uint32_t at = 0;
    for (uint32_t i0 = 0; i0 < b.nbp; i0 += THREADS) {
        const uint32_t c = i0 + tid < b.nbp ? hist[i0 + tid] : 0u;
        uint32_t total;
        const uint32_t x = at + block_excl_scan<uint32_t, THREADS / 64>(c, wsum, &total);
        if (i0 + tid < b.nbp) {
            hist[i0 + tid] = x;
            p.boff[(size_t)blockIdx.x * (b.nbp + 1) + i0 + tid] = (uint16_t)x;
        }
        at += total;
    }
    if (tid == 0) p.boff[(size_t)blockIdx.x * (b.nbp + 1) + b.nbp] = (uint16_t)at;
    if (tid < SMALL_HEAVY_MAX) p.heavy[blockIdx.x * SMALL_HEAVY_MAX + tid] = heavy[tid];
    __syncthreads();
    const uint32_t rbase = b.parts * lbase + part * len;
#pragma unroll
    for (int r = 0; r < SMALL_ITEMS; r++) {
        const uint32_t i = r * THREADS + tid;
        if (i < n_first) {
            const uint32_t w = word[used[i]], pos = w >> 16, cnt = w & 0xFFFFu;
            // batch_show = occurrences (sparse_table_ops.cc:290-293)
            p.recs[rbase + hist[bk[r]] + place[r]] = make_uint2(row[r], pos | (cnt << SMALL_SLOT_BITS));
            p.row_at[lbase + pos] = row[r];
            p.click_at[lbase + pos] = 0;
        }
    }
    for (uint32_t i = tid; i < b.words; i += THREADS) p.bits[(size_t)blockIdx.x * b.words + i] = bits[i];
    if (sh_new) {
        const uint32_t pairs = (uint32_t)(s.D + 1) / 2, work = min(sh_new, (uint32_t)SMALL_NEW) * pairs;
        const float stddev = (float)(1.0 / sqrt((double)s.D));
        for (uint32_t q = tid; q < work; q += THREADS) {
            const uint32_t k = q / pairs;
            init_row_pair(s, o, seed, (uint64_t)keys[new_ent[k]], new_row[k], q - k * pairs, stddev);
        }
    }
}

template <typename Descs>
__global__ __launch_bounds__(SMALL_THREADS) void k_small_slots(SmallShape b, SmallPlan p, Descs descs, uint32_t entries, Store s,
                                                                    OptDev o, uint64_t seed, DevStatus* status,
                                                                    uint64_t* host_words, uint32_t seq) {
    small_slots<SMALL_THREADS>(b, p, descs, entries, s, o, seed, status, host_words, seq);
}
template <typename Descs>
__global__ __launch_bounds__(2 * SMALL_THREADS) void k_small_slots_long(SmallShape b, SmallPlan p, Descs descs,
                                                                             uint32_t entries, Store s, OptDev o, uint64_t seed,
                                                                             DevStatus* status, uint64_t* host_words,
                                                                             uint32_t seq) {
    small_slots<2 * SMALL_THREADS>(b, p, descs, entries, s, o, seed, status, host_words, seq);
}

// What is left of a small pull behind its first launch: small_emit_bucket, a workgroup per bucket, and small_finish.
// Neither needs what the other works out.
template <>
struct EmitArgs<true> {
    static constexpr int THREADS = FINISH_THREADS;
    SmallShape b;
    SmallPlan p;
    uint32_t table;  // entries of the LDS hash table of rows at most: a power of two, 5/4 of the room of a bucket
    uint32_t big_k;
};
inline uint32_t small_emit_table(uint32_t cap) {
    uint32_t n = 64;
    while (n < cap + cap / 4) n *= 2;
    return n;
}
inline size_t small_emit_lds(int N, uint32_t cap, uint32_t table) {
    // per slot: records before it, where its records are, its first lookup; table: row, records / number;
    // per record: row, gi, occurrences | entry, arrival, slot, list
    return align_up((size_t)(N + 1) * 4 + (size_t)N * 8 + (size_t)table * 12 + (size_t)cap * 20, 8);
}

// Workgroups of k_small_pull_rest on a CU, of the eight that its registers let there be: all of them are given the buckets' LDS.
inline uint32_t small_rest_held(size_t emit_lds) {
    constexpr size_t own = (FINISH_THREADS / 64 + 1) * SMALL_WORDS * 8 + SMALL_WORDS * 4 + 64;  // (small_finish, the counters)
    return (uint32_t)std::min<size_t>(8, 160 * 1024 / (emit_lds + own));
}

// The records of a bucket, slot after slot, grouped by row in LDS.
__device__ __forceinline__ void small_emit_bucket(const EmitArgs<true>& a, uint32_t* lds) {
    const SmallShape& b = a.b;
    const SmallPlan& p = a.p;
    const uint32_t N = (uint32_t)b.N;
    uint32_t* spre = lds;                    // [N + 1]
    uint32_t* sstart = spre + N + 1;         // [N]
    uint32_t* slb = sstart + N;              // [N]
    uint32_t* trow = slb + N;                // [table]
    uint32_t* tcnt = trow + a.table;         // [table]
    uint32_t* tinfo = tcnt + a.table;        // [table]: number of the group | first record << 16 (several records)
    uint32_t* rrow = tinfo + a.table;        // [cap]
    uint32_t* rgi = rrow + b.cap;            // [cap]
    uint32_t* rce = rgi + b.cap;             // [cap]: occurrences (14 bits) | entry << 14
    uint32_t* rarr = rce + b.cap;            // [cap]
    uint16_t* rsl = reinterpret_cast<uint16_t*>(rarr + b.cap);  // [cap]
    uint16_t* list = rsl + b.cap;            // [cap]
    __shared__ uint32_t wsum[FINISH_THREADS / 64];
    __shared__ uint32_t n1, nm, nbig, nmem;
    const uint32_t tid = threadIdx.x, c = blockIdx.x, part = c / b.nbp, cl = c % b.nbp;
    if (tid == 0) n1 = nm = nbig = nmem = 0;
    uint32_t m = 0;
    for (uint32_t s0 = 0; s0 < N; s0 += FINISH_THREADS) {
        const uint32_t sl = s0 + tid;
        uint32_t cnt = 0;
        if (sl < N) {
            const uint32_t len = p.descs[sl].len, lbase = p.descs[sl].lbase;
            const uint16_t* off = p.boff + (size_t)(sl * b.parts + part) * (b.nbp + 1) + cl;
            const uint32_t lo = off[0];
            cnt = off[1] - lo;
            sstart[sl] = b.parts * lbase + part * len + lo;
            slb[sl] = lbase;
        }
        uint32_t total;
        const uint32_t x = m + block_excl_scan<uint32_t, FINISH_THREADS / 64>(cnt, wsum, &total);
        if (sl < N) spre[sl] = x;
        m += total;
    }
    if (tid == 0) spre[N] = m;
    if (m > b.cap) {  // more records of few signs than a bucket has room for: a push analyses the batch itself
        if (tid == 0) {
            *p.bad = 1;
            p.head[c] = make_uint4(0, 0, 0, 0);
        }
        return;
    }
    // Of the records there are: half of the entries stay free where the room for the table lets them (with a fifth, 90 to 102 signs in
    // 128 entries, the longest way through it took the launch 14 us of distinct signs in 20 slots of 5500, rows of 8; so 7.7).
    uint32_t table = 64;
    while (table < 2 * m && table < a.table) table *= 2;
    for (uint32_t i = tid; i < table; i += FINISH_THREADS) {
        trow[i] = NO_ROW;
        tcnt[i] = 0;
    }
    __syncthreads();
    for (uint32_t i = tid; i < m; i += FINISH_THREADS) {
        const uint32_t sl = (uint32_t)find_slot(spre, (int)N, i);
        const uint2 r = p.recs[sstart[sl] + i - spre[sl]];
        const uint32_t gi = slb[sl] + (r.y & ((1u << SMALL_SLOT_BITS) - 1u));
        uint32_t e = 0;
        if (r.x != NO_ROW) {  // (a sign the table had no room for: nothing to update)
            e = (r.x * 2654435761u >> 12) & (table - 1);
            for (;;) {  // more entries than records
                uint32_t old = trow[e];
                if (old == NO_ROW) old = atomicCAS(&trow[e], NO_ROW, r.x);
                if (old == NO_ROW || old == r.x) break;
                e = (e + 1) & (table - 1);
            }
            rarr[i] = atomicAdd(&tcnt[e], 1u);
        }
        rrow[i] = r.x;
        rgi[i] = gi;
        rsl[i] = (uint16_t)sl;
        rce[i] = (r.y >> SMALL_SLOT_BITS) | (e << 14);
    }
    __syncthreads();
    const size_t first = (size_t)c * b.cap;
    // signs with one record: numbered and written at once; with several: a number and a stretch of the records for each
    for (uint32_t i = tid; i < m; i += FINISH_THREADS) {
        if (rrow[i] == NO_ROW) continue;
        const uint32_t e = rce[i] >> 14, k = tcnt[e];
        if (k == 1) {
            const uint32_t g = atomicAdd(&n1, 1u);
            p.group[first + g] = make_uint2(rrow[i], g | (1u << 16));
            p.member[first + g] = make_uint4(rgi[i], (uint32_t)rsl[i] << 16, rce[i] & 0x3FFFu, 0u);
        } else if (rarr[i] == 0) {
            tinfo[e] = atomicAdd(is_big(k, a.big_k) ? &nbig : &nm, 1u) | (atomicAdd(&nmem, k) << 16);
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < m; i += FINISH_THREADS) {
        if (rrow[i] == NO_ROW) continue;
        const uint32_t e = rce[i] >> 14, k = tcnt[e];
        if (k > 1) list[(tinfo[e] >> 16) + rarr[i]] = (uint16_t)i;
    }
    __syncthreads();
    for (uint32_t i = tid; i < m; i += FINISH_THREADS) {
        if (rrow[i] == NO_ROW) continue;
        const uint32_t e = rce[i] >> 14, k = tcnt[e];
        if (k == 1) continue;
        const uint32_t at = tinfo[e] >> 16;
        uint32_t place = 0;  // records of the sign in earlier slots
        for (uint32_t j = 0; j < k; j += 8) {  // eight reads in flight (300 slots of 300 lookups: 110 us a step one by one, 97 so)
            uint32_t v[8];
#pragma unroll
            for (uint32_t q = 0; q < 8; q++) v[q] = list[at + min(j + q, k - 1)];
#pragma unroll
            for (uint32_t q = 0; q < 8; q++) place += j + q < k && v[q] < i ? 1u : 0u;
        }
        p.member[first + n1 + at + place] = make_uint4(rgi[i], (uint32_t)rsl[i] << 16, rce[i] & 0x3FFFu, 0u);
        if (rarr[i] == 0) {
            const uint32_t g = tinfo[e] & 0xFFFFu;
            p.group[first + (is_big(k, a.big_k) ? b.cap - 1 - g : n1 + g)] = make_uint2(rrow[i], (n1 + at) | (k << 16));
        }
    }
    if (tid == 0) p.head[c] = make_uint4(n1, nm, nbig, nmem);
}

// Mapped ids (rank of the sign's first lookup) and, for the first lookups, the table row into the variable: a run of `per`
// positions of one slot, a thread per position and part of a row (VEC elements), FINISH_ITEMS of them at most.  Rows of an even
// length go in pairs where they cannot go in fours: 282 k lookups of 47 slots, rows of 8 + 2, 24.0 -> 18.4 us.
// (k_gather_vars moves 240 k such rows in the same time either way.)
constexpr int FINISH_ITEMS = 2;
template <int VEC>
struct FinishPart {
    typedef float type __attribute__((ext_vector_type(VEC)));
};
template <>
struct FinishPart<1> {
    typedef float type;
};
template <int VEC>
__device__ __forceinline__ void small_finish(const SmallShape& b, const SmallPlan& p, uint32_t block, uint32_t chunks,
                                             uint32_t per, const Store& s) {
    using Part = typename FinishPart<VEC>::type;
    constexpr uint32_t WAVES = FINISH_THREADS / 64;
    __shared__ unsigned long long part_bits[WAVES][SMALL_WORDS];
    __shared__ unsigned long long bits[SMALL_WORDS];
    __shared__ uint32_t before[SMALL_WORDS];
    const uint32_t sl = block / chunks;
    const uint32_t C = (uint32_t)(s.wdim / VEC);
    const uint32_t p0 = (block % chunks) * per;
    const SlotDesc d = p.descs[sl];
    if (p0 >= d.len) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, todo = min(per, d.len - p0) * C;
    uint32_t pos[FINISH_ITEMS], c[FINISH_ITEMS], f[FINISH_ITEMS], row[FINISH_ITEMS];
#pragma unroll
    for (int j = 0; j < FINISH_ITEMS; j++) {
        const uint32_t q = j * FINISH_THREADS + tid;
        pos[j] = p0 + q / C;
        c[j] = q % C;
        f[j] = q < todo ? p.first_of[d.lbase + pos[j]] : NO_ROW;
        row[j] = q < todo ? p.row_at[d.lbase + pos[j]] : NO_ROW;  // (of a first lookup only)
    }
    // the parts' first lookups: a wavefront takes every WAVES-th part, then one puts them together
    constexpr uint32_t RUNS = SMALL_WORDS / 64;
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) {
        const uint64_t* w = p.bits + (size_t)sl * b.parts * b.words + r * 64 + lane;
        uint64_t v[SMALL_PARTS_MAX / WAVES];
#pragma unroll
        for (uint32_t k = 0; k < SMALL_PARTS_MAX / WAVES; k++) {
            const uint32_t q = k * WAVES + wave;
            v[k] = q < b.parts && r * 64 + lane < b.words ? w[(size_t)q * b.words] : 0ull;
        }
        uint64_t all = 0;
#pragma unroll
        for (uint32_t k = 0; k < SMALL_PARTS_MAX / WAVES; k++) all |= v[k];
        part_bits[wave][r * 64 + lane] = all;
    }
    Part v[FINISH_ITEMS];
#pragma unroll
    for (int j = 0; j < FINISH_ITEMS; j++) {
        // (NO_ROW, the table is full: never address the table with it)
        if (f[j] != pos[j] || row[j] > s.cap) row[j] = NO_ROW;
        v[j] = Part{};
        if (row[j] != NO_ROW) v[j] = *reinterpret_cast<const Part*>(s.w + (uint64_t)row[j] * s.wstride + c[j] * VEC);
    }
    __syncthreads();
    if (wave == 0) {
        uint32_t done = 0;
#pragma unroll
        for (uint32_t r = 0; r < RUNS; r++) {
            unsigned long long v = 0;
            for (uint32_t q = 0; q < WAVES; q++) v |= part_bits[q][r * 64 + lane];
            const uint32_t n = (uint32_t)__popcll(v);
            uint32_t inc = n;
            for (int x = 1; x < 64; x <<= 1) {
                const uint32_t y = __shfl_up(inc, x);
                if ((int)lane >= x) inc += y;
            }
            bits[r * 64 + lane] = v;
            before[r * 64 + lane] = done + inc - n;
            done += __shfl(inc, 63);
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < FINISH_ITEMS; j++) {
        if (f[j] == NO_ROW) continue;
        const uint32_t rank = before[f[j] >> 6] + (uint32_t)__popcll(bits[f[j] >> 6] & ((1ull << (f[j] & 63)) - 1ull));
        if (c[j] == 0) {
            as_global(d.mapped)[pos[j]] = (int64_t)rank;
            if (f[j] == pos[j]) p.rank_at[d.lbase + pos[j]] = (uint16_t)rank;
        }
        if (row[j] == NO_ROW || (int64_t)rank >= d.rows) continue;  // (the host reports a variable that is too small)
        *(Global<Part>)as_global(d.var + (uint64_t)rank * s.wdim + c[j] * VEC) = v[j];
    }
}

template <int VEC>
__global__ __launch_bounds__(FINISH_THREADS) void k_small_group_finish(SmallShape b, SmallPlan p, uint32_t chunks,
                                                                       uint32_t per, Store s) {
    small_finish<VEC>(b, p, blockIdx.x, chunks, per, s);
}

// Both by one launch: each is a chain of round trips, with the gap between two launches behind it.
template <int VEC>
__global__ __launch_bounds__(FINISH_THREADS) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_small_pull_rest(
    EmitArgs<true> a, uint32_t chunks, uint32_t per, Store s) {
    extern __shared__ uint32_t emit_lds[];
    const uint32_t buckets = a.b.buckets();
    if (blockIdx.x < buckets)
        small_emit_bucket(a, emit_lds);
    else
        small_finish<VEC>(a.b, a.p, blockIdx.x - buckets, chunks, per, s);
}

// First launch of a small push on the last pull's plan: the signs are compared with the plan's copy, and with CLICKS the
// non-zero labels are added to the click sums (sparse_table_ops.cc:283-296; a few thousand lookups do not queue up on
// any entry).  A mismatch also goes to the host (pinned memory); that the comparison is complete, the last launch tells it.
// The workgroups behind those, a wavefront per bucket, put the ranks of the records' first lookups into the records: the
// updates would otherwise read them through rank_at, a round trip more (the pull works ranks and records out side by side).
template <bool CLICKS, typename Descs>
__global__ __launch_bounds__(256) void k_small_verify(SmallShape b, SmallPlan p, Descs descs, uint32_t chunks,
                                                           DevStatus* status, uint32_t* host_mismatch) {
    __shared__ SlotDesc sd;
    if (blockIdx.x >= b.N * chunks) {
        const uint32_t c = (blockIdx.x - b.N * chunks) * 4 + threadIdx.x / 64;
        if (c >= b.buckets()) return;
        const uint4 head = p.head[c];
        uint4* mem = p.member + (size_t)c * b.cap;
        const uint32_t n = min(head.x + head.w, b.cap);
        for (uint32_t i = threadIdx.x & 63; i < n; i += 64) {
            const uint4 m = mem[i];
            mem[i].y = (m.y & 0xFFFF0000u) | p.rank_at[m.x];
        }
        return;
    }
    const int sl = blockIdx.x / chunks;
    const uint32_t p0 = (blockIdx.x % chunks) * SMALL_TILE;
    // what the pull left of these positions is on its way while the descriptor comes in
    const uint32_t lbase = p.descs[sl].lbase, len = p.descs[sl].len;  // (the shape is the pull's)
    constexpr int PER = SMALL_TILE / 256;
    uint64_t now[PER], then[PER];
    int label[PER];
    uint32_t f[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const uint32_t pos = p0 + j * 256 + threadIdx.x;
        then[j] = pos < len ? p.vals_copy[lbase + pos] : 0;
        f[j] = CLICKS && pos < len ? p.first_of[lbase + pos] : 0u;
    }
    DescFetch fetch;
    fetch.start(descs, sl);
    fetch.finish(descs, sl, sd, p0 == 0 ? p.push_descs + sl : nullptr);
    bool bad = false;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        bad = *p.bad != 0;
        status->abort = 0;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const uint32_t pos = p0 + j * 256 + threadIdx.x;
        now[j] = pos < len ? (uint64_t)as_global(sd.values)[pos] : 0;
        label[j] = CLICKS && pos < len ? (int)as_global(sd.labels)[pos] : 0;
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
        bad |= now[j] != then[j];
        if (CLICKS && label[j] != 0) atomicAdd(&p.click_at[lbase + f[j]], label[j]);
    }
    if (bad) {
        atomicOr(&status->mismatch, 1u);
        host_store(host_mismatch, 1u);
    }
}

// Pooled gradients: the gradient of every distinct sign of a slot is the sum over its lookups, in order, of their
// examples' rows times 1 / d(lookups of the example).  2^lp workgroups per slot, each of which looks at the whole slot and
// takes the signs whose first position is its own modulo 2^lp, POOL_ITEMS_MAX lookups at a time (pool_items).
// flat[gi of the sign's first lookup, :] = sum, over the D elements the updates read (rows of `dim`: with the cvm columns).
// 50 slots of 3100 lookups: 39 us (a workgroup of 1024 threads per slot: 43), a push and pull with 512, 1024, 2048 lookups a
// workgroup 142, 136, 136 us.
constexpr uint32_t SMALL_POOL_FILL = 1024;
inline uint32_t small_pool_parts_log2(uint32_t max_len) {
    uint32_t lp = 0;
    while ((max_len >> lp) > SMALL_POOL_FILL) lp++;
    return lp;
}
constexpr uint32_t SMALL_POOL_AHEAD = 4;  // runs of 64 lookups of a wavefront in flight

// The heavy signs of a slot, by position: `heavy` (SMALL_HEAVY_MAX words of LDS), their number.  The workgroups that deal its
// lookups out, and those that add the shares up, all have to have them in the same order.  Ends with a barrier.
__device__ __forceinline__ uint32_t small_heavy(const SmallShape& b, const SmallPlan& p, uint32_t sl, uint32_t* heavy,
                                                uint32_t* found) {
    const uint32_t tid = threadIdx.x;
    if (tid == 0) *found = 0;
    __syncthreads();
    if (tid < b.parts * SMALL_HEAVY_MAX) {
        const uint32_t f = p.heavy[sl * b.parts * SMALL_HEAVY_MAX + tid];
        if (f != SMALL_NONE) heavy[atomicAdd(found, 1u)] = f;
    }
    __syncthreads();
    const uint32_t n = *found, f = tid < n ? heavy[tid] : 0u;
    uint32_t rank = 0;
    for (uint32_t e = 0; e < n; e++) rank += heavy[e] < f ? 1u : 0u;
    __syncthreads();
    if (tid < n) heavy[rank] = f;
    __syncthreads();
    return n;
}
static_assert(SMALL_PARTS_MAX * SMALL_HEAVY_MAX <= POOL_THREADS && SMALL_HEAVY_MAX * 64 == POOL_THREADS, "small_heavy");

// HEAVY: the lookups of the slot's heavy signs are dealt to its workgroups run by run (64 lookups), each of which leaves a share
// of their sums (k_small_pool_shares adds them up).  As one workgroup's such a sign is a chain of rounds (25 us each at 16
// elements a row): 100 slots of 8000 lookups, 80 % of them one sign, a step with rows of 16 237 us, of 64 475;
// so 163 and 266.
// (Four workgroups to a CU, of 64 registers: 100 slots of 6000 lookups 45 us, three 51; 26 of 1000, rows of 64, 33.4 and 33.3.)
template <int LPG, bool ANY, bool HEAVY>
__global__ __launch_bounds__(POOL_THREADS) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_small_pool(SmallShape b, SmallPlan p, const SlotDesc* __restrict__ descs,
                                                             int64_t batch, int dim, int D, int combiner,
                                                             float* __restrict__ flat, DevStatus* status, uint32_t* host_err,
                                                             uint32_t lp, float* __restrict__ shares,
                                                             uint32_t* __restrict__ has) {
    __shared__ PoolLds lds;
    __shared__ uint32_t heavy[HEAVY ? SMALL_HEAVY_MAX : 1], found, have, had;  // have: heavy signs with a sum so far
    __shared__ unsigned long long starts[SMALL_WORDS];  // of the examples
    __shared__ uint32_t bad;
    // The workgroups of a slot, which read the same lookups and rows, on one die (DieShare, an item per workgroup).  Dealt out
    // in turn, the first part of every slot of eight parts, which has the sign that begins it, was the first die's.
    const uint32_t item = blockIdx.x % XCDS * (gridDim.x / XCDS) + blockIdx.x / XCDS;  // (the grid is a multiple of XCDS)
    const uint32_t sl = item >> lp, part = item & ((1u << lp) - 1u);
    if (sl >= (uint32_t)b.N) return;
    const SlotDesc d = descs[sl];
    const uint32_t n = d.len, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (n == 0 || status->mismatch) return;
    const Global<const int64_t> ex = as_global((const int64_t*)d.mapped);
    const Global<const uint16_t> first_of = as_global((const uint16_t*)p.first_of + d.lbase);
    if (tid == 0) bad = have = had = 0;
    const uint32_t n_heavy = HEAVY ? small_heavy(b, p, sl, heavy, &found) : 0u;
    if (!HEAVY) __syncthreads();
    // a wavefront's runs, one behind the other
    const uint32_t words = (n + 63) / 64, per = (words + POOL_WAVES - 1) / POOL_WAVES;
    const uint32_t w0 = wave * per, w1 = min(words, w0 + per), mask = (1u << lp) - 1u;
    const uint32_t others = ((n - 1) >> lp) + 1;  // keys of the signs that are not heavy; the heavy ones' behind them
    // the key of a lookup of sign f at position i, if it is my part's
    auto key_of = [&](uint32_t f, uint32_t i, bool& mine) {
        mine = (f & mask) == part;
        uint32_t key = f >> lp;
        if (HEAVY)
            for (uint32_t e = 0; e < n_heavy; e++)
                if (f == heavy[e]) {
                    mine = ((i >> 6) & mask) == part;
                    key = others + e;
                }
        mine = mine && f != NO_ROW;
        return key;
    };
    uint32_t cnt = 0;
#pragma unroll 1
    for (uint32_t w = w0; w < w1; w += SMALL_POOL_AHEAD) {
        int64_t e[SMALL_POOL_AHEAD], prev[SMALL_POOL_AHEAD];
        uint32_t f[SMALL_POOL_AHEAD];
#pragma unroll
        for (uint32_t j = 0; j < SMALL_POOL_AHEAD; j++) {
            const uint32_t i = (w + j) * 64 + lane;
            const bool there = w + j < w1 && i < n;
            e[j] = there ? ex[i] : -1;
            prev[j] = there && i > 0 ? ex[i - 1] : -1;
            f[j] = there ? (uint32_t)first_of[i] : NO_ROW;
        }
#pragma unroll
        for (uint32_t j = 0; j < SMALL_POOL_AHEAD; j++) {
            const bool there = f[j] != NO_ROW;
            if (there && (e[j] < 0 || e[j] >= batch || prev[j] > e[j])) bad = 1;
            const unsigned long long m = __ballot(there && e[j] != prev[j]);
            if (lane == 0 && w + j < w1) starts[w + j] = m;
            bool mine;
            key_of(f[j], (w + j) * 64 + lane, mine);
            cnt += (uint32_t)__popcll(__ballot(mine));
        }
    }
    if (lane == 0) lds.wsum[wave] = cnt;
    __syncthreads();
    if (bad) {  // unsorted or out-of-range example ids: nothing of this push is applied
        if (tid == 0) {
            status->abort = 1;
            host_store(host_err, 1u);
        }
        return;
    }
    uint32_t first = 0, total = 0;  // of my part: lookups of the wavefronts before, of all
#pragma unroll
    for (uint32_t w = 0; w < POOL_WAVES; w++) {
        if (w < wave) first += lds.wsum[w];
        total += lds.wsum[w];
    }
    const uint32_t top = others - 1 + n_heavy, bits = top ? 32 - (uint32_t)__clz((int)top) : 0u;
#pragma unroll 1
    for (uint32_t done = 0; done < total; done += POOL_ITEMS_MAX) {
        uint32_t at = first - done;  // (of a round before: wraps)
#pragma unroll 1
        for (uint32_t w = w0; w < w1; w += SMALL_POOL_AHEAD) {
            // (read again: kept across the rounds in registers, of which 187 were spilled, 100 slots of 6000 lookups took 151 us
            // here; so 54, and 50 with a slot's workgroups on one die)
            int64_t e[SMALL_POOL_AHEAD];
            uint32_t f[SMALL_POOL_AHEAD];
#pragma unroll
            for (uint32_t j = 0; j < SMALL_POOL_AHEAD; j++) {
                const uint32_t i = (w + j) * 64 + lane;
                const bool there = w + j < w1 && i < n;
                e[j] = there ? ex[i] : 0;
                f[j] = there ? (uint32_t)first_of[i] : NO_ROW;
            }
#pragma unroll
            for (uint32_t j = 0; j < SMALL_POOL_AHEAD; j++) {
                const uint32_t i = (w + j) * 64 + lane;
                bool mine;
                const uint32_t key = key_of(f[j], i, mine);
                const unsigned long long own = __ballot(mine);
                const uint32_t q = at + (uint32_t)__popcll(own & ((1ull << lane) - 1ull));
                if (mine && q < POOL_ITEMS_MAX) {
                    const float count = combiner == POOL_SUM ? 1.f : (float)(bit_above(starts, i, words, n) - bit_at_or_below(starts, i));
                    const float scale = pool_scale(count, combiner);
                    lds.key[q] = key;
                    lds.example[q] = (uint32_t)e[j];
                    lds.scale[q] = f[j] == i ? scale : -scale;
                }
                at += (uint32_t)__popcll(own);
            }
        }
        pool_items<LPG, ANY>(lds, min(POOL_ITEMS_MAX, total - done), bits, d.grads, dim, D,
                             [&](uint32_t key, bool first, bool& add) {
                                 if (HEAVY && key >= others) {
                                     add = ((had >> (key - others)) & 1u) != 0;
                                     atomicOr(&have, 1u << (key - others));
                                     return shares + ((uint64_t)item * SMALL_HEAVY_MAX + (key - others)) * dim;
                                 }
                                 add = !first;
                                 return flat + (uint64_t)(d.lbase + ((key << lp) | part)) * dim;
                             });
        if (HEAVY) {
            if (tid == 0) had = have;
            __syncthreads();
        }
    }
    if (HEAVY && tid == 0) has[item] = have;
}

// The sums of the heavy signs: a workgroup per slot, a wavefront per sign.
template <int LPG, bool ANY>
__global__ __launch_bounds__(64 * SMALL_HEAVY_MAX) void k_small_pool_shares(SmallShape b, SmallPlan p, int dim, int D,
                                                                            float* __restrict__ flat, const DevStatus* status,
                                                                            uint32_t lp, const float* __restrict__ shares,
                                                                            const uint32_t* __restrict__ has) {
    __shared__ uint32_t heavy[SMALL_HEAVY_MAX], found;
    if (status->abort | status->mismatch) return;
    const uint32_t sl = blockIdx.x, e = threadIdx.x / 64, item0 = sl << lp;
    if (e >= small_heavy(b, p, sl, heavy, &found)) return;
    add_shares<LPG, ANY>(
        1u << lp, D, [&](uint32_t q) { return ((has[item0 + q] >> e) & 1u) != 0; },
        [&](uint32_t q) { return shares + ((uint64_t)(item0 + q) * SMALL_HEAVY_MAX + e) * dim; },
        flat + (uint64_t)(p.descs[sl].lbase + heavy[e]) * dim);
}

// Where the update kernels find the gradient of a record: the slots' matrices (in LDS), or the reduced rows of a push
// of pooled gradients, one per first lookup.
struct SmallSrc {
    const float* const* grads;
    const uint32_t* rows;
    const float* flat;
    int32_t* click_at;
    int dim;
    __device__ __forceinline__ const float* gradient(uint4 m) const {
        if (flat) return flat + (uint64_t)m.x * dim;
        const uint32_t sl = m.y >> 16, rank = m.y & 0xFFFFu;
        return rank < rows[sl] ? grads[sl] + (uint64_t)rank * dim : nullptr;  // (the host reports a matrix with too few rows)
    }
    // the record's click sum; zero again for a further push on the plan
    __device__ __forceinline__ int click(uint4 m) const { return click_at[m.x]; }
};

// The records of one sign: entries of the bucket's member list.
struct SmallGroup {
    typedef uint4 Entry;
    SmallSrc src;
    const uint4* mem;
    __device__ __forceinline__ Entry entry(uint32_t j) const { return mem[j]; }
    __device__ __forceinline__ const float* gradient(const Entry& m) const { return src.gradient(m); }
    __device__ __forceinline__ int show(const Entry& m) const { return (int)m.z; }
    __device__ __forceinline__ int click(const Entry& m) const { return src.click(m); }
    __device__ __forceinline__ void taken(uint32_t k, int sub, int lanes) const {
        for (uint32_t j = sub; j < k; j += lanes) src.click_at[mem[j].x] = 0;
    }
};

// One sign with a few records by a group of LPG lanes, AHEAD records at a time: the gradients of the next AHEAD and the
// member entries of the AHEAD after those are in flight meanwhile, so that a chain of k records costs k / AHEAD round
// trips instead of 2 k (a small batch's kernels are as long as their longest chain).  Every load is issued whether its
// record exists or not (past the end: the group's last member again, the row in place of a gradient): a load under a
// condition makes the compiler wait for all loads where the branches join.
// grp: the sign's records -- entry(j) of the j-th (what is fetched ahead), its gradient row (nullptr: it has none) and
// counts, taken(k, sub, lanes) once all have been applied.
// ONCE: the caller says that k <= AHEAD, so nothing is fetched ahead (and registers for 32 words are free).
template <int KIND, int LPG, bool ANY, int AHEAD, bool ONCE, typename Group>
__device__ __forceinline__ void apply_group_ahead(const Store& s, const OptDev& o, const Group& grp, uint32_t row, uint32_t k,
                                                  int sub, float c1, float c2) {
    typedef typename Group::Entry Entry;
    const int D = s.D;
    float* wp = s.w + (uint64_t)row * s.wstride;
    float* sp = s.st + (uint64_t)row * s.sstride;
    float4 w = row_part<ANY>(wp, sub, D);
    float4 a, b;  // Adam m, v / Ftrl z, n
    float g2sum = 0.f, show = 0.f, click = 0.f;
    int delta_show = 0;
    if (KIND == OPT_ADAGRAD) {
        const float4 h = *reinterpret_cast<const float4*>(sp);
        g2sum = h.x;
        show = h.y;
        click = h.z;
    } else {
        a = row_part<ANY>(sp, sub, D);
        b = row_part<ANY>(sp + D, sub, D);
        delta_show = __float_as_int(sp[2 * D + 1]);
    }
    bool any = false;
    Entry m1[AHEAD], m2[AHEAD];
    float4 g0[AHEAD], g1[AHEAD];
    int sh0[AHEAD], ck0[AHEAD], sh1[AHEAD], ck1[AHEAD];
    bool ok0[AHEAD], ok1[AHEAD];
    auto fetch = [&](const Entry (&m)[AHEAD], uint32_t first, float4 (&g)[AHEAD], int (&sh)[AHEAD], int (&ck)[AHEAD],
                     bool (&ok)[AHEAD]) {
#pragma unroll
        for (int q = 0; q < AHEAD; q++) {
            const float* gp = grp.gradient(m[q]);
            ok[q] = gp != nullptr && first + q < k;
            sh[q] = grp.show(m[q]);
            ck[q] = KIND == OPT_ADAGRAD ? grp.click(m[q]) : 0;
            g[q] = row_part<ANY>(ok[q] ? gp : wp, sub, D);
        }
    };
#pragma unroll
    for (int q = 0; q < AHEAD; q++) {
        m1[q] = grp.entry(min((uint32_t)q, k - 1));
        if (!ONCE) m2[q] = grp.entry(min((uint32_t)(AHEAD + q), k - 1));
    }
    fetch(m1, 0, g0, sh0, ck0, ok0);
    if (!ONCE) {
#pragma unroll
        for (int q = 0; q < AHEAD; q++) m1[q] = m2[q];
    }
    for (uint32_t c0 = 0; c0 < (ONCE ? 1 : k); c0 += AHEAD) {
        if (!ONCE) {
#pragma unroll
            for (int q = 0; q < AHEAD; q++) m2[q] = grp.entry(min(c0 + 2 * AHEAD + q, k - 1));
            fetch(m1, c0 + AHEAD, g1, sh1, ck1, ok1);
        }
        if constexpr (KIND == OPT_ADAGRAD) {
            // The records of the window depend on each other through g2sum (one rounded addition per record) and
            // through the row (one subtraction per element and record) only.  Everything else -- the sums of squares
            // with their hand-over from lane to lane, the square roots, the divisions -- is worked out for all records of
            // the window side by side; the two chains then run over the results, in record order.  The same operations
            // on the same operands as record after record.
            float4 sq[AHEAD];
            double mq[AHEAD];
#pragma unroll
            for (int q = 0; q < AHEAD; q++) sq[q] = squares(g0[q]);
            square_sums<LPG>(sq, mq);
#pragma unroll
            for (int q = 0; q < AHEAD; q++) mq[q] = mq[q] / (double)D;
            float g2[AHEAD];
#pragma unroll
            for (int q = 0; q < AHEAD; q++) {
                if (ok0[q]) {
                    any = true;
                    show += (float)sh0[q];
                    click += (float)ck0[q];
                    g2sum = (float)((double)g2sum + mq[q]);
                }
                g2[q] = g2sum;
            }
            float4 st4[AHEAD];
#pragma unroll
            for (int q = 0; q < AHEAD; q++) {
                const float den = o.eps + sqrtf(g2[q]);
                st4[q] = make_float4(o.lr * g0[q].x / den, o.lr * g0[q].y / den, o.lr * g0[q].z / den, o.lr * g0[q].w / den);
            }
#pragma unroll
            for (int q = 0; q < AHEAD; q++) {
                if (!ok0[q]) continue;
                w.x -= st4[q].x;
                w.y -= st4[q].y;
                w.z -= st4[q].z;
                w.w -= st4[q].w;
            }
        } else {
#pragma unroll
            for (int q = 0; q < AHEAD; q++) {
                if (!ok0[q]) continue;
                any = true;
                delta_show += sh0[q];
                if (KIND == OPT_ADAM) {
                    adam_elem(o, c1, c2, g0[q].x, w.x, a.x, b.x);
                    adam_elem(o, c1, c2, g0[q].y, w.y, a.y, b.y);
                    adam_elem(o, c1, c2, g0[q].z, w.z, a.z, b.z);
                    adam_elem(o, c1, c2, g0[q].w, w.w, a.w, b.w);
                } else {
                    ftrl_elem(o, g0[q].x, w.x, a.x, b.x);
                    ftrl_elem(o, g0[q].y, w.y, a.y, b.y);
                    ftrl_elem(o, g0[q].z, w.z, a.z, b.z);
                    ftrl_elem(o, g0[q].w, w.w, a.w, b.w);
                }
            }
        }
        if (ONCE) break;
#pragma unroll
        for (int q = 0; q < AHEAD; q++) {
            g0[q] = g1[q];
            sh0[q] = sh1[q];
            ck0[q] = ck1[q];
            ok0[q] = ok1[q];
            m1[q] = m2[q];
        }
    }
    if (KIND == OPT_ADAGRAD) grp.taken(k, sub, LPG);
    if (!any) return;
    put_row_part<ANY>(wp, sub, D, w);
    if (KIND == OPT_ADAGRAD) {
        if (sub == 0) {
            *reinterpret_cast<float4*>(sp) = make_float4(g2sum, show, click, 0.f);  // no_show_days = 0
            if (o.use_cvm) {
                wp[D] = show;
                wp[D + 1] = logf(click + 1) - logf(show + 1);
            }
        }
    } else {
        put_row_part<ANY>(sp, sub, D, a);
        put_row_part<ANY>(sp + D, sub, D, b);
        if (sub == 0) sp[2 * D + 1] = __int_as_float(delta_show);
    }
}

// Bytes of dynamic LDS of k_small_apply when its launch includes the workgroups for the signs with many records:
// per wavefront the staging and the row of apply_big_groups, then its pointer, count, flag and divisor arrays.
inline size_t small_apply_wave_lds(int D) { return align_up(big_lds_bytes(D), 8) + BIG_CHUNK * (8 + 4); }
// (a sign of a small batch has as many records as the batch has slots at most)
inline int small_gbuf_floats(int D, int N) { return std::min(big_gbuf_floats(D), std::min(N, BIG_CHUNK) * (D + 1)); }

__host__ __device__ inline size_t small_apply_slots_lds(int N) { return ((size_t)N * 12 + 7) / 8 * 8; }

// The next number of a counter in LDS for the whole wavefront, all of whose lanes call it.
__device__ __forceinline__ uint32_t wave_draw(uint32_t* counter) {
    uint32_t r = 0;
    if (__lane_id() == 0) r = atomicAdd(counter, 1u);
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)r);
}

// The updates of a small push by one launch, a workgroup per bucket (three per bucket, one for each kind of sign, were two
// to five times as many workgroups as the chip holds at once, most of their lanes without a sign: 26 slots of 4096 lookups,
// Adam rows of 16, 17.9 us, 15.2 now).  What bounds it is the longest chain of a wavefront.  Its wavefronts take the signs with many records (four
// slots' worth and more) first, one each, the way k_apply_big does; then 64 / LPG signs at a time: those with a few records,
// several records of a sign in flight, then those with one.  Nothing is reported to the host but that this kernel runs,
// which tells it that the comparison of the signs, launched before, is complete: on the plan of the last pull every sign has
// its row, and the host has compared the slots' distinct counts with the rows of the gradient matrices itself.
// BIG: how the signs with many records are applied -- BIG_NONE, the plan lists none; BIG_GROUPS, rows of any length
// (apply_big_groups); else rows of as many elements (apply_big_wave).
enum { BIG_NONE = 0, BIG_GROUPS = -1 };
// Wavefronts a SIMD: AdaGrad rows of 64 with signs of many records fit four (128 registers, none spilled; by itself the compiler
// takes 146): 40 slots of 8192 lookups 46.0 -> 40.0 us, 26 of 1024 14.6 -> 14.1.  Others lose by it: without such signs 12 slots of
// 4000 19.5 -> 21.1, Adam rows of 64 (20 spilled) 50.4 -> 60.8, rows of 32, 26 of 1024, AdaGrad 9.9 -> 10.5, Adam 9.4 -> 10.7.
// Rounds a chunk of apply_big_wave: sixteen, but for Adam rows of 16 and 32, whose chunk (gradients and second moments of 64 or 32
// records, 9 KB) would let a CU hold four workgroups, four.  us with sixteen and with four: 26 slots of 4096 lookups 15.6 and 11.9, rows
// of 32 17.2 and 14.6; of 1200 10.0 and 8.9, 10.7 and 10.4; 80 slots of 2000 32.5 (4000 lookups) and 26.2, 29.9 and 25.5, of 400 15.8
// and 14.5, 18.0 and 17.0; 300 of 300 47.9 and 46.4, 57.8 and 58.1.  Others lose where signs have many records: 300 slots of 300, AdaGrad
// rows of 16 34.1 and 40.6, of 32 44.4 and 62.6, Adam rows of 8 44.2 and 45.6, of 64 73.0 and 90.3; 80 of 400, Ftrl rows of 32 24.0 and 24.7.
constexpr int small_apply_most(int kind, int big) { return kind == OPT_ADAM && (big == 16 || big == 32) ? 4 : 16; }
constexpr int small_apply_waves(int kind, int lpg, int big) { return kind == OPT_ADAGRAD && lpg == 16 && big > 0 ? 4 : 1; }
template <int KIND, int LPG, bool ANY, int BIG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(small_apply_waves(KIND, LPG, BIG), 8))) void k_small_apply(
                                                     SmallShape b, SmallPlan p, const float* flat, Store s,
                                                     OptDev o, const DevStatus* __restrict__ status, uint32_t* host_seq,
                                                     uint32_t seq, int dim, int gbuf_floats, uint32_t wave_lds,
                                                     uint32_t wave_arrays) {
    extern __shared__ unsigned long long apply_lds[];  // the slots' gradient matrices and their rows; then the wavefronts' staging
    __shared__ uint32_t next_round;
    if (blockIdx.x == 0 && threadIdx.x == 0) host_store(host_seq, seq);
    const uint32_t c = blockIdx.x;
    const size_t first = (size_t)c * b.cap;
    const uint4 head = p.head[c];
    const uint2 big0 = p.group[first + b.cap - 1 - (threadIdx.x >> 6)];  // (if there are so many: one round trip less)
    const uint32_t stop = status->mismatch | status->abort;
    const float** grads = reinterpret_cast<const float**>(apply_lds);
    uint32_t* rows = reinterpret_cast<uint32_t*>(grads + (flat ? 0 : b.N));
    if (!flat) {
        for (uint32_t i = threadIdx.x; i < (uint32_t)b.N; i += 256) {
            grads[i] = p.push_descs[i].grads;
            rows[i] = (uint32_t)min(p.push_descs[i].rows, (int64_t)SMALL_SLOT_MAX + 1);
        }
    }
    if (threadIdx.x == 0) next_round = 0;
    __syncthreads();
    // a plan that turned out not to be this batch's: nothing to do (the host analyses the batch itself)
    if (stop) return;
    SmallSrc src;
    src.grads = grads;
    src.rows = rows;
    src.flat = flat;
    src.click_at = p.click_at;
    src.dim = dim;
    const float c1 = 1 - o.beta1, c2 = 1 - o.beta2;
    const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63), sub = lane % LPG;
    auto describe = [](uint2 g) { return make_uint4(g.x, g.y & 0xFFFFu, g.y >> 16, 0u); };
    auto group = [&](uint32_t bi) { return describe(p.group[first + b.cap - 1 - bi]); };
    auto record = [&](const uint4& m, const float*& gp, int& sh, int& ck, bool there) {
        gp = src.gradient(m);
        sh = (int)m.z;
        if (KIND == OPT_ADAGRAD) {
            ck = src.click(m);
            if (there) src.click_at[m.x] = 0;
        }
        return gp != nullptr;
    };
    if constexpr (BIG > 0) {
        __shared__ BigWave<KIND, BIG, small_apply_most(KIND, BIG)> tiles[4];
        apply_big_wave<KIND, BIG>(s, o, tiles[wave], describe(big0), (uint32_t)wave, 4u, head.z, group,
                                  [&](uint32_t at) { return p.member[first + at]; }, record, [] {});
    } else if (BIG == BIG_GROUPS && head.z) {
        char* base = reinterpret_cast<char*>(apply_lds) + small_apply_slots_lds(flat ? 0 : b.N) + (size_t)wave * wave_lds;
        float* gbuf = reinterpret_cast<float*>(base);
        const float** gptr = reinterpret_cast<const float**>(base + wave_arrays);
        float* den = reinterpret_cast<float*>(gptr + BIG_CHUNK);
        apply_big_groups<KIND>(
            s, o, gbuf_floats, gbuf, gptr, den, lane, (uint32_t)wave, 4u, head.z,
            [&](uint32_t bi, uint32_t& row, uint32_t& off, uint32_t& k) {
                const uint4 g = group(bi);
                row = g.x;
                off = g.y;
                k = g.z;
            },
            [&](uint32_t at, const float*& gp, int& sh, int& ck) { return record(p.member[first + at], gp, sh, ck, true); }, [] {},
            [] { wave_sync(); });
    }
    // signs with one record: several rounds of a wavefront on their way at a time where a round has few
    constexpr uint32_t PER = 64 / LPG, AT_ONCE = LPG >= 16 ? 4 : LPG >= 4 ? 2 : 1;
    const uint32_t rounds_multi = (head.y + PER - 1) / PER, rounds = rounds_multi + (head.x + AT_ONCE * PER - 1) / (AT_ONCE * PER);
    // (Nothing leaves the loop's body but through its end: with a `continue` under a condition the compiler makes the lanes
    // that take it a loop of their own, in which lane 0, that draws the next round, does not run.)
    uint32_t r = wave_draw(&next_round);
    while (r < rounds) {
        if (r < rounds_multi) {
            const uint32_t g = r * PER + lane / LPG;
            const uint2 d = g < head.y ? p.group[first + head.x + g] : make_uint2(NO_ROW, 0);
            if (d.x <= s.cap) {  // (no row number at all: never address the table with it)
                const SmallGroup grp{src, p.member + first + (d.y & 0xFFFFu)};
                apply_group_ahead<KIND, LPG, ANY, 4, BIG != BIG_NONE>(s, o, grp, d.x, d.y >> 16, sub, c1, c2);
            }
        } else {
            uint2 d[AT_ONCE];
            uint4 mem[AT_ONCE];
            const float* gp[AT_ONCE];
            RecordRow row[AT_ONCE];
            int ck[AT_ONCE];
            bool ok[AT_ONCE];
#pragma unroll
            for (uint32_t q = 0; q < AT_ONCE; q++) {
                const uint32_t g = ((r - rounds_multi) * AT_ONCE + q) * PER + lane / LPG, at = min(g, b.cap - 1);
                d[q] = p.group[first + at];
                mem[q] = p.member[first + at];
                ok[q] = g < head.x;
            }
            // (what lies behind the last sign is nobody's: row 0 in its place, and nothing written)
#pragma unroll
            for (uint32_t q = 0; q < AT_ONCE; q++) {
                ok[q] = ok[q] && d[q].x <= s.cap;
                if (!ok[q]) {
                    d[q].x = 0;
                    mem[q].x = 0;
                }
                gp[q] = ok[q] ? src.gradient(mem[q]) : nullptr;
                row[q] = fetch_record<KIND, ANY>(s, d[q].x, gp[q] ? gp[q] : s.w, sub);
                ck[q] = KIND == OPT_ADAGRAD ? src.click(mem[q]) : 0;
            }
#pragma unroll
            for (uint32_t q = 0; q < AT_ONCE; q++) {
                if (gp[q])
                    finish_record<KIND, LPG, ANY>(s, o, d[q].x, row[q], (int)mem[q].z, ck[q], sub, c1, c2);
                // (a record without a gradient row, too: the caller may push the batch again on this plan)
                if (KIND == OPT_ADAGRAD && ok[q] && sub == 0) src.click_at[mem[q].x] = 0;
            }
        }
        r = wave_draw(&next_round);
    }
}

}  // namespace tn

#endif  // TN_SMALL_BATCH_H_
