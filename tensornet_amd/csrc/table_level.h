// Pull and push at table level (SparseTable::Pull / Push, core/ps/table/sparse_table.cc:52-83): one array of signs or
// records, in which a sign may occur any number of times, in few launches.
//
//   pull  k_table_pull   probe or insert every sign, its row to the output, a word to the host per workgroup
//         k_report       tells the host that the rows are written
//   push  k_table_part   per tile of records: table row of every record, the records in order of buckets of rows
//         k_table_apply  per bucket: its records, tile after tile, grouped by row in LDS and applied in record order
//
// The push took twelve launches before: a hash table of the records' signs in memory, a compaction of it, arrival
// order, ranks in arrival order, a probe per sign and three update kernels; the pull five and a wait for a copy.  Both
// together, at 60 000 records of 16 elements: 147 us before, 54 us now; at 942 570 records of 10 elements 1250 and 328.
#ifndef TN_TABLE_LEVEL_H_
#define TN_TABLE_LEVEL_H_

#include "small_batch.h"

namespace tn {

// --------------------------------------------------------------------- pull
constexpr uint32_t TABLE_PULL_WORDS = 1024;  // workgroups of k_table_pull at most (the host reads a word of each)
constexpr uint32_t TABLE_PULL_FEW = 256;     // ... as many as there are CUs: with fewer a workgroup takes 64 signs instead of 256

// The m rows of a workgroup's signs, row after row, in pieces, AHEAD of a thread on their way (each written before the next is read,
// as the compiler leaves it -- the output might be the table -- they are a round trip each).  k_table_pull: 60 000 signs, rows of 16
// 9.1 us one by one and 8.4 by eight, of 64 14.7 and 11.4; 300 000, of 16 14.0 and 13.1, of 64 28.3 and 23.8 (four on their way 25.0).
// One by one where a thread has two pieces at most, which it works out eight places for otherwise, in 125 registers instead of 51: 500
// signs, rows of 1 5.1 us by eight and 4.6 so, 5000, of 4 5.7 and 5.1, of 16 5.8 and 4.9, 20 000, of 1 6.4 and 5.6.
constexpr uint32_t PULL_AHEAD = 8, PULL_FEW = 2;
template <uint32_t AHEAD, typename Piece>
__device__ __forceinline__ void table_rows_out(const Store& s, const uint32_t* row, uint32_t m, float* __restrict__ out) {
    constexpr uint32_t VEC = sizeof(Piece) / sizeof(float);
    const uint32_t C = (uint32_t)s.wdim / VEC, pieces = m * C;
    for (uint32_t q0 = threadIdx.x; q0 < pieces; q0 += 256 * AHEAD) {
        Piece v[AHEAD];
#pragma unroll
        for (uint32_t k = 0; k < AHEAD; k++) {
            const uint32_t q = q0 + 256 * k, i = q / C, c = q - i * C, r = q < pieces ? row[i] : NO_ROW;
            v[k] = Piece{};
            if (r != NO_ROW) v[k] = *reinterpret_cast<const Piece*>(s.w + (uint64_t)r * s.wstride + c * VEC);
        }
#pragma unroll
        for (uint32_t k = 0; k < AHEAD; k++) {
            const uint32_t q = q0 + 256 * k;
            if (q < pieces) *reinterpret_cast<Piece*>(out + (uint64_t)q * VEC) = v[k];
        }
    }
}
inline bool table_pull_few(int64_t n, uint32_t per, uint32_t pieces_of_row) {
    return (uint64_t)std::min<int64_t>(n, per) * pieces_of_row <= 256 * PULL_FEW;
}

// `per` signs at a time per workgroup (256 at most): few for a short request, which then has its probes on many CUs.  A
// row that is inserted is filled by all threads of the workgroup that inserted it, before it copies rows out; another
// workgroup that holds the same sign may copy it too early, so a request that inserted anything is copied out once more
// (k_gather_rows, from rows[]).  Every workgroup tells the host itself: rows inserted | out of slots << 31 | seq << 32.
// Bound by the two dependent reads of a row (keys, then weights).
template <uint32_t AHEAD>
__global__ __launch_bounds__(256) void k_table_pull(Store s, OptDev o, uint64_t seed, const uint64_t* __restrict__ signs,
                                                    int64_t n, uint32_t per, int vec, float* __restrict__ out,
                                                    uint32_t* __restrict__ rows, uint64_t* host_words, uint32_t seq) {
    __shared__ uint32_t row[256];
    __shared__ uint8_t fresh[256];
    __shared__ uint32_t n_new, full;
    const uint32_t tid = threadIdx.x;
    uint32_t all_new = 0;
    if (tid == 0) full = 0;
    for (int64_t first = (int64_t)blockIdx.x * per; first < n; first += (int64_t)gridDim.x * per) {
        const uint32_t m = (uint32_t)min((int64_t)per, n - first);
        if (tid == 0) n_new = 0;
        __syncthreads();
        if (tid < m) {
            bool is_new = false;
            const uint32_t r = probe_slot<true>(s, signs[first + tid], is_new);
            row[tid] = r;
            rows[first + tid] = r;
            if (is_new) fresh[atomicAdd(&n_new, 1u)] = (uint8_t)tid;
            if (r == NO_ROW) full = 1;
        }
        __syncthreads();
        if (n_new) {
            const uint32_t pairs = (uint32_t)(s.D + 1) / 2;
            const float stddev = (float)(1.0 / sqrt((double)s.D));
            for (uint32_t q = tid; q < n_new * pairs; q += 256) {
                const uint32_t k = fresh[q / pairs];
                init_row_pair(s, o, seed, signs[first + k], row[k], q % pairs, stddev);
            }
            all_new += n_new;
            __syncthreads();
        }
        if (vec)
            table_rows_out<AHEAD, float4>(s, row, m, out + first * s.wdim);
        else
            table_rows_out<AHEAD, float>(s, row, m, out + first * s.wdim);
        __syncthreads();
    }
    if (tid == 0) {
        if (all_new) atomicAdd(s.count, (unsigned long long)all_new);
        __hip_atomic_store(reinterpret_cast<unsigned long long*>(host_words) + blockIdx.x,
                           (unsigned long long)seq << 32 | (unsigned long long)(full << 31 | all_new), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// --------------------------------------------------------------------- push
constexpr int TABLE_THREADS = 256;
constexpr int TABLE_WAVES = TABLE_THREADS / 64;
constexpr uint32_t TABLE_TILES = 512;        // tiles at most (every bucket's workgroup looks at all of them)
constexpr int TABLE_ITEMS_MAX = 16;          // records per thread of k_table_part
constexpr uint32_t TABLE_BUCKET_RECORDS = 128;  // records per bucket aimed at (64: a second round of workgroups, 54 us for 34)
constexpr uint32_t TABLE_BUCKETS = 2048;     // buckets at most
constexpr uint32_t TABLE_CHUNK = 512;        // records a workgroup of k_table_apply groups at a time
constexpr uint32_t TABLE_ROWS = 1024;        // entries of its LDS hash table of rows
constexpr uint32_t TABLE_BIG = 16;           // records of a chunk from which a sign is applied by a wavefront (64: +4 us)
static_assert(TABLE_ROWS > TABLE_CHUNK, "an insert always ends");

struct TableShape {
    uint32_t n;       // records
    uint32_t tile;    // records per tile: TABLE_THREADS x items
    uint32_t tiles;
    uint32_t nb;      // buckets: equal ranges of table rows
    uint32_t scale;   // nb / (rows of the table), in 2^-32
    uint32_t bits;    // of a bucket number
};

// A tile's records in order of their buckets, and in record order inside a bucket: the place of a record is the number
// of records of earlier buckets, of earlier wavefronts and of earlier lanes, which ballots over the bits of the bucket
// number tell -- no sort, no atomics whose order of arrival would show.  Records of unknown signs are dropped.
// The counters of a bucket's wavefronts stand in LDS behind each other with a free word after every 32 (part_word): the scan gives a
// thread consecutive ones, 32 of them where there are 2048 buckets, which would all be in one bank: k_table_part, 300 000 records
// 33 us and 17, 500 000 35 and 20, 1.3 M 59 and 46, 60 000 (469 buckets) 8.4 and 7.5.
__host__ __device__ constexpr uint32_t part_word(uint32_t k) { return k + (k >> 5); }
template <int ITEMS>
__global__ __launch_bounds__(TABLE_THREADS) void k_table_part(TableShape b, Store s, const tn_sign_info* __restrict__ infos,
                                                              uint2* __restrict__ recs, uint16_t* __restrict__ boff,
                                                              DevStatus* status) {
    extern __shared__ uint32_t cnt[];  // [nb][TABLE_WAVES], by part_word
    __shared__ uint32_t wsum[TABLE_WAVES];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t first = blockIdx.x * b.tile;
    uint32_t row[ITEMS], bk[ITEMS], at[ITEMS];
    bool unknown = false;
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const uint32_t i = first + wave * (64 * ITEMS) + j * 64 + lane;
        row[j] = NO_ROW;
        if (i < b.n) {
            bool is_new;
            row[j] = probe_slot<false>(s, infos[i].sign, is_new);
            unknown |= row[j] == NO_ROW;
        }
        bk[j] = row[j] == NO_ROW ? 0u : (uint32_t)(((uint64_t)row[j] * b.scale) >> 32);
    }
    for (uint32_t i = tid; i < part_word(b.nb * TABLE_WAVES); i += TABLE_THREADS) cnt[i] = 0;
    if (unknown) atomicOr(&status->err, DEV_ERR_UNKNOWN_KEY);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const bool valid = row[j] != NO_ROW;
        unsigned long long same = __ballot(valid);
        for (uint32_t q = 0; q < b.bits; q++) {
            const unsigned long long m = __ballot((bk[j] >> q) & 1u);
            same &= ((bk[j] >> q) & 1u) ? m : ~m;
        }
        at[j] = 0;
        const uint32_t k = part_word(bk[j] * TABLE_WAVES + wave);
        if (valid) at[j] = cnt[k] + (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
        wave_sync();
        if (valid && (uint32_t)__ffsll((long long)same) - 1 == lane) cnt[k] += (uint32_t)__popcll(same);
        wave_sync();
    }
    __syncthreads();
    const uint32_t total = b.nb * TABLE_WAVES, each = (total + TABLE_THREADS - 1) / TABLE_THREADS;
    uint32_t sum = 0;
    for (uint32_t q = 0; q < each; q++) {
        const uint32_t k = tid * each + q;
        sum += k < total ? cnt[part_word(k)] : 0u;
    }
    uint32_t all;
    uint32_t x = block_excl_scan<uint32_t, TABLE_WAVES>(sum, wsum, &all);
    uint16_t* off = boff + (size_t)blockIdx.x * (b.nb + 1);
    for (uint32_t q = 0; q < each; q++) {
        const uint32_t k = tid * each + q;
        if (k >= total) break;
        const uint32_t c = cnt[part_word(k)];
        cnt[part_word(k)] = x;
        if (k % TABLE_WAVES == 0) off[k / TABLE_WAVES] = (uint16_t)x;
        x += c;
    }
    if (tid == 0) off[b.nb] = (uint16_t)all;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; j++)
        if (row[j] != NO_ROW)
            recs[first + cnt[part_word(bk[j] * TABLE_WAVES + wave)] + at[j]] =
                make_uint2(row[j], first + wave * (64 * ITEMS) + j * 64 + lane);
}

// The records of one sign, by their places in LDS.
struct TableGroup {
    typedef uint32_t Entry;  // record number
    const uint16_t* sorted;
    const uint32_t* idx;
    const tn_sign_info* infos;
    const float* grads;
    int dim;
    __device__ __forceinline__ Entry entry(uint32_t j) const { return idx[sorted[j]]; }
    __device__ __forceinline__ const float* gradient(Entry e) const { return grads + (uint64_t)e * dim; }
    __device__ __forceinline__ int show(Entry e) const { return infos[e].batch_show; }
    __device__ __forceinline__ int click(Entry e) const { return infos[e].batch_click; }
    __device__ __forceinline__ void taken(uint32_t, int, int) const {}
};

// Where there are more workgroups than the chip holds of a kernel at once, two or three on a CU, a variant of which a CU holds more.
// Rounds a chunk of apply_big_wave: as in small_apply_most, and four also for Adam rows of 8 and 64, Ftrl rows of 8, 16 and 32, whose
// chunk of sixteen takes 21 to 34 KB.  us with sixteen and with four: 300 000 records of 200 times 1500 signs, Adam rows of 8 98 and 83,
// of 16 130 and 87, of 32 141 and 94, of 64 170 and 138, Ftrl rows of 8 131 and 108, of 32 149 and 127; 104 000 of 40 times 2600, Adam
// rows of 64 46.0 and 35.5, Ftrl rows of 8 37.7 and 27.2; 128 000, Adam 30.9 and 27.1, 36.8 and 27.4, 40.4 and 30.0, 47.2 and 41.3, Ftrl
// rows of 8 38.5 and 31.6, of 32 41.0 and 37.5.  Fewer, 64 000: Adam rows of 8 23.0 and 24.5, of 16 24.0 and 23.8, of 32 27.0 and 25.1,
// Ftrl rows of 32 33.2 and 33.1; 5600 24.8 and 25.4, 24.6 and 24.2, 26.5 and 25.6, 33.9 and 35.3.  Ftrl rows of 64 gain 6 % at 300 000
// and lose 5 at 104 000.  AdaGrad rows lose: of 8 (100 000 records) 45 and 54, of 64 (300 000) 166 and 234.
constexpr int table_apply_most(int kind, int big, bool many) {
    return many && ((kind == OPT_ADAM && (big == 8 || big == 64)) || (kind == OPT_FTRL && (big == 8 || big == 16 || big == 32)))
               ? 4 : small_apply_most(kind, big);
}
// Wavefronts a SIMD.  AdaGrad rows of more than 8 elements take up to 216 registers by themselves, a CU holds two workgroups; held to
// three wavefronts (168 registers, 4 to 27 spilled), us by two and by three: 300 000 records of 200 times 1500 signs, rows of 12 144 and
// 118, of 16 97 and 82, of 32 113 and 95, of 64 149 and 129; 1 040 000 of 26 times 40 000, of 12 169 and 136, of 16 136 and 114; but 60 000
// (469 workgroups) 27.9 and 28.4, 19.4 and 20.3, 22.0 and 23.0, 29.3 and 30.4.  (Four, 31 to 59 spilled: 129, 99, 104 and 164 for the
// first four.)  Rows of more than 64, of which LDS holds two workgroups at most, are the same either way: 300 000, of 66 327 and 331, of
// 128 521 and 517; 520 000 of 26 times 20 000 329 and 323, 451 and 438.
// Ftrl rows of 8 and 16 take 139 and 142, three workgroups; with four, and chunks of four rounds: rows of 16, 104 000
// records 38.3 and 29.9, 240 000 62.4 and 54.6, 300 000 118 and 101, 1 040 000 153 and 140; rows of 8, 240 000 57.4 and 48.7, the others
// the same.
constexpr int table_apply_waves(int kind, int big, int lpg, bool many) {
    return many && kind == OPT_ADAGRAD && lpg > 2 ? 3 : many && kind == OPT_FTRL && (big == 8 || big == 16) ? 4 : 1;
}
// How many workgroups the chip holds of the variant for few.
constexpr uint32_t table_apply_held(int kind) { return kind == OPT_ADAGRAD ? 512 : 768; }

inline size_t table_apply_lists_lds(uint32_t tiles) {
    // per tile: records before it, where they are; table: row, records, first place; per record: row, number, entry |
    // arrival, places in order of arrival and of records, signs with one record, with several
    return align_up((size_t)(2 * tiles + 1) * 4 + TABLE_ROWS * 12 + TABLE_CHUNK * 12 + TABLE_CHUNK * 10, 8);
}

// A bucket's records TABLE_CHUNK at a time, in record order: grouped by row in an LDS hash table, every sign's places
// put in order, the signs applied -- those with TABLE_BIG records or more by a wavefront each, the others by groups of
// LPG lanes, several records in flight.  A sign's records in the next chunk find the row as this chunk left it (the
// workgroup's own stores, behind a barrier), so any number of records of a sign is taken in order.  Bound by chains of
// dependent reads (12 us to group a bucket's records, then the longest sign); the lists are short so that three
// workgroups fit on a CU (a chunk of 1536 records left room for one: 59 us for 34 at 60 000 records).  Rows of a power of two up to
// 64 elements have the long signs taken by apply_big_wave (BIG > 0), the others by apply_big_groups (60 000 records of 40 times
// 1500 signs, AdaGrad rows of 16: 28 us by the latter, 19.5 by the former).
template <int KIND, int LPG, bool ANY, int BIG, int MOST, int WAVES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES, 8))) void k_table_apply(TableShape b, Store s, OptDev o, const tn_sign_info* __restrict__ infos,
                                                     const float* __restrict__ grads, int dim, const uint2* __restrict__ recs,
                                                     const uint16_t* __restrict__ boff, DevStatus* status, uint32_t* host_err,
                                                     int gbuf_floats, uint32_t wave_lds, uint32_t wave_arrays,
                                                     uint32_t lists_lds) {
    extern __shared__ uint32_t lds[];
    uint32_t* spre = lds;                       // [tiles + 1]
    uint32_t* sst = spre + b.tiles + 1;         // [tiles]
    uint32_t* trow = sst + b.tiles;             // [TABLE_ROWS]
    uint32_t* tcnt = trow + TABLE_ROWS;
    uint32_t* toff = tcnt + TABLE_ROWS;
    uint32_t* rrow = toff + TABLE_ROWS;         // [TABLE_CHUNK]
    uint32_t* ridx = rrow + TABLE_CHUNK;
    uint32_t* rent = ridx + TABLE_CHUNK;        // entry | arrival << 16
    uint16_t* arrived = reinterpret_cast<uint16_t*>(rent + TABLE_CHUNK);
    uint16_t* sorted = arrived + TABLE_CHUNK;
    uint16_t* single = sorted + TABLE_CHUNK;
    uint16_t* multi = single + TABLE_CHUNK;     // entries
    uint16_t* big = multi + TABLE_CHUNK;        // [TABLE_CHUNK], entries
    __shared__ uint32_t wsum[4];
    __shared__ uint32_t n_single, n_multi, n_big, n_places, next_round;
    const uint32_t tid = threadIdx.x, bucket = blockIdx.x;
    if (bucket == 0 && tid == 0) {  // the call's errors (the partition has them all) for the host to find when it next waits
        __hip_atomic_store(host_err, status->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        status->err = 0;
    }
    uint32_t m = 0;
    for (uint32_t t0 = 0; t0 < b.tiles; t0 += 256) {
        const uint32_t t = t0 + tid;
        uint32_t c = 0;
        if (t < b.tiles) {
            const uint16_t* off = boff + (size_t)t * (b.nb + 1) + bucket;
            c = (uint32_t)off[1] - off[0];
            sst[t] = t * b.tile + off[0];
        }
        uint32_t total;
        const uint32_t x = m + block_excl_scan<uint32_t, 4>(c, wsum, &total);
        if (t < b.tiles) spre[t] = x;
        m += total;
    }
    if (tid == 0) spre[b.tiles] = m;
    const int sub = tid % LPG;
    const float c1 = 1 - o.beta1, c2 = 1 - o.beta2;
    TableGroup grp;
    grp.idx = ridx;
    grp.infos = infos;
    grp.grads = grads;
    grp.dim = dim;
    for (uint32_t done = 0; done < m; done += TABLE_CHUNK) {
        const uint32_t c = min(TABLE_CHUNK, m - done);
        uint32_t table = 64;
        while (table < c + c / 4) table *= 2;
        for (uint32_t i = tid; i < table; i += 256) {
            trow[i] = NO_ROW;
            tcnt[i] = 0;
        }
        if (tid == 0) n_single = n_multi = n_big = n_places = next_round = 0;
        __syncthreads();
        for (uint32_t i = tid; i < c; i += 256) {
            const uint32_t t = (uint32_t)find_slot(spre, (int)b.tiles, done + i);
            const uint2 r = recs[sst[t] + (done + i - spre[t])];
            uint32_t e = ((r.x * 2654435761u) >> 12) & (table - 1);
            for (;;) {  // more entries than records
                uint32_t old = trow[e];
                if (old == NO_ROW) old = atomicCAS(&trow[e], NO_ROW, r.x);
                if (old == NO_ROW || old == r.x) break;
                e = (e + 1) & (table - 1);
            }
            rrow[i] = r.x;
            ridx[i] = r.y;
            rent[i] = e | (atomicAdd(&tcnt[e], 1u) << 16);
        }
        __syncthreads();
        for (uint32_t i = tid; i < c; i += 256) {
            const uint32_t e = rent[i] & 0xFFFFu, k = tcnt[e];
            if (k == 1) {
                single[atomicAdd(&n_single, 1u)] = (uint16_t)i;
            } else if ((rent[i] >> 16) == 0) {
                toff[e] = atomicAdd(&n_places, k);
                if (k >= TABLE_BIG)
                    big[atomicAdd(&n_big, 1u)] = (uint16_t)e;
                else
                    multi[atomicAdd(&n_multi, 1u)] = (uint16_t)e;
            }
        }
        __syncthreads();
        for (uint32_t i = tid; i < c; i += 256) {
            const uint32_t e = rent[i] & 0xFFFFu;
            if (tcnt[e] > 1) arrived[toff[e] + (rent[i] >> 16)] = (uint16_t)i;
        }
        __syncthreads();
        for (uint32_t i = tid; i < c; i += 256) {
            const uint32_t e = rent[i] & 0xFFFFu, k = tcnt[e];
            if (k == 1) continue;
            const uint32_t at = toff[e];
            uint32_t place = 0;
            for (uint32_t j = 0; j < k; j += 8) {  // eight reads in flight
                uint32_t v[8];
#pragma unroll
                for (uint32_t q = 0; q < 8; q++) v[q] = arrived[at + min(j + q, k - 1)];
#pragma unroll
                for (uint32_t q = 0; q < 8; q++) place += j + q < k && v[q] < i ? 1u : 0u;
            }
            sorted[at + place] = (uint16_t)i;
        }
        __syncthreads();
        // The wavefronts take the long signs first, then 64 / LPG short ones at a time: those that have no long sign
        // (10 us for 40 records) go on meanwhile.
        const int wave = (int)(tid >> 6), lane = (int)(tid & 63);
        if constexpr (BIG > 0) {
            __shared__ BigWave<KIND, BIG, MOST> tiles[TABLE_WAVES];
            auto group = [&](uint32_t bi) {
                const uint32_t e = big[bi];
                return make_uint4(trow[e], toff[e], tcnt[e], 0u);
            };
            apply_big_wave<KIND, BIG>(
                s, o, tiles[wave], (uint32_t)wave < n_big ? group((uint32_t)wave) : make_uint4(NO_ROW, 0, 0, 0), (uint32_t)wave,
                (uint32_t)TABLE_WAVES, n_big, group, [&](uint32_t at) { return ridx[sorted[at]]; },
                [&](uint32_t e, const float*& gp, int& sh, int& ck, bool) {
                    gp = grads + (uint64_t)e * dim;
                    sh = infos[e].batch_show;
                    ck = infos[e].batch_click;
                    return true;
                },
                [] {});
        } else if (n_big) {
            char* base = reinterpret_cast<char*>(lds) + lists_lds + (size_t)wave * wave_lds;
            float* gbuf = reinterpret_cast<float*>(base);
            const float** gptr = reinterpret_cast<const float**>(base + wave_arrays);
            float* den = reinterpret_cast<float*>(gptr + BIG_CHUNK);
            apply_big_groups<KIND>(
                s, o, gbuf_floats, gbuf, gptr, den, lane, (uint32_t)wave, (uint32_t)TABLE_WAVES, n_big,
                [&](uint32_t bi, uint32_t& row, uint32_t& off, uint32_t& k) {
                    const uint32_t e = big[bi];
                    row = trow[e];
                    off = toff[e];
                    k = tcnt[e];
                },
                [&](uint32_t at, const float*& gp, int& sh, int& ck) {
                    const uint32_t e = ridx[sorted[at]];
                    gp = grads + (uint64_t)e * dim;
                    sh = infos[e].batch_show;
                    ck = infos[e].batch_click;
                    return true;
                },
                [] {}, [] { wave_sync(); });
        }
        const uint32_t rounds_multi = (n_multi + 64 / LPG - 1) / (64 / LPG);
        const uint32_t rounds = rounds_multi + (n_single + 64 / LPG - 1) / (64 / LPG);
        for (;;) {
            uint32_t r = 0;
            if (lane == 0) r = atomicAdd(&next_round, 1u);
            r = (uint32_t)__builtin_amdgcn_readfirstlane((int)r);
            if (r >= rounds) break;
            if (r < rounds_multi) {
                const uint32_t g = r * (64 / LPG) + lane / LPG;
                if (g < n_multi) {
                    const uint32_t e = multi[g];
                    grp.sorted = sorted + toff[e];
                    apply_group_ahead<KIND, LPG, ANY, 4, false>(s, o, grp, trow[e], tcnt[e], sub, c1, c2);
                }
            } else {
                const uint32_t g = (r - rounds_multi) * (64 / LPG) + lane / LPG;
                if (g < n_single) {
                    const uint32_t i = single[g], e = ridx[i];
                    apply_one_record<KIND, LPG, ANY>(s, o, rrow[i], grads + (uint64_t)e * dim, infos[e].batch_show,
                                                     infos[e].batch_click, sub, c1, c2);
                }
            }
        }
        __syncthreads();
    }
}

}  // namespace tn

#endif  // TN_TABLE_LEVEL_H_
