// The backward half of the combiner in LDS: up to POOL_ITEMS_MAX lookups of a slot, in the order of their positions, are
// sorted by their sign and every sign's pooled rows summed.  What both paths of a push of pooled gradients are made of
// (k_reduce_pooled, k_small_pool).
#ifndef TN_POOL_ITEMS_H_
#define TN_POOL_ITEMS_H_

#include "sparse_kernels.h"

namespace tn {

constexpr int POOL_THREADS = 512;
constexpr uint32_t POOL_ITEMS_MAX = 2048;
constexpr uint32_t POOL_ITEMS = POOL_ITEMS_MAX / POOL_THREADS;
constexpr uint32_t POOL_WAVES = POOL_THREADS / 64;
constexpr uint32_t POOL_RUN = POOL_ITEMS_MAX / POOL_WAVES;  // consecutive places of a wavefront, of all of them
constexpr uint32_t POOL_WORDS = POOL_ITEMS_MAX / 64;
constexpr uint32_t POOL_PIECE = 16;  // places of a piece; a half, a quarter where there are half, a quarter as many items
constexpr uint32_t POOL_PIECES = POOL_ITEMS_MAX / POOL_PIECE;
constexpr uint32_t POOL_AHEAD = 4;  // rows of a group of lanes in flight (eight: the registers of a workgroup of four do not hold them)
constexpr uint32_t POOL_DIGIT = 7;  // (10, one pass for most slots, whose 8192 counters take longer: 44 -> 47 us, 175 -> 184)
static_assert(POOL_AHEAD == 4 && POOL_PIECE / 4 % POOL_AHEAD == 0, "items are read four at a time");
enum { POOL_SUM = 0, POOL_MEAN = 1, POOL_SQRTN = 2 };  // (the combiners of the C ABI)
static_assert(POOL_RUN == 64 * POOL_ITEMS && 64 % POOL_PIECE == 0, "whole wavefronts, pieces inside a word");

// 37 KB: four workgroups of eight wavefronts to a CU (45 KB and three of them: 4.9 M lookups 161 us, so 148; twice the size in
// workgroups of sixteen: one to a CU, 2.5 times as long).  The sort's last pass moves the items themselves, so that its orders
// and what the pieces leave can share their room, and a piece's own sum stays in its lanes' registers.
struct PoolLds {
    alignas(16) uint32_t key[POOL_ITEMS_MAX];      // the lookup's sign (in the end the lookups are in the order of their signs)
    alignas(16) uint32_t example[POOL_ITEMS_MAX];  // its example
    alignas(16) float scale[POOL_ITEMS_MAX];       // 1 / d(lookups of the example); negative: not its sign's first lookup
    uint16_t ord[POOL_ITEMS_MAX];      // while sorting: the order after every other pass,
    union {
        struct {
            uint16_t half[POOL_ITEMS_MAX];             // ... after the others,
            uint16_t digit[POOL_WAVES << POOL_DIGIT];  // counters
        };
        float4 part[POOL_PIECES][4];  // then: what a piece has of a sign that began before it
        uint32_t list[2 * POOL_THREADS + 1];  // (before: k_reduce_pooled's tiles)
    };
    unsigned long long heads[POOL_WORDS];  // starts of the signs in the order
    uint32_t wsum[POOL_WAVES];
};

// Last set bit at or below i, first one above it (or `none`), in a bitmap in LDS.
__device__ __forceinline__ uint32_t bit_at_or_below(const unsigned long long* bm, uint32_t i) {
    uint32_t w = i >> 6;
    unsigned long long v = bm[w] & (~0ull >> (63 - (i & 63)));
    while (v == 0) v = bm[--w];  // (bit 0 is set)
    return w * 64 + 63 - (uint32_t)__clzll((long long)v);
}
__device__ __forceinline__ uint32_t bit_above(const unsigned long long* bm, uint32_t i, uint32_t words, uint32_t none) {
    uint32_t w = i >> 6;
    unsigned long long v = (i & 63) == 63 ? 0ull : bm[w] & (~0ull << ((i & 63) + 1));
    while (v == 0) {
        if (++w >= words) return none;
        v = bm[w];
    }
    return w * 64 + (uint32_t)__ffsll((long long)v) - 1;
}

__device__ __forceinline__ float pool_scale(float count, int combiner) {
    return combiner == POOL_SUM ? 1.f : 1.f / (combiner == POOL_MEAN ? count : sqrtf(count));
}

// lds.key, example, scale [0, n) are filled, keys of `bits` bits, n > 0.  A stable radix sort (passes of up to 7 bits,
// a wavefront's lanes told apart by ballots); then every group of LPG lanes takes a piece of consecutive places of the order,
// whatever signs they hold, POOL_AHEAD rows in flight, sixteen elements of them at a time (LPG 4).  (A group per sign has one
// row in flight where most signs have one lookup, and waits for the longest of its wavefront: twice as long.)  A sign
// with lookups in several pieces: their shares are added in order.  row(key, first, add): where its sum goes, and whether it
// is added to what stands there; first: the sign's first lookup is among those summed.
template <int LPG, bool ANY, typename Row>
__device__ __forceinline__ void pool_items(PoolLds& lds, uint32_t n, uint32_t bits, const float* __restrict__ pooled, int dim,
                                           int D, Row row) {
    static_assert(LPG <= 4, "PoolLds::part");
    uint32_t tid = threadIdx.x;
    // (addresses worked out from here on stay inside the round: held in registers across the caller's loop they cost a
    // workgroup of the four)
    asm volatile("" : "+v"(tid));
    const uint32_t lane = tid & 63, wave = tid >> 6;
    // Turns of 64 items that the wavefronts take, and the consecutive items of one: as few as n asks for, so that all wavefronts have
    // their share of them.  (Always four of each: 349 lookups in one slot, k_small_pool 17.4 us, 20 slots of 500 16.1; so 11.8 and
    // 12.0, with the shorter pieces below.  k_reduce_pooled, 4.9 M lookups in parts of 1600 on average, 151 and 139.)
    const uint32_t turns = (n + POOL_THREADS - 1) / POOL_THREADS, run = turns * 64;
    const uint32_t passes = (bits + POOL_DIGIT - 1) / POOL_DIGIT, width = passes ? (bits + passes - 1) / passes : 0u;
    __syncthreads();
    for (uint32_t pass = 0; pass < passes; pass++) {
        uint16_t* const to = pass & 1u ? lds.ord : lds.half;
        const uint16_t* const from = pass & 1u ? lds.half : lds.ord;  // (the first pass takes them as they are)
        for (uint32_t i = tid; i < POOL_WAVES << width >> 1; i += POOL_THREADS) reinterpret_cast<uint32_t*>(lds.digit)[i] = 0;
        __syncthreads();
        uint32_t item[POOL_ITEMS], dg[POOL_ITEMS], at[POOL_ITEMS];
#pragma unroll
        for (uint32_t j = 0; j < POOL_ITEMS; j++) {
            const uint32_t i = wave * run + j * 64 + lane;
            item[j] = j < turns && i < n ? (pass == 0 ? i : (uint32_t)from[i]) : 0u;
        }
#pragma unroll
        for (uint32_t j = 0; j < POOL_ITEMS; j++) {
            dg[j] = at[j] = 0;
            if (j >= turns) continue;
            const bool valid = wave * run + j * 64 + lane < n;
            dg[j] = (lds.key[item[j]] >> (pass * width)) & ((1u << width) - 1u);
            unsigned long long same = __ballot(valid);
            for (uint32_t q = 0; q < width; q++) {
                const unsigned long long m = __ballot((dg[j] >> q) & 1u);
                same &= ((dg[j] >> q) & 1u) ? m : ~m;
            }
            const uint32_t k = dg[j] * POOL_WAVES + wave;
            if (valid) at[j] = lds.digit[k] + (uint32_t)__popcll(same & ((1ull << lane) - 1ull));  // (before this round)
            wave_sync();
            if (valid && (uint32_t)__ffsll((long long)same) - 1 == lane) lds.digit[k] += (uint16_t)__popcll(same);
            wave_sync();
        }
        __syncthreads();
        {  // digit by digit and wavefront by wavefront: where they go
            const uint32_t all = POOL_WAVES << width, each = (all + POOL_THREADS - 1) / POOL_THREADS, k0 = tid * each;
            uint32_t sum = 0;
            for (uint32_t k = k0; k < min(k0 + each, all); k++) sum += lds.digit[k];
            uint32_t x = block_excl_scan<uint32_t, POOL_WAVES>(sum, lds.wsum, nullptr);
            for (uint32_t k = k0; k < min(k0 + each, all); k++) {
                const uint32_t c = lds.digit[k];
                lds.digit[k] = (uint16_t)x;
                x += c;
            }
        }
        if (pass + 1 < passes) {
            __syncthreads();
#pragma unroll
            for (uint32_t j = 0; j < POOL_ITEMS; j++)
                if (j < turns && wave * run + j * 64 + lane < n) to[lds.digit[dg[j] * POOL_WAVES + wave] + at[j]] = (uint16_t)item[j];
        } else {  // the last one moves the items themselves
            uint32_t key[POOL_ITEMS], example[POOL_ITEMS];
            float scale[POOL_ITEMS];
#pragma unroll
            for (uint32_t j = 0; j < POOL_ITEMS; j++) {
                key[j] = lds.key[item[j]];
                example[j] = lds.example[item[j]];
                scale[j] = lds.scale[item[j]];
            }
            __syncthreads();
#pragma unroll
            for (uint32_t j = 0; j < POOL_ITEMS; j++) {
                if (j >= turns || wave * run + j * 64 + lane >= n) continue;
                const uint32_t place = lds.digit[dg[j] * POOL_WAVES + wave] + at[j];
                lds.key[place] = key[j];
                lds.example[place] = example[j];
                lds.scale[place] = scale[j];
            }
        }
        __syncthreads();
    }
    // starts of the signs in the order (and what lies behind it)
#pragma unroll
    for (uint32_t j = 0; j < POOL_ITEMS; j++) {
        const uint32_t i = wave * POOL_RUN + j * 64 + lane;
        const bool head = i >= n || i == 0 || lds.key[i] != lds.key[i - 1];
        const unsigned long long m = __ballot(head);
        if (lane == 0) lds.heads[i >> 6] = m;
    }
    __syncthreads();
    // (a piece is a chain of round trips: shorter ones where the groups of lanes are enough for them)
    const uint32_t piece = n > POOL_ITEMS_MAX / 2 ? POOL_PIECE : n > POOL_ITEMS_MAX / 4 ? POOL_PIECE / 2 : POOL_PIECE / 4;
    const uint32_t pieces = (n + piece - 1) / piece;
    asm volatile("" : "+v"(tid));
    const int sub = tid % LPG;
    auto put = [&](uint32_t key, bool first, int c0, float4 v) {
        bool add;
        float* out = row(key, first, add) + c0;
        if (add) {
            const float4 w = row_part<ANY>(out, sub, D - c0);
            v = make_float4(w.x + v.x, w.y + v.y, w.z + v.z, w.w + v.w);
        }
        put_row_part<ANY>(out, sub, D - c0, v);
    };
    // a piece per group of lanes
    static_assert(POOL_THREADS / 4 >= POOL_PIECES, "there are as many");
    const uint32_t q = tid / LPG, lo = q * piece, hi = lo + piece;
    for (int c0 = 0; c0 < D; c0 += 4 * LPG) {
        bool began = false, goes_on = false;  // the running sum's sign: began in the piece, goes on behind it
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        if (q < pieces) {
            // which places start a sign, and the one behind the piece (those behind the last lookup do)
            uint32_t hb = (uint32_t)(lds.heads[lo >> 6] >> (lo & 63)) & ((1u << piece) - 1u);
            if (hi >= n || ((lds.heads[hi >> 6] >> (hi & 63)) & 1ull)) hb |= 1u << piece;
            bool first = false;  // (the running sum has its sign's first lookup)
#pragma unroll 1
            for (uint32_t j0 = 0; j0 < piece && lo + j0 < n; j0 += POOL_AHEAD, hb >>= POOL_AHEAD) {
                float4 g[POOL_AHEAD];
                const uint4 e4 = *reinterpret_cast<const uint4*>(lds.example + lo + j0);
                const float4 s4 = *reinterpret_cast<const float4*>(lds.scale + lo + j0);
                const uint32_t example[POOL_AHEAD] = {e4.x, e4.y, e4.z, e4.w};
                const float sc[POOL_AHEAD] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
                for (uint32_t w = 0; w < POOL_AHEAD; w++) {
                    const uint32_t e = lo + j0 + w < n ? example[w] : 0u;  // (behind the last item: some row or other)
                    g[w] = row_part<ANY>(pooled + (uint64_t)e * dim + c0, sub, D - c0);
                }
#pragma unroll
                for (uint32_t w = 0; w < POOL_AHEAD; w++) {
                    if (lo + j0 + w >= n) break;
                    if ((hb >> w) & 1u) {
                        acc = make_float4(0.f, 0.f, 0.f, 0.f);
                        began = true;
                        first = sc[w] > 0.f;
                    }
                    const float scale = fabsf(sc[w]);
                    acc.x += g[w].x * scale;
                    acc.y += g[w].y * scale;
                    acc.z += g[w].z * scale;
                    acc.w += g[w].w * scale;
                    if ((hb >> (w + 1)) & 1u) {  // the sign ends here
                        if (began)
                            put(lds.key[lo + j0 + w], first, c0, acc);
                        else
                            lds.part[q][sub] = acc;
                    }
                }
            }
            goes_on = !(hb & 1u);
            if (goes_on && !began) lds.part[q][sub] = acc;
        }
        __syncthreads();
        if (goes_on && began) {  // with what the pieces behind have of it, in order
            const uint32_t from = bit_at_or_below(lds.heads, hi - 1);
            const uint32_t end = bit_above(lds.heads, hi, POOL_WORDS, n), last = (end - 1) / piece;
            for (uint32_t r = q + 1; r <= last; r += 4) {
                float4 g[4];
#pragma unroll
                for (uint32_t w = 0; w < 4; w++) g[w] = lds.part[min(r + w, last)][sub];
#pragma unroll
                for (uint32_t w = 0; w < 4; w++) {
                    if (r + w > last) break;
                    acc.x += g[w].x;
                    acc.y += g[w].y;
                    acc.z += g[w].z;
                    acc.w += g[w].w;
                }
            }
            put(lds.key[from], lds.scale[from] > 0.f, c0, acc);
        }
        __syncthreads();
    }
}

// The sum of a sign whose lookups were dealt to `parts` workgroups, by a wavefront: its groups of LPG lanes take every so many of
// the parts in turn and then add their sums up by halves.  has(q): part q has a share; share(q): its row.
template <int LPG, bool ANY, typename Has, typename Share>
__device__ __forceinline__ void add_shares(uint32_t parts, int D, Has has, Share share, float* __restrict__ out) {
    const uint32_t group = (uint32_t)__lane_id() / LPG;
    const int sub = (int)__lane_id() % LPG;
    for (int c0 = 0; c0 < D; c0 += 4 * LPG) {
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        for (uint32_t q = group; q < parts; q += 64 / LPG) {
            if (!has(q)) continue;
            const float4 v = row_part<ANY>(share(q) + c0, sub, D - c0);
            acc.x += v.x;
            acc.y += v.y;
            acc.z += v.z;
            acc.w += v.w;
        }
#pragma unroll
        for (int o = 32; o >= LPG; o >>= 1) {
            acc.x += __shfl_xor(acc.x, o);
            acc.y += __shfl_xor(acc.y, o);
            acc.z += __shfl_xor(acc.z, o);
            acc.w += __shfl_xor(acc.w, o);
        }
        if (group == 0) put_row_part<ANY>(out + c0, sub, D - c0, acc);
    }
}

}  // namespace tn

#endif  // TN_POOL_ITEMS_H_
