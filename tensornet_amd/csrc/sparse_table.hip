// SparseTable host side: registry, HBM storage management and the launch
// sequences of pull / push at table level (core/ps/table/sparse_table.cc:52-83)
// and at operator level (core/kernels/sparse_table_ops.cc:170-265,317-368).
#include "apply_launch.h"
#include "combine_kernels.h"
#include "host_work.h"
#include "remap_lds.h"
#include "row_width.h"
#include "table_level.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <thread>
#include <type_traits>

// Device memory of tn_sparse_table_pull_static, the one entry point that allocates nothing: the call's
// status block, then the row number and the new-row list of every requested sign.  Every GPU the library
// runs on holds its own copy until the process ends; host code reaches it through the address that
// hipGetSymbolAddress returns for the current device (static_scratch below), never through this name.
constexpr int64_t TN_STATIC_MAX_SIGNS = 1 << 20;
constexpr size_t TN_STATIC_STATUS_BYTES = 256;
constexpr size_t TN_STATIC_SCRATCH_BYTES = TN_STATIC_STATUS_BYTES + 2 * (size_t)TN_STATIC_MAX_SIGNS * sizeof(uint32_t);
static __device__ __align__(256) unsigned char scratch[TN_STATIC_SCRATCH_BYTES];

namespace tn {

namespace {

constexpr double MAX_LOAD = 0.75;                       // optimizer_kernel.h:266
constexpr double RESERVE_LOAD = 0.5;                    // what a reservation is sized for where memory allows
constexpr uint64_t DEFAULT_SLOTS = 8ull * 15485863ull;  // optimizer_kernel.h:43,263
constexpr uint64_t MAX_SLOTS_PER_TABLE = 0xFFFFFFF0ull; // rows are addressed with 32 bits
constexpr size_t DETACH_LOOKUPS = 3u << 20;  // lookups of a push from which its updates may be detached
constexpr uint32_t SELF_SCAN_TILES = 8192;  // tiles of the ranking pass up to which no scan kernel runs between its launches
constexpr int GRID_CAP = 256 * 8;                       // 256 CUs x 8 workgroups of 256 threads
constexpr int TILE_GRID = 256 * 4;                      // workgroups of k_tile_dedup: what the chip holds of it at once
constexpr size_t PULL_WORDS = std::max<size_t>(SMALL_WORKGROUPS, TABLE_PULL_WORDS);
constexpr uint32_t COMBINE_EXAMPLES = 64;  // examples per workgroup of k_combine_fwd at least
constexpr int COMBINE_DIRECT = 1024;       // workgroups of it up to which they read the slots' descriptors from pinned host memory
constexpr size_t LDS_MIN_LOOKUPS = 1024;  // from here on the remap through LDS wins: it also takes fewer launches (cfg1, 8 k lookups: 0.154 -> 0.136 ms)

// Which batches take the path of few launches (small_batch.h), beside those its arrays have room for (SMALL_SLOT_MAX
// lookups a slot, SMALL_SLOTS slots, the LDS its kernels may have).  Up to SMALL_MAX_LOOKUPS lookups, and where the other
// path groups through LDS (GRP_SLOTS slots), up to SMALL_WORK slots x lookups: every bucket's workgroup looks at all
// slots, and a slot has one workgroup from 129 slots on, so that both grow with slots x lookups where the other path
// grows with the lookups.  Push and pull of rows of 16 elements under AdaGrad, us, few launches / the other path:
//   lookups a slot    1024        2048        3072        4096
//    26 slots        42 / 114    46 / 112    53 / 122    60 / 119   (the limit of 4096 is that of the field widths)
//    64              54 / 115    68 / 117    78 / 126    85 / 126
//   128              81 / 132   104 / 135   120 / 152   133 / 151
//   192             110 / 149   139 / 159   201 / 189   231 / 195
//   254             148 / 167   220 / 182   275 / 226   339 / 242
// Slots of more than 4096 lookups (k_small_slots_long): 20 slots of 6000, AdaGrad rows of 16, 52 / 128 us, 40 of 8192, Ftrl rows
// of 1, 71 / 142, 100 of 8000, Adam rows of 16, 138 / 171.  Up to SMALL_SPLIT_SLOTS of them stay with the other path, where
// tests/test_gpu_small.py wants 3 and 8 slots of 4097.  They lose by it: AdaGrad rows of 16, one slot of 4097 to 8192 lookups
// 32 to 37 us here and 92 to 96 there, two 34 to 40 and 95 to 113, four 35 to 43 and 100 to 115, eight 38 to 48 and 101 to 115.
// They cross at 89 to 106 M slots x lookups (160 to 254 slots; rows of 64: 58 to 90, of 8 under Adam: 120; pulls alone: 115).
// With pooled gradients, whose reduction is shorter here, at 180 M (192 slots, 700 k lookups: 1.08 times as fast, 254 and
// 700 k: 1.02, 850 k: 0.96).  A pull does not know what push will follow: it goes by the table's last one.
// With more than GRP_SLOTS slots the other path is 1.2 to 2.2 times as long wherever this one has room (260 slots, 1 M
// lookups: 1.29; 300, 850 k: 1.24; 400, 400 k: 1.28; 512, 131 k: 1.47).
constexpr size_t SMALL_MAX_LOOKUPS = 1u << 20;
constexpr size_t SMALL_WORK = 100'000'000, SMALL_WORK_POOLED = 180'000'000;

// A small batch of at most this many slots leaves every sign to the lane groups of k_small_apply.  With more slots a
// sign with SMALL_BIG_GROUP records or more is taken by a wavefront of its own: a small batch's kernels are as long as
// their longest chain, and the records of a sign applied one after the other by a lane group (four elements per lane)
// take four times as long as by a wavefront with a lane per element (measured, 4096 x 26 slots, Adam: the updates take
// 0.040 ms with every sign left to the lane groups, 0.020 ms with the threshold at 5; 1024 x 8 slots: no difference
// between 4 and 12 slots here).
constexpr int SMALL_NO_BIG_SLOTS = 12;
constexpr uint32_t SMALL_BIG_GROUP = 5;  // (k_small_apply takes the signs with fewer in one go)
constexpr uint32_t BIG_GROUP_DEFAULT = 16;

// What a small pull has left to do behind its first launch takes one launch (k_small_pull_rest: 26 slots of 4096 lookups
// 8.7 us, as two launches 7.0 + 7.2 and the gap), unless the buckets' workgroups want so much dynamic LDS, which all
// workgroups of a launch are given, that fewer than four would be on a CU.  Up to SMALL_SPLIT_SLOTS slots it stays two
// launches, the sequence tests/test_gpu_small.py wants at 8 slots, which one would beat there, too: a step of 4 slots of 256
// lookups 32.8 us as two launches, 32.0 as one, of 8 of 1024 36.3 and 34.4, of 8 of 4096 42.0 and 39.4.
constexpr int SMALL_SPLIT_SLOTS = 8;  // (up to as many, slots are short, too: small_batch_shape)
// Parts of rows from which a thread of small_finish takes two: up to here more workgroups are the shorter way.
constexpr size_t FINISH_FULL = 1 << 17;
constexpr size_t SMALL_SHARED_LDS = 36 * 1024;

struct HostStatus {
    DevStatus st;
    uint32_t ubase[MAX_SLOTS + 1];
};

struct SparseTable {
    std::shared_ptr<OptConf> opt;
    std::string name, group;
    int dim = 0, use_cvm = 0, shard_num = 1, self_shard_id = 0;
    uint32_t handle = 0;
    int device = 0;
    uint64_t seed = 0x243F6A8885A308D3ull;
    uint64_t reserve_keys = 0;
    bool allocated = false;
    Store store{};
    uint64_t count_upper = 0;  // upper bound of resident keys known without a device read
    uint64_t booked = 0;       // part of count_upper booked for the inserts of the pending call

    DevBuf ws;                      // per-call scratch
    DevBuf plan_buf;                // what the last pull op worked out about its batch (see Plan)
    bool plan_valid = false;
    bool plan_has_show = false;     // the plan already holds batch_show of every distinct sign
    int plan_N = 0;
    std::vector<int64_t> plan_lens;
    uint64_t epoch = 0;             // bumped whenever rows move (growth)
    uint64_t plan_epoch = 0;
    DevStatus* dstatus = nullptr;   // device: status of table-level calls
    DevStatus* dplan = nullptr;     // device: status / counts of the op-level plan
    DevStatus* dtpush = nullptr;    // device: error flags of a table-level push (zero between calls)
    DevStatus* dcomb = nullptr;     // device: error flags of a combine op (zero between calls)
    DevStatus* dpush = nullptr;     // device: status of a push that reuses the plan (the plan's counts, flags of its own)
    HostStatus* hpull = nullptr;    // pinned
    HostStatus* hpush = nullptr;    // pinned
    unsigned long long* hcount = nullptr;  // pinned: the number of resident keys is read into it
    char* hstage = nullptr;         // pinned staging of slot descriptors
    size_t hstage_bytes = 0;
    hipEvent_t stage_ev = nullptr;  // staging buffer free again
    DevBuf comb_buf;                // slot descriptors of a combine op
    DevBuf pooled_ws;               // scratch of a push of pooled gradients (items of the lookups, reduced rows)
    // The path of few launches for small batches: the words in pinned memory its kernels report through (hwords: one
    // per workgroup of a small pull's first launch, or of a table-level pull's; hseq [0] a large pull's status is on the host, [1] a push's signs are
    // compared) with the numbers the host expects there next, the dynamic LDS its kernels may have.
    uint64_t* hwords = nullptr;
    uint64_t* hcomb = nullptr;         // pinned: what a combine op reports (k_report), and that a table-level pull has ended
    uint32_t seq_comb = 0;
    uint32_t* hseq = nullptr;
    uint32_t seq_pull = 0, seq_verify = 0;
    bool plan_heavy = false;        // the pull that left the plan (small, or through LDS) found a sign with HEAVY_LOOKUPS lookups in a slot
    std::vector<int64_t> plan_counts;  // distinct signs per slot of the pull that left the plan
    SmallShape small_shape{};          // how that pull laid its batch out
    size_t small_lds = 0, small_emit_lds = 0;
    bool table_lds[4] = {};  // k_table_apply (rows in 16-byte pieces / any, few / many workgroups) has been told how much it may have
    bool plan_small = false;   // the plan was left by a small pull: a push may take the small path, too
    bool plan_prints = false;  // the plan holds fingerprints of the batch's signs, not a copy of them
    bool exact_verify = false; // pulls that leave fingerprints keep a copy of the signs as well, pushes compare that
    bool plan_exact = false;   // the plan holds such a copy
    uint32_t plan_big_k = BIG_GROUP_DEFAULT;  // records from which the plan lists a sign as one for k_apply_big
    bool plan_big_desc = false;               // the plan's big_desc goes with its big_list (a pull grouped through LDS)
    hipStream_t side = nullptr;     // the signs with several records of detached updates are applied here
    hipStream_t aux = nullptr;      // k_apply_single of detached updates runs here
    hipEvent_t fork_ev = nullptr;   // detached updates may start
    hipEvent_t apply_ev = nullptr;  // the detached updates on the auxiliary stream are done
    // Detached updates (tn_sparse_table_set_detached_updates): the update kernels of a large push run on the
    // table's own streams and the caller's stream does not wait for them, so that whatever the caller queues next
    // -- above all the analysis of the next pull's batch, which touches no table row -- runs beside them.
    // upd_ev marks their end (and that of the push's status); every call on the table orders its stream behind
    // it before it touches a row, the plan's groups or the table's memory (order_after_updates).
    bool detach_updates = false;
    bool detached_now = false;      // the push being queued has its updates detached
    bool upd_pending = false;       // upd_ev has been recorded and no host-side wait has covered it since
    hipEvent_t upd_ev = nullptr;
    // what the detached kernels read of the plan buffer: the slot arrays at its head (laid out by the slot count)
    // and the groups from upd_groups_off on, less the first upd_slack bytes (the groups' signs, which they leave alone)
    int upd_N = 0;
    size_t upd_groups_off = 0, upd_slack = 0;
    bool push_on_side = false;  // the pending push's updates end on the side stream (detached)
    // A pull whose status is final before its last kernel (the gather) publishes it by that kernel's first workgroup
    // and returns when it is there: tail_ev = the gather is done (what a call on another stream has to wait for).
    hipEvent_t tail_ev = nullptr;
    bool tail_recorded = false;
    bool tail_owed = false;         // ... was on the default stream, which is there for good: recorded when another stream asks
    bool several_streams = false;   // a call has come on another stream than the one before it
    bool plan_clicks_dirty = false;  // a push has added clicks to the member lists of the current plan
    // Distinct records per lookup seen by the recent pulls (1 = every lookup distinct, the safe start):
    // sizes the number of second-level buckets, whose room is fixed.  A batch with more distinct
    // records than expected overflows a bucket and takes the fallback path once; the estimate is then reset.
    double distinct_est = 1.0;
    // Records a tile of the remap through LDS hands to the first-level buckets per lookup (1 = no sign repeats
    // inside a tile, the safe start), for the slot where that share is largest: sizes the first-level buckets,
    // whose room is fixed, with the same fallback as above.
    double tile_est = 1.0;
    uint64_t pull_lookups = 0;  // lookups of the pull whose status is pending
    // The staging buffer is being read by a call that has not waited for that: stage_ev has been recorded behind it, or
    // (a call that was to wait and failed before) not.
    bool stage_pending = false, stage_recorded = false;
    bool push_pending = false;      // hpush holds an unchecked status
    bool pull_pending = false;
    int pull_slots = 0, push_slots = 0;  // N of the pending calls
    std::vector<int64_t> pending_rows;  // var rows of a pending async pull
    int async_pull = 0;
    bool pooled_pushes = false;     // the last push had pooled gradients
    bool small_path = true;         // small batches take the path of few launches (tn_sparse_table_set_small_batch_path)
    int latched = TN_OK;
    std::string latched_msg;
    std::vector<int64_t> last_counts;
    hipStream_t last_stream = nullptr;  // of the table's last call, if it had one (nullptr is the default stream)
    bool had_call = false;
    std::mutex mu;
};

std::mutex g_tables_mu;
std::vector<SparseTable*> g_tables;

SparseTable* get_table(uint32_t h) {
    std::lock_guard<std::mutex> lk(g_tables_mu);
    if (h >= g_tables.size()) return nullptr;
    return g_tables[h];
}

OptDev make_optdev(const SparseTable* t) {
    const OptConf& c = *t->opt;
    OptDev o{};
    o.kind = c.kind;
    o.zero_init = c.sparse_zero_init;
    o.use_cvm = t->use_cvm;
    o.lr = c.learning_rate;
    o.eps = c.epsilon;
    o.initial_g2sum = c.initial_g2sum;
    o.initial_scale = c.initial_scale;
    o.beta1 = c.beta1;
    o.beta2 = c.beta2;
    o.beta = c.beta;
    o.lambda1 = c.lambda1;
    o.lambda2 = c.lambda2;
    return o;
}

int round4(int x) { return (x + 3) & ~3; }
constexpr size_t LINE_BYTES = 128;  // L2 line: what a random access to the table moves

void layout(const SparseTable* t, Store& s) {
    s.D = t->dim;
    s.wdim = t->dim + (t->use_cvm ? 2 : 0);
    bool vec = (t->dim % 4) == 0;
    s.wlen = vec ? round4(s.wdim) : s.wdim;
    int sf = (t->opt->kind == OPT_ADAGRAD) ? 4 : 2 * t->dim + 2;
    s.slen = vec ? round4(sf) : sf;
    s.wstride = s.wlen;
    s.sstride = s.slen;
}

// Weights and state of a row share one 128-byte line (or a power-of-two part of one) when they fit and the table stays
// below half of the device memory that way (dim-16 AdaGrad: 136 instead of 88 bytes per slot);
// an update then touches one line of the table instead of two.
void choose_strides(Store& s, uint64_t cap) {
    if (s.wlen % 4 != 0 || (s.wlen + s.slen) * sizeof(float) > LINE_BYTES) return;
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) return;
    size_t pitch = 32;  // a power of two, so that no row straddles a line
    while (pitch < (s.wlen + s.slen) * sizeof(float)) pitch *= 2;
    if ((cap + 1) * (pitch + sizeof(uint64_t)) > total_b / 2) return;
    s.wstride = s.sstride = (int)(pitch / sizeof(float));
}

bool interleaved(const Store& s) { return s.wstride != s.wlen; }

int state_floats(const SparseTable* t) { return (t->opt->kind == OPT_ADAGRAD) ? 4 : 2 * t->dim + 2; }

void free_store(Store& s);

int alloc_store(const SparseTable* t, uint64_t cap, Store& s, hipStream_t st) {
    layout(t, s);
    if (cap < 64) cap = 64;
    cap = (cap + PROBE_WIDTH - 1) / PROBE_WIDTH * PROBE_WIDTH;  // probing goes by aligned groups of slots
    if (cap > MAX_SLOTS_PER_TABLE) return fail(TN_ERR_UNSUPPORTED, "sparse table: more than 2^32 slots");
    s.cap = cap;
    choose_strides(s, cap);
    const size_t rows = (size_t)cap + 1;
    // whatever was allocated before a failure is released again: the caller keeps no half-built store
    auto oom = [&](const char* what, hipError_t e) {
        const std::string msg = std::string("hipMalloc ") + what + ": " + hipGetErrorString(e);
        free_store(s);
        return fail(TN_ERR_OUT_OF_MEMORY, msg);
    };
    hipError_t e;
    e = hipMalloc((void**)&s.keys, rows * sizeof(uint64_t) + 64);
    if (e != hipSuccess) return oom("keys", e);
    e = hipMalloc((void**)&s.w, rows * s.wstride * sizeof(float));
    if (e != hipSuccess) return oom("weights", e);
    if (interleaved(s)) {
        s.st = s.w + s.wlen;
    } else {
        e = hipMalloc((void**)&s.st, rows * s.sstride * sizeof(float));
        if (e != hipSuccess) return oom("state", e);
    }
    void* small = nullptr;
    e = hipMalloc(&small, 64);
    if (e != hipSuccess) return oom("counters", e);
    s.count = (unsigned long long*)small;
    s.special = (uint32_t*)((char*)small + 8);
    e = hipMemsetAsync(small, 0, 64, st);
    if (e == hipSuccess) e = hipMemsetAsync(s.keys, 0xFF, rows * sizeof(uint64_t), st);
    if (e != hipSuccess) {
        const std::string msg = std::string("hipMemsetAsync (new table): ") + hipGetErrorString(e);
        free_store(s);
        return fail(TN_ERR_HIP, msg);
    }
    return TN_OK;
}

void free_store(Store& s) {
    if (s.keys) (void)hipFree(s.keys);
    if (s.w) (void)hipFree(s.w);
    if (s.st && !interleaved(s)) (void)hipFree(s.st);
    if (s.count) (void)hipFree(s.count);
    s = Store{};
}

int ensure_side_buffers(SparseTable* t) {
    if (t->dstatus) return TN_OK;
    TN_HIP(hipMalloc((void**)&t->dstatus, 5 * sizeof(DevStatus)));
    TN_HIP(hipMemset(t->dstatus, 0, 5 * sizeof(DevStatus)));
    t->dplan = t->dstatus + 1;
    t->dpush = t->dstatus + 2;
    t->dcomb = t->dstatus + 3;
    t->dtpush = t->dstatus + 4;
    TN_HIP(hipHostMalloc((void**)&t->hpull, sizeof(HostStatus), hipHostMallocDefault));
    TN_HIP(hipHostMalloc((void**)&t->hpush, sizeof(HostStatus), hipHostMallocDefault));
    std::memset(t->hpull, 0, sizeof(HostStatus));
    std::memset(t->hpush, 0, sizeof(HostStatus));
    TN_HIP(hipHostMalloc((void**)&t->hcount, 64, hipHostMallocDefault));
    TN_HIP(hipHostMalloc((void**)&t->hseq, 64, hipHostMallocDefault));
    std::memset(t->hseq, 0, 64);
    TN_HIP(hipHostMalloc((void**)&t->hwords, PULL_WORDS * sizeof(uint64_t), hipHostMallocDefault));
    std::memset(t->hwords, 0, PULL_WORDS * sizeof(uint64_t));
    TN_HIP(hipHostMalloc((void**)&t->hcomb, 64, hipHostMallocDefault));
    std::memset(t->hcomb, 0, 64);
    t->hstage_bytes = (size_t)MAX_SLOTS * sizeof(SlotDesc) + (MAX_SLOTS + 1) * sizeof(uint32_t);
    TN_HIP(hipHostMalloc((void**)&t->hstage, t->hstage_bytes, hipHostMallocDefault));
    TN_HIP(hipEventCreateWithFlags(&t->stage_ev, hipEventDisableTiming));
    TN_HIP(hipEventCreateWithFlags(&t->fork_ev, hipEventDisableTiming));
    TN_HIP(hipEventCreateWithFlags(&t->tail_ev, hipEventDisableTiming));
    TN_HIP(hipEventCreateWithFlags(&t->apply_ev, hipEventDisableTiming));
    TN_HIP(hipEventCreateWithFlags(&t->upd_ev, hipEventDisableTiming));
    TN_HIP(hipStreamCreateWithFlags(&t->side, hipStreamNonBlocking));  // default priority
    TN_HIP(hipStreamCreateWithFlags(&t->aux, hipStreamNonBlocking));
    return TN_OK;
}

// Slots for a reservation of `keys` signs.  Growth starts at a load of 0.75 (optimizer_kernel.h:266); a reservation
// is sized for a load of 0.5 where that keeps the table (with its rows interleaved) below half of the device
// memory: probe chains are shorter there (cfg3: the probes of a pull take 0.078 instead of 0.096 ms).
uint64_t reserved_slots(const SparseTable* t, uint64_t keys) {
    const uint64_t tight = (uint64_t)((double)keys / MAX_LOAD) + 64;
    const uint64_t roomy = (uint64_t)((double)keys / RESERVE_LOAD) + 64;
    Store s{};
    layout(t, s);
    size_t pitch = 32;
    while (pitch < (s.wlen + s.slen) * sizeof(float)) pitch *= 2;
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) return tight;
    return (roomy + 1) * (pitch + sizeof(uint64_t)) <= total_b / 2 ? roomy : tight;
}

// Orders `st` behind the detached updates of the last push, if any (a wait for an event that has completed
// costs nothing on the device).
int order_after_updates(SparseTable* t, hipStream_t st) {
    if (t->upd_pending) TN_HIP(hipStreamWaitEvent(st, t->upd_ev, 0));
    return TN_OK;
}

// (The default stream is one like any other here: streams made with hipStreamNonBlocking are not ordered behind it.)
bool other_stream(const SparseTable* t, hipStream_t st) { return t->had_call && t->last_stream != st; }

void set_last_stream(SparseTable* t, hipStream_t st) {
    t->last_stream = st;
    t->had_call = true;
}

// A call on another stream than the table's last one: what that call left running there (a pull's gather, a small
// push's updates, a decay: tail_ev) is waited for on the device, and a call whose status is still pending on the host.
int order_after_other_stream(SparseTable* t, hipStream_t st) {
    if (!other_stream(t, st)) return TN_OK;
    t->several_streams = true;
    if (t->tail_owed) {
        TN_HIP(hipEventRecord(t->tail_ev, nullptr));
        t->tail_owed = false;
        t->tail_recorded = true;
    }
    if (t->tail_recorded) TN_HIP(hipStreamWaitEvent(st, t->tail_ev, 0));
    if (t->push_pending || t->pull_pending) TN_HIP(hipStreamSynchronize(t->last_stream));
    return TN_OK;
}

// What the last kernel of a call signals for calls on other streams.  On the default stream nothing as long as the table has had no
// calls on others: that one can neither be destroyed nor captured, so the event can be recorded there by the call that needs
// it.  That one call waits for whatever has been queued there meanwhile; from then on every call leaves its event again, so that
// calls on a stream of their own beside a training loop on the default one wait for the table's kernels alone.  (A launch with an
// event takes the host 1.6 us longer, in front of the kernel.)
hipEvent_t tail_event(SparseTable* t, hipStream_t st) {
    t->tail_owed = st == nullptr && !t->several_streams;
    if (t->tail_owed) return nullptr;
    t->tail_recorded = true;
    return t->tail_ev;
}

// The same as an event recorded behind the last kernel.  That is a small pull's form: a program that waits for the pulled rows waits
// longer where the kernel itself signals.  Push and pull of 1024 x 8, 4096 x 26 and 3001 x 47 x 2 lookups on a stream of the
// caller's, us, one step after the other, and each waited for: events recorded behind both calls 42.3, 51.6, 76.4, and 44.1, 59.0,
// 80.8; signals of both calls' last kernels 38.4, 50.0, 73.0, and 45.0, 61.8, 82.6; the push's a signal, the pull's recorded
// 39.2, 51.0, 74.7, and 41.5, 58.0, 78.9.  (Pull and combine of 256 x 26 x 3: 40.0 and 51.5, 37.9 and 48.4, 38.5 and 50.0.)
int record_tail(SparseTable* t, hipStream_t st) {
    hipEvent_t tail = tail_event(t, st);
    if (tail) TN_HIP(hipEventRecord(tail, st));
    return TN_OK;
}

// beside_updates: the caller (the pull op) orders its stream behind detached updates itself, as late as it can.
int ensure_allocated(SparseTable* t, hipStream_t st, bool beside_updates = false) {
    TN_TRY(ensure_side_buffers(t));
    if (!beside_updates) TN_TRY(order_after_updates(t, st));
    TN_TRY(order_after_other_stream(t, st));
    if (t->allocated) return TN_OK;
    uint64_t cap = DEFAULT_SLOTS;
    if (t->reserve_keys) cap = reserved_slots(t, t->reserve_keys);
    TN_TRY(alloc_store(t, cap, t->store, st));
    t->allocated = true;
    t->count_upper = 0;
    return TN_OK;
}

const char* dev_err_text(uint32_t err) {
    if (err & DEV_ERR_TABLE_FULL) return "sparse table is full";
    if (err & DEV_ERR_UNKNOWN_KEY) return "embedding of a pushed sign not created yet (push before pull)";
    if (err & DEV_ERR_VAR_CAPACITY) return "distinct signs of a slot exceed the rows of its variable";
    if (err & DEV_ERR_GRAD_ROWS) return "gradient matrix of a slot has fewer rows than the slot has distinct signs";
    return "";
}

int dev_err_code(uint32_t err) {
    if (err & DEV_ERR_TABLE_FULL) return TN_ERR_TABLE_FULL;
    if (err & DEV_ERR_UNKNOWN_KEY) return TN_ERR_UNKNOWN_KEY;
    if (err & DEV_ERR_VAR_CAPACITY) return TN_ERR_VAR_CAPACITY;
    if (err & DEV_ERR_GRAD_ROWS) return TN_ERR_INVALID_ARGUMENT;
    return TN_OK;
}

void latch(SparseTable* t, int code, const std::string& msg) {
    if (code != TN_OK && t->latched == TN_OK) {
        t->latched = code;
        t->latched_msg = msg;
    }
}

// CHECK_LT(signs.size(), max_var_count), sparse_table_ops.cc:136
void latch_var_capacity(SparseTable* t, int slot, int64_t rows) {
    latch(t, TN_ERR_VAR_CAPACITY,
          "sparse pull: slot " + std::to_string(slot) + " has " + std::to_string(t->last_counts[slot]) +
              " distinct signs, its variable only " + std::to_string(rows) + " rows");
}

// The share of distinct records among a pull's lookups: rises at once, falls within about ten pulls.
void note_distinct_share(SparseTable* t, double now) {
    t->distinct_est = std::min(1.0, std::max(now, 0.75 * t->distinct_est + 0.25 * now));
}

// Examines the status blocks of finished calls (the stream must have been synchronised).
void harvest(SparseTable* t) {
    // a pending push is older than a pending pull (a push collects everything before it starts)
    if (t->push_pending) {
        t->push_pending = false;
        if (t->push_on_side) {
            t->push_on_side = false;
            const hipError_t e = hipStreamSynchronize(t->side);
            if (e != hipSuccess) latch(t, TN_ERR_HIP, std::string("sparse push: ") + hipGetErrorString(e));
            t->upd_pending = false;
        }
        const HostStatus& h = *t->hpush;
        int N = t->push_slots;
        if (N > 0) {
            t->last_counts.assign(N, 0);
            for (int s = 0; s < N; s++) t->last_counts[s] = (int64_t)h.ubase[s + 1] - (int64_t)h.ubase[s];
        }
        latch(t, dev_err_code(h.st.err), std::string("sparse push: ") + dev_err_text(h.st.err));
    }
    if (t->pull_pending) {
        t->pull_pending = false;
        const HostStatus& h = *t->hpull;
        int N = t->pull_slots;
        // the call booked room for every sign it could have inserted; keep what it did insert
        if (t->booked >= h.st.n_new) t->count_upper -= t->booked - h.st.n_new;
        t->booked = 0;
        t->last_counts.assign(N, 0);
        for (int s = 0; s < N; s++) t->last_counts[s] = (int64_t)h.ubase[s + 1] - (int64_t)h.ubase[s];
        if (N > 0) {  // (a pull of the table or a load of rows has no slots: the last pull's plan stands, and so does what is known of it)
            t->plan_heavy = h.st.heavy != 0;
            t->plan_counts = t->last_counts;
            note_distinct_share(t, (double)h.ubase[N] / (double)t->pull_lookups);
            if (h.st.tile_share_q16 != 0) {  // (a pull through LDS with a slot of more than one bucket)
                const double share = (double)h.st.tile_share_q16 / 65536.0;
                t->tile_est = std::min(1.0, std::max(share, 0.75 * t->tile_est + 0.25 * share));
            }
        }
        latch(t, dev_err_code(h.st.err), std::string("sparse pull: ") + dev_err_text(h.st.err));
        for (int s = 0; s < N && s < (int)t->pending_rows.size(); s++)
            if (t->last_counts[s] >= t->pending_rows[s]) latch_var_capacity(t, s, t->pending_rows[s]);
    }
}

int take_latched(SparseTable* t) {
    int code = t->latched;
    if (code != TN_OK) {
        set_error(t->latched_msg);
        t->latched = TN_OK;
        t->latched_msg.clear();
    }
    return code;
}

int sync_table(SparseTable* t, hipStream_t st) {
    if (t->upd_pending) {
        TN_HIP(hipEventSynchronize(t->upd_ev));
        t->upd_pending = false;
    }
    TN_HIP(hipStreamSynchronize(st));
    if (other_stream(t, st)) TN_HIP(hipStreamSynchronize(t->last_stream));
    harvest(t);
    return take_latched(t);
}

// Moves every resident row into a freshly allocated table of `cap` slots.
int grow_to(SparseTable* t, uint64_t cap, hipStream_t st) {
    Store& s = t->store;
    if (cap > MAX_SLOTS_PER_TABLE) cap = MAX_SLOTS_PER_TABLE;
    if (cap <= s.cap) return fail(TN_ERR_TABLE_FULL, "sparse table cannot grow beyond 2^32 slots");
    Store bigger{};
    int rc = alloc_store(t, cap, bigger, st);
    if (rc != TN_OK) {
        free_store(bigger);
        return rc;
    }
    TN_LAUNCH(k_reset_status, dim3(1), dim3(64), st, t->dstatus, 0u, 0u);
    TN_LAUNCH(k_rehash, dim3(launch_grid((int64_t)s.cap + 1, 256, GRID_CAP * 4)), dim3(256), st, s, bigger, t->dstatus);
    TN_HIP(hipMemcpyAsync(bigger.count, s.count, sizeof(unsigned long long), hipMemcpyDeviceToDevice, st));
    TN_HIP(hipStreamSynchronize(st));
    free_store(s);
    s = bigger;
    t->epoch++;  // cached row numbers are stale now
    return TN_OK;
}

// The number of resident keys, read on the stream `st` itself (a copy on the null stream would wait for,
// and hold up, every blocking stream of the process: other tables' calls).
int read_count(SparseTable* t, hipStream_t st, uint64_t* out) {
    TN_HIP(hipMemcpyAsync(t->hcount, t->store.count, sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
    TN_HIP(hipStreamSynchronize(st));
    t->count_upper = *t->hcount;
    *out = *t->hcount;
    return TN_OK;
}

// Makes room for up to `incoming` new keys: grows (re-inserts into a larger
// table) when the load factor could pass MAX_LOAD (optimizer_kernel.h:266).
// Callers have collected the status of earlier calls (t->booked == 0).
int ensure_room(SparseTable* t, uint64_t incoming, hipStream_t st) {
    Store& s = t->store;
    if ((double)(t->count_upper + incoming) > MAX_LOAD * (double)s.cap) {
        TN_TRY(order_after_updates(t, st));  // growing moves the rows
        uint64_t cnt = 0;  // the bound may be loose: read the true count
        TN_TRY(read_count(t, st, &cnt));
        if ((double)(cnt + incoming) > MAX_LOAD * (double)s.cap) {
            uint64_t need = (uint64_t)((double)(cnt + incoming) / MAX_LOAD) + 64;
            TN_TRY(grow_to(t, std::max<uint64_t>(need, s.cap * 2), st));
        }
    }
    t->count_upper += incoming;
    t->booked = incoming;
    return TN_OK;
}

// ---------------------------------------------------------------- workspace
struct Carver {
    char* base;
    size_t off = 0;
    template <typename T>
    T* take(size_t n) {
        off = align_up(off, 256);
        T* p = reinterpret_cast<T*>(base + off);
        off += n * sizeof(T);
        return p;
    }
};

// Results of analysing one batch.  For an op-level call they live in the
// table's plan buffer and survive until the next op-level call, so that a push
// of the same batch can reuse them; a table-level push carves the group part
// from the per-call scratch.
struct Plan {
    SlotDesc* descs;
    SlotDesc* push_descs;  // descriptors of the push that reuses the plan (the pull's gather may still read `descs`)
    uint32_t* push_ubase;  // ... and its copy of ubase (the next pull rewrites ubase, detached updates may still run then)
    uint32_t* lbase;
    uint32_t* ubase;
    uint64_t* vals_copy;   // signs of every lookup, concatenated; after a pull through LDS their fingerprints instead
    uint32_t* u_of_gi;     // lookup -> index of its distinct sign
    uint64_t* uniq_sign;   // per-slot distinct signs, slot-major, first-occurrence order
    uint32_t* uniq_slot;
    uint32_t* ushow;       // batch_show per distinct sign, when the remap already knows it
    uint64_t* grp_sign;    // distinct signs over all slots
    uint32_t* grp_row;     // their table rows
    uint32_t* grp_off;
    uint32_t* grp_cnt;
    Member* list;          // members of every group, ascending (with their show / click counts)
    uint2* where_u;        // record -> {its place in `list`, its group}
    uint32_t* big_list;    // groups with BIG_GROUP records or more
    uint4* big_desc;       // {row, first member, records, group} of those groups (emit_buckets writes it, the other groupings do not)
    uint32_t big_cap;      // entries of big_list / big_desc
    const float** gaddr;   // gradient row of every record of the groups with several records (a push fills it)
    uint64_t* vals_exact;  // copy of the signs beside their fingerprints (tn_sparse_table_set_exact_verify), else nullptr
};

// Per-call scratch of the analysis.
struct Scratch {
    DedupEntry* dt;
    size_t dt_entries;
    uint32_t* tidx;
    uint8_t* flag8;
    uint32_t* tilesum;
    uint32_t* tileoff;
    uint32_t ntiles;
    // LDS remap
    uint32_t nbuckets;
    uint32_t span_cap;   // first-level buckets the widest tile touches (LDS counters of k_tile_dedup)
    uint32_t* bcursor;   // per first-level bucket: records handed in
    ulonglong2* prec;    // the tiles' records by bucket, L1_ROOM each: {sign, position | occurrences | slot}
    uint32_t* first_of;
    uint32_t* cnt_at;
    uint32_t* wordpre;  // first occurrences before every 64-lookup word
    // grouping through LDS (second-level buckets)
    uint32_t nb2;
    uint32_t* cursor2;
    GroupRec* recs;
    uint2* aux;
    uint32_t* rrow;      // per distinct record: table row of its sign
    uint32_t* newrec;    // per second-level bucket: its records whose rows the pull inserted ...
    uint32_t* newcnt;    // ... and how many
    uint4* bcounts;
    uint4* bbase;
    void* gt;  // GroupEntry[] or MaskEntry[]
    uint32_t* gidx;
    uint32_t* ord;
    uint32_t* arrival;
};

size_t group_cap(size_t n) { return std::max<size_t>(16, n + n / 2); }

// Signs with this many records or more are applied by one wavefront each
// (k_apply_big); rows too wide for its LDS staging stay with the lane groups.
constexpr uint32_t BIG_GROUP = BIG_GROUP_DEFAULT;
uint32_t big_threshold(const Store& s) { return s.D <= BIG_DIM_MAX ? BIG_GROUP : 0xFFFFFFFFu; }

void carve_groups(Carver& c, Plan& p, size_t n) {
    p.grp_sign = c.take<uint64_t>(n);
    p.grp_row = c.take<uint32_t>(n);
    p.grp_off = c.take<uint32_t>(n);
    p.grp_cnt = c.take<uint32_t>(n);
    p.list = c.take<Member>(n);
    p.where_u = c.take<uint2>(n);
    p.big_cap = (uint32_t)(n / BIG_GROUP + 64);
    p.big_list = c.take<uint32_t>(p.big_cap);
    p.big_desc = c.take<uint4>(p.big_cap);
    p.gaddr = c.take<const float*>(n);
}

void carve_group_scratch(Carver& c, Scratch& w, size_t n) {
    w.gt = c.take<MaskEntry>(group_cap(n) + 1);  // the larger of the two entry types
    w.gidx = c.take<uint32_t>(n);
    w.ord = c.take<uint32_t>(n);
    w.arrival = c.take<uint32_t>(n);
}

size_t carve_plan(char* base, Plan& p, int N, size_t L, bool exact = false) {
    Carver c{base};
    p.descs = c.take<SlotDesc>(N);
    p.push_descs = c.take<SlotDesc>(N);
    p.lbase = c.take<uint32_t>(N + 1);
    p.ubase = c.take<uint32_t>(N + 1);
    p.push_ubase = c.take<uint32_t>(N + 1);
    p.vals_copy = c.take<uint64_t>(std::max<size_t>(L, 16));  // (the fingerprints of a short batch: 64 bytes a tile)
    p.u_of_gi = c.take<uint32_t>(L);
    p.uniq_sign = c.take<uint64_t>(L);
    p.uniq_slot = c.take<uint32_t>(L);
    p.ushow = c.take<uint32_t>(L);
    carve_groups(c, p, L);
    p.vals_exact = exact ? c.take<uint64_t>(L) : nullptr;  // last: the other arrays keep their places either way
    return align_up(c.off, 256);
}

// Second-level buckets of a batch of L lookups: GRP_TARGET records each on average if the batch has the
// expected share of distinct records plus a quarter (GRP_CAP is the room of a bucket).
uint32_t second_level_buckets(size_t L, double distinct_est, size_t target) {
    const double expected = std::min(1.0, distinct_est * 1.25) * (double)L;
    return (uint32_t)std::max<size_t>(1, ((size_t)expected + target - 1) / target);
}

// dt_entries: entries of the global dedup table, or (use_lds) the number of buckets.
// First-level buckets of a slot of `len` lookups whose tiles hand on `share` records per lookup: L1_FILL records
// each on average (L1_ROOM is the room of a bucket); a slot that fits one bucket whatever its signs has one.
constexpr size_t L1_FILL = 1150;
constexpr double L1_MARGIN = 1.15;
size_t first_level_buckets(size_t len, double share) {
    if (len <= (size_t)L1_ROOM) return 1;
    return ((size_t)((double)len * std::min(1.0, share * L1_MARGIN)) + L1_FILL - 1) / L1_FILL;
}

size_t carve_scratch(char* base, Scratch& w, size_t L, size_t dt_entries, bool use_lds, double distinct_est = 1.0,
                     int N = 0) {
    Carver c{base};
    if (use_lds) {
        w.nbuckets = (uint32_t)dt_entries;
        const size_t target = N <= GRP_NARROW ? GRP_TARGET : GRP_TARGET_WIDE;
        w.nb2 = second_level_buckets(L, distinct_est, target);
        // room for the buckets of a batch of distinct signs only: a call that overflows is repeated with that
        // many, and must not pay for a larger buffer then (freeing and allocating waits for the whole device)
        const size_t nb2_room = std::max<size_t>(w.nb2, (L + target - 1) / target);
        const size_t nb1_room = std::max<size_t>(dt_entries, L / L1_FILL + (size_t)N + 1);
        w.bcursor = c.take<uint32_t>(nb1_room + 1 + nb2_room);  // (the part in use is zeroed together)
        w.cursor2 = w.bcursor + dt_entries + 1;
        w.recs = c.take<GroupRec>(nb2_room * GRP_CAP);
        w.aux = c.take<uint2>(nb2_room * GRP_CAP);
        w.rrow = c.take<uint32_t>(nb2_room * GRP_CAP);
        w.newrec = c.take<uint32_t>(nb2_room * GRP_CAP);
        w.newcnt = c.take<uint32_t>(nb2_room);
        w.bcounts = c.take<uint4>(nb2_room);
        w.bbase = c.take<uint4>(nb2_room);
        w.prec = c.take<ulonglong2>(nb1_room * (size_t)L1_ROOM);
        w.first_of = c.take<uint32_t>(L);
        w.cnt_at = c.take<uint32_t>(L);
        w.wordpre = c.take<uint32_t>(L / 64 + 2);
        w.dt = nullptr;
        w.dt_entries = 0;
        w.tidx = nullptr;
    } else {
        w.dt = c.take<DedupEntry>(dt_entries);
        w.dt_entries = dt_entries;
        w.tidx = c.take<uint32_t>(L);
    }
    w.flag8 = c.take<uint8_t>(L / REMAP_ITEMS + REMAP_THREADS);
    w.ntiles = (uint32_t)((L + REMAP_TILE - 1) / REMAP_TILE);
    w.tilesum = c.take<uint32_t>(w.ntiles + 1);
    w.tileoff = c.take<uint32_t>(w.ntiles + 1);
    carve_group_scratch(c, w, L);
    return align_up(c.off, 256);
}

// Validates the slot arrays of an op and fills the descriptors; returns L.
// With *use_lds set on entry the slots are laid out for the LDS remap if the batch
// qualifies (tbase/tcap = first bucket / number of buckets of the slot, dt_entries =
// number of buckets); otherwise *use_lds comes back false and tbase/tcap describe the
// slot's region of the global dedup table.
int stage_slots(SparseTable* t, int N, const int64_t* const* values, const int64_t* lens, std::vector<SlotDesc>& descs,
                std::vector<uint32_t>& lbase, size_t& L, size_t& dt_entries, const char* what, bool* use_lds,
                uint32_t* span_cap = nullptr) {
    if (N <= 0 || !values || !lens) return fail(TN_ERR_INVALID_ARGUMENT, std::string(what) + ": no slots");
    if (N > MAX_SLOTS)
        return fail(TN_ERR_UNSUPPORTED, std::string(what) + ": more than " + std::to_string(MAX_SLOTS) + " slots");
    descs.assign(N, SlotDesc{});
    lbase.assign(N + 1, 0);
    size_t l = 0, te = 0;
    for (int s = 0; s < N; s++) {
        if (lens[s] < 0 || (lens[s] > 0 && !values[s]))
            return fail(TN_ERR_INVALID_ARGUMENT, std::string(what) + ": bad values tensor of slot " + std::to_string(s));
        SlotDesc& d = descs[s];
        d.values = values[s];
        d.len = (uint32_t)lens[s];
        d.lbase = (uint32_t)l;
        d.tbase = (uint32_t)te;
        size_t tcap = (size_t)lens[s] + (size_t)lens[s] / 2 + 8;
        d.tcap = (uint32_t)tcap;
        lbase[s] = (uint32_t)l;
        l += (size_t)lens[s];
        te += tcap + 1;
        if (l > 0x7FFFFFF0ull || te > 0xFFFFFFF0ull)
            return fail(TN_ERR_UNSUPPORTED, std::string(what) + ": more than 2^31 lookups in one call");
    }
    lbase[N] = (uint32_t)l;
    L = l;
    dt_entries = te;
    if (use_lds && *use_lds) {
        bool ok = l >= LDS_MIN_LOOKUPS;
        for (int s = 0; s < N && ok; s++) ok = (size_t)lens[s] <= (size_t)LDS_MAX_SUB * L1_FILL;
        *use_lds = ok;
        if (ok) {
            // The buckets have fixed room for the records the tiles hand in (one per distinct sign of a tile):
            // sized from the share of such records the recent pulls had, with a margin; a batch that overflows
            // them is repeated with buckets for a batch without repeats.
            size_t nb = 0;
            for (int s = 0; s < N; s++) {
                const size_t sub = first_level_buckets((size_t)lens[s], t->tile_est);
                descs[s].tbase = (uint32_t)nb;
                descs[s].tcap = (uint32_t)sub;
                nb += sub;
            }
            dt_entries = nb;
            // buckets the widest tile of the partition kernel touches: first bucket of the slot of
            // its first lookup .. last bucket of the slot of its last lookup
            size_t widest = 1;
            int s0 = 0, s1 = 0;
            for (size_t g0 = 0; g0 < l; g0 += LDS_TILE) {
                const size_t g1 = std::min(l, g0 + (size_t)LDS_TILE) - 1;
                while (s0 + 1 < N && lbase[s0 + 1] <= g0) s0++;
                if (s1 < s0) s1 = s0;
                while (s1 + 1 < N && lbase[s1 + 1] <= g1) s1++;
                widest = std::max<size_t>(widest, (size_t)descs[s1].tbase + descs[s1].tcap - descs[s0].tbase);
            }
            if (span_cap) *span_cap = (uint32_t)std::min<size_t>(widest, LDS_SPAN);
        }
    }
    return TN_OK;
}

// The staging buffer may be written again.
int staging_free(SparseTable* t) {
    if (t->stage_pending) TN_HIP(t->stage_recorded ? hipEventSynchronize(t->stage_ev) : hipDeviceSynchronize());
    t->stage_pending = false;
    return TN_OK;
}

// Slot descriptors to the device (dst_descs; the slots' first lookups to dst_lbase unless nullptr); the same
// launch prepares the call's status block `ds` (status_mode) and clears `zero[0 .. n_zero)`.
// waited: the caller waits for something behind it, and then says that the staging buffer is free; else an event says so.
int upload_slots(SparseTable* t, SlotDesc* dst_descs, uint32_t* dst_lbase, DevStatus* ds,
                 const std::vector<SlotDesc>& descs, const std::vector<uint32_t>& lbase, hipStream_t st,
                 bool waited, int status_mode, uint32_t* zero = nullptr, uint32_t n_zero = 0,
                 const uint32_t* copy_src = nullptr, uint32_t* copy_dst = nullptr, uint32_t copy_n = 0) {
    TN_TRY(staging_free(t));
    const size_t db = descs.size() * sizeof(SlotDesc);
    const size_t lb = dst_lbase ? lbase.size() * sizeof(uint32_t) : 0;
    std::memcpy(t->hstage, descs.data(), db);
    if (lb) std::memcpy(t->hstage + db, lbase.data(), lb);
    TN_LAUNCH(k_stage_in, dim3(launch_grid((int64_t)std::max<size_t>((db + lb) / 4, n_zero), 256, 64)), dim3(256), st,
              reinterpret_cast<const uint32_t*>(t->hstage), reinterpret_cast<uint32_t*>(dst_descs), (uint32_t)(db / 4), dst_lbase,
              (uint32_t)(lb / 4), ds, status_mode, zero, n_zero, (const DevStatus*)t->dplan, copy_src, copy_dst, copy_n);
    if (!waited) TN_HIP(hipEventRecord(t->stage_ev, st));
    t->stage_recorded = !waited;
    t->stage_pending = true;
    return TN_OK;
}

// own_copies: the source of a push on the last pull's plan, whose kernels may still run (detached updates) or
// be staged (the next pull's descriptors go in beside them) while the next pull rewrites p.descs and p.ubase:
// it reads the push's own descriptors and its own copy of the slots' distinct bases.
PushSrc op_source(const Plan& p, int dim, bool own_copies = false) {
    PushSrc src{};
    src.uniq_sign = p.uniq_sign;
    src.uniq_slot = p.uniq_slot;
    src.ubase = own_copies ? p.push_ubase : p.ubase;
    src.descs = own_copies ? p.push_descs : p.descs;
    src.dim = dim;
    return src;
}

// Groups n records (n_host of them, or status->n_unique) by sign: group arrays
// and member lists in ascending record order.  Works for any records: arrival
// order by atomics, then every record finds its place among its group's members.
void launch_grouping(const Plan& p, const Scratch& w, const PushSrc& src, int64_t n_host, int64_t n_upper,
                     uint32_t big_k, const uint32_t* ushow, DevStatus* ds, hipStream_t st) {
    const uint32_t* n_dev = src.infos ? nullptr : &ds->n_unique;
    GroupEntry* gt = static_cast<GroupEntry*>(w.gt);
    const int gblocks = launch_grid(n_upper, 256, GRID_CAP * 2);
    const int tblocks = launch_grid((int64_t)group_cap(n_upper) + 1, 256, GRID_CAP * 2);
    TN_LAUNCH(k_fill_groups, dim3(tblocks), dim3(256), st, gt, ds);
    TN_LAUNCH(k_group_insert, dim3(gblocks), dim3(256), st, src, n_host, ds, gt, w.gidx, w.ord);
    TN_LAUNCH(k_group_compact, dim3(launch_grid((int64_t)group_cap(n_upper) / COMPACT_ITEMS + 1, 256, GRID_CAP)),
              dim3(256), st, ds, gt, p.grp_sign, p.grp_off, p.grp_cnt, p.big_list, big_k, (uint32_t)n_upper);
    TN_LAUNCH(k_group_fill, dim3(gblocks), dim3(256), st, n_host, n_dev, gt, p.grp_off, w.gidx, w.ord, w.arrival);
    TN_LAUNCH(k_group_rank, dim3(gblocks), dim3(256), st, n_host, n_dev, gt, p.grp_off, w.gidx, w.arrival,
              src.uniq_slot, ushow, p.list, p.where_u);
}

constexpr int MASK_SLOTS = 128;

// The same result for the distinct signs of an op with at most MASK_SLOTS slots, from slot masks.  (Where the signs are not
// grouped through LDS: a pull that does not wait for its stream, a push that analyses its batch itself.)
void launch_mask_grouping(const Plan& p, const Scratch& w, int64_t n_upper, uint32_t big_k, const uint32_t* ushow,
                          DevStatus* ds, hipStream_t st) {
    MaskEntry* gt = static_cast<MaskEntry*>(w.gt);
    const int gblocks = launch_grid(n_upper, 256, GRID_CAP * 2);
    const int tblocks = launch_grid(2 * (int64_t)group_cap(n_upper) + 2, 256, GRID_CAP * 2);
    TN_LAUNCH(k_fill_masks, dim3(tblocks), dim3(256), st, gt, ds);
    TN_LAUNCH(k_mask_insert, dim3(gblocks), dim3(256), st, p.uniq_sign, p.uniq_slot, ds, gt, w.gidx);
    TN_LAUNCH(k_mask_compact, dim3(launch_grid((int64_t)group_cap(n_upper) / COMPACT_ITEMS + 1, 256, GRID_CAP)),
              dim3(256), st, ds, gt, p.grp_sign, p.grp_off, p.grp_cnt, p.big_list, big_k, (uint32_t)n_upper);
    TN_LAUNCH(k_mask_fill, dim3(gblocks), dim3(256), st, ds, gt, w.gidx, p.uniq_slot, ushow, p.list, p.where_u);
}

// Analyses the batch staged in p.descs: per-slot distinct signs and mapped ids,
// groups of equal signs, and the table row of every group (inserting absent
// signs for a pull).  use_lds picks the remap through LDS (pull only).  The
// upload of the descriptors has cleared the status block and, for the LDS path,
// the bucket counters.
int launch_build_plan(SparseTable* t, const Plan& p, const Scratch& w, int N, uint32_t L, bool for_pull, bool use_lds,
                      hipStream_t st) {
    DevStatus* ds = t->dplan;
    const Store& s = t->store;
    const int lblocks = launch_grid(L, 256, GRID_CAP * 2);
    const bool lds_groups = use_lds && N <= GRP_SLOTS;
    // second-level buckets up to which emit_buckets adds up the bucket counts itself (one bucket per workgroup)
    const bool own_offsets = w.nb2 <= (uint32_t)GRID_CAP * 4;
    if (use_lds) {
        // (as many workgroups as the chip holds of this kernel at once -- four per CU --, each taking its tiles in turn)
        const int tiles = launch_grid((int64_t)(L + LDS_TILE - 1) / LDS_TILE, 1, TILE_GRID);
        const size_t tile_lds = tile_dedup_lds(N, w.span_cap);
        TN_LAUNCH_LDS(k_tile_dedup, dim3(tiles), dim3(TILE_THREADS), tile_lds, st, p.descs, p.lbase, N, L, w.bcursor, w.prec,
                      reinterpret_cast<ulonglong2*>(p.vals_copy), p.vals_exact, w.first_of, ds, w.span_cap);
        if (lds_groups)
            TN_LAUNCH((k_lds_dedup<true>), dim3(launch_grid(w.nbuckets, 1, GRID_CAP * 2)), dim3(DEDUP_THREADS), st, w.bcursor,
                      w.nbuckets, w.prec, w.first_of, w.cnt_at, ds, w.nb2, w.cursor2, w.recs);
        else
            TN_LAUNCH((k_lds_dedup<false>), dim3(launch_grid(w.nbuckets, 1, GRID_CAP * 2)), dim3(DEDUP_THREADS), st, w.bcursor,
                      w.nbuckets, w.prec, w.first_of, w.cnt_at, ds, w.nb2, w.cursor2, w.recs);
        // up to SELF_SCAN_TILES tiles the ranking pass adds up the tile counts itself
        const uint32_t* own_sums = w.ntiles <= SELF_SCAN_TILES ? w.tilesum : nullptr;
        const size_t lb_lds = ((size_t)N + 1) * sizeof(uint32_t);
        if (lds_groups) {
            GroupProbeArgs ga;
            ga.nb2 = w.nb2, ga.ntiles = w.ntiles, ga.L = L;
            ga.cursor2 = w.cursor2;
            ga.recs = w.recs;
            ga.big_k = big_threshold(s);
            ga.aux = w.aux;
            ga.bcounts = w.bcounts;
            ga.rrow = w.rrow, ga.newrec = w.newrec, ga.newcnt = w.newcnt;
            ga.first_of = w.first_of;
            ga.flag8 = w.flag8;
            ga.tilesum = w.tilesum;
            ga.descs = p.descs;
            ga.N = N;
            ga.bcursor = w.bcursor;
            const dim3 gblocks = item_grid(2 * (uint64_t)w.nb2 + (w.ntiles + 1) / 2 + ((uint32_t)N + 7) / 8);
            if (N <= GRP_NARROW)
                TN_LAUNCH((k_group_probe<2>), gblocks, dim3(GRP_THREADS), st, ga, s, ds);
            else
                TN_LAUNCH((k_group_probe<4>), gblocks, dim3(GRP_THREADS), st, ga, s, ds);
            if (!own_offsets) TN_LAUNCH(k_group_offsets, dim3(1), dim3(1024), st, w.bcounts, w.bbase, w.nb2, ds);
        } else {
            TN_LAUNCH(k_lds_flags, dim3(w.ntiles), dim3(REMAP_THREADS), st, L, w.first_of, w.flag8, w.tilesum, p.descs, N,
                      w.bcursor, ds);
        }
        if (!own_sums)
            TN_LAUNCH(k_scan_tiles, dim3(1), dim3(1024), st, w.tilesum, w.tileoff, w.ntiles, p.lbase, p.ubase, N, L, ds);
        if (lds_groups) {
            InitArgs ia;
            ia.seed = t->seed;
            ia.recs = w.recs;
            ia.rrow = w.rrow;
            ia.nb2 = w.nb2;
            ia.newrec = w.newrec, ia.newcnt = w.newcnt;
            ia.parts = std::max<uint32_t>(1, (uint32_t)GRID_CAP / w.nb2);
            const int iblocks = launch_grid((int64_t)w.nb2 * ia.parts, 1, GRID_CAP);
            TN_LAUNCH_LDS(k_assign_init, dim3(w.ntiles + iblocks), dim3(REMAP_THREADS), lb_lds, st, p.descs, p.lbase, N, L, w.ntiles,
                          w.flag8, w.tileoff, w.wordpre, p.ubase, own_sums, s, make_optdev(t), ia, ds);
        } else {
            TN_LAUNCH_LDS((k_lds_assign<true>), dim3(w.ntiles), dim3(REMAP_THREADS), lb_lds, st, p.descs, p.lbase, N, L,
                          w.flag8, w.tileoff, w.cnt_at, w.wordpre, p.ubase, p.uniq_sign, p.uniq_slot, p.ushow, own_sums, ds);
            TN_LAUNCH_LDS(k_lds_mapped, dim3(lblocks), dim3(256), lb_lds, st, p.descs, p.lbase, p.ubase, N, L, w.first_of,
                          w.flag8, w.wordpre, p.u_of_gi);
        }
    } else {
        TN_LAUNCH(k_fill_ff, dim3(launch_grid((int64_t)w.dt_entries, 256, GRID_CAP * 2)), dim3(256), st,
                  reinterpret_cast<uint4*>(w.dt), w.dt_entries);
        TN_LAUNCH(k_remap_insert, dim3(lblocks), dim3(256), st, p.descs, p.lbase, N, L, w.dt, w.tidx, p.vals_copy);
        TN_LAUNCH(k_flag_count, dim3(w.ntiles), dim3(REMAP_THREADS), st, p.lbase, N, L, w.dt, w.tidx, w.flag8,
                  w.tilesum);
        TN_LAUNCH(k_scan_tiles, dim3(1), dim3(1024), st, w.tilesum, w.tileoff, w.ntiles, p.lbase, p.ubase, N, L, ds);
        TN_LAUNCH(k_assign_rank, dim3(w.ntiles), dim3(REMAP_THREADS), st, p.descs, p.lbase, N, L, w.dt, w.tidx, w.flag8,
                  w.tileoff, p.ubase, p.uniq_sign, p.uniq_slot);
        TN_LAUNCH(k_write_mapped, dim3(lblocks), dim3(256), st, p.descs, p.lbase, p.ubase, N, L, w.dt, w.tidx, w.flag8,
                  p.u_of_gi, for_pull ? 1 : 0);
    }
    const uint32_t* ushow = use_lds ? p.ushow : nullptr;
    // from here on the groups and member lists are written, which detached updates of the push before still read
    TN_TRY(order_after_updates(t, st));
    if (lds_groups) {
        const int bblocks = launch_grid(w.nb2, 1, GRID_CAP * 4);
        EmitArgs<false> ea;
        ea.nb2 = w.nb2;
        ea.cursor2 = w.cursor2;
        ea.recs = w.recs;
        ea.aux = w.aux;
        ea.bbase = own_offsets ? nullptr : w.bbase;
        ea.bcounts = w.bcounts;
        ea.flag8 = w.flag8;
        ea.wordpre = w.wordpre;
        ea.ids_cap = L;
        ea.big_k = big_threshold(s);
        ea.singles = row_share(s, true).lanes == 0;
        ea.grp_off = p.grp_off;
        ea.grp_cnt = p.grp_cnt;
        ea.big_list = p.big_list;
        ea.big_desc = p.big_desc;
        ea.list = p.list;
        ea.where_u = p.where_u;
        ea.rrow = w.rrow;
        ea.grp_row = p.grp_row;
        ea.status = ds;
        const MapArgs ma{p.descs, p.lbase, p.ubase, N, L, w.first_of, p.u_of_gi};
        const int mblocks = launch_grid(((int64_t)L + 3) / 4, EMIT_THREADS, GRID_CAP);
        TN_LAUNCH_LDS(k_emit_mapped, dim3(bblocks + mblocks), dim3(EMIT_THREADS), ((size_t)N + 1) * sizeof(uint32_t), st, ea, ma,
                      (uint32_t)bblocks);
        t->plan_big_desc = true;
        return TN_OK;  // the rows were found beside the grouping
    } else if (N <= MASK_SLOTS)
        launch_mask_grouping(p, w, (int64_t)L, big_threshold(s), ushow, ds, st);
    else
        launch_grouping(p, w, op_source(p, 0), 0, (int64_t)L, big_threshold(s), ushow, ds, st);
    if (for_pull)
        TN_LAUNCH((k_probe<true>), dim3(lblocks), dim3(256), st, s, p.grp_sign, (int64_t)0, ds, L, p.grp_row,
                  (uint32_t*)nullptr, ds, (uint32_t)DEV_ERR_TABLE_FULL, make_optdev(t), t->seed);
    else
        TN_LAUNCH((k_probe<false>), dim3(lblocks), dim3(256), st, s, p.grp_sign, (int64_t)0, ds, L, p.grp_row,
                  (uint32_t*)nullptr, ds, (uint32_t)DEV_ERR_UNKNOWN_KEY, make_optdev(t), t->seed);
    return TN_OK;
}

// workgroups of k_apply_all for the signs with many records at most (a wavefront each in turn)
constexpr int ALL_BIG_GRID = 1024;

// The signs with many records, with a few and with one: one launch (k_apply_all) where a row fits the lanes of a wavefront half.
// Above 3 M lookups they were three launches on two streams until the pull needed no second stream: 4.9 M of 100 slots, rows of
// 16, a step 527 us and 516 as one launch, with pooled gradients 881 and 856; 3.2 M of 70 slots over 300 signs 168 and 132;
// 3.5 M of 88 over 250 k, rows of 64, 1107 and 1132, the only batch found that loses.  (With a launch of their own for the signs
// with many records ahead of the others': 3.2 M of 70 slots over 150 signs, rows of 16 127 and 123, of 64 133 and 135; 4 M of 40
// over 350, rows of 32, 154 and 151; 4.9 M of 100 over 50, rows of 8, 143 and 143.)
//
// detach: the three kernels one by one on streams of the table's own, which the caller's does not wait for -- k_apply_single on
// the auxiliary stream, the others on the side stream; the caller of this function records their end (SparseTable::upd_ev).
// `behind`: an event that the last kernel on `st` signals.
template <int KIND>
int launch_apply_kind(SparseTable* t, RowShare share, const Store& s, const OptDev& o, const PushSrc& src, DevStatus* ds,
                      const Plan& p, int64_t n_upper, hipStream_t st, bool addr_ready, uint32_t big_k, bool detach,
                      bool big_desc, hipEvent_t behind) {
    const uint32_t ids_cap = (uint32_t)n_upper;
    const bool with_big = big_k != 0xFFFFFFFFu;
    const float* const* gaddr = (with_big && !src.infos && !src.flat) ? p.gaddr : nullptr;
    detach = detach && share.lanes != 0;
    t->detached_now = detach;
    // op-level gradients: their addresses for the records of the groups with several records, once, in a
    // coalesced pass ahead of everything (beside k_apply_single it would take several times as long)
    if (with_big && gaddr && !addr_ready) {
        behind = detach ? t->fork_ev : nullptr;
        TN_LAUNCH_EVENT(behind, k_member_grads, dim3(launch_grid(n_upper, 256, GRID_CAP * 2)), dim3(256), st, src, ds, p.list,
                        p.gaddr, ids_cap);
    }
    if (detach) {
        if (!behind) {
            behind = t->fork_ev;
            TN_HIP(hipEventRecord(behind, st));
        }
        TN_HIP(hipStreamWaitEvent(t->side, behind, 0));
        TN_HIP(hipStreamWaitEvent(t->aux, behind, 0));
    }
    // rows of a power-of-two dim on a plan that describes its frequent signs: apply_big_wave (detached AdaGrad's from 4 on only)
    const bool tiled = big_desc && s.D <= 64 && (s.D & (s.D - 1)) == 0 && (!detach || (KIND == OPT_ADAGRAD && s.D >= 4));
    const bool all = with_big && !detach && share.lanes != 0;
    if (with_big && !all) {
        const int gfloats = big_gbuf_floats(s.D);
        const int big_blocks = launch_grid(n_upper / BIG_GROUP + 1, 1, 16384);
        hipStream_t bst = detach ? t->side : st;
#define TN_LAUNCH_BIG_ADAGRAD(DIM)                                                                                  \
    TN_LAUNCH((k_apply_big_adagrad<DIM>), dim3(big_blocks), dim3(64), bst, s, o, src, ds, (const uint4*)p.big_desc, \
              p.big_cap, p.list, gaddr)
        if (tiled && s.D == 4) TN_LAUNCH_BIG_ADAGRAD(4);
        else if (tiled && s.D == 8) TN_LAUNCH_BIG_ADAGRAD(8);
        else if (tiled && s.D == 16) TN_LAUNCH_BIG_ADAGRAD(16);
        else if (tiled && s.D == 32) TN_LAUNCH_BIG_ADAGRAD(32);
        else if (tiled && s.D == 64) TN_LAUNCH_BIG_ADAGRAD(64);
        else
            TN_LAUNCH_LDS((k_apply_big<KIND>), dim3(big_blocks), dim3(64), big_lds_bytes(s.D), bst, s, o, src, ds,
                          p.big_list, p.grp_row, p.grp_off, p.grp_cnt, p.list, gfloats, gaddr);
#undef TN_LAUNCH_BIG_ADAGRAD
    }
    if (all) {
        ApplyAll a;
        a.big_blocks = (uint32_t)launch_grid((n_upper / BIG_GROUP + 4) / 4, 1, ALL_BIG_GRID);
        a.multi_blocks = (uint32_t)launch_grid(n_upper * share.lanes / 2, 256, GRID_CAP * 2);
        const uint32_t singles = (uint32_t)launch_grid(n_upper * share.lanes, 256, GRID_CAP * 2);
        a.grp_row = p.grp_row, a.grp_off = p.grp_off, a.grp_cnt = p.grp_cnt, a.big_list = p.big_list;
        a.big_desc = p.big_desc;
        a.big_cap = p.big_cap, a.big_k = big_k, a.ids_cap = ids_cap;
        a.list = p.list;
        a.gaddr = gaddr;
        a.gbuf_floats = std::min(big_gbuf_floats(s.D), ALL_GBUF);
        a.wave_arrays = (uint32_t)align_up((size_t)(a.gbuf_floats + 3 * s.D) * sizeof(float), 8);
        a.wave_lds = a.wave_arrays + BIG_CHUNK * (8 + 4);
#define TN_LAUNCH_ALL_BY(LPG, ANY, TILE)                                                                                   \
    do {                                                                                                                   \
        const dim3 grid(a.big_blocks + a.multi_blocks + singles);                                                          \
        if (tiled && TILE != 0)                                                                                            \
            TN_LAUNCH((k_apply_all<KIND, LPG, ANY, TILE>), grid, dim3(256), st, s, o, src, ds, a);                         \
        else                                                                                                               \
            TN_LAUNCH_LDS((k_apply_all<KIND, LPG, ANY, 0>), grid, dim3(256), 4 * a.wave_lds, st, s, o, src, ds, a);        \
    } while (0)
#define TN_LAUNCH_ALL_ANY(LPG, ANY)  /* (rows of 1 and 2 are a lane's, which they do not fill) */                       \
    do {                                                                                                               \
        constexpr int TILE = big_tile(KIND, LPG);                                                                      \
        if (LPG == 1 && ANY && s.D == 1) TN_LAUNCH_ALL_BY(LPG, ANY, (LPG == 1 && ANY ? 1 : TILE));                     \
        else if (LPG == 1 && ANY && s.D == 2) TN_LAUNCH_ALL_BY(LPG, ANY, (LPG == 1 && ANY ? 2 : TILE));                \
        else TN_LAUNCH_ALL_BY(LPG, ANY, TILE);                                                                         \
    } while (0)
#define TN_LAUNCH_ALL(LPG)                    \
    do {                                      \
        if (share.any)                        \
            TN_LAUNCH_ALL_ANY(LPG, true);     \
        else                                  \
            TN_LAUNCH_ALL_ANY(LPG, false);    \
    } while (0)
        switch (share.lanes) {
            case 1: TN_LAUNCH_ALL(1); break;
            case 2: TN_LAUNCH_ALL(2); break;
            case 4: TN_LAUNCH_ALL(4); break;
            case 8: TN_LAUNCH_ALL(8); break;
            case 16: TN_LAUNCH_ALL(16); break;
            default: TN_LAUNCH_ALL(32); break;
        }
#undef TN_LAUNCH_ALL
#undef TN_LAUNCH_ALL_ANY
#undef TN_LAUNCH_ALL_BY
        return TN_OK;
    }
#define TN_LAUNCH_VEC_ANY(LPG, ANY)                                                                                \
    do {                                                                                                          \
        TN_LAUNCH_EVENT(detach ? t->apply_ev : nullptr, (k_apply_single<KIND, LPG, ANY>),                          \
                        dim3(launch_grid(n_upper * LPG, 256, GRID_CAP * 4)), dim3(256), detach ? t->aux : st, s, o, src, ds, \
                        p.grp_row, p.list);                                                                       \
        TN_LAUNCH((k_apply_vec<KIND, LPG, ANY>), dim3(launch_grid(n_upper * LPG / 2, 256, GRID_CAP * 4)), dim3(256), \
                  detach ? t->side : st, s, o, src, ds, p.grp_row, p.grp_off, p.grp_cnt, p.list, big_k, ids_cap,  \
                  gaddr);                                                                                         \
    } while (0)
#define TN_LAUNCH_VEC(LPG)                        \
    do {                                          \
        if (share.any)                            \
            TN_LAUNCH_VEC_ANY(LPG, true);         \
        else                                      \
            TN_LAUNCH_VEC_ANY(LPG, false);        \
    } while (0)
    switch (share.lanes) {
        case 1: TN_LAUNCH_VEC(1); break;
        case 2: TN_LAUNCH_VEC(2); break;
        case 4: TN_LAUNCH_VEC(4); break;
        case 8: TN_LAUNCH_VEC(8); break;
        case 16: TN_LAUNCH_VEC(16); break;
        case 32: TN_LAUNCH_VEC(32); break;
        default:
            TN_LAUNCH((k_apply_scalar<KIND>), dim3(launch_grid(n_upper, 256, GRID_CAP * 2)), dim3(256), st, s, o, src, ds,
                      p.grp_row, p.grp_off, p.grp_cnt, p.list, big_k, ids_cap);
    }
#undef TN_LAUNCH_VEC
#undef TN_LAUNCH_VEC_ANY
    return TN_OK;
}

// Applies the grouped records; n_upper bounds the number of records.
// addr_ready: p.gaddr already holds the gradient addresses of the multi-record groups' records.
// big_k: the number of records from which the plan's grouping listed a sign for k_apply_big (0: the table's default).
// big_desc: p.big_desc describes the signs of p.big_list (the plan of a pull that grouped through LDS).
int launch_apply(SparseTable* t, const Plan& p, const PushSrc& src, DevStatus* ds, int64_t n_upper, bool vec_ok,
                 hipStream_t st, bool addr_ready = false, uint32_t big_k = 0, bool detach = false, bool big_desc = false,
                 hipEvent_t behind = nullptr) {
    const Store& s = t->store;
    const OptDev o = make_optdev(t);
    const RowShare share = row_share(s, vec_ok);
    if (big_k == 0) big_k = big_threshold(s);
    switch (o.kind) {
        case OPT_ADAGRAD: return launch_apply_kind<OPT_ADAGRAD>(t, share, s, o, src, ds, p, n_upper, st, addr_ready, big_k, detach, big_desc, behind);
        case OPT_ADAM: return launch_apply_kind<OPT_ADAM>(t, share, s, o, src, ds, p, n_upper, st, addr_ready, big_k, detach, big_desc, behind);
        default: return launch_apply_kind<OPT_FTRL>(t, share, s, o, src, ds, p, n_upper, st, addr_ready, big_k, detach, big_desc, behind);
    }
}

// The updates of a small push, one launch (k_small_apply), with the signs with many records if the plan lists such.  flat: the
// reduced rows of pooled gradients, else nullptr.
void launch_small_apply(SparseTable* t, RowShare share, const SmallPlan& p, const float* flat, int dim, hipStream_t st,
                        uint32_t* host_seq, uint32_t seq, hipEvent_t done) {
    const SmallShape& b = t->small_shape;
    const bool with_big = t->plan_big_k != 0xFFFFFFFFu && (uint32_t)b.N >= t->plan_big_k;
    const SmallApplyCall c{b, p, flat, t->store, make_optdev(t), t->dplan, host_seq, seq, dim, share, with_big, st, done};
    switch (c.o.kind) {
        case OPT_ADAGRAD: return tn::launch_small_apply<OPT_ADAGRAD>(c);
        case OPT_ADAM: return tn::launch_small_apply<OPT_ADAM>(c);
        default: return tn::launch_small_apply<OPT_FTRL>(c);
    }
}

// LAUNCH(lanes, any) for the kernels that reduce pooled rows by pool_items: rows of up to 4, 8 or more elements; any: they do
// not fill the lanes, or stand at other than 16-byte boundaries (row_part<true>).
#define TN_POOL_LANES(LAUNCH, D, ALIGNED)                          \
    do {                                                           \
        const int lanes = (D) <= 4 ? 1 : (D) <= 8 ? 2 : 4;         \
        const bool any = !(ALIGNED) || (D) % (4 * lanes) != 0;     \
        if (any && lanes == 1) LAUNCH(1, true);                    \
        else if (any && lanes == 2) LAUNCH(2, true);               \
        else if (any) LAUNCH(4, true);                             \
        else if (lanes == 1) LAUNCH(1, false);                     \
        else if (lanes == 2) LAUNCH(2, false);                     \
        else LAUNCH(4, false);                                     \
    } while (0)

// Where the reduction of a small push's pooled gradients leaves its sums.
struct SmallPool {
    uint32_t lp, blocks;  // workgroups of a slot (2^lp), of the launch
    bool spread;          // heavy signs are dealt to all of a slot's (in one round's lookups none is a chain)
    float *flat, *shares;
    uint32_t* has;
};
int small_pool_room(SparseTable* t, int dim, SmallPool& r) {
    const SmallShape& b = t->small_shape;
    r.lp = small_pool_parts_log2(b.max_len);
    r.blocks = (uint32_t)align_up((size_t)b.N << r.lp, XCDS);
    r.spread = t->plan_heavy && b.max_len > POOL_ITEMS_MAX;
    auto carve = [&](char* base) {
        Carver c{base};
        r.flat = c.take<float>((size_t)b.L * dim);
        r.shares = c.take<float>(r.spread ? (size_t)r.blocks * SMALL_HEAVY_MAX * dim : 0);
        r.has = c.take<uint32_t>(r.spread ? r.blocks : 0);
        return align_up(c.off, 256);
    };
    TN_TRY(t->pooled_ws.ensure(carve(nullptr)));
    carve((char*)t->pooled_ws.p);
    return TN_OK;
}

// The gradients of a small push's distinct signs from pooled ones (k_small_pool).
void launch_small_pool(SparseTable* t, bool aligned, const SmallPlan& p, int64_t batch, int dim, int combiner, const SmallPool& r,
                       hipStream_t st, uint32_t* host_err) {
    static_assert((int)POOL_SUM == (int)COMBINE_SUM && (int)POOL_MEAN == (int)COMBINE_MEAN && (int)POOL_SQRTN == (int)COMBINE_SQRTN, "");
    const SmallShape& b = t->small_shape;
#define TN_LAUNCH_POOL(LPG, ANY)                                                                                           \
    TN_LAUNCH((k_small_pool<LPG, ANY, false>), dim3(r.blocks), dim3(POOL_THREADS), st, b, p, p.push_descs, batch, dim,     \
              t->store.D, combiner, r.flat, t->dplan, host_err, r.lp, r.shares, r.has)
#define TN_LAUNCH_SPREAD(LPG, ANY)                                                                                         \
    TN_LAUNCH((k_small_pool<LPG, ANY, true>), dim3(r.blocks), dim3(POOL_THREADS), st, b, p, p.push_descs, batch, dim,      \
              t->store.D, combiner, r.flat, t->dplan, host_err, r.lp, r.shares, r.has)
#define TN_LAUNCH_SHARES(LPG, ANY)                                                                                         \
    TN_LAUNCH((k_small_pool_shares<LPG, ANY>), dim3((uint32_t)b.N), dim3(64 * SMALL_HEAVY_MAX), st, b, p, dim, t->store.D, \
              r.flat, t->dplan, r.lp, r.shares, r.has)
    if (r.spread) {
        TN_POOL_LANES(TN_LAUNCH_SPREAD, t->store.D, aligned);
        TN_POOL_LANES(TN_LAUNCH_SHARES, t->store.D, dim % 4 == 0);
    } else {
        TN_POOL_LANES(TN_LAUNCH_POOL, t->store.D, aligned);
    }
#undef TN_LAUNCH_SHARES
#undef TN_LAUNCH_SPREAD
#undef TN_LAUNCH_POOL
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

size_t carve_small(char* base, SmallPlan& p, const SmallShape& b) {
    Carver c{base};
    const size_t L = b.L, segments = (size_t)b.N * b.parts;
    p.descs = c.take<SlotDesc>(b.N);
    p.push_descs = c.take<SlotDesc>(b.N);
    p.vals_copy = c.take<uint64_t>(L);
    p.first_of = c.take<uint16_t>(L);
    p.row_at = c.take<uint32_t>(L);
    p.rank_at = c.take<uint16_t>(L);
    p.click_at = c.take<int32_t>(L);
    p.bits = c.take<uint64_t>(segments * b.words);
    p.recs = c.take<uint2>(L * b.parts);
    p.boff = c.take<uint16_t>(segments * (b.nbp + 1));
    p.head = c.take<uint4>(b.buckets());
    p.group = c.take<uint2>((size_t)b.buckets() * b.cap);
    p.member = c.take<uint4>((size_t)b.buckets() * b.cap);
    p.heavy = c.take<uint16_t>(segments * SMALL_HEAVY_MAX);
    p.bad = c.take<uint32_t>(1);
    return align_up(c.off, 256);
}

// The updates of a table-level push (k_table_apply).
void launch_table_apply(SparseTable* t, RowShare share, const TableShape& b, const tn_sign_info* infos, const float* grads,
                        int dim, const uint2* recs, const uint16_t* boff, DevStatus* ds, hipStream_t st) {
    const TableApplyCall c{b, t->store, make_optdev(t), infos, grads, dim, recs, boff, ds, &t->hpush->st.err, share, st,
                           t->table_lds};
    switch (c.o.kind) {
        case OPT_ADAGRAD: return tn::launch_table_apply<OPT_ADAGRAD>(c);
        case OPT_ADAM: return tn::launch_table_apply<OPT_ADAM>(c);
        default: return tn::launch_table_apply<OPT_FTRL>(c);
    }
}

// Does the batch qualify for the path of few launches, and how is it laid out on it?
bool small_batch_shape(SparseTable* t, int N, const int64_t* lens, SmallShape& b) {
    if (!t->small_path || t->async_pull || N <= 0 || N > SMALL_SLOTS || t->dim > 128) return false;
    size_t L = 0, max_len = 0;
    const int64_t longest = N > SMALL_SPLIT_SLOTS ? SMALL_SLOT_MAX : SMALL_SLOT_SHORT;
    for (int s = 0; s < N; s++) {
        if (lens[s] < 0 || lens[s] > longest) return false;
        L += (size_t)lens[s];
        max_len = std::max<size_t>(max_len, (size_t)lens[s]);
    }
    if (L == 0 || L > SMALL_MAX_LOOKUPS) return false;
    if (N <= GRP_SLOTS && (size_t)N * L > (t->pooled_pushes ? SMALL_WORK_POOLED : SMALL_WORK)) return false;
    b.N = N;
    b.L = (uint32_t)L;
    b.max_len = (uint32_t)max_len;
    b.words = (uint32_t)((max_len + 63) / 64);
    b.parts = (uint32_t)std::min<size_t>(SMALL_PARTS_MAX, (max_len + SMALL_PART_LOOKUPS - 1) / SMALL_PART_LOOKUPS);
    while (b.parts > 1 && (size_t)N * b.parts > (size_t)SMALL_SEGMENTS) b.parts--;
    // (every bucket's workgroup looks at all slots: fewer buckets where there are many)
    const size_t most = std::min<size_t>({(L + SMALL_BUCKET_RECORDS - 1) / SMALL_BUCKET_RECORDS, (size_t)SMALL_BUCKETS_MAX,
                                          std::max<size_t>(64, (size_t)(1 << 18) / N)});
    // room for twice the records expected of a batch of distinct signs and for four signs that are in every slot
    auto lay_out = [&](size_t want) {
        // (as many as the chip holds, and not a few more)
        b.nbp = (uint32_t)std::max<size_t>(1, (want + (want < SMALL_BUCKETS_FEW ? b.parts - 1 : 0)) / b.parts);
        b.cap = (uint32_t)align_up(2 * (L / b.buckets()) + 64 + 4 * (size_t)N, 64);
        return small_emit_lds(N, b.cap, small_emit_table(b.cap));
    };
    const uint32_t wide_held = t->dim > 32 ? small_rest_held(lay_out(most)) : 0;
    for (size_t want = std::min(most, std::max<size_t>(SMALL_BUCKETS_FEW, L / small_bucket_lookups(t->dim)));;
         want = std::min(most, want + want / 4)) {
        // no fewer than let the pull's second half be one launch, and a CU hold as many workgroups of it where rows are wide
        const size_t lds = lay_out(want);
        if (want == most || (lds <= SMALL_SHARED_LDS && small_rest_held(lds) >= wide_held)) break;
    }
    if (!t->small_lds) {
        t->small_lds = 144 * 1024;
        for (const void* k : {(const void*)k_small_slots<ArgDescs>, (const void*)k_small_slots<HostDescs>,
                              (const void*)k_small_slots_long<ArgDescs>, (const void*)k_small_slots_long<HostDescs>})
            t->small_lds = std::min(t->small_lds, big_lds_bytes_for(k, 144 * 1024));
        t->small_emit_lds = big_lds_bytes_for(reinterpret_cast<const void*>(k_group_emit<true>), 144 * 1024);
    }
    return small_slots_lds(small_entries(b.max_len, b.parts), b.max_len, b.nbp) <= t->small_lds &&
           small_emit_lds(N, b.cap, small_emit_table(b.cap)) <= t->small_emit_lds;
}

thread_local void (*waiting_fn)(void*) = nullptr;
thread_local void* waiting_arg = nullptr;

// The launches are queued and the host is about to wait for them.
void do_host_work() {
    if (void (*fn)(void*) = waiting_fn) {
        waiting_fn = nullptr;
        fn(waiting_arg);
    }
}

// Waits for kernels on `st` to report through pinned memory: there() looks whether they have.  It is polled for a
// while (a word arrives a few microseconds after it is written, well before a wait on the stream or on an event
// returns).  A caller's stream with much else to do ahead of the call is looked at now and then from there on: until the
// report is there, whatever is queued behind it, or the stream has ended without, which also brings a failed launch to light.
template <typename There>
int wait_until(There there, hipStream_t st, const char* what) {
    const auto t0 = std::chrono::steady_clock::now();
    for (uint32_t spins = 1;; spins++) {
        if (there()) break;
        __builtin_ia32_pause();
        if ((spins & 255u) || std::chrono::steady_clock::now() - t0 < std::chrono::milliseconds(2)) continue;
        const hipError_t state = hipStreamQuery(st);
        if (state == hipErrorNotReady) {
            std::this_thread::sleep_for(std::chrono::microseconds(20));
            continue;
        }
        TN_HIP(state);
        if (!there()) return fail(TN_ERR_HIP, std::string(what) + ": the device did not report");
        break;
    }
    std::atomic_thread_fence(std::memory_order_acquire);  // what the device wrote before the report is read after it
    return TN_OK;
}
int wait_reported(const uint32_t* flag, uint32_t want, hipStream_t st, const char* what) {
    const volatile uint32_t* f = flag;
    return wait_until([&] { return *f == want; }, st, what);
}

// The same for the words of a small pull's first launch: hwords[0 .. n) all carry `seq`.
int wait_words(const uint64_t* words, uint32_t n, uint32_t seq, hipStream_t st, const char* what) {
    do_host_work();
    const volatile uint64_t* w = words;
    uint32_t i = 0;
    return wait_until(
        [&] {
            while (i < n && (uint32_t)(w[i] >> 32) == seq) i++;
            return i == n;
        },
        st, what);
}

// SparseTablePull of a small batch laid out as `b` (the caller has validated the call and made room in the table).
int small_pull(SparseTable* t, const SmallShape& b, const int64_t* const* values, const int64_t* lens, float* const* vars,
               const int64_t* var_rows, int wdim, int64_t* const* mapped, hipStream_t st) {
    const Store& s = t->store;
    TN_TRY(order_after_updates(t, st));
    SmallPlan p{};
    const size_t bytes = carve_small(nullptr, p, b);
    // (a plan buffer that has to grow is freed first: not under detached updates that still read it)
    if (t->upd_pending && bytes > t->plan_buf.bytes) TN_HIP(hipEventSynchronize(t->upd_ev));
    TN_TRY(t->plan_buf.ensure(bytes));
    carve_small((char*)t->plan_buf.p, p, b);
    t->plan_valid = false;
    const bool by_value = b.N <= ARG_SLOTS;
    if (!by_value) TN_TRY(staging_free(t));
    ArgDescs args;
    SlotDesc* descs = by_value ? args.slot : reinterpret_cast<SlotDesc*>(t->hstage);
    int width = row_width(wdim, s.wstride);
    uint32_t at = 0;
    for (int i = 0; i < b.N; i++) {
        SlotDesc d{};
        d.values = values[i];
        d.mapped = mapped[i];
        d.var = vars[i];
        d.rows = var_rows[i];
        d.len = (uint32_t)lens[i];
        d.lbase = at;
        descs[i] = d;
        at += d.len;
        width = row_width_at(width, vars[i]);
    }
    const uint32_t seq = ++t->seq_pull, workgroups = (uint32_t)b.N * b.parts, entries = small_entries(b.max_len, b.parts);
    const size_t slots_lds = small_slots_lds(entries, b.max_len, b.nbp);
    auto launch_slots = [&](const auto& by) {
        using Descs = std::decay_t<decltype(by)>;
        // (the names the profiler knows them by)
        constexpr auto k_small_slots = tn::k_small_slots<Descs>;
        constexpr auto k_small_slots_long = tn::k_small_slots_long<Descs>;
        if (b.max_len <= SMALL_SLOT_SHORT)
            TN_LAUNCH_LDS(k_small_slots, dim3(workgroups), dim3(SMALL_THREADS), slots_lds, st, b, p, by, entries, s, make_optdev(t),
                          t->seed, t->dplan, t->hwords, seq);
        else
            TN_LAUNCH_LDS(k_small_slots_long, dim3(workgroups), dim3(2 * SMALL_THREADS), slots_lds, st, b, p, by, entries, s,
                          make_optdev(t), t->seed, t->dplan, t->hwords, seq);
    };
    if (by_value)
        launch_slots(args);
    else
        launch_slots(HostDescs{descs});
    const uint32_t C = (uint32_t)(wdim / width), items = (size_t)b.L * C > FINISH_FULL ? FINISH_ITEMS : 1;
    const uint32_t per = items * FINISH_THREADS / C, chunks = (b.max_len + per - 1) / per;
    EmitArgs<true> ea;
    ea.b = b;
    ea.p = p;
    ea.table = small_emit_table(b.cap);
    ea.big_k = t->plan_big_k = b.N <= SMALL_NO_BIG_SLOTS ? 0xFFFFFFFFu : SMALL_BIG_GROUP;
    const size_t emit_lds = small_emit_lds(b.N, b.cap, ea.table);
    const uint32_t finish = (uint32_t)b.N * chunks;
    if (b.N > SMALL_SPLIT_SLOTS && emit_lds <= SMALL_SHARED_LDS) {
#define TN_LAUNCH_REST(VEC)                                                                                              \
    TN_LAUNCH_LDS((k_small_pull_rest<VEC>), dim3(b.buckets() + finish), dim3(FINISH_THREADS), emit_lds, st, ea, chunks, per, s)
        if (width == 4) TN_LAUNCH_REST(4);
        else if (width == 2) TN_LAUNCH_REST(2);
        else TN_LAUNCH_REST(1);
#undef TN_LAUNCH_REST
    } else {
#define TN_LAUNCH_FINISH(VEC) \
    TN_LAUNCH((k_small_group_finish<VEC>), dim3(finish), dim3(FINISH_THREADS), st, b, p, chunks, per, s)
        if (width == 4) TN_LAUNCH_FINISH(4);
        else if (width == 2) TN_LAUNCH_FINISH(2);
        else TN_LAUNCH_FINISH(1);
#undef TN_LAUNCH_FINISH
        TN_LAUNCH_LDS((k_group_emit<true>), dim3(b.buckets()), dim3(FINISH_THREADS), emit_lds, st, ea);
    }
    TN_TRY(record_tail(t, st));
    TN_HIP(hipGetLastError());
    // the call returns when the first launch has reported: what follows is complete in stream order
    t->small_shape = b;
    t->plan_valid = true;
    t->plan_small = true;
    t->plan_clicks_dirty = false;
    t->plan_has_show = true;
    t->plan_prints = false;
    t->plan_exact = false;
    t->plan_big_desc = false;
    t->plan_N = b.N;
    t->plan_lens.assign(lens, lens + b.N);
    t->plan_epoch = t->epoch;
    TN_TRY(wait_words(t->hwords, workgroups, seq, st, "SparseTablePull"));
    harvest(t);  // (a push before this call)
    uint64_t n_new = 0, n_distinct = 0;
    bool full = false;
    t->plan_heavy = false;
    constexpr uint64_t MASK = (1u << SMALL_REPORT_BITS) - 1u;
    t->last_counts.assign(b.N, 0);
    for (uint32_t i = 0; i < workgroups; i++) {
        const uint64_t w = t->hwords[i];
        t->last_counts[i / b.parts] += (int64_t)(w & MASK);
        n_new += (w >> SMALL_REPORT_BITS) & MASK;
        full |= ((w >> (2 * SMALL_REPORT_BITS)) & 1u) != 0;
        t->plan_heavy |= ((w >> (2 * SMALL_REPORT_BITS)) & 2u) != 0;
    }
    // the call booked room for every sign it could have inserted; keep what it did insert
    t->count_upper -= t->booked - n_new;
    t->booked = 0;
    if (full) latch(t, TN_ERR_TABLE_FULL, std::string("sparse pull: ") + dev_err_text(DEV_ERR_TABLE_FULL));
    for (int i = 0; i < b.N; i++) {
        n_distinct += (uint64_t)t->last_counts[i];
        if (t->last_counts[i] >= var_rows[i]) latch_var_capacity(t, i, var_rows[i]);
    }
    note_distinct_share(t, (double)n_distinct / (double)b.L);
    t->plan_counts = t->last_counts;
    return take_latched(t);
}

// A push on the plan of a small pull (same shape, same table).  *other_batch: its signs turned out to be others.
int small_push(SparseTable* t, const int64_t* const* values, const float* const* grads, const int64_t* grad_rows, int dim,
               const int64_t* const* labels, const int64_t* const* example_ids, int64_t batch, int combiner, bool vec,
               hipStream_t st, bool* other_batch) {
    const SmallShape& b = t->small_shape;
    const bool pooled = example_ids != nullptr, clicks = t->opt->kind == OPT_ADAGRAD;  // (the only optimizer that reads batch_click)
    SmallPlan p{};
    carve_small((char*)t->plan_buf.p, p, b);
    SmallPool pool{};
    if (pooled) TN_TRY(small_pool_room(t, dim, pool));
    const bool by_value = b.N <= ARG_SLOTS;
    if (!by_value) TN_TRY(staging_free(t));
    ArgDescs args;
    SlotDesc* descs = by_value ? args.slot : reinterpret_cast<SlotDesc*>(t->hstage);
    uint32_t at = 0;
    for (int i = 0; i < b.N; i++) {
        SlotDesc d{};
        d.values = values[i];
        d.labels = labels[i];
        d.grads = grads[i];
        d.rows = pooled ? batch : grad_rows[i];
        if (pooled) d.mapped = const_cast<int64_t*>(example_ids[i]);
        d.len = (uint32_t)t->plan_lens[i];
        d.lbase = at;
        descs[i] = d;
        at += d.len;
    }
    t->hpush->st.mismatch = 0;
    t->hpush->st.abort = 0;
    const uint32_t seq = ++t->seq_verify, chunks = (b.max_len + SMALL_TILE - 1) / SMALL_TILE;
    // (the records of pooled gradients go by their first lookups, not by rank)
    const uint32_t verify_blocks = (uint32_t)b.N * chunks + (pooled ? 0u : (b.buckets() + 3) / 4);
    auto launch_verify = [&](const auto& by) {
        using Descs = std::decay_t<decltype(by)>;
#define TN_VERIFY(KERNEL, CLICKS)                                                                                          \
    do {                                                                                                                   \
        if (g_profile_on) prof_begin(KERNEL, st);                                                                          \
        hipLaunchKernelGGL((k_small_verify<CLICKS, Descs>), dim3(verify_blocks), dim3(256), 0, st, b, p, by, chunks, \
                           t->dplan, &t->hpush->st.mismatch);                                                              \
        if (g_profile_on) prof_end(st);                                                                                    \
    } while (0)
        if (clicks)
            TN_VERIFY("k_small_verify<true>", true);
        else
            TN_VERIFY("k_small_verify<false>", false);
#undef TN_VERIFY
    };
    if (by_value)
        launch_verify(args);
    else
        launch_verify(HostDescs{descs});
    const bool rows16 = dim % 4 == 0 && t->store.wstride % 4 == 0;
    if (pooled)
        launch_small_pool(t, vec, p, batch, dim, combiner, pool, st, &t->hpush->st.abort);
    // (tail_ev is what a call on another stream has to wait for: the updates are still running when this call returns)
    launch_small_apply(t, row_share(t->store, (pooled || vec) && rows16), p, pool.flat, dim, st, t->hseq + 1, seq,
                       tail_event(t, st));
    TN_HIP(hipGetLastError());
    // the outcome of the comparison: the updates are queued behind it and do nothing on a mismatch
    TN_TRY(wait_reported(t->hseq + 1, seq, st, "SparseTablePush"));
    *other_batch = t->hpush->st.mismatch != 0;
    if (*other_batch) return TN_OK;
    t->last_counts = t->plan_counts;
    if (pooled) {
        if (t->hpush->st.abort) {  // reported by the next call that waits, like the other errors of a push's device work
            t->plan_valid = false;  // (its click sums have been added and not taken up)
            latch(t, TN_ERR_INVALID_ARGUMENT, std::string("sparse push: ") + dev_err_text(DEV_ERR_GRAD_ROWS));
        }
        return TN_OK;
    }
    // (the records without a gradient row were left out by the update kernel, as on the other paths)
    for (int i = 0; i < b.N; i++)
        if (grad_rows[i] < t->plan_counts[i])
            return fail(TN_ERR_INVALID_ARGUMENT, std::string("sparse push: ") + dev_err_text(DEV_ERR_GRAD_ROWS) + " (slot " +
                                                     std::to_string(i) + ")");
    return TN_OK;
}

}  // namespace
}  // namespace tn

using namespace tn;

extern "C" {

int tn_sparse_table_create(tn_opt_t opt, const char* name, int dimension, int use_cvm, int shard_num,
                           int self_shard_id, const char* embedding_group, uint32_t* handle) {
    if (!handle) return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_create: handle is NULL");
    auto conf = get_opt(opt);
    if (!conf) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_create: unknown optimizer handle");
    if (dimension <= 0 || dimension > 4096)
        return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_create: dimension must be in [1, 4096]");
    if (shard_num != 1 || self_shard_id != 0)
        return fail(TN_ERR_UNSUPPORTED, "tn_sparse_table_create: one worker only (shard_num 1, self_shard_id 0)");
    std::string group = embedding_group ? embedding_group : "";
    std::lock_guard<std::mutex> lk(g_tables_mu);
    if (!group.empty()) {  // sparse_table.cc:175-180
        for (SparseTable* t : g_tables)
            if (t->group == group) {
                *handle = t->handle;
                return TN_OK;
            }
    }
    SparseTable* t = new SparseTable();
    t->opt = conf;
    t->name = name ? name : "";
    t->group = group;
    t->dim = dimension;
    // only the AdaGrad row maintains the cvm columns (ada_grad_kernel.cc:99-102,123-128)
    t->use_cvm = (use_cvm && conf->kind == OPT_ADAGRAD) ? 1 : 0;
    t->shard_num = shard_num;
    t->self_shard_id = self_shard_id;
    if (hipGetDevice(&t->device) != hipSuccess) t->device = 0;
    t->handle = (uint32_t)g_tables.size();
    g_tables.push_back(t);
    *handle = t->handle;
    return TN_OK;
}

int tn_sparse_table_reserve(uint32_t handle, uint64_t max_keys) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_reserve: bad table handle " + std::to_string(handle));
    std::lock_guard<std::mutex> lk(t->mu);
    if (!t->allocated) {
        t->reserve_keys = max_keys;
        return TN_OK;
    }
    hipStream_t st = t->last_stream;
    if (t->push_pending || t->pull_pending) {
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    uint64_t want = reserved_slots(t, max_keys);
    if (want <= t->store.cap) return TN_OK;
    return grow_to(t, want, st);
}

int tn_sparse_table_clear(uint32_t handle) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_clear: bad table handle " + std::to_string(handle));
    std::lock_guard<std::mutex> lk(t->mu);
    if (!t->allocated) return TN_OK;
    // everything the table has queued, on whichever stream
    TN_HIP(hipStreamSynchronize(t->last_stream));
    TN_HIP(hipStreamSynchronize(t->side));
    TN_HIP(hipStreamSynchronize(t->aux));
    harvest(t);
    free_store(t->store);
    t->ws.release();
    t->plan_buf.release();
    t->comb_buf.release();
    t->pooled_ws.release();
    t->allocated = false;
    t->plan_valid = false;
    t->tail_recorded = false;
    t->tail_owed = false;
    t->count_upper = 0;
    t->booked = 0;
    t->epoch++;
    t->latched = TN_OK;
    t->latched_msg.clear();
    return TN_OK;
}

int tn_sparse_table_set_seed(uint32_t handle, uint64_t seed) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_set_seed: bad table handle " + std::to_string(handle));
    std::lock_guard<std::mutex> lk(t->mu);
    t->seed = seed;
    return TN_OK;
}

int tn_sparse_table_key_count(uint32_t handle, uint64_t* count) {
    SparseTable* t = get_table(handle);
    if (!t || !count) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_key_count: bad table handle");
    std::lock_guard<std::mutex> lk(t->mu);
    *count = 0;
    if (!t->allocated) return TN_OK;
    // Only this table's own work is waited for: the count is kept by kernels on the stream of the table's last
    // call (a pull has waited for its status before it returned).
    if (t->push_pending || t->pull_pending) {
        TN_HIP(hipStreamSynchronize(t->last_stream));
        harvest(t);
    }
    uint64_t cnt = 0;
    TN_TRY(read_count(t, t->last_stream, &cnt));
    *count = cnt;
    return TN_OK;
}

int tn_sparse_table_capacity(uint32_t handle, uint64_t* slots) {
    SparseTable* t = get_table(handle);
    if (!t || !slots) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_capacity: bad table handle");
    std::lock_guard<std::mutex> lk(t->mu);
    *slots = t->allocated ? t->store.cap : 0;
    return TN_OK;
}

int tn_sparse_table_row_layout(uint32_t handle, int* weight_floats, int* state_floats_out) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_row_layout: bad table handle");
    if (weight_floats) *weight_floats = t->dim + (t->use_cvm ? 2 : 0);
    if (state_floats_out) *state_floats_out = state_floats(t);
    return TN_OK;
}

int tn_sparse_table_set_async(uint32_t handle, int async_pull) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_set_async: bad table handle");
    std::lock_guard<std::mutex> lk(t->mu);
    t->async_pull = async_pull ? 1 : 0;
    return TN_OK;
}

int tn_sparse_table_set_small_batch_path(uint32_t handle, int enable) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "bad sparse table handle");
    std::lock_guard<std::mutex> lk(t->mu);
    t->small_path = enable != 0;
    return TN_OK;
}

int tn_sparse_table_set_exact_verify(uint32_t handle, int enable) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "bad sparse table handle");
    std::lock_guard<std::mutex> lk(t->mu);
    t->exact_verify = enable != 0;
    return TN_OK;
}

int tn_sparse_table_set_detached_updates(uint32_t handle, int enable) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "bad sparse table handle");
    std::lock_guard<std::mutex> lk(t->mu);
    t->detach_updates = enable != 0;
    return TN_OK;
}

int tn_sparse_table_sync(uint32_t handle) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_sync: bad table handle " + std::to_string(handle));
    std::lock_guard<std::mutex> lk(t->mu);
    if (!t->allocated) return TN_OK;
    return sync_table(t, t->last_stream);
}

int tn_sparse_table_last_unique_counts(uint32_t handle, int N, int64_t* counts) {
    SparseTable* t = get_table(handle);
    if (!t || !counts) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_last_unique_counts: bad table handle");
    std::lock_guard<std::mutex> lk(t->mu);
    if (t->pull_pending || t->push_pending) {
        TN_HIP(hipStreamSynchronize(t->last_stream));
        harvest(t);
    }
    if ((int)t->last_counts.size() != N)
        return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_last_unique_counts: last op had " +
                                                 std::to_string(t->last_counts.size()) + " slots");
    for (int s = 0; s < N; s++) counts[s] = t->last_counts[s];
    return TN_OK;
}

// ------------------------------------------------------------ table level
int tn_sparse_table_pull(uint32_t handle, const uint64_t* signs, int64_t n, int dim, float* out, void* stream) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_pull: bad table handle " + std::to_string(handle));
    if (n < 0 || (n > 0 && (!signs || !out))) return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_pull: NULL buffer");
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    TN_TRY(ensure_allocated(t, st));
    const int wdim = t->dim + (t->use_cvm ? 2 : 0);
    if (dim != wdim)
        return fail(TN_ERR_DIM_MISMATCH,
                    "tn_sparse_table_pull: dim " + std::to_string(dim) + " but table rows hold " + std::to_string(wdim));
    if (n > 0x7FFFFFF0LL) return fail(TN_ERR_UNSUPPORTED, "tn_sparse_table_pull: more than 2^31 signs");
    // a push pending on this stream is collected behind this call's own wait
    if (t->pull_pending || (t->push_pending && other_stream(t, st))) {
        if (other_stream(t, st)) TN_HIP(hipStreamSynchronize(t->last_stream));
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    set_last_stream(t, st);
    if (n == 0) return sync_table(t, st);
    TN_TRY(ensure_room(t, (uint64_t)n, st));
    TN_TRY(t->ws.ensure(align_up((size_t)n * sizeof(uint32_t), 256)));
    uint32_t* rows = (uint32_t*)t->ws.p;
    const Store& s = t->store;
    const bool vec = wdim % 4 == 0 && s.wstride % 4 == 0 && aligned16(out);
    const uint32_t per = n > 64 * (int64_t)TABLE_PULL_FEW ? 256 : 64;
    const uint32_t workgroups = (uint32_t)std::min<int64_t>((n + per - 1) / per, TABLE_PULL_WORDS);
    const uint32_t seq = ++t->seq_pull;
    const auto k_table_pull =
        table_pull_few(n, per, (uint32_t)(vec ? wdim / 4 : wdim)) ? tn::k_table_pull<1> : tn::k_table_pull<PULL_AHEAD>;
    TN_LAUNCH(k_table_pull, dim3(workgroups), dim3(256), st, s, make_optdev(t), t->seed, signs, n, per, vec ? 1 : 0, out, rows,
              t->hwords, seq);
    // The rows are written when the call returns, for readers on any stream: a launch behind the pull says that it has
    // ended.  (A workgroup's own word does not: its other wavefronts' rows may still be on their way.  60 000 signs of 16
    // elements pushed and pulled: 52 us by the workgroups' words alone, 54 with this, 61 with a wait for the stream.)
    const uint32_t end_seq = ++t->seq_comb;
    TN_LAUNCH(k_report, dim3(1), dim3(64), st, t->dcomb, t->hcomb, end_seq);
    TN_HIP(hipGetLastError());
    TN_TRY(wait_words(t->hcomb, 1, end_seq, st, "tn_sparse_table_pull"));
    TN_TRY(wait_words(t->hwords, workgroups, seq, st, "tn_sparse_table_pull"));
    uint64_t n_new = 0;
    uint32_t err = 0;
    for (uint32_t i = 0; i < workgroups; i++) {
        n_new += t->hwords[i] & 0x7FFFFFFFu;
        if ((t->hwords[i] >> 31) & 1u) err = DEV_ERR_TABLE_FULL;
    }
    harvest(t);
    // the call booked room for every sign it could have inserted; keep what it did insert
    t->count_upper -= t->booked - n_new;
    t->booked = 0;
    t->last_counts.clear();
    latch(t, dev_err_code(err), std::string("sparse pull: ") + dev_err_text(err));
    if (n_new) {  // a sign that occurs several times may have been copied out before its new row was filled
        if (vec)
            TN_LAUNCH((k_gather_rows<4>), dim3(launch_grid(n * (wdim / 4), 256, GRID_CAP * 4)), dim3(256), st, s, rows, n, out);
        else
            TN_LAUNCH((k_gather_rows<1>), dim3(launch_grid(n * wdim, 256, GRID_CAP * 4)), dim3(256), st, s, rows, n, out);
        TN_HIP(hipGetLastError());
        TN_HIP(hipStreamSynchronize(st));
    }
    if (t->upd_pending) return sync_table(t, st);  // (an earlier push's updates on streams of their own)
    return take_latched(t);
}

namespace {
constexpr int STATIC_MAX_DEVICES = 64;
std::mutex g_static_mu;  // one call at a time uses a GPU's scratch array
unsigned char* g_static_ptr[STATIC_MAX_DEVICES] = {};

// Address of the current device's copy of `scratch`, looked up once per device.
int static_scratch(int* device, unsigned char** out) {
    int dev = 0;
    TN_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= STATIC_MAX_DEVICES)
        return fail(TN_ERR_UNSUPPORTED, "tn_sparse_table_pull_static: device number beyond " + std::to_string(STATIC_MAX_DEVICES));
    if (!g_static_ptr[dev]) {
        unsigned char* ptr = nullptr;
        TN_HIP(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
        if (!ptr) return fail(TN_ERR_HIP, "tn_sparse_table_pull_static: no address for the scratch array");
        g_static_ptr[dev] = ptr;
    }
    *device = dev;
    *out = g_static_ptr[dev];
    return TN_OK;
}
}  // namespace

int tn_sparse_table_pull_static(uint32_t handle, const uint64_t* signs, int64_t n, int dim, float* out, void* stream) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_pull_static: bad table handle " + std::to_string(handle));
    if (n < 0 || (n > 0 && (!signs || !out)))
        return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_pull_static: NULL buffer");
    if (n > TN_STATIC_MAX_SIGNS)
        return fail(TN_ERR_UNSUPPORTED, "tn_sparse_table_pull_static: " + std::to_string(n) + " signs, at most " +
                                            std::to_string(TN_STATIC_MAX_SIGNS) + " per call (use tn_sparse_table_pull)");
    std::lock_guard<std::mutex> sk(g_static_mu);
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    int dev = 0;
    unsigned char* ptr = nullptr;
    TN_TRY(static_scratch(&dev, &ptr));
    if (!t->allocated)
        return fail(TN_ERR_UNSUPPORTED, "tn_sparse_table_pull_static: the table has no storage yet (its first call through "
                                        "another entry point allocates it); this entry point allocates nothing");
    if (dev != t->device)
        return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_pull_static: the table lives on device " +
                                                 std::to_string(t->device) + ", the current device is " + std::to_string(dev));
    // the prologue every entry point shares (ensure_allocated), less the allocation
    TN_TRY(order_after_updates(t, st));
    TN_TRY(order_after_other_stream(t, st));
    const int wdim = t->dim + (t->use_cvm ? 2 : 0);
    if (dim != wdim)
        return fail(TN_ERR_DIM_MISMATCH, "tn_sparse_table_pull_static: dim " + std::to_string(dim) +
                                             " but table rows hold " + std::to_string(wdim));
    if (t->push_pending || t->pull_pending) {
        if (other_stream(t, st)) TN_HIP(hipStreamSynchronize(t->last_stream));
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    set_last_stream(t, st);
    if (n == 0) return sync_table(t, st);
    const Store& s = t->store;
    // every requested sign may be new; a table that would have to grow for them needs a new allocation
    if ((double)(t->count_upper + (uint64_t)n) > MAX_LOAD * (double)s.cap) {
        uint64_t cnt = 0;  // the bound may be loose: read the true count (pinned memory, no allocation)
        TN_TRY(read_count(t, st, &cnt));
        if ((double)(cnt + (uint64_t)n) > MAX_LOAD * (double)s.cap)
            return fail(TN_ERR_TABLE_FULL, "tn_sparse_table_pull_static: the table would have to grow for " +
                                               std::to_string(n) + " more signs, which needs an allocation "
                                               "(tn_sparse_table_reserve beforehand, or tn_sparse_table_pull)");
    }
    t->count_upper += (uint64_t)n;
    t->booked = (uint64_t)n;
    DevStatus* ds = reinterpret_cast<DevStatus*>(ptr);
    uint32_t* rows = reinterpret_cast<uint32_t*>(ptr + TN_STATIC_STATUS_BYTES);
    uint32_t* newlist = rows + TN_STATIC_MAX_SIGNS;
    const OptDev o = make_optdev(t);
    const int blocks = launch_grid(n, 256, GRID_CAP * 2);
    // the array keeps the last call's contents: the status block is cleared here, rows[0 .. n) and
    // newlist[0 .. new rows) are written by this call's probe before anything reads them
    TN_LAUNCH(k_reset_status, dim3(1), dim3(64), st, ds, (uint32_t)n, 0u);
    TN_LAUNCH((k_probe<true>), dim3(blocks), dim3(256), st, s, signs, n, (const DevStatus*)nullptr, 0u, rows, newlist, ds,
              (uint32_t)DEV_ERR_TABLE_FULL, o, t->seed);
    TN_LAUNCH(k_init_rows, dim3(blocks), dim3(256), st, s, o, t->seed, signs, rows, newlist, ds);
    TN_LAUNCH(k_finish_insert, dim3(1), dim3(64), st, s, ds);
    if (wdim % 4 == 0 && s.wstride % 4 == 0 && aligned16(out))
        TN_LAUNCH((k_gather_rows<4>), dim3(launch_grid(n * (wdim / 4), 256, GRID_CAP * 4)), dim3(256), st, s, rows, n, out);
    else
        TN_LAUNCH((k_gather_rows<1>), dim3(launch_grid(n * wdim, 256, GRID_CAP * 4)), dim3(256), st, s, rows, n, out);
    TN_HIP(hipGetLastError());
    TN_HIP(hipMemcpyAsync(&t->hpull->st, ds, sizeof(DevStatus), hipMemcpyDeviceToHost, st));
    t->hpull->ubase[0] = 0;
    t->pull_pending = true;
    t->pull_slots = 0;
    t->pending_rows.clear();
    return sync_table(t, st);  // the scratch array is free again when the lock is released
}

int tn_sparse_table_push(uint32_t handle, const tn_sign_info* infos, const float* grads, int64_t n, int dim,
                         void* stream) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_push: bad table handle " + std::to_string(handle));
    if (n < 0 || (n > 0 && (!infos || !grads))) return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_push: NULL buffer");
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    TN_TRY(ensure_allocated(t, st));
    const int wdim = t->dim + (t->use_cvm ? 2 : 0);
    if (dim != wdim)
        return fail(TN_ERR_DIM_MISMATCH,
                    "tn_sparse_table_push: dim " + std::to_string(dim) + " but table rows hold " + std::to_string(wdim));
    if (n > 0x7FFFFFF0LL) return fail(TN_ERR_UNSUPPORTED, "tn_sparse_table_push: more than 2^31 records");
    if (n > 0 && (t->push_pending || t->pull_pending)) {  // one status block per direction: collect the previous one first
        if (other_stream(t, st)) TN_HIP(hipStreamSynchronize(t->last_stream));
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    set_last_stream(t, st);
    if (n == 0) return TN_OK;
    const Store& s = t->store;
    const RowShare share = row_share(s, aligned16(grads) && dim % 4 == 0 && s.wstride % 4 == 0);
    DevStatus* ds = t->dtpush;
    if (share.lanes != 0 && n <= (int64_t)TABLE_TILES * TABLE_THREADS * TABLE_ITEMS_MAX) {
        // two launches (table_level.h), for rows of up to 128 elements (a wavefront half holds no more) and up to 2 M
        // records (a bucket's workgroup looks at every tile, and a tile holds what a workgroup keeps in registers)
        TableShape b{};
        b.n = (uint32_t)n;
        b.tile = TABLE_THREADS;
        while (b.tile < (uint32_t)(TABLE_THREADS * TABLE_ITEMS_MAX) && (n + b.tile - 1) / b.tile > (int64_t)TABLE_TILES) b.tile *= 4;
        b.tiles = (uint32_t)((n + b.tile - 1) / b.tile);
        b.nb = (uint32_t)std::min<int64_t>({(n + TABLE_BUCKET_RECORDS - 1) / TABLE_BUCKET_RECORDS, (int64_t)TABLE_BUCKETS,
                                            (int64_t)(s.cap / 64)});
        b.scale = (uint32_t)((((uint64_t)b.nb << 32)) / (s.cap + 1));
        while ((1u << b.bits) < b.nb) b.bits++;
        auto carve = [&](Carver& c, uint2*& recs, uint16_t*& boff) {
            recs = c.take<uint2>((size_t)b.tiles * b.tile);
            boff = c.take<uint16_t>((size_t)b.tiles * (b.nb + 1));
        };
        uint2* recs = nullptr;
        uint16_t* boff = nullptr;
        Carver room{nullptr};
        carve(room, recs, boff);
        TN_TRY(t->ws.ensure(align_up(room.off, 256) + 256));
        Carver c{(char*)t->ws.p};
        carve(c, recs, boff);
        const size_t part_lds = ((size_t)part_word(b.nb * TABLE_WAVES) + 1) * sizeof(uint32_t);
        if (b.tile == TABLE_THREADS)
            TN_LAUNCH_LDS((k_table_part<1>), dim3(b.tiles), dim3(TABLE_THREADS), part_lds, st, b, s, infos, recs, boff, ds);
        else if (b.tile == 4 * TABLE_THREADS)
            TN_LAUNCH_LDS((k_table_part<4>), dim3(b.tiles), dim3(TABLE_THREADS), part_lds, st, b, s, infos, recs, boff, ds);
        else
            TN_LAUNCH_LDS((k_table_part<16>), dim3(b.tiles), dim3(TABLE_THREADS), part_lds, st, b, s, infos, recs, boff, ds);
        t->hpush->st.err = 0;
        launch_table_apply(t, share, b, infos, grads, dim, recs, boff, ds, st);
        TN_HIP(hipGetLastError());
        t->push_pending = true;
        t->push_slots = 0;
        return TN_OK;
    }
    Plan p{};
    Scratch w{};
    {
        Carver probe{nullptr};
        carve_groups(probe, p, (size_t)n);
        carve_group_scratch(probe, w, (size_t)n);
        TN_TRY(t->ws.ensure(align_up(probe.off, 256) + 256));
        Carver c{(char*)t->ws.p};
        carve_groups(c, p, (size_t)n);
        carve_group_scratch(c, w, (size_t)n);
    }
    PushSrc src{};
    src.infos = infos;
    src.grads = grads;
    src.dim = dim;
    ds = t->dstatus;
    TN_LAUNCH(k_reset_status, dim3(1), dim3(64), st, ds, (uint32_t)n, (uint32_t)group_cap((size_t)n));
    launch_grouping(p, w, src, n, n, big_threshold(t->store), nullptr, ds, st);
    TN_LAUNCH((k_probe<false>), dim3(launch_grid(n, 256, GRID_CAP * 2)), dim3(256), st, t->store, p.grp_sign,
              (int64_t)0, ds, (uint32_t)n, p.grp_row, (uint32_t*)nullptr, ds, (uint32_t)DEV_ERR_UNKNOWN_KEY, make_optdev(t), t->seed);
    TN_TRY(launch_apply(t, p, src, ds, n, aligned16(grads) && dim % 4 == 0, st));
    TN_HIP(hipGetLastError());
    TN_HIP(hipMemcpyAsync(&t->hpush->st, t->dstatus, sizeof(DevStatus), hipMemcpyDeviceToHost, st));
    t->push_pending = true;
    t->push_slots = 0;
    return TN_OK;
}

int tn_sparse_table_load_rows(uint32_t handle, const uint64_t* signs, const float* w, const float* state, int64_t n,
                              void* stream) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_load_rows: bad table handle " + std::to_string(handle));
    if (n < 0 || (n > 0 && (!signs || !w))) return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_load_rows: NULL buffer");
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    TN_TRY(ensure_allocated(t, st));
    set_last_stream(t, st);
    if (n == 0) return TN_OK;
    if (n > 0x7FFFFFF0LL) return fail(TN_ERR_UNSUPPORTED, "tn_sparse_table_load_rows: more than 2^31 rows per call");
    if (t->push_pending || t->pull_pending) {
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    TN_TRY(ensure_room(t, (uint64_t)n, st));
    TN_TRY(t->ws.ensure(2 * align_up((size_t)n * sizeof(uint32_t), 256)));
    Carver c{(char*)t->ws.p};
    uint32_t* rows = c.take<uint32_t>(n);
    uint32_t* newlist = c.take<uint32_t>(n);
    const Store& s = t->store;
    const int blocks = launch_grid(n, 256, GRID_CAP * 4);
    TN_LAUNCH(k_reset_status, dim3(1), dim3(64), st, t->dstatus, (uint32_t)n, 0u);
    TN_LAUNCH((k_probe<true>), dim3(blocks), dim3(256), st, s, signs, n, (const DevStatus*)nullptr, 0u, rows, newlist, t->dstatus, (uint32_t)DEV_ERR_TABLE_FULL, make_optdev(t), t->seed);
    TN_LAUNCH(k_finish_insert, dim3(1), dim3(64), st, s, t->dstatus);
    TN_LAUNCH(k_load_rows, dim3(blocks), dim3(256), st, s, make_optdev(t), rows, n, w, state);
    TN_HIP(hipGetLastError());
    TN_HIP(hipMemcpyAsync(&t->hpull->st, t->dstatus, sizeof(DevStatus), hipMemcpyDeviceToHost, st));
    t->pull_pending = true;
    t->pull_slots = 0;
    t->pending_rows.clear();
    return sync_table(t, st);
}

int tn_sparse_table_export_rows(uint32_t handle, const uint64_t* signs, int64_t n, float* w, float* state,
                                uint8_t* found, void* stream) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_export_rows: bad table handle " + std::to_string(handle));
    if (n < 0 || (n > 0 && !signs)) return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_export_rows: NULL buffer");
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    TN_TRY(ensure_allocated(t, st));
    set_last_stream(t, st);
    if (n == 0) return TN_OK;
    if (n > 0x7FFFFFF0LL) return fail(TN_ERR_UNSUPPORTED, "tn_sparse_table_export_rows: more than 2^31 rows per call");
    if (t->push_pending || t->pull_pending) {
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    TN_TRY(t->ws.ensure(align_up((size_t)n * sizeof(uint32_t), 256)));
    uint32_t* rows = (uint32_t*)t->ws.p;
    const Store& s = t->store;
    const int blocks = launch_grid(n, 256, GRID_CAP * 4);
    TN_LAUNCH((k_probe<false>), dim3(blocks), dim3(256), st, s, signs, n, (const DevStatus*)nullptr, 0u, rows, (uint32_t*)nullptr, t->dstatus, 0u, make_optdev(t), t->seed);
    TN_LAUNCH(k_export_rows, dim3(blocks), dim3(256), st, s, make_optdev(t), rows, n, w, state, found);
    TN_HIP(hipGetLastError());
    TN_HIP(hipStreamSynchronize(st));
    return TN_OK;
}

namespace {
DecayConf make_decayconf(const SparseTable* t) {
    const OptConf& c = *t->opt;
    DecayConf d{};
    d.kind = c.kind;
    d.rate = c.show_decay_rate;
    d.show_threshold = c.show_threshold;
    d.no_show_days = c.no_show_days;
    d.elimination_logic = c.elimination_logic;
    return d;
}
}  // namespace

int tn_sparse_table_export_range(uint32_t handle, uint64_t first_slot, uint64_t n_slots, int skip_eliminated,
                                 uint64_t* signs, float* w, float* state, uint64_t* count, void* stream) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_export_range: bad table handle " + std::to_string(handle));
    if (!count || (n_slots > 0 && (!signs || !w || !state)))
        return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_export_range: NULL buffer");
    if (n_slots > 0x7FFFFFF0ull) return fail(TN_ERR_UNSUPPORTED, "tn_sparse_table_export_range: more than 2^31 slots per call");
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    TN_TRY(ensure_allocated(t, st));
    if (t->push_pending || t->pull_pending) {
        if (other_stream(t, st)) TN_HIP(hipStreamSynchronize(t->last_stream));
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    set_last_stream(t, st);
    *count = 0;
    const Store& s = t->store;
    if (n_slots == 0 || first_slot > s.cap) return TN_OK;
    TN_LAUNCH(k_reset_status, dim3(1), dim3(64), st, t->dstatus, 0u, 0u);
    TN_LAUNCH(k_export_range, dim3(launch_grid((int64_t)n_slots, 256, GRID_CAP * 4)), dim3(256), st, s, make_decayconf(t),
              first_slot, n_slots, skip_eliminated, signs, w, state, &t->dstatus->n_new);
    TN_HIP(hipGetLastError());
    TN_HIP(hipMemcpyAsync(&t->hpull->st, t->dstatus, sizeof(DevStatus), hipMemcpyDeviceToHost, st));
    TN_HIP(hipStreamSynchronize(st));
    *count = t->hpull->st.n_new;
    return TN_OK;
}

int tn_sparse_table_name(uint32_t handle, char* name, int cap) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_name: bad table handle " + std::to_string(handle));
    if (!name || cap <= 0) return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_name: NULL buffer");
    std::snprintf(name, (size_t)cap, "%s", t->name.c_str());
    return TN_OK;
}

int tn_sparse_table_optimizer(uint32_t handle, int* kind, int* use_cvm) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_optimizer: bad table handle " + std::to_string(handle));
    if (kind) *kind = t->opt->kind;
    if (use_cvm) *use_cvm = t->use_cvm ? 1 : 0;
    return TN_OK;
}

int tn_sparse_table_show_decay(uint32_t handle, int delta_days, void* stream) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_show_decay: bad table handle " + std::to_string(handle));
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    TN_TRY(ensure_allocated(t, st));
    if (t->push_pending || t->pull_pending) {
        if (other_stream(t, st)) TN_HIP(hipStreamSynchronize(t->last_stream));
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    set_last_stream(t, st);
    if (t->opt->kind == OPT_ADAM) return TN_OK;  // adam_kernel.h:67
    const Store& s = t->store;
    TN_LAUNCH(k_show_decay, dim3(launch_grid((int64_t)s.cap + 1, 256, GRID_CAP * 8)), dim3(256), st, s, make_decayconf(t),
              delta_days);
    TN_HIP(hipEventRecord(t->tail_ev, st));  // (still running when this call returns)
    t->tail_recorded = true;
    t->tail_owed = false;
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int tn_sparse_table_delete_by_show(uint32_t handle, const uint64_t* signs, int64_t n, uint8_t* out, void* stream) {
    SparseTable* t = get_table(handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "tn_sparse_table_delete_by_show: bad table handle " + std::to_string(handle));
    if (n < 0 || (n > 0 && (!signs || !out))) return fail(TN_ERR_INVALID_ARGUMENT, "tn_sparse_table_delete_by_show: NULL buffer");
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    TN_TRY(ensure_allocated(t, st));
    set_last_stream(t, st);
    if (n == 0) return TN_OK;
    if (n > 0x7FFFFFF0LL) return fail(TN_ERR_UNSUPPORTED, "tn_sparse_table_delete_by_show: more than 2^31 rows per call");
    if (t->push_pending || t->pull_pending) {
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    TN_TRY(t->ws.ensure(align_up((size_t)n * sizeof(uint32_t), 256)));
    uint32_t* rows = (uint32_t*)t->ws.p;
    const Store& s = t->store;
    const int blocks = launch_grid(n, 256, GRID_CAP * 4);
    TN_LAUNCH((k_probe<false>), dim3(blocks), dim3(256), st, s, signs, n, (const DevStatus*)nullptr, 0u, rows,
              (uint32_t*)nullptr, t->dstatus, 0u, make_optdev(t), t->seed);
    TN_LAUNCH(k_delete_by_show, dim3(blocks), dim3(256), st, s, make_decayconf(t), rows, n, out);
    TN_HIP(hipGetLastError());
    TN_HIP(hipStreamSynchronize(st));
    return TN_OK;
}

// --------------------------------------------------------------- op level
int tn_sparse_table_pull_op(uint32_t table_handle, int N, const int64_t* const* values, const int64_t* value_lens,
                            float* const* vars, const int64_t* var_rows, int var_dim, int64_t* const* mapped_values,
                            void* stream) {
    SparseTable* t = get_table(table_handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "SparseTablePull: bad table handle " + std::to_string(table_handle));
    if (!vars || !var_rows || !mapped_values) return fail(TN_ERR_INVALID_ARGUMENT, "SparseTablePull: NULL argument");
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    // (detached updates of the push before: the analysis of this call's batch runs beside them; the stream is
    // ordered behind them where the call first touches what they read or write)
    TN_TRY(ensure_allocated(t, st, true));
    const int wdim = t->dim + (t->use_cvm ? 2 : 0);
    if (var_dim != wdim)
        return fail(TN_ERR_DIM_MISMATCH, "SparseTablePull: variable dim " + std::to_string(var_dim) +
                                             " but table rows hold " + std::to_string(wdim));
    // An earlier push on the same stream need not be waited for: this call runs behind it and
    // collects its status when it waits for its own work.
    const bool same_stream = !other_stream(t, st);
    if (!same_stream || t->async_pull) TN_TRY(order_after_updates(t, st));
    if (t->pull_pending || (t->push_pending && (t->async_pull || !same_stream))) {
        if (!same_stream) TN_HIP(hipStreamSynchronize(t->last_stream));
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    set_last_stream(t, st);
    // The remap through LDS needs the call's status on the host to fall back if a
    // bucket overflowed, so it is only used when the pull waits for its stream anyway.
    bool use_lds = !t->async_pull;
    SmallShape shape{};
    if (values && value_lens && small_batch_shape(t, N, value_lens, shape)) {
        for (int s = 0; s < N; s++)
            if (var_rows[s] < 0 || !vars[s] || (value_lens[s] > 0 && (!values[s] || !mapped_values[s])))
                return fail(TN_ERR_INVALID_ARGUMENT, "SparseTablePull: bad tensors of slot " + std::to_string(s));
        TN_TRY(ensure_room(t, (uint64_t)shape.L, st));
        return small_pull(t, shape, values, value_lens, vars, var_rows, wdim, mapped_values, st);
    }
    for (int attempt = 0; attempt < 3; attempt++) {
        const double est_used = std::min(t->distinct_est, t->tile_est);  // what this attempt's buckets are sized from
        std::vector<SlotDesc> descs;
        std::vector<uint32_t> lbase;
        size_t L = 0, dt_entries = 0;
        uint32_t span_cap = 0;
        TN_TRY(stage_slots(t, N, values, value_lens, descs, lbase, L, dt_entries, "SparseTablePull", &use_lds,
                           &span_cap));
        bool vec = (wdim % 4 == 0) && (t->store.wstride % 4 == 0);
        for (int s = 0; s < N; s++) {
            if (var_rows[s] < 0 || !vars[s] || (value_lens[s] > 0 && !mapped_values[s]))
                return fail(TN_ERR_INVALID_ARGUMENT,
                            "sparse pull variable must Matrix(sign_id_cnt, dim), slot " + std::to_string(s));
            descs[s].var = vars[s];
            descs[s].rows = var_rows[s];
            descs[s].mapped = mapped_values[s];
            vec = vec && aligned16(vars[s]);
        }
        if (L == 0) {
            t->last_counts.assign(N, 0);
            return take_latched(t);
        }
        TN_TRY(ensure_room(t, (uint64_t)L, st));
        Plan p{};
        Scratch w{};
        const bool exact = t->exact_verify && use_lds;
        // (a plan buffer that has to grow is freed first: not under detached updates that still read it)
        if (t->upd_pending && carve_plan(nullptr, p, N, L, exact) > t->plan_buf.bytes)
            TN_HIP(hipEventSynchronize(t->upd_ev));
        TN_TRY(t->plan_buf.ensure(carve_plan(nullptr, p, N, L, exact)));
        carve_plan((char*)t->plan_buf.p, p, N, L, exact);
        TN_TRY(t->ws.ensure(carve_scratch(nullptr, w, L, dt_entries, use_lds, t->distinct_est, N)));
        carve_scratch((char*)t->ws.p, w, L, dt_entries, use_lds, t->distinct_est, N);
        w.span_cap = span_cap;
        t->plan_valid = false;
        // Detached updates of the push before read its plan in this same buffer.  A batch of the same slot count
        // and about the same size lays its plan out over it array by array, and what this call writes before it
        // orders itself behind them (the per-lookup arrays) stays clear of what they read; any other batch waits.
        // So does a call that keeps a copy of its signs for the exact comparison: the copy lies behind the group
        // arrays, where a batch of another size puts it on top of the gradient addresses the updates still read,
        // and the call's first kernel writes it.
        if (t->upd_pending && (exact || N != t->upd_N ||
                               (size_t)((const char*)p.grp_sign - (const char*)t->plan_buf.p) >
                                   t->upd_groups_off + t->upd_slack))
            TN_TRY(order_after_updates(t, st));
        t->plan_small = false;
        t->plan_big_k = big_threshold(t->store);
        t->plan_big_desc = false;
        TN_TRY(upload_slots(t, p.descs, p.lbase, t->dplan, descs, lbase, st, !t->async_pull, STATUS_NEW_PLAN,
                            use_lds ? w.bcursor : nullptr, use_lds ? w.nbuckets + 1 + w.nb2 : 0));

        const Store& s = t->store;
        DevStatus* ds = t->dplan;
        TN_TRY(launch_build_plan(t, p, w, N, (uint32_t)L, true, use_lds, st));
        // The grouping through LDS leaves the row of every distinct record in where_u itself, and the
        // call's status (counts, new rows, errors) is final before the gather starts: it is published
        // by the gather's first workgroup, and the call returns when the host has it, through a word in pinned memory: the
        // host prepares the push while the gather runs.  The
        // variables are complete in stream order, as the outputs of any call that takes a stream.  (No sooner: the mapped ids,
        // which are there when the call returns, and the plan's counts of groups are k_emit_mapped's.  Published beside that
        // one, 2.1 M lookups of 64 slots took 172.3 us a step instead of 174.2, a pooled step of 211 slots 287 instead of 294.)
        const bool final_early = use_lds && N <= GRP_SLOTS && !t->async_pull;
        const uint32_t seq = final_early ? ++t->seq_pull : 0;
        const uint32_t* rows_of_groups = (use_lds && N <= GRP_SLOTS) ? nullptr : p.grp_row;
        Publish pub{};
        if (final_early) pub = {reinterpret_cast<uint32_t*>(t->hpull), s.count, t->hseq + 0, seq};
        hipEvent_t tail = final_early ? tail_event(t, st) : nullptr;
        if (vec)
            TN_LAUNCH_EVENT(tail, (k_gather_vars<4>), dim3(1 + launch_grid((int64_t)L * (wdim / 4), 256, GRID_CAP * 4)), dim3(256),
                            st, s, ds, rows_of_groups, p.where_u, p.ubase, N, p.descs, pub);
        else
            TN_LAUNCH_EVENT(tail, (k_gather_vars<1>), dim3(1 + launch_grid((int64_t)L * wdim, 256, GRID_CAP * 4)), dim3(256), st,
                            s, ds, rows_of_groups, p.where_u, p.ubase, N, p.descs, pub);
        TN_HIP(hipGetLastError());
        if (!final_early)
            TN_LAUNCH(k_publish, dim3(1), dim3(256), st, ds, p.ubase, (uint32_t)(N + 1), reinterpret_cast<uint32_t*>(t->hpull),
                      s.count);
        t->pull_pending = true;
        t->pull_slots = N;
        t->pull_lookups = (uint64_t)L;
        t->pending_rows.assign(var_rows, var_rows + N);
        // a push of the same batch may reuse the analysis
        t->plan_valid = true;
        t->plan_clicks_dirty = false;  // a new plan's click sums start at zero
        t->plan_has_show = use_lds;
        t->plan_prints = use_lds;
        t->plan_exact = exact;
        t->plan_N = N;
        t->plan_lens.assign(value_lens, value_lens + N);
        t->plan_epoch = t->epoch;
        if (t->async_pull) return TN_OK;
        do_host_work();
        if (final_early)
            TN_TRY(wait_reported(t->hseq + 0, seq, st, "SparseTablePull"));
        else
            TN_HIP(hipStreamSynchronize(st));
        t->stage_pending = false;
        if (use_lds && (t->hpull->st.err & DEV_ERR_REMAP_OVERFLOW)) {
            // rows the failed attempt inserted belong to signs of this batch; keep them counted
            t->hpull->st.err &= ~DEV_ERR_REMAP_OVERFLOW;
            harvest(t);
            // The batch had more distinct records than the buckets were sized for (the share of the recent pulls
            // plus a quarter).  Sized for a batch of distinct signs only, a bucket cannot overflow short of an
            // adversarial hash (first level: 768 lookups for 2048 entries; second level: 1024 records expected
            // in room for 1536), so the call is repeated through LDS once more -- at the cost of a pull, not of
            // the global-table path, which remains for the batch that overflows even then.
            if (est_used >= 1.0) use_lds = false;
            t->distinct_est = 1.0;
            t->tile_est = 1.0;
            t->latched = TN_OK;
            t->latched_msg.clear();
            continue;
        }
        if (final_early) {
            harvest(t);
            return take_latched(t);
        }
        return sync_table(t, st);
    }
    return fail(TN_ERR_HIP, "SparseTablePull: remap fell back three times");
}

}  // extern "C"

namespace {

// SparseTablePush.  With example_ids the gradients are pooled ([batch, dim] per slot, one row per
// example): they are first reduced to one row per distinct sign (the gradient of the combiner).
int push_op_impl(uint32_t table_handle, int N, const int64_t* const* values, const int64_t* value_lens,
                 const float* const* grads, const int64_t* grad_rows, int grad_dim,
                 const int64_t* const* feature_labels, const int64_t* const* example_ids, int64_t batch, int combiner,
                 void* stream) {
    SparseTable* t = get_table(table_handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "SparseTablePush: bad table handle " + std::to_string(table_handle));
    if (!grads || (!grad_rows && !example_ids) || !feature_labels)
        return fail(TN_ERR_INVALID_ARGUMENT, "SparseTablePush: NULL argument");
    const bool pooled = example_ids != nullptr;
    if (pooled && (batch <= 0 || combiner < COMBINE_SUM || combiner > COMBINE_SQRTN))
        return fail(TN_ERR_INVALID_ARGUMENT, "SparseTablePush (pooled): bad batch size or combiner");
    // an item of the reduction has 32 bits for its example: lookups of examples beyond are refused as those beyond the batch are
    if (pooled) batch = std::min(batch, (int64_t)1 << 32);
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    TN_TRY(ensure_allocated(t, st));
    const int wdim = t->dim + (t->use_cvm ? 2 : 0);
    if (grad_dim != wdim)
        return fail(TN_ERR_DIM_MISMATCH, "SparseTablePush: gradient dim " + std::to_string(grad_dim) +
                                             " but table rows hold " + std::to_string(wdim));
    std::vector<SlotDesc> descs;
    std::vector<uint32_t> lbase;
    size_t L = 0, dt_entries = 0;
    TN_TRY(stage_slots(t, N, values, value_lens, descs, lbase, L, dt_entries, "SparseTablePush", nullptr));
    bool vec = (grad_dim % 4 == 0);
    for (int s = 0; s < N; s++) {
        const int64_t rows = pooled ? batch : grad_rows[s];
        if (rows < 0 || (rows > 0 && !grads[s]) || (value_lens[s] > 0 && !feature_labels[s]) ||
            (pooled && value_lens[s] > 0 && !example_ids[s]))
            return fail(TN_ERR_INVALID_ARGUMENT,
                        "sparse push grad must Matrix(sign_id_cnt, dim), slot " + std::to_string(s));
        descs[s].grads = grads[s];
        descs[s].rows = rows;
        descs[s].labels = feature_labels[s];
        if (pooled) descs[s].mapped = const_cast<int64_t*>(example_ids[s]);  // example index of every lookup
        vec = vec && aligned16(grads[s]);
    }
    if (t->push_pending || t->pull_pending) {
        // a call pending on another stream (an asynchronous pull) builds the plan this push reads
        if (other_stream(t, st)) TN_HIP(hipStreamSynchronize(t->last_stream));
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    set_last_stream(t, st);
    if (L == 0) return TN_OK;
    t->pooled_pushes = pooled;
    Plan p{};
    Scratch w{};
    // Same batch as the last pull?  Necessary conditions on the host, the signs
    // themselves are compared on the device.
    bool reuse = t->plan_valid && t->plan_epoch == t->epoch && t->plan_N == N &&
                 std::equal(value_lens, value_lens + N, t->plan_lens.begin());
    // A push on the last pull's plan has its own descriptors and status block (the plan's counts, flags of its
    // own): the pull's gather may still be running, and the next pull may stage its slots while this push's
    // updates run.  A push that analyses its batch itself uses the plan's.
    DevStatus* ds = reuse ? t->dpush : t->dplan;
    const SlotDesc* pd = nullptr;  // set with the plan
    const int lblocks = launch_grid(L, 256, GRID_CAP * 2);
    const bool with_click = t->opt->kind == OPT_ADAGRAD;  // the only optimizer that reads batch_click
    // show / click counts of the batch into the member lists of a plan that has none
    auto launch_counts = [&]() -> int {
        TN_LAUNCH(k_reset_counts, dim3(lblocks), dim3(256), st, p.list, ds, (uint32_t)L, 0);
        TN_LAUNCH(k_count_show, dim3(launch_grid((int64_t)(L + COUNT_TILE - 1) / COUNT_TILE, 1, GRID_CAP)), dim3(256),
                  st, pd, p.lbase, N, (uint32_t)L, p.u_of_gi, p.where_u, p.list, with_click ? 1 : 0);
        return TN_OK;
    };
    // Where the apply kernels find the gradient of a record.  Pooled gradients are first reduced
    // to one row per distinct sign.
    PushSrc src{};
    uint32_t compared_seq = 0;    // with a plan of the last pull's: what the host waits for in hseq[1]
    auto prepare_src = [&]() -> int {
        src = op_source(p, grad_dim, pd == p.push_descs);
        const HostWord compared{reuse ? t->hseq + 1 : nullptr, compared_seq};
        uint32_t* host_err = reuse ? &t->hpush->st.err : nullptr;
        if (!pooled) {
            src.compared = compared;
            src.host_err = host_err;
            return TN_OK;
        }
        size_t max_len = 0;
        for (int s = 0; s < N; s++) max_len = std::max<size_t>(max_len, (size_t)value_lens[s]);
        const PoolShare share((uint32_t)max_len, !reuse || !t->plan_has_show || t->plan_heavy);
        const uint32_t tiles = PoolShare::first_tile((uint32_t)N, (uint32_t)L);
        const uint32_t blocks = (PoolShare::first_part((uint32_t)N, (uint32_t)L) + XCDS - 1) / XCDS * XCDS;
        Carver c{nullptr};
        uint2* pool;
        uint16_t* poff;
        float *flat, *shares;
        uint64_t* has;
        uint32_t* extra;
        const bool spread = share.spreads((uint32_t)max_len);
        auto carve = [&](Carver& cv) {
            pool = cv.take<uint2>(L);
            poff = cv.take<uint16_t>((size_t)tiles * (share.parts_max + 1));
            flat = cv.take<float>(L * (size_t)grad_dim);
            shares = cv.take<float>(spread ? (size_t)blocks * POOL_SHARES * grad_dim : 0);
            has = cv.take<uint64_t>(spread ? (size_t)blocks * (POOL_SHARES / 64) : 0);
            extra = cv.take<uint32_t>(spread ? (size_t)N * (POOL_EXTRA + 1) : 0);
        };
        carve(c);
        TN_TRY(t->pooled_ws.ensure(align_up(c.off, 256)));
        Carver c2{(char*)t->pooled_ws.p};
        carve(c2);
        if (spread) TN_LAUNCH(k_pool_frequent, dim3((uint32_t)N), dim3(POOL_THREADS), st, p.lbase, p.ubase, p.u_of_gi, share, extra);
        TN_LAUNCH_LDS(k_lookup_keys, dim3(tiles), dim3(256), pool_tile_lds(share.parts_max), st, pd, p.lbase, p.ubase, (uint32_t)N,
                      p.u_of_gi, batch, pool, poff, share, extra, ds, compared, host_err);
#define TN_REDUCE(LPG, ANY)                                                                                                \
    TN_LAUNCH((k_reduce_pooled<LPG, ANY>), dim3(blocks), dim3(POOL_THREADS), st, pd, p.lbase, p.ubase, (uint32_t)N, pool,  \
              poff, grad_dim, t->store.D, combiner, ds, flat, share, extra, shares, has)
        TN_POOL_LANES(TN_REDUCE, t->store.D, vec);
#undef TN_REDUCE
        if (spread) {
#define TN_REDUCE(LPG, ANY)                                                                                                \
    TN_LAUNCH((k_reduce_pooled_shares<LPG, ANY>), dim3((uint32_t)N * (POOL_SPREAD / 4)), dim3(256), st, p.lbase, p.ubase,  \
              grad_dim, t->store.D, ds, shares, has, flat, share, extra)
            TN_POOL_LANES(TN_REDUCE, t->store.D, grad_dim % 4 == 0);
#undef TN_REDUCE
        }
        src.flat = flat;
        return TN_OK;
    };
    if (reuse && t->plan_small) {
        bool other_batch = false;
        TN_TRY(small_push(t, values, grads, grad_rows, grad_dim, feature_labels, example_ids, batch, combiner, vec, st,
                          &other_batch));
        if (!other_batch) return TN_OK;
        reuse = false;  // another batch than the last pull's: analysed below
    } else if (reuse) {
        carve_plan((char*)t->plan_buf.p, p, N, L, t->plan_exact);
        pd = p.push_descs;
        TN_TRY(upload_slots(t, p.push_descs, nullptr, ds, descs, lbase, st, true, STATUS_REUSE_PLAN, nullptr, 0, p.ubase,
                            p.push_ubase, (uint32_t)(N + 1)));
        // On a plan with show counts the verify pass also sums the clicks; they start at zero
        // after the pull, a further push on the same plan clears them first.
        const bool clicks = t->plan_has_show && with_click;
        const int vblocks = launch_grid((int64_t)(L + VERIFY_TILE - 1) / VERIFY_TILE, 1, GRID_CAP * 2);
        const size_t vlds = ((size_t)N + 1) * sizeof(uint32_t);
        // the outcome comes back through pinned host memory, written by the verify kernel itself; that it has come, by a
        // word from the kernels behind it
        compared_seq = ++t->seq_verify;
        const bool detach = t->detach_updates && !pooled && L >= DETACH_LOOKUPS;
        hipEvent_t behind = detach && t->plan_has_show ? t->fork_ev : nullptr;
        t->hpush->st.mismatch = 0;
        t->hpush->st.err = 0;
        uint32_t* host_mismatch = &t->hpush->st.mismatch;
        // op-level gradients (not pooled): the verify pass also works out the gradient addresses of the records
        // of the groups with several records (see k_member_grads)
        const PushSrc vsrc = op_source(p, grad_dim, true);
        const bool addr_in_verify = !pooled && t->plan_big_k != 0xFFFFFFFFu;
        const float** vgaddr = addr_in_verify ? p.gaddr : nullptr;
#define TN_VERIFY_BY(CLICKS, COPY, THREADS)                                                                         \
    do {                                                                                                            \
        if (g_profile_on) prof_begin("k_verify_values<" #CLICKS ", " #COPY ">", st);                                \
        launch_signalling(behind, k_verify_values<CLICKS, COPY, THREADS>, dim3(vblocks), dim3(THREADS), vlds, st, pd, p.lbase, N, \
                          (uint32_t)L, then_vals, ds, p.u_of_gi, p.where_u, p.list, host_mismatch, vsrc, vgaddr);    \
        if (g_profile_on) prof_end(st);                                                                             \
    } while (0)
#define TN_VERIFY(CLICKS, COPY)                                      \
    do {                                                             \
        if (few)                                                     \
            TN_VERIFY_BY(CLICKS, COPY, VERIFY_THREADS_FEW);          \
        else                                                         \
            TN_VERIFY_BY(CLICKS, COPY, VERIFY_THREADS);              \
    } while (0)
        const bool few = (L + VERIFY_TILE - 1) / VERIFY_TILE <= (size_t)VERIFY_FEW_TILES;
        const bool copy = !t->plan_prints || t->plan_exact;
        const uint64_t* then_vals = t->plan_exact ? p.vals_exact : p.vals_copy;
        if (clicks) {
            if (t->plan_clicks_dirty)
                TN_LAUNCH(k_reset_counts, dim3(lblocks), dim3(256), st, p.list, ds, (uint32_t)L, 1);
            t->plan_clicks_dirty = true;
            if (copy)
                TN_VERIFY(true, true);
            else
                TN_VERIFY(true, false);
        } else if (copy) {
            TN_VERIFY(false, true);
        } else {
            TN_VERIFY(false, false);
        }
#undef TN_VERIFY_BY
#undef TN_VERIFY
        // Counts and apply kernels are queued before the host knows the outcome: the counts only
        // touch the plan's member lists, which a mismatch discards anyway, and the apply kernels
        // return at once when the mismatch flag is set.  The device never waits for the host.
        if (!t->plan_has_show) TN_TRY(launch_counts());
        TN_TRY(prepare_src());
        TN_TRY(launch_apply(t, p, src, ds, (int64_t)L, vec, st, addr_in_verify, t->plan_big_k, detach, t->plan_big_desc, behind));
        // their end, for whoever touches the table next; the status goes out behind them (below)
        if (t->detached_now) TN_HIP(hipStreamWaitEvent(t->side, t->apply_ev, 0));
        TN_TRY(wait_reported(t->hseq + 1, compared_seq, t->detached_now ? t->side : st, "SparseTablePush"));
        t->stage_pending = false;
        reuse = t->hpush->st.mismatch == 0;
        if (t->detached_now && !reuse) {
            // (the update kernels return at once on a mismatch; what follows works on the caller's stream)
            TN_HIP(hipEventRecord(t->upd_ev, t->side));
            t->upd_pending = true;
            t->detached_now = false;
            TN_TRY(order_after_updates(t, st));
        }
    }
    if (!reuse) {
        // another batch than the last pull's: analyse it here, on the global-table path
        // (its status cannot be waited for, a push only enqueues)
        t->plan_valid = false;
        ds = t->dplan;
        TN_TRY(t->plan_buf.ensure(carve_plan(nullptr, p, N, L)));
        carve_plan((char*)t->plan_buf.p, p, N, L);
        pd = p.descs;
        TN_TRY(t->ws.ensure(carve_scratch(nullptr, w, L, dt_entries, false)));
        carve_scratch((char*)t->ws.p, w, L, dt_entries, false);
        TN_TRY(upload_slots(t, p.descs, p.lbase, ds, descs, lbase, st, false, STATUS_NEW_PLAN));
        TN_TRY(launch_build_plan(t, p, w, N, (uint32_t)L, false, false, st));
        TN_TRY(launch_counts());
        TN_TRY(prepare_src());
        TN_TRY(launch_apply(t, p, src, ds, (int64_t)L, vec, st));
    }
    TN_HIP(hipGetLastError());
    const bool detached = reuse && t->detached_now;  // (the side stream is behind all update kernels already)
    t->detached_now = false;
    if (reuse)
        t->last_counts = t->plan_counts;  // (its errors reach the host by themselves)
    else
        TN_LAUNCH(k_publish, dim3(1), dim3(256), st, ds, p.ubase, (uint32_t)(N + 1), reinterpret_cast<uint32_t*>(t->hpush),
                  (unsigned long long*)nullptr);
    if (detached) {
        TN_HIP(hipEventRecord(t->upd_ev, t->side));
        t->upd_pending = true;
        t->upd_N = N;
        t->upd_groups_off = (size_t)((const char*)p.grp_sign - (const char*)t->plan_buf.p);
        t->upd_slack = (size_t)((const char*)p.grp_row - (const char*)p.grp_sign);
    }
    t->push_pending = true;
    t->push_on_side = detached;
    t->push_slots = reuse ? 0 : N;
    return TN_OK;
}

}  // namespace

extern "C" {

int tn_sparse_table_push_op(uint32_t table_handle, int N, const int64_t* const* values, const int64_t* value_lens,
                            const float* const* grads, const int64_t* grad_rows, int grad_dim,
                            const int64_t* const* feature_labels, void* stream) {
    return push_op_impl(table_handle, N, values, value_lens, grads, grad_rows, grad_dim, feature_labels, nullptr, 0, 0,
                        stream);
}

int tn_sparse_table_push_pooled_op(uint32_t table_handle, int N, const int64_t* const* values,
                                   const int64_t* value_lens, const int64_t* const* example_ids,
                                   const float* const* pooled_grads, int64_t batch, int grad_dim, int combiner,
                                   const int64_t* const* feature_labels, void* stream) {
    if (!example_ids) return fail(TN_ERR_INVALID_ARGUMENT, "SparseTablePush (pooled): NULL argument");
    return push_op_impl(table_handle, N, values, value_lens, pooled_grads, nullptr, grad_dim, feature_labels, example_ids,
                        batch, combiner, stream);
}

int tn_sparse_table_combine_op(uint32_t table_handle, int N, const int64_t* const* mapped_values,
                               const int64_t* value_lens, const int64_t* const* example_ids, const float* const* vars,
                               const int64_t* var_rows, int dim, int64_t batch, int combiner, float* const* out,
                               void* stream) {
    SparseTable* t = get_table(table_handle);
    if (!t) return fail(TN_ERR_BAD_HANDLE, "embedding combine: bad table handle " + std::to_string(table_handle));
    if (!mapped_values || !value_lens || !example_ids || !vars || !var_rows || !out || N <= 0)
        return fail(TN_ERR_INVALID_ARGUMENT, "embedding combine: NULL argument");
    if (N > MAX_SLOTS) return fail(TN_ERR_UNSUPPORTED, "embedding combine: too many slots");
    if (dim <= 0 || batch <= 0 || combiner < COMBINE_SUM || combiner > COMBINE_SQRTN)
        return fail(TN_ERR_INVALID_ARGUMENT, "embedding combine: bad dim, batch size or combiner");
    std::lock_guard<std::mutex> lk(t->mu);
    hipStream_t st = (hipStream_t)stream;
    TN_TRY(ensure_allocated(t, st));
    std::vector<SlotDesc> descs(N, SlotDesc{});
    size_t L = 0;
    int64_t max_len = 0;
    bool vec = dim % 4 == 0;
    for (int s = 0; s < N; s++) {
        if (value_lens[s] < 0 || var_rows[s] < 0 || !out[s] ||
            (value_lens[s] > 0 && (!mapped_values[s] || !example_ids[s] || !vars[s])))
            return fail(TN_ERR_INVALID_ARGUMENT, "embedding combine: bad tensors of slot " + std::to_string(s));
        SlotDesc& d = descs[s];
        d.values = mapped_values[s];
        d.mapped = const_cast<int64_t*>(example_ids[s]);
        d.grads = vars[s];
        d.var = out[s];
        d.rows = var_rows[s];
        d.len = (uint32_t)value_lens[s];
        L += (size_t)value_lens[s];
        max_len = std::max<int64_t>(max_len, value_lens[s]);
        if (L > 0x7FFFFFF0ull) return fail(TN_ERR_UNSUPPORTED, "embedding combine: more than 2^31 lookups in one call");
        vec = vec && aligned16(vars[s]) && aligned16(out[s]);
    }
    // an earlier call's status is collected first
    if (t->push_pending || t->pull_pending) {
        if (other_stream(t, st)) TN_HIP(hipStreamSynchronize(t->last_stream));
        TN_HIP(hipStreamSynchronize(st));
        harvest(t);
    }
    set_last_stream(t, st);
    // A workgroup per COMBINE_EXAMPLES examples of a slot where the chip holds them all at once, else per more of them, as long
    // as their lookups' rows fit in LDS: every workgroup pays for finding its lookups.  (211 slots of 2039 examples, 256 a
    // workgroup 21 us, 128 25, 64 32; 100 slots of 16384: 1024, which do not fit 167, 512 100, 256 108, 128 127.)
    uint32_t per = COMBINE_EXAMPLES;
    while (per < 512 && (int64_t)N * ((batch + per - 1) / per) > GRID_CAP &&
           (double)max_len * (2 * per) <= 0.8 * COMBINE_IDS * (double)batch)
        per *= 2;
    const uint32_t per_slot = (uint32_t)((batch + per - 1) / per);
    const int64_t items = (int64_t)N * per_slot;
    if (items > 0x7FFFFFF0LL) return fail(TN_ERR_UNSUPPORTED, "embedding combine: too many examples");
    const int grid = launch_grid(items, 1, GRID_CAP * 4);
    ArgDescs args;
    const SlotDesc* ddescs = nullptr;
    const NoDescs none;
    const bool by_value = N <= ARG_SLOTS;
    if (by_value) {
        std::copy(descs.begin(), descs.end(), args.slot);
    } else {
        TN_TRY(staging_free(t));
        std::memcpy(t->hstage, descs.data(), (size_t)N * sizeof(SlotDesc));
        ddescs = reinterpret_cast<const SlotDesc*>(t->hstage);
    }
    if (!by_value && grid > COMBINE_DIRECT) {  // (few workgroups read their slot's descriptor from the host's buffer themselves: a launch less)
        const size_t db = (size_t)N * sizeof(SlotDesc);
        TN_TRY(t->comb_buf.ensure(align_up(db, 256)));
        TN_LAUNCH(k_stage_in, dim3(launch_grid((int64_t)db / 4, 256, 64)), dim3(256), st,
                  reinterpret_cast<const uint32_t*>(t->hstage), reinterpret_cast<uint32_t*>(t->comb_buf.p), (uint32_t)(db / 4),
                  (uint32_t*)nullptr, 0u, (DevStatus*)nullptr, (int)STATUS_KEEP, (uint32_t*)nullptr, 0u,
                  (const DevStatus*)nullptr, (const uint32_t*)nullptr, (uint32_t*)nullptr, 0u);
        ddescs = (const SlotDesc*)t->comb_buf.p;
    }
    int lanes = 1;
    while (lanes < 32 && 4 * lanes < dim) lanes *= 2;
    const bool any = !vec || dim % (4 * lanes) != 0;
#define TN_LAUNCH_COMBINE_BY(LPG, ANY, BY)                                                                                \
    do {                                                                                                                  \
        if (g_profile_on) prof_begin("k_combine_fwd<" #LPG ", " #ANY ">", st);                                            \
        hipLaunchKernelGGL((k_combine_fwd<LPG, ANY, std::decay_t<decltype(BY)>>), dim3(grid), dim3(256), (size_t)per * 8, \
                           st, BY, ddescs, (uint32_t)items, per_slot, per, dim, batch, combiner, t->dcomb);                       \
        if (g_profile_on) prof_end(st);                                                                                   \
    } while (0)
#define TN_LAUNCH_COMBINE_ANY(LPG, ANY)                \
    do {                                               \
        if (by_value)                                  \
            TN_LAUNCH_COMBINE_BY(LPG, ANY, args);      \
        else                                           \
            TN_LAUNCH_COMBINE_BY(LPG, ANY, none);      \
    } while (0)
#define TN_LAUNCH_COMBINE(LPG)                  \
    do {                                        \
        if (any)                                \
            TN_LAUNCH_COMBINE_ANY(LPG, true);   \
        else                                    \
            TN_LAUNCH_COMBINE_ANY(LPG, false);  \
    } while (0)
    switch (lanes) {
        case 1: TN_LAUNCH_COMBINE(1); break;
        case 2: TN_LAUNCH_COMBINE(2); break;
        case 4: TN_LAUNCH_COMBINE(4); break;
        case 8: TN_LAUNCH_COMBINE(8); break;
        case 16: TN_LAUNCH_COMBINE(16); break;
        default: TN_LAUNCH_COMBINE(32); break;
    }
#undef TN_LAUNCH_COMBINE
#undef TN_LAUNCH_COMBINE_ANY
#undef TN_LAUNCH_COMBINE_BY
    const uint32_t seq = ++t->seq_comb;
    TN_LAUNCH(k_report, dim3(1), dim3(64), st, t->dcomb, t->hcomb, seq);
    TN_HIP(hipGetLastError());
    TN_TRY(wait_words(t->hcomb, 1, seq, st, "embedding combine"));
    const uint32_t err = (uint32_t)*t->hcomb;
    if (err & DEV_ERR_VAR_CAPACITY) return fail(TN_ERR_VAR_CAPACITY, "embedding combine: a mapped id is not a row of its variable");
    if (err & DEV_ERR_GRAD_ROWS)
        return fail(TN_ERR_INVALID_ARGUMENT, "embedding combine: example ids must be non-decreasing and in [0, batch)");
    return TN_OK;
}

void tn_while_waiting(void (*fn)(void*), void* arg) {
    waiting_fn = fn;
    waiting_arg = arg;
}

}  // extern "C"
