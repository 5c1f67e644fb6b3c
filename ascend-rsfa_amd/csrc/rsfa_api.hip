// C ABI of the gfx950 FlashAttention-2 forward library (declared in include/rsfa.h).
//
// Replaces the host half of the reference operator
// (ascend_rsfa/flash_attention_forward.py): argument checks of
// _attention.forward (551-556), the dispatch to the small / causal-split /
// persistent kernels (564-610), _run_causal_split (493-541), get_tiling
// (624-665) and get_num_compute_cores (19-21).
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <mutex>
#include <unordered_map>

#include "../../include/rsfa.h"
#include "fa_fwd_kernel.hpp"
#include "kernel_table.hpp"

namespace rsfa {

// The no-allocation entry point's buffer: queue counters in the first 4 KiB,
// then the workspace.  Host code never uses this name as an address (on the
// host it only stands for the symbol): rsfa_attention_fwd_noalloc looks the
// device address up once per device with hipGetSymbolAddress.
constexpr size_t kScratchCounterBytes = 4096;
static __device__ __align__(256) char scratch[kScratchCounterBytes + RSFA_NOALLOC_WORKSPACE_BYTES];

namespace {

constexpr int kMaxDevices = 64;
constexpr int kTicketSlots = 256;       // concurrent streams with a dynamic queue
constexpr int kQueues = 8;              // task queues per launch (one per XCD)
constexpr int kTicketStrideWords = 16;  // one 64-byte line per counter
constexpr int kSlotWords = kQueues * kTicketStrideWords;
static_assert(kSlotWords * sizeof(uint32_t) <= kScratchCounterBytes, "the counters fit the scratch head");
constexpr int kLdsPerCu = 160 * 1024;   // gfx950
constexpr int kMaxKernels = 512;        // instantiations in all kernel lists

KernelList all_lists[] = {kernels_d16(), kernels_d32(), kernels_d64(), kernels_d128(), kernels_d256()};

template <class F>
void for_each_kernel(F&& f) {
    for (const KernelList& l : all_lists)
        for (int i = 0; i < l.count; ++i) f(l.entries[i]);
}

const KernelEntry* find_kernel(int dtype, int d, int bn, int bm, int causal, int mode) {
    const KernelEntry* hit = nullptr;
    for_each_kernel([&](const KernelEntry& e) {
        if (e.dtype == dtype && e.d == d && e.bn == bn && e.bm == bm && e.causal == causal && e.mode == mode && e.kg == 1)
            hit = &e;
    });
    return hit;
}

bool valid_head_dim(int64_t d) { return d == 16 || d == 32 || d == 64 || d == 128 || d == 256; }
bool is_pow2(int64_t x) { return x > 0 && (x & (x - 1)) == 0; }

struct DeviceState {
    std::mutex mu;
    int num_cus = 0;              // 0 until queried
    uint32_t* tickets = nullptr;  // kTicketSlots counters, allocated by the first dynamic launch
    std::unordered_map<void*, int> stream_slot;
    std::atomic<int> occupancy[kMaxKernels] = {};  // by kernel_index: resident workgroups per CU, 0 = not yet queried
    void* scratch = nullptr;                        // this device's address of `scratch` (no-allocation entry point)
};

DeviceState g_dev[kMaxDevices];

int current_device(int* dev) {
    if (hipGetDevice(dev) != hipSuccess) return RSFA_E_DEVICE;
    if (*dev < 0 || *dev >= kMaxDevices) return RSFA_E_DEVICE;
    return RSFA_OK;
}

// Compute units of `dev`, queried once.  A failed query is not remembered, so
// a later call retries it.
int device_cus(DeviceState& ds, int dev, int* cus) {
    std::lock_guard<std::mutex> lock(ds.mu);
    if (ds.num_cus <= 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            return RSFA_E_DEVICE;
        ds.num_cus = n;
    }
    *cus = ds.num_cus;
    return RSFA_OK;
}

// CU count the tile search plans for: the current device's, or a whole
// MI355X (256) where no device is visible, so get_tiling answers the same as
// the launcher on a GPU and still answers without one.
int planning_cus() {
    int dev = 0, cus = 0;
    if (current_device(&dev) == RSFA_OK && device_cus(g_dev[dev], dev, &cus) == RSFA_OK) return cus;
    return 256;
}

// Whether a launch on `stream` may use a dynamic ticket counter.  The counter
// is found by the stream handle and relies on the stream running its launches
// one after another, which fails for launches recorded into a graph (replays
// of graphs captured on one stream may run concurrently on other streams) and
// for hipStreamPerThread (one handle for every thread's stream): those use the
// static schedule, which gives bitwise the same results.
bool dynamic_schedule_allowed(void* stream) {
    if ((hipStream_t)stream == hipStreamPerThread) return false;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing((hipStream_t)stream, &cs) != hipSuccess) return false;
    return cs == hipStreamCaptureStatusNone;
}

// Counter for launches on `stream`.  Launches on one stream run in order, and
// each launch leaves its counter at 0 when it ends, so a stream can reuse its
// counter; distinct streams get distinct counters.  The counters are allocated
// (and zeroed) by the first call; returns null when that fails or all counters
// are taken (the launch then uses the static schedule; a failed allocation is
// retried by the next call).
uint32_t* stream_ticket(DeviceState& ds, void* stream) {
    std::lock_guard<std::mutex> lock(ds.mu);
    if (!ds.tickets) {
        void* buf = nullptr;
        const size_t bytes = sizeof(uint32_t) * kTicketSlots * kSlotWords;
        if (hipMalloc(&buf, bytes) != hipSuccess) return nullptr;
        if (hipMemset(buf, 0, bytes) != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
            (void)hipFree(buf);
            return nullptr;
        }
        ds.tickets = (uint32_t*)buf;
    }
    auto it = ds.stream_slot.find(stream);
    int slot;
    if (it != ds.stream_slot.end()) {
        slot = it->second;
    } else {
        if ((int)ds.stream_slot.size() >= kTicketSlots) return nullptr;
        slot = (int)ds.stream_slot.size();
        ds.stream_slot.emplace(stream, slot);
    }
    return ds.tickets + (size_t)slot * kSlotWords;
}

// Task queues of a launch: one per XCD (8) when every queue gets whole heads
// in near-equal numbers, else a single queue.  The kernel's queue x holds the
// heads bh % nq == x and is served by workgroups b % nq == x.
int32_t queue_count(int64_t num_heads, int64_t grid) {
    if (grid < kQueues || num_heads < kQueues) return 1;
    if (num_heads % kQueues != 0 && num_heads < 8 * kQueues) return 1;
    return kQueues;
}

// Whether a causal fused launch hands out its query blocks in pairs (nmb-1-i,
// then i, as one ticket: every ticket the same length, nmb + 1 block-lengths
// of key tiles).  Pairs run in lockstep rounds and fetch fewer K/V bytes past
// L2, but a last round that the pairs fill only partly idles workgroups for a
// whole pair, where single blocks served longest-first end closer together.
// Makespans per queue in block-lengths, with Wq workgroups: pairs
// ceil(heads * nmb / 2 / Wq) * (nmb + 1), single blocks about their total
// work / Wq + 1/2; pairs win ties within 3 %.  Every tile takes them: at head
// dim 256, whose tasks load Q at their start, interleaved against single
// blocks: B=64 H=8 S=1024 +1.2 % (8 % fewer bytes fetched past L2), B=128
// S=2048 +2.0 %, B=16 S=2048 +4.3 %, B=8 S=4096 +5.5 %.  Only for an even
// nmb, whose pairs are all whole (B=64 H=8 S=1792 D=128: 1.5 % slower with
// the middle blocks alone).
int32_t use_pairs(int64_t num_heads, int32_t nmb, int64_t grid, int32_t nq) {
    if (nmb < 2 || (nmb & 1)) return 0;
    const int64_t wq = grid / nq;                  // workgroups per queue
    const int64_t hq = (num_heads + nq - 1) / nq;  // heads of the fullest queue
    if (wq < 1) return 0;
    const double rounds = (double)hq * nmb / 2.0 / (double)wq;
    if (rounds < 1.0) return 0;
    const double len = nmb + 1.0;
    const double paired = std::ceil(rounds - 1e-9) * len;
    const double single = rounds * len + 0.5;
    return paired <= 1.03 * single ? 1 : 0;
}

// Whether a launch hands out more tickets than the workgroups' first ones (each
// serves its rank in its queue without drawing).  Where every queue has a
// workgroup per ticket, the counters are left out: the atomic that draws a
// ticket past the end is then no part of a task (one 64-key tile on 8 heads
// 5.7 -> 5.5 us, four 197-key ones on 128 heads 10.0 -> 9.4).  Nor where equal
// tasks (`equal`: non-causal) go to three or more workgroups per CU (`wgs`) in at
// most two rounds, or in three of which the last is half full or more: drawn, the
// tasks of a last round that is not full gather on the CUs that ask first, where
// three share what one could have, while strided by rank they spread over all.
// Head dim 32, drawn and strided: B*H = 20 S=8192 (1.7 rounds) 330 and 259 us,
// 256 S=777 (1.75) 48.6 and 41.2, 32 S=8192 (2.7) 442 and 412; head dim 16, 36
// S=4096 (1.5) 135 and 107.  Otherwise the queue evens out what the rounds drift
// apart by: 36 S=6348 (2.3) 306 and 317, 1024 S=333 (3) 36.6 and 39.2, 40 S=8192
// (3.3) 491 and 509.
bool queue_needed(const FwdParams& p, int64_t grid, bool equal, int wgs) {
    const int64_t heads = (p.num_heads + p.nq - 1) / p.nq;  // of the fullest queue
    const int64_t tickets = heads * (p.pairs ? (p.nmb + 1) / 2 : p.nmb);
    const int64_t slots = grid / p.nq;
    if (equal && wgs >= 3 && (tickets <= 2 * slots || (2 * tickets >= 5 * slots && tickets < 3 * slots))) return false;
    return tickets > slots;
}

// Position of an instantiation in the kernel lists (a fixed-size cache index).
int kernel_index(const KernelEntry& e) {
    int base = 0;
    for (const KernelList& l : all_lists) {
        if (&e >= l.entries && &e < l.entries + l.count) return base + (int)(&e - l.entries);
        base += l.count;
    }
    return -1;
}

// Resident workgroups per CU of an instantiation, queried once per device
// (a fixed array: no host memory is allocated for it).
int resident_wgs(DeviceState& ds, const KernelEntry& e) {
    const int idx = kernel_index(e);
    if (idx >= 0 && idx < kMaxKernels) {
        const int cached = ds.occupancy[idx].load(std::memory_order_relaxed);
        if (cached > 0) return cached;
    }
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, e.fn, e.nw * 64, 0) != hipSuccess || nb <= 0) nb = 1;
    if (idx >= 0 && idx < kMaxKernels) ds.occupancy[idx].store(nb, std::memory_order_relaxed);
    return nb;
}

// ---------------------------------------------------------------------------
// Tile search.  The reference's get_tiling is a table of Ascend UB tilings
// (flash_attention_forward.py:628-664) and its search tool times every
// (BM, BN) pair (tiling/search_optimal_tiling.py:47-81).  Here the candidates
// are the compiled instantiations for (dtype, head dim), each built for a
// stated number of waves per SIMD; each is checked against gfx950's per-CU LDS
// and scored with a
// cost model: the persistent grid's makespan in key-tile steps, where a step of
// a BM x BN tile costs its MFMA cycles plus a fixed per-tile synchronisation
// overhead, and workgroups sharing a CU share its four SIMDs.
// ---------------------------------------------------------------------------
struct TileCost {
    bool feasible;
    double cycles;
};

// SIMD-cycle model of one wave's key-tile step, measured on MI355X: the two
// contractions (32 x BN x D each at 1024 flop/cycle) plus the softmax VALU work
// (~9.5 cycles per score of the lane's 32 x BN tile share) plus workgroup
// synchronisation, which costs an 8-wave workgroup (one per CU, two waves of
// it per SIMD) about a third of what two 4-wave workgroups per CU pay.  The
// ping-pong schedule hides about a quarter of the softmax work behind the
// other wave's MFMAs.
double wave_tile_cycles(const KernelEntry& e) {
    const int dp = e.d < 32 ? 32 : e.d;
    const double mfma = 2.0 * 2.0 * 32.0 * e.bn * dp / 1024.0;
    const double valu = (9.5 * e.bn / 2.0 + 300.0 * e.bn / 64.0) * (e.pp ? 0.75 : 1.0);
    const double sync = e.nw >= 8 ? 100.0 : 300.0;
    return mfma + valu + sync;
}

TileCost tile_cost(const KernelEntry& e, int64_t z, int64_t h, int64_t n, int num_cus) {
    TileCost tc{false, 0.0};
    const int dp = e.d < 32 ? 32 : e.d;
    // Each instantiation was compiled for `occ` waves per SIMD (the compiler
    // fits its registers to that), so only the LDS budget is checked here.
    const int lds = (e.pp ? 3 : 2) * 2 * e.bn * dp * 2;
    if (lds > kLdsPerCu) return tc;
    const int wg_by_waves = (4 * e.occ) / e.nw;
    const int wg_by_lds = kLdsPerCu / lds;
    const int wg_per_cu = std::max(1, std::min(wg_by_waves, wg_by_lds));
    const int bm = e.bm;
    const int64_t nmb = (n + bm - 1) / bm;
    // workgroups that actually share a CU: fewer tasks than CUs leave each alone
    const int64_t ntask = z * h * nmb;
    const int64_t conc = std::min<int64_t>(wg_per_cu, (ntask + num_cus - 1) / num_cus);
    const int waves_per_simd = (int)std::max<int64_t>(1, conc * e.nw / 4);
    const int64_t tiles_full = (n + e.bn - 1) / e.bn;
    const double step = wave_tile_cycles(e);
    // Makespan of the persistent grid: total wave work over the 4 SIMDs of
    // every CU, but no shorter than the longest task, whose waves each share
    // a SIMD with waves_per_simd - 1 others.
    double work = 0.0, longest = 0.0;
    // task setup / epilogue; the wait for the first tile, of the few a short
    // row has, decides between the 64- and the 128-key tiles of head dims 16
    // and 32 (B=32 H=16 S=333 D=32: 23.1 and 24.4 us)
    const double setup = 600.0 + (e.d <= 32 ? 16.0 * e.bn : 0.0);
    for (int64_t mb = 0; mb < nmb; ++mb) {
        const int64_t tiles = e.causal ? std::min<int64_t>(tiles_full, ((mb + 1) * bm + e.bn - 1) / e.bn) : tiles_full;
        const double c = tiles * step + setup;
        work += c * e.nw;
        longest = std::max(longest, c * waves_per_simd);
    }
    work *= (double)(z * h);
    // SIMDs with work: each wave of a running task sits on its own SIMD
    // until all 4 * num_cus are taken
    const double busy_simds = std::min<double>(4.0 * num_cus, (double)ntask * e.nw);
    tc.feasible = true;
    tc.cycles = std::max(work / busy_simds, longest);
    return tc;
}

// ---------------------------------------------------------------------------
// Key-split variants (fa_fwd_keysplit.hpp).  A launch whose blocks are too few
// or too unequal to fill the CUs runs shorter with smaller blocks whose keys
// the waves of a workgroup share: twice as many tasks of half the length at
// the same rate per CU (128 rows, two key groups), or four times as many (64
// rows, four groups) that load K and V once per 64 rows.  Which one ends first
// is read off this model: a task costs `task` + `step` per key tile (of all its
// groups), in microseconds at the clock of a part-filled chip, the shared pair
// where several workgroups of it sit on a CU; a launch takes as long as its
// longest task, no less than its work spread over the workgroups, and, filled,
// no less than 1.5 times that, since the board then runs at its power limit
// (1.3 times for causal launches at head dim 128, whose short tasks leave the
// matrix cores idle more; between the two 32 of 573 choices differ, where 1.3
// is up to 1.30 times as fast, B*H = 16, S=4096, and down to 0.82, B*H = 40,
// S=512, in the mean of all 0.1 %).  Against the times of 3372 shapes (1 to 256
// heads, 64 to 8192 keys, fp16; part of them in
// profiles/fa_fwd_keysplit_choice.csv) it is off by 10 to 13 % rms.  (Head dim
// 256 has no variant: 128 rows of its Q do not fit the buffers that are free at
// a task's start.)
// ---------------------------------------------------------------------------
struct LaunchCost {
    int d, rows, bn, kg;  // rows and keys per step of a workgroup
    int wgs;              // workgroups per CU
    double task, step, task_shared, step_shared;
};
constexpr double LAUNCH_US = 4.0;
constexpr LaunchCost launch_costs[] = {
    {128, 256, 64, 1, 1, 3.00, 1.34, 0, 0},   {128, 128, 64, 1, 2, 2.04, 1.15, 3.44, 1.48},
    {128, 128, 128, 2, 1, 2.90, 1.49, 0, 0},  {128, 64, 128, 4, 1, 2.85, 0.82, 0, 0},
    {64, 256, 128, 1, 1, 3.03, 1.49, 0, 0},   {64, 128, 64, 1, 2, 1.07, 0.79, 2.31, 0.90},
    {64, 128, 256, 2, 1, 2.92, 1.72, 0, 0},   {64, 64, 256, 4, 1, 2.36, 0.86, 0, 0},
    {32, 128, 64, 1, 4, 0.23, 0.61, 1.25, 0.83}, {32, 128, 128, 1, 3, 0.23, 1.10, 1.25, 1.50},
    {32, 64, 256, 4, 1, 2.06, 0.57, 0, 0},
};

// Predicted microseconds of a launch, or 0 where the model has no entry.
double launch_us(const KernelEntry& e, int64_t heads, int64_t n, int num_cus) {
    for (const LaunchCost& c : launch_costs) {
        if (c.d != e.d || c.rows != e.rows || c.kg != e.kg || c.bn != e.keys * e.kg) continue;
        const int64_t nmb = (n + c.rows - 1) / c.rows;
        const int64_t tasks = heads * nmb;
        const int64_t conc = std::max<int64_t>(1, std::min<int64_t>(c.wgs, (tasks + num_cus - 1) / num_cus));
        const double task = conc > 1 ? c.task_shared : c.task, step = conc > 1 ? c.step_shared : c.step;
        const int64_t slots = num_cus * conc;
        const double longest = task + step * (double)((n + c.bn - 1) / c.bn);
        double total = longest * (double)tasks, span;
        if (e.causal) {
            // block m has ceil((m + 1) rows / bn) steps: on average (nmb + 1) / 2
            // blocks' worth and half a step of rounding up where a step is longer
            const double rounding = c.bn > c.rows ? 0.5 * (1.0 - (double)c.rows / c.bn) : 0.0;
            const double steps = std::min(0.5 * (double)(nmb + 1) * c.rows, (double)n) / c.bn + rounding;
            total = (double)tasks * (task + step * std::max(1.0, steps));
            span = std::max(longest, total / (double)std::min(slots, tasks));
        } else {
            span = (double)((tasks + slots - 1) / slots) * longest;
        }
        return LAUNCH_US + std::max(span, total / (double)slots * (e.causal && e.d == 128 ? 1.3 : 1.5));
    }
    return 0.0;
}

// The key-split variant that runs `base`'s shape at least a tenth shorter than
// `base` (head dim 32, whose predictions are looser: 15 %), or `base`.  Of the
// 3372 shapes 1371 run one, 1.41 to 1.60 times as fast as `base` in the geometric
// mean by head dim and mask; 17 of them are slower, by up to a tenth (B*H = 32,
// S=1200, D=32 causal 16.6 -> 18.3 us).  Always the fastest would be 1 to 4 % more.
const KernelEntry* keysplit_or(const KernelEntry* base, int64_t heads, int64_t n, int num_cus) {
    const KernelEntry* best = base;
    // (0 without an entry: no variant is shorter)
    double limit = launch_us(*base, heads, n, num_cus) * (base->d == 32 ? 0.85 : 0.9);
    for_each_kernel([&](const KernelEntry& e) {
        if (e.kg == 1 || e.dtype != base->dtype || e.d != base->d || e.causal != base->causal) return;
        const double us = launch_us(e, heads, n, num_cus);
        if (us > 0.0 && us < limit) {
            best = &e;
            limit = us;
        }
    });
    return best;
}

int choose_tiling(int64_t z, int64_t h, int64_t n, int64_t d, int causal, int dtype, int num_cus,
                  const KernelEntry** out) {
    const KernelEntry* best = nullptr;
    double best_cycles = 0.0;
    for_each_kernel([&](const KernelEntry& e) {
        if (e.dtype != dtype || e.d != d || e.causal != (causal ? 1 : 0) || e.mode != MODE_FUSED || e.kg > 1) return;
        const TileCost tc = tile_cost(e, z, h, n, num_cus);
        if (!tc.feasible) return;
        if (!best || tc.cycles < best_cycles - 1e-6 ||
            (std::fabs(tc.cycles - best_cycles) <= 1e-6 && e.bn > best->bn)) {
            best = &e;
            best_cycles = tc.cycles;
        }
    });
    if (!best) return RSFA_E_TILE;
    *out = keysplit_or(best, z * h, n, num_cus);
    return RSFA_OK;
}

// choose_tiling's answer for a launch, kept per thread for the shapes last asked
// for: the search takes 1.7 us, as long as the rest of a launch's checks.  (The C
// library allocates the table, 2.5 KB, at a thread's first launch.  A table shared
// by all threads, behind a mutex or sequence numbers, left attention() at 13.9 us
// instead of 12.5: this library's own thread-local access brings the thread's
// table of such storage up to date, and other libraries' accesses stay fast.)
int choose_tiling_kept(int64_t z, int64_t h, int64_t n, int64_t d, int causal, int dtype, int num_cus,
                       const KernelEntry** out) {
    struct Kept {
        int64_t zh, n;
        int32_t d, causal, dtype, num_cus;
        const KernelEntry* e;
    };
    static thread_local Kept kept[64] = {};
    const int64_t zh = z * h;
    Kept& k = kept[((uint64_t)(zh * 1000003 + n * 8191 + d * 31 + causal * 7 + dtype) * 0x9E3779B97F4A7C15ull) >> 58];
    if (!(k.e && k.zh == zh && k.n == n && k.d == d && k.causal == causal && k.dtype == dtype && k.num_cus == num_cus)) {
        const KernelEntry* e = nullptr;
        const int st = choose_tiling(z, h, n, d, causal, dtype, num_cus, &e);
        if (st != RSFA_OK) return st;
        k = Kept{zh, n, (int32_t)d, causal, dtype, num_cus, e};
    }
    *out = k.e;
    return RSFA_OK;
}

// A requested (BLOCK_M, BLOCK_N) must follow the reference's rules (powers of
// two in [16, 512], BLOCK_M * BLOCK_N <= 65536, tiling/search_optimal_tiling.py:
// 47-81) and, when causal, BLOCK_N <= BLOCK_M, which the reference silently
// breaks on (NaN, benchmarks/run_correctness_test.py:24-25).
int validate_request(int causal, int req_bm, int req_bn) {
    if (!is_pow2(req_bm) || !is_pow2(req_bn) || req_bm < 16 || req_bn < 16 || req_bm > 512 || req_bn > 512 ||
        (int64_t)req_bm * req_bn > 65536)
        return RSFA_E_TILE;
    if (causal && req_bn > req_bm) return RSFA_E_TILE;
    return RSFA_OK;
}

// The compiled instantiation nearest to a valid request (log distance in BM
// and BN; ties go to the larger BN).  This is what a launch with a request runs.
int resolve_exact(int64_t d, int causal, int dtype, int req_bm, int req_bn, const KernelEntry** out) {
    const int st = validate_request(causal, req_bm, req_bn);
    if (st != RSFA_OK) return st;
    if ((*out = find_kernel(dtype, (int)d, req_bn, req_bm, causal, MODE_FUSED)) != nullptr) return RSFA_OK;
    const KernelEntry* best = nullptr;
    double best_dist = 0.0;
    for_each_kernel([&](const KernelEntry& e) {
        if (e.dtype != dtype || e.d != d || e.causal != (causal ? 1 : 0) || e.mode != MODE_FUSED || e.kg > 1) return;
        const double dist = std::fabs(std::log2((double)e.bm / req_bm)) + std::fabs(std::log2((double)e.bn / req_bn));
        if (!best || dist < best_dist - 1e-9 || (std::fabs(dist - best_dist) <= 1e-9 && e.bn > best->bn)) {
            best = &e;
            best_dist = dist;
        }
    });
    if (!best) return RSFA_E_TILE;
    *out = best;
    return RSFA_OK;
}

bool valid_dtype(int dt) {
    return dt == RSFA_DTYPE_F16 || dt == RSFA_DTYPE_BF16 || dt == RSFA_DTYPE_F16_V8E5M2;
}

// `mult`: required multiple (elements) of the outer strides: 8 for 2-byte
// elements, 16 for a float8 V, i.e. 16-byte rows either way.
int check_tensor(const void* ptr, const int64_t st[4], int mult = 8) {
    if (((uintptr_t)ptr & 15) != 0) return RSFA_E_ALIGN;
    if (st[3] != 1) return RSFA_E_ALIGN;
    for (int i = 0; i < 3; ++i)
        if (st[i] < 0 || (st[i] % mult) != 0) return RSFA_E_ALIGN;
    return RSFA_OK;
}

// The K/V loader of a tile (and the Q loader of the ping-pong tiles that stage
// Q through LDS) keeps one uniform 64-bit base per tile and per-lane 32-bit
// byte offsets that span the tile's BN rows: ((BN - 1) * row stride +
// row width) * 2 bytes must stay below 2^32, or the offsets would wrap.
bool loader_offsets_fit(const KernelEntry& e, int64_t row_stride) {
    const int64_t dp = e.d < 32 ? 32 : e.d;
    return ((int64_t)(e.keys - 1) * row_stride + dp) * 2 < (int64_t(1) << 32);
}

// Zeroes `words` 32-bit words (the no-allocation entry point's queue
// counters) in stream order; a kernel rather than a memset so that graph
// capture records a kernel node.
__global__ void __launch_bounds__(64) clear_words(uint32_t* __restrict__ p, int words) {
    for (int i = threadIdx.x; i < words; i += blockDim.x) p[i] = 0u;
}

}  // namespace
}  // namespace rsfa

using namespace rsfa;

extern "C" {

int rsfa_abi_version(void) { return RSFA_ABI_VERSION; }

const char* rsfa_strerror(int status) {
    switch (status) {
        case RSFA_OK: return "success";
        case RSFA_E_NULL: return "a required pointer is NULL";
        case RSFA_E_SHAPE: return "invalid shape: Z, H and N_CTX must be >= 1 and fit the 32-bit task index "
                                  "(split mode: Z*H*N_CTX below 2^31 rows)";
        case RSFA_E_HEADDIM: return "head_dim must be one of 16, 32, 64, 128, 256";
        case RSFA_E_DTYPE: return "dtype must be float16 or bfloat16 (q, k, v, o), or float16 q, k, o with a float8_e5m2 v";
        case RSFA_E_TILE: return "invalid BLOCK_M/BLOCK_N: powers of two in [16, 512], BLOCK_M*BLOCK_N <= 65536, "
                                 "and BLOCK_N <= BLOCK_M when causal";
        case RSFA_E_ALIGN: return "tensors need a unit last-dim stride, other strides multiple of 8 elements, "
                                  "16-byte aligned base pointers, and K/V row strides that keep a key tile "
                                  "within 4 GiB";
        case RSFA_E_DEVICE: return "HIP runtime error while preparing the device";
        case RSFA_E_LAUNCH: return "kernel launch failed";
        case RSFA_E_ABI: return "rsfa_fwd_args.struct_size does not match this library";
        case RSFA_E_SCRATCH:
            return "the problem needs more workspace (split state) than the no-allocation "
                   "entry point's fixed buffer (RSFA_NOALLOC_WORKSPACE_BYTES)";
        case RSFA_E_WORKSPACE:
            return "workspace missing or smaller than rsfa_split_workspace_bytes() (causal split mode)";
        default: return "unknown rsfa status";
    }
}

int rsfa_get_num_compute_cores(int device) {
    int dev = device;
    if (dev < 0) {
        const int st = current_device(&dev);
        if (st != RSFA_OK) return st;
    }
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return RSFA_E_DEVICE;
    return cus;
}

int rsfa_resolve_tiling(int64_t head_dim, int32_t causal, int32_t dtype, int32_t req_block_m, int32_t req_block_n,
                        int32_t* block_m, int32_t* block_n) {
    if (!block_m || !block_n) return RSFA_E_NULL;
    if (!valid_head_dim(head_dim)) return RSFA_E_HEADDIM;
    if (!valid_dtype(dtype)) return RSFA_E_DTYPE;
    const KernelEntry* e = nullptr;
    const int st = resolve_exact(head_dim, causal, dtype, req_block_m, req_block_n, &e);
    if (st != RSFA_OK) return st;
    *block_m = e->bm;
    *block_n = e->bn;
    return RSFA_OK;
}

int rsfa_get_tiling(int64_t z, int64_t h, int64_t n_ctx, int64_t head_dim, int32_t causal, int32_t dtype,
                    int32_t* block_m, int32_t* block_n) {
    if (!block_m || !block_n) return RSFA_E_NULL;
    if (z < 1 || h < 1 || n_ctx < 1) return RSFA_E_SHAPE;
    if (!valid_head_dim(head_dim)) return RSFA_E_HEADDIM;
    if (!valid_dtype(dtype)) return RSFA_E_DTYPE;
    // the same CU count the launcher plans with (256 where no device is visible)
    const KernelEntry* e = nullptr;
    const int st = choose_tiling(z, h, n_ctx, head_dim, causal, dtype, planning_cus(), &e);
    if (st != RSFA_OK) return st;
    *block_m = e->bm;
    *block_n = e->bn;
    return RSFA_OK;
}

// The kernels read a float8 V's bytes at every head dim: no copy, no workspace.
uint64_t rsfa_v8_workspace_bytes(int64_t, int64_t, int64_t, int64_t) { return 0; }

uint64_t rsfa_split_workspace_bytes(int64_t z, int64_t h, int64_t n_ctx, int64_t head_dim, int32_t block_m) {
    if (z < 1 || h < 1 || n_ctx < 1 || block_m < 1 || !valid_head_dim(head_dim)) return 0;
    const int64_t nmb = (n_ctx + block_m - 1) / block_m;
    // per query row: m and l, then the un-normalised accumulator (head_dim floats)
    return (uint64_t)(z * h * nmb * block_m) * (uint64_t)(2 + head_dim) * sizeof(float);
}

// Whether a kernel's loaders can address the call's rows (below).
static bool loaders_fit(const KernelEntry& e, const rsfa_fwd_args* a) {
    const bool q_loader = e.kg > 1 || uses_q_buffer(e.d, e.bn, e.nw, e.causal != 0, e.mode);  // Q through LDS
    return loader_offsets_fit(e, a->k_stride[2]) && loader_offsets_fit(e, a->v_stride[2]) &&
           (!q_loader || loader_offsets_fit(e, a->q_stride[2]));
}

// Kernels that a call whose rows they cannot address leaves for a tile with
// fewer keys per load: the key-split variants, and the 128-key tiles of head dims
// 16 and 32 (their rows may lie twice as far apart with 64).
static bool has_stand_in(const KernelEntry& e) { return e.kg > 1 || (e.d <= 32 && e.bn > 64); }

// The kernel a launch runs: for a request (block_m, block_n), that of the
// nearest compiled tile, as the reference's BLOCK_M / BLOCK_N select its
// kernel's tile; under RSFA_FLAG_TILE_HINT (unless RSFA_FLAG_EXACT_TILE) and
// without a request, the tile search's choice for `num_cus` CUs.  Where that
// choice is a key-split variant, a request for its tile runs it too, unless it
// is exact; exact requests, split mode, and rows the variant cannot address,
// run the tile's plain kernel.
static int launch_tile(const rsfa_fwd_args* a, int num_cus, const KernelEntry** e) {
    const int causal = a->causal != 0;
    const bool exact = a->flags & RSFA_FLAG_EXACT_TILE;
    const bool requested = (a->block_m != 0 || a->block_n != 0) && (exact || !(a->flags & RSFA_FLAG_TILE_HINT));
    const bool split = causal && (a->flags & RSFA_FLAG_CAUSAL_SPLIT);
    int st;
    if (requested && (st = resolve_exact(a->head_dim, causal, a->dtype, a->block_m, a->block_n, e)) != RSFA_OK)
        return st;
    if (!requested || !(split || exact)) {
        const KernelEntry* best = nullptr;
        if ((st = choose_tiling_kept(a->z, a->h, a->n_ctx, a->head_dim, causal, a->dtype, num_cus, &best)) != RSFA_OK)
            return st;
        if (!requested || (best->kg > 1 && best->bm == (*e)->bm && best->bn == (*e)->bn)) *e = best;
    }
    if (has_stand_in(**e) && ((split && (*e)->kg > 1) || !loaders_fit(**e, a)))
        *e = find_kernel(a->dtype, (int)a->head_dim, (*e)->kg > 1 ? (*e)->bn : 64, (*e)->bm, causal, MODE_FUSED);
    return *e ? RSFA_OK : RSFA_E_TILE;  // (null: a build without the tile that stands in)
}

// Shared body of the launch entry points.  `ws` / `ws_bytes` is the
// workspace the launch may use (float8 V copy, split state).  With
// `tickets_given`, `tickets` holds the dynamic queue counters (kSlotWords
// words, cleared here on `stream` before use) and the dynamic schedule is
// used even under graph capture; otherwise the launch takes this stream's
// counter from the library's allocation when the stream allows it.
static int fwd_launch(const rsfa_fwd_args* a, void* stream, void* ws, uint64_t ws_bytes, uint32_t* tickets,
                      bool tickets_given) {
    if (!a) return RSFA_E_NULL;
    if (a->struct_size != sizeof(rsfa_fwd_args)) return RSFA_E_ABI;
    if (!a->q || !a->k || !a->v || !a->o) return RSFA_E_NULL;
    if (!valid_dtype(a->dtype)) return RSFA_E_DTYPE;
    const bool v8 = a->dtype == RSFA_DTYPE_F16_V8E5M2;
    if (!valid_head_dim(a->head_dim)) return RSFA_E_HEADDIM;
    if (a->z < 1 || a->h < 1 || a->n_ctx < 1 || a->n_ctx > (1 << 30) || a->z * a->h > (1 << 30))
        return RSFA_E_SHAPE;
    int st;
    if ((st = check_tensor(a->q, a->q_stride)) != RSFA_OK) return st;
    if ((st = check_tensor(a->k, a->k_stride)) != RSFA_OK) return st;
    if ((st = check_tensor(a->v, a->v_stride, v8 ? 16 : 8)) != RSFA_OK) return st;
    if ((st = check_tensor(a->o, a->o_stride)) != RSFA_OK) return st;
    if (((uintptr_t)a->lse & 3) != 0) return RSFA_E_ALIGN;
    const bool causal = a->causal != 0;
    const bool split = causal && (a->flags & RSFA_FLAG_CAUSAL_SPLIT);
    if ((a->block_m != 0 || a->block_n != 0) &&
        (st = validate_request(causal ? 1 : 0, a->block_m, a->block_n)) != RSFA_OK)
        return st;
    // Limits of the kernels' index arithmetic, checked for every tile the
    // launch could pick (before any device work): the K/V loader's per-lane
    // 32-bit offsets, and the split state's 32-bit rows (task * BLOCK_M + row
    // <= Z*H*N_CTX rounded up to the largest BLOCK_M, 256).
    // (a float8 V's byte offsets are half those of the two-byte check)
    for_each_kernel([&](const KernelEntry& e) {
        if (st == RSFA_OK && !has_stand_in(e) && e.dtype == a->dtype && e.d == a->head_dim && !loaders_fit(e, a))
            st = RSFA_E_ALIGN;
    });
    if (st != RSFA_OK) return st;
    if (split && a->z * a->h * ((a->n_ctx + 255) / 256 * 256) >= (int64_t(1) << 31)) return RSFA_E_SHAPE;

    int dev = 0;
    if ((st = current_device(&dev)) != RSFA_OK) return st;
    DeviceState& ds = g_dev[dev];
    int num_cus = 0;
    if ((st = device_cus(ds, dev, &num_cus)) != RSFA_OK) return st;

    // A valid (BLOCK_M, BLOCK_N) request runs the nearest compiled tile, a
    // hint (RSFA_FLAG_TILE_HINT) or no request the tile the search picks.
    const KernelEntry* e = nullptr;
    if ((st = launch_tile(a, num_cus, &e)) != RSFA_OK) return st;
    const int bm = e->rows;

    FwdParams p{};
    p.q = a->q;
    p.k = a->k;
    p.v = a->v;
    p.o = a->o;
    p.lse = a->lse;
    p.q_sz = a->q_stride[0], p.q_sh = a->q_stride[1], p.q_sm = a->q_stride[2];
    p.k_sz = a->k_stride[0], p.k_sh = a->k_stride[1], p.k_sn = a->k_stride[2];
    p.v_sz = a->v_stride[0], p.v_sh = a->v_stride[1], p.v_sn = a->v_stride[2];
    p.o_sz = a->o_stride[0], p.o_sh = a->o_stride[1], p.o_sm = a->o_stride[2];
    p.H = (int32_t)a->h;
    p.n_ctx = (int32_t)a->n_ctx;
    p.nmb = (int32_t)((a->n_ctx + bm - 1) / bm);
    p.num_heads = (int32_t)(a->z * a->h);
    if ((int64_t)p.num_heads * p.nmb > (int64_t(1) << 30)) return RSFA_E_SHAPE;
    p.num_tasks = p.num_heads * p.nmb;
    const float sc = a->sm_scale;
    p.c = std::fabs(sc) * 1.4426950408889634f;
    // Masked scores are -inf and the kernel forms exp2(s * c - m): with c == 0
    // that is -inf * 0 = NaN.  FLT_MIN scales every finite fp16/bf16 score
    // product (|s| < 2^40) below 2^-86, so exp2 of it is exactly 1.0f, the
    // value sm_scale == 0 gives, while masked keys still get exp2(-inf) = 0.
    if (p.c < FLT_MIN) p.c = FLT_MIN;
    p.neg = sc < 0.0f ? 1u : 0u;

    // workspace: the split state
    if (split) {
        const uint64_t need = rsfa_split_workspace_bytes(a->z, a->h, a->n_ctx, a->head_dim, bm);
        if (!ws || ws_bytes < need) return RSFA_E_WORKSPACE;
        if (((uintptr_t)ws & 3) != 0) return RSFA_E_ALIGN;
        // (m, l) of every row, then the rows' fp32 accumulators
        p.state = (float*)ws;
        p.acc = p.state + 2 * (int64_t)p.num_tasks * bm;
    }

    const int modes[2] = {split ? MODE_PREFIX : MODE_FUSED, MODE_DIAG};
    const int launches = split ? 2 : 1;
    bool cleared = false;
    for (int li = 0; li < launches; ++li) {
        const KernelEntry* k = modes[li] == MODE_FUSED ? e
                               : find_kernel(a->dtype, (int)a->head_dim, e->bn, e->bm, causal ? 1 : 0, modes[li]);
        if (!k) return RSFA_E_TILE;
        int wgs = resident_wgs(ds, *k);
        int64_t grid = 0;
        for (;;) {
            grid = std::max<int64_t>(1, std::min<int64_t>((int64_t)num_cus * wgs, p.num_tasks));
            p.nq = queue_count(p.num_heads, grid);
            p.pairs = causal && modes[li] == MODE_FUSED && !(a->flags & RSFA_FLAG_SINGLE_BLOCKS)
                          ? use_pairs(p.num_heads, p.nmb, grid, p.nq)
                          : 0;
            // Long pairs at head dim 32 in exactly two rounds of four workgroups per
            // CU come too staggered in the second: two per CU (B*H = 128 S=4096
            // 253 -> 240 us, 64 S=8192 462 -> 448, 32 S=16384 930 -> 878, 16
            // S=32768 1587 -> 1697).  Not shorter ones (256 S=2048 137 and 152),
            // nor another number of rounds: one (32 S=8192 226 and 281), three
            // (96 S=8192 673 and 704), four (128 S=8192 844 and 963); nor a float8 V
            // (64 S=8192 446 and 479).
            const int64_t pairs_per_queue = (int64_t)((p.num_heads + p.nq - 1) / p.nq) * (p.nmb / 2);
            if (!(p.pairs && e->d == 32 && !v8 && a->n_ctx >= 4096 && wgs > 2 && pairs_per_queue == 2 * (grid / p.nq))) break;
            wgs = 2;
        }
        p.ticket = nullptr;
        if (!(a->flags & RSFA_FLAG_STATIC_SCHEDULE) && queue_needed(p, grid, !causal, wgs)) {
            if (!tickets_given) {
                if (dynamic_schedule_allowed(stream)) p.ticket = stream_ticket(ds, stream);
            } else {
                p.ticket = tickets;
                if (!cleared) {
                    // caller-placed counters start at zero in the first launch
                    // of a call that takes them (a launch leaves them at zero,
                    // but the caller's buffer may hold anything)
                    hipLaunchKernelGGL(clear_words, dim3(1), dim3(64), 0, (hipStream_t)stream, tickets, kSlotWords);
                    if (hipGetLastError() != hipSuccess) return RSFA_E_LAUNCH;
                    cleared = true;
                }
            }
        }
        void* args[] = {&p};
        if (hipLaunchKernel(k->fn, dim3((unsigned)grid), dim3((unsigned)(k->nw * 64)), args, 0,
                            (hipStream_t)stream) != hipSuccess)
            return RSFA_E_LAUNCH;
    }
    return RSFA_OK;
}

int rsfa_attention_fwd_noalloc(const rsfa_fwd_args* a, void* stream) {
    if (!a) return RSFA_E_NULL;
    if (a->struct_size != sizeof(rsfa_fwd_args)) return RSFA_E_ABI;
    // Workspace this call needs, checked before any device work (fwd_launch
    // repeats every other check).
    if (valid_dtype(a->dtype) && valid_head_dim(a->head_dim) && a->z >= 1 && a->h >= 1 && a->n_ctx >= 1) {
        const bool split = a->causal != 0 && (a->flags & RSFA_FLAG_CAUSAL_SPLIT);
        uint64_t need = 0;
        if (split) {
            const KernelEntry* e = nullptr;
            if (launch_tile(a, planning_cus(), &e) == RSFA_OK)
                need += rsfa_split_workspace_bytes(a->z, a->h, a->n_ctx, a->head_dim, e->bm);
        }
        if (need > RSFA_NOALLOC_WORKSPACE_BYTES) return RSFA_E_SCRATCH;
    }
    int dev = 0, st;
    if ((st = current_device(&dev)) != RSFA_OK) return st;
    DeviceState& ds = g_dev[dev];
    {
        // set-up, once per device, with that device current
        std::lock_guard<std::mutex> lock(ds.mu);
        if (!ds.scratch) {
            void* ptr = nullptr;
            if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return RSFA_E_DEVICE;
            ds.scratch = ptr;
        }
    }
    char* const base = (char*)ds.scratch;
    return fwd_launch(a, stream, base + kScratchCounterBytes, RSFA_NOALLOC_WORKSPACE_BYTES, (uint32_t*)base, true);
}

int rsfa_attention_fwd(const rsfa_fwd_args* a, void* stream) {
    if (!a) return RSFA_E_NULL;
    if (a->struct_size != sizeof(rsfa_fwd_args)) return RSFA_E_ABI;
    return fwd_launch(a, stream, a->workspace, a->workspace_bytes, nullptr, false);
}

}  // extern "C"
