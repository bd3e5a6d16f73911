// C ABI of the MI355X signature library: the four hot entry points of the
// reference's GPU plugin (siglib/cusig/cu_signature.cu:3494-3545) plus its
// lifecycle symbols, re-implemented on the gfx950 tree kernels.
//
// Every entry point is synchronous (device work has completed on return), never
// throws across the ABI, returns the reference's status codes
// (siglib/cusig/cu_macros.h:27-89) and leaves a message in a thread-local buffer
// (siglib/shared/last_error.h:22-41).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <charconv>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/cusig_amd.h"
#include "sig_chen_adjoint.h"
#include "sig_deep.h"
#include "sig_heads.h"
#include "sig_rows.h"
#include "sig_degree2.h"
#include "sig_degree2_waves.h"
#include "sig_degree3.h"
#include "sig_host.h"
#include "sig_kernels.h"
#include "sig_registry.h"

namespace sigamd {

thread_local char g_last_error[4096] = {0};

// ---------------------------------------------------------------------------
// kernel table
// ---------------------------------------------------------------------------
struct Table {
    // several partitions (tail, k) of one shape may be compiled; the first listed is the default
    std::map<std::tuple<int, int, int>, std::vector<const KernelEntry*>> fwd, bwd;
    std::map<std::tuple<int, int, int>, const KernelEntry*> fine_fwd, fine_bwd;     // for launches that leave SIMDs without work
    Table()
    {
        int n = 0;
        const EntryList* lists = all_entry_lists(&n);
        for (int i = 0; i < n; ++i)
            for (int j = 0; j < lists[i].count; ++j) {
                const KernelEntry* e = &lists[i].entries[j];
                auto key = std::make_tuple(e->is_f64, e->D, e->N);
                if (e->fine) {
                    (e->fwd ? fine_fwd : fine_bwd)[key] = e;
                    continue;
                }
                auto& slot = e->fwd ? fwd[key] : bwd[key];
                if (e->preferred && !e->staged) slot.insert(slot.begin(), e);
                else slot.push_back(e);
            }
    }
};

// Process-wide hooks (tuning, tests, measurement) may be set by one thread while another is inside a call: atomics,
// read once where a call needs a consistent value.
using Hook = std::atomic<int>;
// the tuning and test hooks below only take effect after cusig_amd_enable_test_hooks(1): a caller that merely links
// the library cannot reroute the kernels of other threads by accident
static Hook g_test_hooks{0};
// tuning hook: when set (tail > 0), prefer the compiled partition with this (tail, k)
static Hook g_force_tail{0}, g_force_k{0};
static Hook g_ignore_table{0};          // tuning hook: every shape runs the run-time-dimension kernels, as if it had no compiled instance
static Hook g_force_run_time_wide{0};   // with a forced partition: take the run-time-dimension kernel in the wide layout

static const Table& table()
{
    static const Table t;
    return t;
}

static int simd_count();
static const KernelEntry* find_entry(bool backward, bool f64, uint64_t d, uint64_t degree);
static double sweep_estimate(const KernelEntry* e, int d, int64_t batch, int64_t L, bool backward);

// The specialised partition of a shape is tuned for a full chip; with few paths its few, heavy lanes make every
// one of the L dependent steps slow.  Then the run-time-dimension kernel (one word prefix per lane, many light
// lanes) finishes sooner even though it issues more instructions in total.
static const KernelEntry* choose_entry(bool backward, bool f64, uint64_t d, uint64_t degree, uint64_t batch, uint64_t L)
{
    const KernelEntry* spec = find_entry(backward, f64, d, degree);
    if (!spec || spec->D == 0 || g_force_tail > 0) return spec;
    const auto& m = backward ? table().bwd : table().fwd;
    auto it = m.find(std::make_tuple(int(f64), 0, int(degree)));
    if (it == m.end() || it->second.empty()) return spec;
    const KernelEntry* gen = it->second.front();
    return sweep_estimate(gen, int(d), int64_t(batch), int64_t(L), backward) <
                   0.7 * sweep_estimate(spec, int(d), int64_t(batch), int64_t(L), backward)
               ? gen
               : spec;
}

// Cutting a path in pieces costs scratch for their signatures.  Where the finer partition cuts more often than the call would
// be cut without it (or an instance more often than the run-time kernel in its place, or the sweep with shared prefix chains is taken, which has a
// table of its own) and the device cannot hold
// that, the call is served without it: it needs no more memory than it ever did.
static thread_local bool tl_no_fine = false, tl_fine_more_pieces = false;

// Where choose_entry's estimate asks for the run-time kernel and no finer partition takes its place, the instance after all (else null): time pieces and
// the staged twin make it the sooner one of 28000 random calls in that state, but where this rule says (0.80 of the run-time kernel's time on average, four calls
// 1.03 to 1.05 times as long, 59 x 6384 x 4, degree 3, the longest; 571 paths x 6136 steps x 12 channels, degree 3, double, backward 14.6 -> 4.0 ms;
// 1 x 15 x 29, degree 4, single 0.26 -> 0.06):
// - forward, lanes that hold one level, or few steps: 0.92 on average, but up to 1.47 (3 x 731 x 13, degree 3);
// - backward, lanes that hold four levels and more: 135 x 80 x 2, degree 9, single 0.19 -> 0.34;
// - backward, few steps: 40 us -> 47 (5 x 4 x 32, degree 3), in single precision where a prefix's last lane lacks letters up to 15 (3 x 14 x 32, degree 3:
//   44 -> 48);
// - many steps in all of few coefficients: 116 x 13224 x 2, degree 4, 0.39 -> 0.59; a few times ten paths of the longest, 3 channels, degree 4: 1.02 on average of
//   13, up to 1.16 (64 x 8480: 255 us -> 296);
// - few paths of 128 to 511 steps, which instances do not cut yet: 2 x 345 x 8, degree 4, double 0.13 -> 0.19; up to 16 paths at 8 channels, degree 4, from 256
//   steps, where the run-time kernel cuts them, to 399 (10 x 348: 140 us -> 168; 10 x 224: 207 -> 116, 9 x 508: 164 -> 120).
static const KernelEntry* instance_after_all(const KernelEntry* e, bool backward, uint64_t d, uint64_t degree, uint64_t batch, uint64_t L)
{
    if (e->D != 0 || g_force_tail > 0 || tl_no_fine) return nullptr;
    const KernelEntry* spec = find_entry(backward, e->is_f64 != 0, d, degree);
    if (!spec || spec->D <= 0) return nullptr;
    if (!backward) return L >= 256 && spec->tail >= 2 ? spec : nullptr;
    if (L < 8 || spec->tail >= 4) return nullptr;
    if (L < 16 && batch < 16 && !spec->is_f64 && d % uint64_t(spec->k) != 0) return nullptr;
    const int64_t top = ipow64(int64_t(d), int(degree));
    if (top <= 32 && batch * L > 100000) return nullptr;
    if (top == 81 && L >= 6900 && batch < 84) return nullptr;
    if (top >= 4096 && batch <= 8 && L >= 128 && L < 512) return nullptr;
    if (top >= 4096 && degree == 4 && d <= 8 && batch <= 16 && L >= 256 && L < 400) return nullptr;
    return spec;
}

// Shapes without a specialised instance run a run-time-dimension kernel.  Its default carries few depth-1 letters
// per lane in the packed layout, which suits the few lanes of small shapes.  Up to degree 10 there are variants with
// more letters per lane (the chain work of a lane is shared by more top-level updates), most of them in the wide
// layout (one letter group of one path per wave, the group's increments arriving through scalar loads), which needs
// at least 48 word prefixes.  Measured for d = 41 .. 80 at degree 4, 21 .. 32 at degree 5, 9 .. 16 at degree 6,
// 6 .. 8 at degree 7 and 5 .. 6 at degree 8: 2-16x faster forward, 1.5-5x backward than the default.
static const KernelEntry* pick_run_time_entry(bool backward, bool f64, int d, int degree)
{
    const auto& m = backward ? table().bwd : table().fwd;
    auto packed = m.find(std::make_tuple(int(f64), 0, degree));
    if (packed == m.end() || packed->second.empty()) return nullptr;
    const KernelEntry* best = packed->second.front();
    const KernelEntry* packed_many = nullptr;
    for (const KernelEntry* e : packed->second)
        if (e->k > best->k && !e->staged && (!packed_many || e->k > packed_many->k)) packed_many = e;
    auto wide = m.find(std::make_tuple(int(f64), -1, degree));
    if (wide == m.end() || wide->second.empty() || ipow64(d, degree - 1) < 48)
        return d >= 12 && packed_many ? packed_many : best;
    // single precision backward at 9 .. 15 channels: the packed 16-letter variant is ~10 % ahead of the wide one,
    // whose only letter group is then partly empty
    if (backward && !f64 && d > 8 && d < 16 && packed_many) return packed_many;
    // letters per lane: a partly empty last group costs more than the longer chain share of a smaller K
    // (forward, 32 letters: single precision only -- a double-precision row of 32 does not fit the scalar registers twice)
    const int want = d <= 8 ? 8 : backward ? (d <= 32 ? 16 : 32) : (d % 32 == 0 && !f64 ? 32 : 16);
    const KernelEntry* pick = nullptr;
    for (const KernelEntry* e : wide->second) {
        if (e->staged) continue;
        // the largest letter count up to `want`, else the smallest there is
        if (!pick || (e->k <= want ? (pick->k > want || e->k > pick->k) : (pick->k > want && e->k < pick->k))) pick = e;
    }
    return pick ? pick : best;
}

static const KernelEntry* find_entry(bool backward, bool f64, uint64_t d, uint64_t degree)
{
    const auto& m = backward ? table().bwd : table().fwd;
    if (d <= 0x7fffffff && degree <= 0x7fffffff) {
        auto it = m.find(std::make_tuple(int(f64), int(d), int(degree)));
        const bool run_time = it == m.end() || g_ignore_table != 0;
        if (run_time) it = m.find(std::make_tuple(int(f64), 0, int(degree)));
        if (it != m.end() && !it->second.empty()) {
            if (g_force_tail > 0) {
                auto forced = [](const std::vector<const KernelEntry*>& from) -> const KernelEntry* {
                    for (const KernelEntry* e : from)
                        if (e->tail == g_force_tail && e->k == g_force_k && !e->staged) return e;
                    return nullptr;
                };
                // a partition that an instance does not have: the run-time kernels' one
                const KernelEntry* e = run_time ? nullptr : forced(it->second);
                if (!e) {
                    const bool wide = g_force_run_time_wide && ipow64(int64_t(d), int(degree) - 1) >= 48;
                    auto rt = m.find(std::make_tuple(int(f64), wide ? -1 : 0, int(degree)));
                    if (wide && rt == m.end()) rt = m.find(std::make_tuple(int(f64), 0, int(degree)));
                    if (rt != m.end()) e = forced(rt->second);
                }
                if (e) return e;
            }
            if (run_time) return pick_run_time_entry(backward, f64, int(d), int(degree));
            return it->second.front();
        }
    }
    return nullptr;
}

// Rough VALU instruction count of one forward step of one lane for partition (tail, k); the backward costs a
// near-constant multiple of it, so the same figure ranks partitions for both sweeps.
static double lane_step_cost(int d, int n, int tail, int k)
{
    const int m = n - tail;
    double cost = m;
    for (int t = 1; t <= n; ++t) {
        if (t == 1) cost += 1;
        else if (t <= m) cost += 2.0 * (t - 1);
        else {
            cost += 1 + 2.0 * (m - 1);
            double nodes = k;
            for (int e = 1; e <= t - m; ++e) {
                cost += (e == t - m) ? nodes : 2.0 * nodes + nodes / (e == 1 ? k : d);
                nodes *= d;
            }
        }
    }
    return cost;
}

static TreeGeom geom_of(const KernelEntry* e, int d) { return make_geom(d, e->N - e->tail, e->k, layout_of(e->D, e->staged != 0)); }

// A sweep is a chain of dependent steps: its duration is their number times the longer of one lane-step (latency
// of a lone wave) and the chip-wide issue time of all waves' steps.  Long paths of an under-filled launch are cut
// in time (about two waves per SIMD, segments of at least 32 resp. 48 steps), which divides the chain and multiplies
// the waves.  Returns a relative figure.
static double sweep_estimate(const KernelEntry* e, int d, int64_t batch, int64_t L, bool backward)
{
    const TreeGeom g = geom_of(e, d);
    const double waves = double(total_waves(g, batch));
    const double simds = double(simd_count());
    double cuts = 1.0;
    if (waves * 2 <= simds) cuts = std::max(1.0, std::min({2.0 * simds / waves, double(L / (backward ? 32 : 48)), backward ? 64.0 : 32.0}));
    const double per_step = lane_step_cost(d, e->N, e->tail, e->k) * (e->D > 0 ? 1.0 : 1.15);
    return per_step / cuts * std::max(1.0, waves * cuts / simds * 0.8);
}

// the LDS-staged twin of a kernel instance (same partition), if one was compiled
static const KernelEntry* staged_twin(bool backward, const KernelEntry* base)
{
    const auto& m = backward ? table().bwd : table().fwd;
    auto it = m.find(std::make_tuple(base->is_f64, base->D, base->N));
    if (it == m.end()) return nullptr;
    for (const KernelEntry* e : it->second)
        if (e->staged && e->tail == base->tail && e->k == base->k) return e;
    return nullptr;
}

// ---------------------------------------------------------------------------
// per-device workspace (grow-only; released by cusig_shutdown).  The mutex also
// serialises concurrent host threads on the shared buffers, as the reference
// does for its backward workspaces (siglib/cusig/cu_signature.cu:2971).
// ---------------------------------------------------------------------------
struct Workspace {
    void* ptr = nullptr;
    size_t bytes = 0;
};
std::atomic<int> g_force_wide_index{0};
std::atomic<int> g_chen_adjoint_mode{0};
std::atomic<int> g_chen_low_levels{1};
std::atomic<int> g_row_forms{1};
thread_local int tl_row_form = 0, tl_chen_both = 0;
std::mutex g_ws_mutex;
static std::map<std::pair<int, int>, Workspace> g_ws;   // (device, slot)

// test hooks: workspace requests above this many bytes, and those that would make the device's pool larger than this, fail as if
// the device were out of memory (0: no limit)
static std::atomic<uint64_t> g_alloc_limit{0}, g_pool_limit{0};
static std::atomic<int> g_alloc_retries{0};     // calls split in two after a failed workspace allocation

static uint64_t pool_bytes(int dev)
{
    uint64_t total = 0;
    for (const auto& kv : g_ws)
        if (kv.first.first == dev) total += kv.second.bytes;
    return total;
}

static void give_back(Workspace& w)     // hipFree waits for the device, and so for whatever still uses the buffer
{
    if (!w.ptr) return;
    void* const ptr = w.ptr;
    w.ptr = nullptr;
    w.bytes = 0;
    SIG_HIP(hipFree(ptr));
}

static thread_local uint64_t tl_grown = 0;      // slots that grew since fine_if_it_fits began this thread's call
constexpr int kHeadsSlot = 20;

void* workspace(int slot, size_t bytes)
{
    int dev = 0;
    SIG_HIP(hipGetDevice(&dev));
    Workspace& w = g_ws[{dev, slot}];
    if (w.bytes < bytes) {
        give_back(w);
        const size_t want = (bytes + bytes / 8 + 255) & ~size_t(255);
        auto allocate = [&] {
            const uint64_t limit = g_alloc_limit, pool = g_pool_limit;
            if ((limit && want > limit) || (pool && pool_bytes(dev) + want > pool) || hipMalloc(&w.ptr, want) != hipSuccess) {
                (void)hipGetLastError();
                w.ptr = nullptr;
                return false;
            }
            w.bytes = want;
            return true;
        };
        if (!allocate()) {
            // the table of the sweeps with shared prefix chains, up to 1.1 GiB, was the last thing its call asked for, so no call that is under
            // way here holds it: a call that fits without it gets that room
            Workspace& table = g_ws[{dev, kHeadsSlot}];
            if (slot == kHeadsSlot || !table.ptr) throw std::bad_alloc();
            give_back(table);
            if (!allocate()) throw std::bad_alloc();
        }
        tl_grown |= uint64_t(1) << slot;
    }
    return w.ptr;
}

// The increment-gradient accumulators of backward sweeps that form their own increments (no pre-pass launch that could
// clear one): two buffers per device take turns.  The launch that turns a call's accumulator into the path gradient also
// clears whatever the other buffer still holds, so the next call finds its accumulator zero.  `dirty` counts the leading
// bytes that may be non-zero (everything after an allocation; a failed call leaves its buffer dirty and `next`
// unchanged, and the next call clears it with a launch of its own).  Guarded by the workspace mutex.
struct DzPair {
    void* ptr[2] = {nullptr, nullptr};
    size_t capacity[2] = {0, 0};
    size_t dirty[2] = {0, 0};
    int next = 0;
};
static std::map<int, DzPair> g_dz;      // per device
constexpr int kDzSlot[2] = {16, 17};

static void* dz_pair_buffer(DzPair& st, int which, size_t bytes)
{
    int dev = 0;
    SIG_HIP(hipGetDevice(&dev));
    void* p = workspace(kDzSlot[which], bytes);
    const size_t capacity = g_ws[{dev, kDzSlot[which]}].bytes;
    if (p != st.ptr[which] || capacity != st.capacity[which]) {     // fresh memory: all of it may be non-zero
        st.ptr[which] = p;
        st.capacity[which] = capacity;
        st.dirty[which] = capacity;
    }
    return p;
}

// what the thread's call has grown since fine_if_it_fits began it goes back to the device
static void give_back_grown()
{
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    int dev = 0;
    SIG_HIP(hipGetDevice(&dev));
    for (int slot = 0; slot < 64; ++slot) {
        if (!(tl_grown >> slot & 1)) continue;
        auto it = g_ws.find({dev, slot});
        if (it != g_ws.end()) give_back(it->second);
        if (slot == kDzSlot[0] || slot == kDzSlot[1]) g_dz.erase(dev);      // what it knows of their contents
    }
    tl_grown = 0;
}

static int* g_flag_host = nullptr;     // pinned word the forward kernels report NaN / infinity through

static void release_workspaces() noexcept
{
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    for (auto& kv : g_ws) {
        if (kv.second.ptr) {
            int cur = 0;
            if (hipGetDevice(&cur) == hipSuccess && hipSetDevice(kv.first.first) == hipSuccess) {
                (void)hipFree(kv.second.ptr);
                (void)hipSetDevice(cur);
            }
        }
    }
    g_ws.clear();
    g_dz.clear();
    rocblas_release();
    if (g_flag_host) {
        (void)hipHostFree(g_flag_host);
        g_flag_host = nullptr;
    }
    (void)hipGetLastError();
}

// ---------------------------------------------------------------------------
// kernel timing hook for the benchmark
// ---------------------------------------------------------------------------
static std::atomic<bool> g_profile{false};
static std::atomic<float> g_last_ms{-1.f};
// name and events are only touched under the workspace mutex (every timer lives inside a locked region)
static char g_last_name[128] = {0};
static hipEvent_t g_ev0 = nullptr, g_ev1 = nullptr;

struct MainKernelTimer {
    hipStream_t s;
    bool on;
    MainKernelTimer(hipStream_t stream, const char* name, bool allowed = true) : s(stream), on(g_profile && allowed)
    {
        if (!on) return;
        if (!g_ev0) {
            SIG_HIP(hipEventCreate(&g_ev0));
            SIG_HIP(hipEventCreate(&g_ev1));
        }
        std::snprintf(g_last_name, sizeof g_last_name, "%s", name);
        SIG_HIP(hipEventRecord(g_ev0, s));
    }
    // defer: only mark the end; read() fetches the duration later, so that kernels enqueued after the timed one do
    // not wait for a host round trip
    void stop(bool defer = false)
    {
        if (!on) return;
        SIG_HIP(hipEventRecord(g_ev1, s));
        if (!defer) read();
    }
    void read()
    {
        if (!on) return;
        SIG_HIP(hipEventSynchronize(g_ev1));
        float ms = -1.f;
        SIG_HIP(hipEventElapsedTime(&ms, g_ev0, g_ev1));
        g_last_ms = ms;
    }
};

// Stream-ordered mode (off by default): signature_cuda / sig_backprop_cuda only enqueue their kernels on the null
// stream and return; neither the device-wide wait on entry nor the wait for completion is made.  Correct for callers
// whose producers and consumers are ordered with the null stream (PyTorch's default stream is the null stream, and
// blocking streams synchronise with it implicitly); it removes the host round trip between consecutive calls.
static Hook g_stream_ordered{0};
static void entry_sync()
{
    if (!g_stream_ordered) SIG_HIP(hipDeviceSynchronize());
}
static void exit_sync(hipStream_t stream)
{
    if (!g_stream_ordered) SIG_HIP(hipStreamSynchronize(stream));
}

// ---------------------------------------------------------------------------
// NaN / infinity report of the forward pass
// ---------------------------------------------------------------------------
// The kernels that store a signature set a flag when a stored value is not finite, so that callers who must warn
// about overflow (pysiglib/sig.py:299-311 scans the result for NaN and Inf) need no pass of their own over the
// output.  The flag is one word of pinned host memory mapped into the device: it costs nothing to read after the
// call's final synchronisation.  Calls are serialised by the workspace mutex; each thread keeps its own last answer.
static thread_local int tl_sig_nonfinite = -1;     // -1: the last forward call on this thread did not report

static int* nonfinite_flag()
{
    if (!g_flag_host) SIG_HIP(hipHostMalloc(reinterpret_cast<void**>(&g_flag_host), 64, hipHostMallocMapped | hipHostMallocPortable));
    int* dev = nullptr;
    SIG_HIP(hipHostGetDevicePointer(reinterpret_cast<void**>(&dev), g_flag_host, 0));
    return dev;
}

// ---------------------------------------------------------------------------
// time segmentation of the forward sweep
// ---------------------------------------------------------------------------
static Hook g_force_segments{0};   // tuning hook (0 = automatic)
static thread_local int tl_last_segments = 0;   // pieces per path of the last forward sweep on this thread (0: no sweep ran)
static Hook g_point_fed{1};        // tuning hook: 0 always computes the increments in a kernel of their own
static Hook g_lead_lag_sparse{1};  // tuning hook: 0 sweeps lead-lag paths like any other (every letter of every step)

static int simd_count()
{
    static int cached = 0;
    if (!cached) {
        int dev = 0, cus = 0;
        SIG_HIP(hipGetDevice(&dev));
        SIG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        cached = 4 * (cus > 0 ? cus : 256);
    }
    return cached;
}

// Cutting every path into g pieces of 1/g of the steps multiplies the waves and divides the chain of dependent
// steps; it costs one signature write per piece plus the Chen folds.  Two situations pay:
//  * under-filled: whole-path sweeps leave SIMDs without a wave (few paths);
//  * unevenly filled: a few waves per SIMD, and the fullest SIMD holds one more than most (1280 waves on 1024 SIMDs
//    that hold two each run as long as 2048 would); the launch lasts as long as its fullest SIMD needs, and shorter
//    pieces even the load out.
// A small model picks g: the fullest SIMD works through its waves `waves_per_simd` at a time, a SIMD with two or
// more resident waves issuing `pair_rate` times as fast as with one; a step of a lone wave takes 2.4 ns per
// instruction of lane_step_cost, and at least 240 ns when its increments come straight from memory instead of the
// LDS ring (lane_step(g) says which, for the launch g pieces make); the folds cost a fixed 8 us, 10 us per launch
// and 2.2 signature sets of traffic per piece at 4 TB/s (measured: d = 12, degree 4, 48 paths of 300 steps: whole
// 92 us, 2 pieces 77, 3: 76, 4: 94, 6: 101 us).  Pieces keep at least 48 steps and 256 MB of segment signatures at most, and a
// split must promise 7 % (batch 128, length 1024, d = 5, degree 7, f32: 0.587 -> 0.523 ms with three pieces).
struct SplitPlan {
    int pieces;
    double seconds;     // what the model expects the call to take
    double folds;       // the part of it that putting the pieces together takes
};

// Waves of an instance that fit a SIMD, a property of the compiled kernel: asked for once (the query takes 5 us, an eighth of a
// short call: 86 paths of 2 steps, 48 channels, degree 3).  Called under the workspace mutex.
static int resident_waves(const KernelEntry* e)
{
    static std::map<const KernelEntry*, int> known;
    auto it = known.find(e);
    if (it == known.end()) it = known.emplace(e, e->waves_per_simd()).first;
    return it->second;
}

template <typename LaneStep>
static SplitPlan choose_segments(int64_t waves, int64_t L, int waves_per_simd, uint64_t sig_bytes_all_paths, LaneStep&& lane_step,
                           bool f64)
{
    const int64_t simds = simd_count();
    if (waves <= 0 || sig_bytes_all_paths == 0) return {1, 0.0, 0.0};
    const int occ = std::max(1, waves_per_simd);
    const double pair_rate = f64 ? 1.2 : 1.35;
    auto folds = [&](int g) {
        int launches = 0;
        for (int m = g; m > 1; m = (m + 1) / 2) ++launches;
        return g > 1 ? 8e-6 + 10e-6 * launches + 2.2 * g * double(sig_bytes_all_paths) / 4e12 : 0.0;
    };
    auto estimate = [&](int g) {
        const int64_t fullest = (waves * g + simds - 1) / simds;          // waves of the fullest SIMD
        const int64_t rounds = fullest / occ, rest = fullest % occ;
        double steps = double(rounds) * occ / (occ > 1 ? pair_rate : 1.0);
        if (rest) steps += double(rest) / (rest > 1 ? pair_rate : 1.0);
        return double((L + g - 1) / g) * lane_step(g) * steps + folds(g);
    };
    int best = 1;
    double best_t = estimate(1);
    const double whole = best_t;
    if (waves > 4 * simds * occ) return {1, whole, 0.0};
    // (one very long path of few channels: hundreds of pieces, each further doubling one more 10 us fold)
    for (int g : {2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512, 768, 1024}) {
        if (L / g < 48 || uint64_t(g) * sig_bytes_all_paths > (uint64_t(256) << 20)) break;
        const double t = estimate(g);
        if (t < best_t) { best = g; best_t = t; }
    }
    if (best_t < 0.93 * whole) return {best, best_t, folds(best)};
    return {1, whole, 0.0};
}

// The backward sweep can be cut in time as well: the state at the end of segment g is the Chen product of the
// segment signatures up to g, and the adjoint of that state is the upstream gradient pulled back through the product
// with the remaining segments.  That costs a segmented forward sweep, two chains of Chen products and one product
// adjoint, all over (path, segment) rows.
static Hook g_force_bwd_segments{0};   // tuning hook (0 = automatic)
// test hooks, the by-row sweeps of many channels: 0 never, 1 by the rules below, 2 wherever they apply; backward also 3,
// wherever they apply, single precision in the form without matrix units
static Hook g_rows_forward{1};
static Hook g_rows_backward{1};
static thread_local int tl_matrix_form = 0;     // whether the last sweep on this thread was a by-row sweep on the matrix units

// g pieces are chosen by the same kind of model as for the forward sweep (fullest SIMD, `pair_rate`, lane_step(g) =
// seconds per step of a lone wave).  The extra work is larger here: the segmented forward sweep (a third of the
// backward's arithmetic), 2 ceil(log2 g) + 2 launches of about 10 us each on top of a fixed 30 us, and the
// traffic of the scans and of the product adjoint over g rows per path, fitted at 4.2 + 0.64 ceil(log2 g) ps per
// byte of segment signatures (48 paths of 300 steps, d = 12, degree 4, f64: whole 0.225 ms, 2 pieces 0.270,
// 8: 0.578, 64: 4.65 ms; 8 paths of 4000 steps, d = 6, degree 4, f32: whole 3.42 ms, 32 pieces 0.249 ms).
template <typename LaneStep>
static SplitPlan choose_bwd_segments(int64_t waves, int64_t L, int waves_per_simd, uint64_t sig_bytes_all_paths, LaneStep&& lane_step,
                               bool f64)
{
    const int64_t simds = simd_count();
    if (waves <= 0 || sig_bytes_all_paths == 0) return {1, 0.0, 0.0};
    const int occ = std::max(1, waves_per_simd);
    const double pair_rate = f64 ? 1.2 : 1.35;
    auto estimate = [&](int g) {
        const int64_t fullest = (waves * g + simds - 1) / simds;
        const int64_t rounds = fullest / occ, rest = fullest % occ;
        double steps = double(rounds) * occ / (occ > 1 ? pair_rate : 1.0);
        if (rest) steps += double(rest) / (rest > 1 ? pair_rate : 1.0);
        double t = double((L + g - 1) / g) * lane_step(g) * steps;
        if (g > 1) {
            int lg = 0;
            while ((1 << lg) < g) ++lg;
            t *= 1.31;
            t += 30e-6 + 10e-6 * (2 * lg + 2) + double(g) * double(sig_bytes_all_paths) * (4.2e-12 + 0.64e-12 * lg);
        }
        return t;
    };
    int best = 1;
    double best_t = estimate(1);
    const double whole = best_t;
    if (waves > 2 * simds * occ) return {1, whole, 0.0};
    for (int g : {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512}) {
        if (L / g < 32 || uint64_t(g) * sig_bytes_all_paths > (uint64_t(64) << 20)) break;
        const double t = estimate(g);
        if (t < best_t) { best = g; best_t = t; }
    }
    if (best_t < 0.93 * whole) return {best, best_t, 0.0};
    return {1, whole, 0.0};
}

// With at most two waves per SIMD the LDS-staged twin (all-VGPR FMAs, HBM latency hidden by a chunk of
// arithmetic) is the faster way to feed increments.  With more resident waves it depends (measured over d = 4..24,
// degrees 4..6, 3-9 waves per SIMD): the f32 forward is always faster staged (1.2-1.8x: SGPR-operand FMAs issue
// slower than all-VGPR ones), the f32 backward up to 13 channels and both f64 sweeps up to 8 (1.05-1.3x), while with
// more channels the ring's LDS reads cost them 3-30 % (f64 at 10-12 channels is mixed).
static Hook g_force_staged{-1};   // tuning hook: -1 automatic, 0 never, 1 whenever compiled

// lead_lag_sparse: the path is a lead-lag path and staged twins that skip a step's still letters may be used.  Those
// twins do about 40 % less arithmetic, which outweighs what the tuned choice for dense paths says: measured on 144
// lead-lag shapes (2-20 raw channels, both precisions), the forward twin is faster wherever it exists (mean 0.82x), the
// backward twin in single precision and, in double precision, up to 13 augmented channels (mean 0.85x; beyond, its
// register pressure costs more than the skipped work saves, and the general rules below decide; the scalar-fed
// backward kernels of those dimensions have a lead-lag form of their own).
static const KernelEntry* pick_variant(bool backward, const KernelEntry* base, int64_t waves, bool lead_lag_sparse = false)
{
    if (lead_lag_sparse && g_force_staged < 0) {
        const KernelEntry* twin = base->staged ? base : staged_twin(backward, base);
        if (twin && (backward ? (twin->bwd_lead_lag && (!twin->is_f64 || twin->D <= 13)) : twin->fwd_lead_lag != nullptr))
            return twin;
    }
    const bool small_dim = base->D > 0 && base->D <= (base->is_f64 ? 8 : 13);
    const bool want = g_force_staged >= 0 ? g_force_staged != 0
                      : base->stage_policy == 1 ? true
                      : base->stage_policy == 2 ? false
                      : base->stage_policy == 3 ? waves <= 2 * int64_t(simd_count())
                                                : waves <= 2 * int64_t(simd_count()) || small_dim ||
                                                      (!backward && !base->is_f64);
    if (!want) return base;
    const KernelEntry* twin = staged_twin(backward, base);
    return twin ? twin : base;
}

// The by-row forward sweep in single precision against a compiled instance of the same shape, at degree 3: both are
// estimated, the path length included, since only the instance's paths can be cut in time.  Seconds beside what the calls
// have in common.
// By rows: a wave alone on its SIMD takes 148 ns a step (long paths of 48 .. 128 channels, degree 3: 139-152), a full SIMD
// 37 ns a wave and step plus 11.2 ns per product of 32 x 32 (8 waves per SIMD: 82 ns measured at 64 and 97 channels, 62 at
// 72 and 96, whose tiles are partly empty).
static double rows_fwd_seconds(uint64_t d, uint64_t batch, uint64_t L)
{
    const double tiles = double((d + kWave - 1) / kWave), halves = double((d + 31) / 32);
    const double waves = double(batch) * double(d) * tiles * tiles;
    const double per_wave = 37e-9 + 11.2e-9 * halves * halves / (tiles * tiles);
    return double(L) * std::max(148e-9, per_wave * std::ceil(waves / double(simd_count())));
}
// The instance: `run` is the kernel that would be launched.  Scalar-fed sweeps of many channels wait for their loads: 170 ns a
// step and 1.8 ns per instruction and wave of a SIMD (80 channels, 2.7 / 10.2 waves per SIMD: 288 / 589 ns), 1.3 times as
// long where an odd channel count leaves the rows unaligned.  LDS-fed ones follow the model of choose_segments at two
// subtree levels, at one they take 1.7 times as long (49 channels, 21 paths of 8000 steps: 0.94 / 1.74 ms).
// Fitted to 17 channel counts of 48 .. 128 at 0.1 .. 8 waves per SIMD and 8 .. 8000 steps; time-split estimates scatter by
// an eighth and are taken down by it, so that the instance keeps what it may win.  Paths of 8000 steps, degree 3, instance
// in pieces / by rows: 4 x 72 channels 0.58 / 1.13 ms, 22 x 48: 1.13 / 1.40, 13 x 80: 2.1 / 2.4; 22 x 96: 6.1 / 4.1,
// 19 x 112: 14.9 / 5.5.
static double instance_fwd_seconds(const KernelEntry* run, const SplitPlan& plan, int64_t waves, uint64_t d, uint64_t L)
{
    if (run->staged) return (run->tail > 1 ? 1.0 : 1.7) * plan.seconds;
    const double per_simd = double(waves) * plan.pieces / double(simd_count());
    const double step = (170e-9 + 1.8e-9 * lane_step_cost(int(d), run->N, run->tail, run->k) * per_simd) * (d % 2 ? 1.3 : 1.0);
    const double t = std::ceil(double(L) / plan.pieces) * step + plan.folds;
    return plan.pieces > 1 ? 0.88 * t : t;
}

// The same choice for the backward of 33 .. 47 channels, degree 3.  By rows, a step takes 355 ns while no CU holds more than
// one block of four waves and 488 ns with two, which is all it can hold (33 .. 47 channels, 2000 and 8000 steps: 353-368 and
// 477-499 ns; 2.07 rounds of blocks 1.32 us, 2.2 rounds 1.46).  Up to sixteen steps cost alike; from 39 channels on the
// instances start so much slower that eight are counted (9 points: 118 x 35 channels 56 / 68 us, 96 x 43: 84 / 69).
static double rows_bwd_seconds(uint64_t d, uint64_t batch, uint64_t L)
{
    const uint64_t cus = uint64_t(simd_count()) / 4, blocks = batch * ((d + 3) / 4);
    const uint64_t rounds = blocks / (2 * cus), rest = blocks % (2 * cus);
    const double last = rest == 0 ? 0.0 : (rounds == 0 ? rest <= cus : rest <= 48) ? 355e-9 : 488e-9;
    const uint64_t least = d < 39 ? 16 : 8;
    return double((L + least - 1) / least * least) * (488e-9 * double(rounds) + last);
}
// The instances take longer than the model of choose_bwd_segments has it: whole paths 1.6 times (1.5-1.9 at 33 .. 47
// channels), fewer than eight pieces 1.05 times (1.03-1.2), from 39 channels on 1.35 times (1.25-1.5); of more pieces, few
// paths' way to fill the chip, it is 0.85 at the least.  Paths of 8000 steps,
// instance in pieces / by rows: 16 x 33 channels 1.34 / 2.86 ms, 63 x 33: 4.38 / 7.99, 26 x 40: 2.93 / 3.83; 44 x 47,
// whole: 12.1 / 6.9.
static double instance_bwd_seconds(const SplitPlan& plan, uint64_t d)
{
    return plan.seconds * (plan.pieces == 1 ? 1.6 : plan.pieces >= 8 ? 0.85 : d < 39 ? 1.05 : 1.35);
}

// The by-row reverse sweep in single precision on the matrix units or off them.  The matrix form works on sixteen steps at a
// time and its smaller blocks add three times as many pieces to the gradient rows, which shows on paths of a few steps whose
// tiles of 64 x 64 are partly empty (8 paths of 3 / 9 / 12 steps, 65 channels, a quarter filled, degree 4: off / on
// 0.84 / 1.15, 1.24 / 1.33, 1.40 / 1.38 ms; 32 x 1 / 10, 65, degree 3: 76 / 87, 111 / 97 us; 8 x 1 / 4, 72, a third filled,
// degree 4: 1.24 / 1.32, 1.43 / 1.34 ms; 1 x 2 / 4 / 8, 33, degree 5: 278 / 314, 310 / 315, 393 / 320 us).  Tiles filled to
// nine sixteenths win from one step on where several waves share a SIMD (8 x 1, 49, degree 4: 187 / 166 us; 1 x 2, 96:
// 397 / 377; but 1 x 1, 48: 60 / 66) and at degree 3 (1 x 1, 200: 100 / 79 us), full tiles always (8 x 1, 64, degree 4:
// 441 / 389 us), and so do launches of up to two waves per SIMD at degree 3 (4 x 1, 96: 55 / 53 us).
static bool rows_bwd_mfma_wins(uint64_t d, uint64_t degree, uint64_t batch, uint64_t L)
{
    const uint64_t groups = (d + kWave - 1) / kWave, tile = groups * kWave, simds = uint64_t(simd_count());
    const double waves = double(batch) * std::pow(double(d), double(degree) - 2) * double(groups * groups);
    const bool shared = degree == 3 || waves >= 4.0 * double(simds);
    if (L >= (degree == 3 ? 6u : 12u) || 16 * d * d >= (shared ? 9 : 14) * tile * tile) return true;
    if (L >= 3 && (groups == 1 || 16 * d * d >= 5 * tile * tile)) return true;
    return degree == 3 && waves <= 2.0 * double(simds);
}

// ---------------------------------------------------------------------------
// a shape's second, finer partition (gen_instances.py: fine_partition)
// ---------------------------------------------------------------------------
static Hook g_fine{1};      // test hook: 0 never, 1 by the estimates below, 2 wherever there is one

template <typename F>
static void fine_if_it_fits(F&& run)
{
    tl_fine_more_pieces = false;
    tl_grown = 0;
    try {
        run();
    } catch (const std::bad_alloc&) {
        if (!tl_fine_more_pieces) throw;
        give_back_grown();          // the retry has the memory that it would have had without the attempt
        struct Off {
            Off() { tl_no_fine = true; }
            ~Off() { tl_no_fine = false; }
        } off;
        run();
    }
}

static const KernelEntry* fine_entry(bool backward, bool f64, uint64_t d, uint64_t degree)
{
    if (g_fine == 0 || tl_no_fine || g_force_tail > 0 || g_force_staged >= 0 || g_ignore_table != 0 || d > 0x7fffffff || degree > 0x7fffffff) return nullptr;
    const auto& m = backward ? table().fine_bwd : table().fine_fwd;
    auto it = m.find(std::make_tuple(int(f64), int(d), int(degree)));
    return it == m.end() ? nullptr : it->second;
}

// Seconds per step of a launch: a wave alone on its SIMD pays the latency of its step, several share the issue slots; backward,
// every channel beyond four costs a row of the LDS tile of the increment gradient, more in double precision without the
// half-wave sums (one subtree level).  Fitted to 110 partitions of 2 .. 24 channels, degrees 3 .. 8, both precisions, at a thousandth to 8
// waves per SIMD; most within 15 % (ns a step measured / model, one wave per SIMD and eight; single precision: forward d = 4,
// degree 6, 1 level x 4 letters 106 / 104, 361 / 424, 3 x 4 letters 277 / 309, 1299 / 1416; backward 4, 6, 2 x 2: 443 / 443, 1465 / 1556;
// 10, 4, 1 x 10: 474 / 490, 2125 / 1898; 17, 4, 2 x 6: 1028 / 984, 4454 / 4855; double, backward 10, 5, 2 x 5: 619 / 685, 4492 / 5128).
// Scalar-fed forward steps take at least 130 ns (of four and more levels no longer than staged ones: 1325 paths of 2 channels, degree 9, 5 x 1: 285 /
// 288), those of the run-time-dimension kernels about 2.2 times as long (one path of 4 channels, degree 5, double: 270 / 120 ns).  Forward, from 17 channels on: the letters of a staged step come from LDS, and every one
// beyond four that a lane reads costs that again; groups of which the last is not whole guard each read (staged: from four groups
// on); lead-lag sweeps take half of the top level and its letters, unless there are four and more groups of a single level.  Degree 3, ns a step measured / model, one wave
// per SIMD and six: single precision, 27 channels, 27 letters 150 / 141, 678 / 667; 7 letters 134 / 125, 271 / 283; lead-lag 27 letters 108 / 94, 406 /
// 367; 34 channels, lead-lag, 34 letters 122 / 106, 491 / 445; 9 letters 147 / 133, 333 / 327; double, 32 channels, 32 letters 279 / 263, 1451 / 1450; 8
// letters 102 / 89, 462 / 442 (the measured ones with 20 ns of the launch).
struct StepModel {
    double lone, issue;         // ns: a step of a wave on its own; what each of several waves on a SIMD adds
    int64_t occ, simds;
    TreeGeom geom;
    bool backward;
    double elem;
    StepModel(const KernelEntry* e, int d, bool backward_, bool sparse_ll = false)
        : occ(std::max(1, resident_waves(e))), simds(simd_count()), geom(geom_of(e, d)), backward(backward_), elem(e->is_f64 ? 8.0 : 4.0)
    {
        double c = lane_step_cost(d, e->N, e->tail, e->k);
        const double m = double(e->N - e->tail), wide = std::max(0, d - 4), tile = std::max(0, d - 3);
        const bool f64 = e->is_f64 != 0, no_pairs = f64 && e->tail == 1;
        if (backward) {
            lone = 200.0 + 3.2 * c + 6.0 * m * m + (no_pairs ? 40.0 : 26.0) * wide;
            issue = f64 ? 50.0 + 4.6 * (c + m * m) + (no_pairs ? 40.0 * (d - 1) : 22.0 * tile) : (2.0 + 3.0 / d) * c + 2.9 * m * m + 22.0 * tile;
            if (!e->staged) lone *= 1.15;
        } else {
            const int groups = (d + e->k - 1) / e->k;
            double beyond = 0.0, guards = 0.0;
            if (d > kPointFedMaxDim && e->D > 0) {
                double letters = e->tail == 1 ? e->k : groups <= 3 ? d : d + e->k;
                if (sparse_ll && e->staged && e->fwd_lead_lag && (groups <= 3 || e->tail > 1)) {
                    c -= 0.5 * e->k * std::pow(double(d), e->tail - 1);
                    letters *= 0.5;
                }
                if (e->staged) beyond = std::max(0.0, letters - 4.0);
                if (d % e->k && groups > (e->staged ? 3 : 1)) guards = e->staged ? 55.0 : 190.0;
            }
            lone = 40.0 + 1.65 * c + (f64 ? 5.6 : 1.9) * beyond + guards;
            issue = f64 ? 24.0 + 1.8 * c + 5.2 * beyond : 14.0 + c + 2.7 * beyond;
            if (!e->staged) { lone = std::max(130.0, (e->tail >= 4 ? 1.0 : 1.15) * lone); issue += 20.0; }
            else if (guards > 0.0) issue += 10.0;
        }
        if (e->D <= 0) { lone *= 2.2; issue *= 1.5; }
    }
    double step(int64_t items) const
    {
        const int64_t fullest = (total_waves(geom, items) + simds - 1) / simds, rest = fullest % occ;
        return 1e-9 * (double(fullest / occ) * std::max(lone, issue * double(occ)) + (rest ? std::max(lone, issue * double(rest)) : 0.0));
    }
    double sweep(int64_t batch, int64_t L, int g, uint64_t sig_bytes_all_paths) const;
};

// Whole sweep in g pieces per path, beside what every call pays.  A fold launch takes 6 us (one path of 1024 points, 4 channels,
// degree 6, 16 pieces: 25 us of folds).  Backward: 10 us, and 4 to 6 us by the length of the rows for each launch of the two
// scans, beside the forward sweep of the pieces, a third of the backward's, and traffic as in choose_bwd_segments (calls of one
// path of 1024 points in 32 pieces less their sweeps: 3 channels, degree 5: 56 us; 4, 5: 71; 4, 6: 82).
double StepModel::sweep(int64_t batch, int64_t L, int g, uint64_t sig_bytes_all_paths) const
{
    int lg = 0;
    while ((1 << lg) < g) ++lg;
    const double t = double((L + g - 1) / g) * step(batch * g);
    if (g <= 1) return t;
    const double bytes = double(g) * double(sig_bytes_all_paths);
    if (!backward) return t + 2e-6 + 6e-6 * lg + 2.2 * bytes / 4e12;
    const double launch = 3.8e-6 + 0.55e-6 * std::log2(std::max(1.0, double(sig_bytes_all_paths) / (double(batch) * elem * 363.0)));
    return 1.31 * t + 10e-6 + launch * (2 * lg + 2) + bytes * (4.2e-12 + 0.64e-12 * lg);
}

// The finer partition in as many pieces as serve it best (of at least 16 steps; 256 MB of segment signatures forward, 64 MB per
// buffer backward), if that promises 8 % (backward 12 %, of whole lead-lag paths, whose steps skip half of what the estimates count, 16 %: single
// precision, 10 channels, degree 4, 147 paths of 105 points, promised 15 %: 151 -> 174 us; 11, 4, 130 of 26, 13 %: 62 -> 71) against `now`, the
// choice made without it.  On return `e` is the kernel to launch.
static SplitPlan with_fine(const KernelEntry*& e, const KernelEntry* run_now, const SplitPlan& now, bool backward, uint64_t d, uint64_t degree,
                           uint64_t batch, uint64_t L, uint64_t sig_bytes_all_paths, bool sparse_ll, int forced_pieces, bool whole_only = false)
{
    const KernelEntry* f = fine_entry(backward, e->is_f64 != 0, d, degree);
    if (!f || (forced_pieces > 0 && g_fine != 2)) return now;
    const int64_t steps = int64_t(L), paths = int64_t(batch);
    const StepModel model(f, int(d), backward, sparse_ll);
    SplitPlan best{forced_pieces > 0 ? now.pieces : 1, 0.0, 0.0};
    best.seconds = model.sweep(paths, steps, best.pieces, sig_bytes_all_paths);
    if (forced_pieces <= 0 && !whole_only) {
        const uint64_t most = uint64_t(backward ? 64 : 256) << 20;
        for (int g : {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512}) {
            if (steps / g < 16 || uint64_t(g) * sig_bytes_all_paths > most) break;
            const double t = model.sweep(paths, steps, g, sig_bytes_all_paths);
            if (t < 0.95 * best.seconds) best = SplitPlan{g, t, 0.0};
        }
    }
    if (g_fine != 2 && best.seconds > (!backward ? 0.92 : sparse_ll && best.pieces == 1 ? 0.84 : 0.88) * StepModel(run_now, int(d), backward, sparse_ll).sweep(paths, steps, now.pieces, sig_bytes_all_paths)) return now;
    tl_fine_more_pieces = tl_fine_more_pieces || best.pieces > now.pieces;
    e = f;
    return best;
}

// ---------------------------------------------------------------------------
// degree 2 in closed form (matrix cores): taken for paths of many channels, where no specialised sweep exists
// ---------------------------------------------------------------------------
static Hook g_force_degree2{-1};    // tuning hook: -1 automatic, 0 never, 1 whenever the degree is 2
static Hook g_degree2_staged{1};    // tuning hook: 0 keeps the operands of the degree-2 products out of LDS

// Measured against the sweeps for d = 3 .. 256: the backward wins everywhere (1.4x at d = 4, 20x at d = 64), the
// forward from about 12 channels on and for small dimensions whenever the sweeps cannot fill the chip.
static Hook g_force_degree3{-1};    // tuning hook: -1 automatic, 0 never, 1 whenever the degree is 3
// rows buffer [paths of a chunk][L][d^2] of the degree-3 matrix form: paths are taken in chunks that fit this many bytes
constexpr uint64_t kDeg3BufBytes = uint64_t(1) << 30;

// degree 3 as library matrix products around a scan (sig_degree3.h): two products backward, in double precision also one
// forward (1.3x at 128 channels, slower at 80; in single precision the by-row sweep on the matrix units takes half the
// products' time: 200 paths of 256 steps, 112 channels 4.4 / 2.2 ms, 128: 5.4 / 2.3).  Backward, library / by rows (which
// needs neither the library nor the rows buffer), whole calls at batch 512, length 257 (256 paths from 97 channels on):
// float32 48 channels 3.04 / 1.68 ms, 64: 3.74 / 2.31, 65: 7.00 / 9.49, 80: 8.64 / 11.7, 96: 9.07 / 14.4, 97: 6.07 / 7.25,
// 128: 9.14 / 9.87; float64 64: 6.84 / 9.77, 80: 13.4 / 34.9, 128: 25.7 / 40.8 (below 48 channels the compiled float64
// instances: 1.3x from 36).  The scan needs a wave per SIMD to be worth it (a wave: 8 rows x 64 columns of one path's
// level 2).  In float32 that line still gives the library what the by-row sweep does sooner: 96 paths of 128 channels
// 4.23 / 3.75, and short paths (32 x 16 steps, 128 channels 1.15 / 0.24; 128 x 64, 80: 1.05 / 0.93).
static bool want_degree3_gemm(uint64_t d_aug, uint64_t degree, uint64_t L, uint64_t batch, bool f64, bool backward)
{
    if (degree != 3 || d_aug < 2 || d_aug > uint64_t(kDeg3MaxDim) || L > 0x7fffffff) return false;
    // one path's rows must fit the buffer (longer paths stay with the sweeps, which need B * L * d elements)
    if (L > kDeg3BufBytes / (d_aug * d_aug * (f64 ? 8 : 4))) return false;
    if (!backward && !f64) return false;
    if (g_force_degree3 >= 0) return g_force_degree3 != 0;
    const uint64_t waves = ((d_aug + kWave - 1) / kWave) * ((d_aug + kDeg3RowsPerThread - 1) / kDeg3RowsPerThread) * batch;
    const uint64_t from = backward ? (f64 ? 36u : 65u) : 112u;
    return d_aug >= from && waves >= 1024;
}

static bool use_degree2(bool backward, uint64_t d_aug, uint64_t degree, uint64_t batch)
{
    if (degree != 2 || d_aug < 2 || d_aug > 0x7fff) return false;
    if (g_force_degree2 >= 0) return g_force_degree2 != 0;
    return backward || d_aug >= 12 || batch * 8 <= uint64_t(simd_count());
}

// Steps from which the forward kernel of sig_degree2_waves.h serves a plain path.  A block of it takes four waves and an exchange
// through LDS whatever the number of steps, which short paths do not repay, in double precision (two blocks a CU) less than in
// single; and channel counts that the TN channels of a lane do not divide cost it 2 TN loads a point.  Whole calls of 5000 paths,
// us, the kernels of sig_degree2.h / this one:
//  * up to 32 channels, 24: 8 steps 34 / 36, 16: 38 / 36; double 8: 38 / 42, 16: 45 / 42;
//  * up to 48, 40: 8 steps 44 / 51, 16: 53 / 51; double 8: 50 / 82, 24: 78 / 82, 28: 86 / 82;
//  * more, TN dividing, single: 96: 4 steps 125 / 128, 8: 136 / 128; double, TN = 3, 96: 20 steps 243 / 242, 24: 269 / 261, 32: 353 / 263,
//    TN = 4, 112: 24 steps 281 / 340, 40: 359 / 399, 56: 425 / 463, 64: 592 / 475;
//  * more, not dividing, TN = 3, 95: 24 steps 119 / 154, 48: 196 / 163; double 40 steps 273 / 360, 56: 327 / 369, 64: 446 / 370;
//  * TN = 4, one group, 61: 16 steps 48 / 58, 64: 74 / 69; double 48 steps 102 / 120, 72: 138 / 150, 80: 152 / 151; several, 111:
//    4 steps 89 / 211, 64: 290 / 298, 112: 350 / 429, 1500 paths 208 steps 1.04, 256: 0.79 of the time; double 64 steps 481 / 503, 80: 486 / 557,
//    1500 paths 136: 1.03, 144: 0.90.
static uint64_t degree2_waves_from(uint64_t d, bool f64)
{
    const uint64_t groups = (d + 63) / 64, tn = (d + 16 * groups - 1) / (16 * groups);
    if (d <= 32) return 16;
    if (d <= 48) return f64 ? 28 : 16;
    if (d % tn == 0) return !f64 ? 1 : tn == 3 ? 24 : 64;
    if (tn == 3) return f64 ? 64 : 48;
    if (groups == 1) return f64 ? 80 : 64;
    return f64 ? 140 : 224;
}

// The kernels of sig_degree2_waves.h, plain paths only.  Forward at any channel count, but beyond 48 channels not where few paths
// would have to be cut into slices (their 64 x 64 sums then meet in 16-byte pieces of atomics: 1 x 8192 points x 64 channels
// 32 -> 52 us, 16 x 4096: 39 -> 65; up to 48 it wins there too: 1 x 8000 x 8: 41 -> 31, 64 x 1000 x 32: 44 -> 32, 1 x 8000 x 48: 45 -> 41; worst of
// 250 cut shapes 2 x 8000 x 48 in double precision, 50 -> 53), nor for the shortest paths (degree2_waves_from).  Backward up to 48
// channels: with 64 the registers of A leave too few waves (2048 x 256 x 64: 124 -> 143, double 190 -> 240).
static bool degree2_by_waves(bool backward, uint64_t d, uint64_t L, uint64_t batch, size_t elem_bytes, bool augmented)
{
    if (augmented || g_degree2_staged == 0 || (L + 1) * d >= (uint64_t(1) << 31)) return false;
    if (backward) return d <= 48;
    if (g_degree2_staged == 2) return true;
    const uint64_t groups = (d + 63) / 64;
    const bool sliced = batch * groups * groups * 4 < uint64_t(simd_count()) && L >= 128;
    return L >= degree2_waves_from(d, elem_bytes == 8) && !(sliced && d > 48);
}

// Paths that one launch of those kernels takes: HIP numbers the threads of a launch with 32 bits along x, and their blocks serve
// one path each where the kernels of sig_degree2.h put four short ones into a block.
static int64_t degree2_paths_per_launch(int64_t blocks_per_path) { return std::max<int64_t>(1, ((int64_t(1) << 32) / kBlock - 1) / blocks_per_path); }

// ---------------------------------------------------------------------------
// degrees beyond the instance table: run-time-degree sweeps (sig_deep.hip)
// ---------------------------------------------------------------------------
static Hook g_force_deep{0};        // test hook: 1 takes the run-time-degree sweeps wherever they apply

static bool use_deep(uint64_t d_aug, uint64_t degree)
{
    if (!deep_supported(d_aug, degree)) return false;
    return degree > 16 || g_force_deep != 0;
}

// the reference's run-time-degree kernels stop at degree 64 (siglib/cusig/cu_signature.cu:400,3022-3025)
static void check_degree_limit(uint64_t d_aug, uint64_t degree, const char* who)
{
    if (d_aug >= 2 && degree > uint64_t(kDeepMaxDegree))
        throw std::invalid_argument(std::string(who) + " requires degree <= 64. Use CPU or reduce the truncation level.");
}

// ---------------------------------------------------------------------------
// shared argument handling
// ---------------------------------------------------------------------------
static void validate_correction(const void* correction, uint64_t correction_len, uint64_t dimension,
                                uint64_t degree, bool lead_lag)
{
    // siglib/cpsig/cp_signature.h:229-256
    if (correction == nullptr && correction_len != 0)
        throw std::invalid_argument("correction pointer is null but correction_len is nonzero");
    if (lead_lag && correction_len != 0)
        throw std::invalid_argument("correction cannot be used with lead_lag=true");
    if (correction_len == 0) return;
    if (degree < 2) throw std::invalid_argument("correction must be empty when degree < 2");
    uint64_t offset = 0, level_size = dimension;
    bool ok = false;
    for (uint64_t level = 2; level <= degree; ++level) {
        level_size *= dimension;
        offset += level_size;
        if (offset == correction_len) { ok = true; break; }
        if (offset > correction_len) break;
    }
    if (!ok) throw std::invalid_argument("correction length must be a prefix of tensor levels 2..degree");
    throw std::runtime_error("per-segment correction is not implemented in this build");
}

struct Shape {
    uint64_t d_aug, len_aug, L, full_len, stride;
};

static Shape make_shape(uint64_t dimension, uint64_t length, uint64_t degree, bool time_aug, bool lead_lag,
                        bool scalar_term)
{
    Shape s;
    s.d_aug = (lead_lag ? 2 * dimension : dimension) + (time_aug ? 1 : 0);
    s.len_aug = (lead_lag && length > 0) ? 2 * length - 1 : length;
    s.L = s.len_aug > 0 ? s.len_aug - 1 : 0;
    s.full_len = sig_length_u64(s.d_aug, degree);
    if (s.full_len == 0) throw std::overflow_error("signature length overflows 64 bits");
    s.stride = scalar_term ? s.full_len : s.full_len - 1;
    return s;
}

template <typename T, typename Z = T>
static void compute_increments(const T* path, T* inc, uint64_t batch, uint64_t dimension, uint64_t length,
                               bool time_aug, bool lead_lag, T end_time, const Shape& s, hipStream_t stream,
                               Z* zero_out = nullptr, uint64_t zero_count = 0)
{
    const T time_step = s.len_aug > 1 ? end_time / T(s.len_aug - 1) : T(0);
    (void)zero_count;       // always the whole increment gradient of the batch: batch * L * d elements
    const uint64_t per = (s.L + 2) * s.d_aug;
    launch_indexed(per, (per + 1) / 2, batch, [&](auto ix, dim3 grid) {
        using I = decltype(ix);
        hipLaunchKernelGGL((increments_kernel<T, I, Z>), grid, dim3(kBlock), 0, stream, path, inc, int64_t(batch), int64_t(length),
                           int(dimension), int(time_aug), int(lead_lag), time_step, zero_out, DivBy<I>(s.d_aug));
    });
    SIG_HIP(hipGetLastError());
}

// Everything the degree-3 matrix form needs from the device, taken before anything is launched: when the device
// cannot provide it (or rocBLAS cannot create its handle) `ok` stays false and the caller sweeps the shape instead,
// which needs B * L * d elements of workspace where this form needs up to kDeg3BufBytes more.
template <typename T>
struct Degree3Buffers {
    bool ok = false;
    uint64_t chunk = 0;     // paths per pass over the rows buffer
    T* inc = nullptr;
    T* dzinc = nullptr;     // backward only
    T* r1 = nullptr;        // backward only
    T* rows = nullptr;
    RocBlas::Handle handle = nullptr;

    void acquire(uint64_t batch, const Shape& s, hipStream_t stream, bool backward)
    {
        try {
            const uint64_t inc_elems = checked_mul(checked_mul(batch, s.L + 2, "increments"), s.d_aug, "increments");
            const uint64_t dz_elems = checked_mul(checked_mul(batch, s.L, "increments"), s.d_aug, "increments");
            const uint64_t per_path = checked_mul(checked_mul(s.L, s.d_aug * s.d_aug, "level-2 rows"), sizeof(T), "level-2 rows");
            if (per_path == 0 || per_path > kDeg3BufBytes) return;
            chunk = std::max<uint64_t>(1, std::min<uint64_t>(std::min<uint64_t>(batch, 65535), kDeg3BufBytes / per_path));
            inc = static_cast<T*>(workspace(0, checked_mul(inc_elems, sizeof(T), "increments")));
            if (backward) {
                dzinc = static_cast<T*>(workspace(1, checked_mul(dz_elems, sizeof(T), "increments")));
                r1 = static_cast<T*>(workspace(18, checked_mul(dz_elems, sizeof(T), "increments")));
            }
            rows = static_cast<T*>(workspace(19, checked_mul(chunk, per_path, "level-2 rows")));
            handle = rocblas_handle_for(stream);
            ok = true;
        } catch (const std::bad_alloc&) {
        } catch (const std::runtime_error&) {       // no rocBLAS handle
        }
    }
};

// ---------------------------------------------------------------------------
// few channels to high degrees in double precision: shared prefix chains (sig_heads.hip)
// ---------------------------------------------------------------------------
static Hook g_heads{1};     // test hook: 0 never, 1 by the estimates below, 2 wherever there is such a sweep
// the table of fractions; paths are taken in chunks that fit (test hook: cusig_amd_set_heads_table_limit)
constexpr uint64_t kHeadsTableBytes = uint64_t(1) << 30;
static std::atomic<uint64_t> g_heads_table{kHeadsTableBytes};

// Paths whose table fits, 0 if not even one's does.  A row beyond the paths' own ends the table.
static uint64_t heads_chunk(const HeadsEntry* e, uint64_t L)
{
    const uint64_t rows = g_heads_table / (uint64_t(e->row) * sizeof(double));
    return rows > 1 ? (rows - 1) / L : 0;
}

// Pieces per path of such a sweep if that promises 10 % against `now`, the sweep of `run` chosen without it; 0 if not.  Blocks run in rounds of
// what the compute units hold, chunk of paths by chunk: where a chunk is a few long paths, each of its launches leaves most of the chip idle
// (186 x 155309 x 3, degree 9, in chunks of 53: 279 ms, tree kernels 86).  A step that is shorter than a row of the table takes from memory waits for
// it once the table is too large for the last cache (tables of 120 / 500 MB, ns a step: 3 channels, degree 9, one block a compute unit 324 / 453, four 635 /
// 736; 3, 10: 311 / 438, 697 / 753; 4, 9: 462 / 533; 5, 8: 377 / 444; 11, 6: 326 / 426; 3, 12: 583 / 586).  With both counted, of 1155 random calls up
// to 300000 steps 489 take this form, 0.75 of the tree kernels' time on average.  Beside the sweep a call
// lays out the table, and its lanes store runs of a few values each.  Lead-lag twins of the tree kernels skip half of what the estimate of theirs counts.
static int heads_pieces(const HeadsEntry* e, const KernelEntry* run, const SplitPlan& now, uint64_t d, uint64_t batch, uint64_t L, uint64_t sig_bytes_all_paths,
                        bool sparse_ll)
{
    const int mode = g_heads, forced = g_force_segments;
    if (!e || mode == 0 || tl_no_fine || g_force_tail > 0 || g_force_staged >= 0 || g_ignore_table != 0 || L >= (uint64_t(1) << 30) ||
        batch > (uint64_t(1) << 40) / uint64_t(e->blocks))
        return 0;
    const uint64_t chunk = std::min(batch, heads_chunk(e, L));
    if (chunk == 0) return 0;
    if (forced > 0) return mode == 2 ? int(std::min<uint64_t>(std::min<uint64_t>(uint64_t(forced), L), uint64_t(e->most_blocks / e->blocks))) : 0;
    const int64_t cus = simd_count() / 4;
    const double wait = e->lone_ns < 500 && double(chunk) * double(L) * e->row * sizeof(double) > 140e6 ? 100.0 : 0.0;
    auto step_of = [&](uint64_t paths, int g) {      // ns of a step of one launch
        const int64_t fullest = (int64_t(paths) * g * e->blocks + cus - 1) / cus, rest = fullest % e->resident;
        return double(fullest / e->resident) * (e->step_ns + (e->resident > 2 ? 0.6 : 1.0) * wait) +
               (rest ? wait + std::max(double(e->lone_ns), double(e->step_ns) * double(rest) / e->resident) : 0.0);
    };
    auto seconds = [&](int g) {
        const double step = double(batch / chunk) * step_of(chunk, g) + step_of(batch % chunk, g);
        int lg = 0;
        while ((1 << lg) < g) ++lg;
        const double folds = g > 1 ? 2e-6 + 6e-6 * lg + 2.2 * g * double(sig_bytes_all_paths) / 4e12 : 0.0;
        return 12e-6 + double((L + g - 1) / g) * step * 1e-9 + double(batch * L) * e->row * 8.0 / 3e12 + double(sig_bytes_all_paths) * g / 4e12 + folds;
    };
    int best = 1;
    double best_t = seconds(1);
    for (int g : {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64}) {
        if (L / uint64_t(g) < 48 || uint64_t(g) * sig_bytes_all_paths > (uint64_t(256) << 20)) break;
        const double t = seconds(g);
        if (t < 0.95 * best_t) { best = g; best_t = t; }
    }
    if (mode == 2) return best;
    double old = StepModel(run, int(d), false, sparse_ll).sweep(int64_t(batch), int64_t(L), now.pieces, sig_bytes_all_paths);
    if (sparse_ll && run->staged && run->fwd_lead_lag) old *= 0.6;
    return best_t < 0.9 * old ? best : 0;
}

// ---------------------------------------------------------------------------
// forward  (dispatch mirrors siglib/cpsig/cp_signature.h:740-851 and
// siglib/cusig/cu_signature.cu:2592-2657)
// ---------------------------------------------------------------------------
template <typename T>
static void signature_impl(const T* path, T* out, uint64_t batch, uint64_t dimension, uint64_t length,
                           uint64_t degree, bool time_aug, bool lead_lag, T end_time, bool /*horner*/,
                           bool scalar_term, const T* correction, uint64_t correction_len)
{
    if (dimension == 0) throw std::invalid_argument("signature_cuda received path of dimension 0");
    validate_correction(correction, correction_len, dimension, degree, lead_lag);
    if (batch == 0) return;
    if (dimension > 0x3fffffff || degree > 0x7fffffff || length > (uint64_t(1) << 40))
        throw std::invalid_argument("signature_cuda: shape out of range");
    const Shape s = make_shape(dimension, length, degree, time_aug, lead_lag, scalar_term);
    check_degree_limit(s.d_aug, degree, "signature on this GPU build");
    checked_mul(checked_mul(batch, s.stride, "signature output"), sizeof(T), "signature output");
    hipStream_t stream = nullptr;
    entry_sync();   // inputs may have been produced on any stream

    // everything below runs under the workspace mutex: one flag serves all callers
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    tl_sig_nonfinite = -1;
    tl_matrix_form = 0;
    int* flag = nullptr;
    if (!g_stream_ordered) {
        flag = nonfinite_flag();
        *g_flag_host = 0;
    }

    const int sc = scalar_term ? 1 : 0;
    Degree3Buffers<T> d3;
    if (s.len_aug > 1 && s.d_aug > 1 && want_degree3_gemm(s.d_aug, degree, s.L, batch, sizeof(T) == 8, false) && rocblas_ready())
        d3.acquire(batch, s, stream, false);
    if (s.len_aug <= 1) {
        if (s.stride)
            hipLaunchKernelGGL((fill_trivial_kernel<T>), dim3(grid_for(batch * s.stride)), dim3(kBlock), 0, stream,
                               out, int64_t(batch), int64_t(s.stride), sc);
    } else if (degree == 0) {
        if (scalar_term)
            hipLaunchKernelGGL((fill_trivial_kernel<T>), dim3(grid_for(batch)), dim3(kBlock), 0, stream, out,
                               int64_t(batch), int64_t(1), 1);
    } else if (s.d_aug == 1) {
        hipLaunchKernelGGL((dim_one_fwd_kernel<T>), dim3(grid_for(batch)), dim3(kBlock), 0, stream, path, out,
                           int64_t(batch), int64_t(length), int(degree), sc, flag);
    } else if (degree == 1) {
        const T time_step = end_time / T(s.len_aug - 1);
        hipLaunchKernelGGL((degree_one_fwd_kernel<T>), dim3(grid_for(batch * s.stride)), dim3(kBlock), 0, stream,
                           path, out, int64_t(batch), int64_t(length), int(dimension), int(time_aug),
                           int(lead_lag), time_step, sc, flag);
    } else if (d3.ok) {
        if constexpr (sizeof(T) == 8) {      // single precision: the by-row sweep on the matrix units
            const int d = int(s.d_aug);
            const int64_t L = int64_t(s.L);
            const uint64_t chunk = d3.chunk;
            T* inc = d3.inc;
            T* rows = d3.rows;
            compute_increments(path, inc, batch, dimension, length, time_aug, lead_lag, end_time, s, stream);
            RocBlas::Handle h = d3.handle;
            tl_last_segments = 1;
            MainKernelTimer timer(stream, "degree3_fwd_gemm_f64");
            const int64_t dd = int64_t(d) * d;
            const int groups = (d + kDeg3RowsPerThread - 1) / kDeg3RowsPerThread;
            for (uint64_t first = 0; first < batch; first += chunk) {
                const int nb = int(std::min<uint64_t>(chunk, batch - first));
                const dim3 sgrid(unsigned((d + kWave - 1) / kWave), unsigned(nb), unsigned((groups + kWavesPerBlock - 1) / kWavesPerBlock));
                hipLaunchKernelGGL((degree3_fwd_scan_kernel<T>), sgrid, dim3(kBlock), 0, stream, (const T*)inc, rows, out, L, d,
                                   int64_t(s.stride), sc, int64_t(first));
                // level 3 (row-major d^2 x d) = V^T Z; column-major: [d x d^2] = Z^T (stored: d x L) * (V^T stored: d^2 x L)^T
                gemm_col_major<T>(h, false, true, d, int(dd), int(L), inc + (first * (s.L + 2) + 1) * s.d_aug, d, (L + 2) * d,
                                  (const T*)rows, int(dd), L * dd, T(0), out + first * s.stride + sc + d + dd, d, int64_t(s.stride), nb);
            }
            timer.stop();
            if (flag)
                hipLaunchKernelGGL((finite_rows_kernel<T>), dim3(grid_for(batch * s.stride)), dim3(kBlock), 0, stream, out,
                                   int64_t(batch * s.stride), flag);
        }
    } else if (use_degree2(false, s.d_aug, degree, batch) && degree2_by_waves(false, s.d_aug, s.L, batch, sizeof(T), time_aug || lead_lag)) {
        const int d = int(s.d_aug), groups = (d + 63) / 64, tn = (d + 16 * groups - 1) / (16 * groups);
        // few paths: two blocks per CU through slices of the steps, at least 64 steps each, that add into the cleared output
        const int64_t whole = int64_t(batch) * groups * groups;
        int64_t slices = whole * 4 >= simd_count() ? 1 : std::min<int64_t>(simd_count() / (2 * whole), int64_t(s.L) / 64);
        slices = std::max<int64_t>(slices, 1);
        const int64_t slice_len = (int64_t(s.L) + slices - 1) / slices;
        slices = (int64_t(s.L) + slice_len - 1) / slice_len;
        const int64_t per_path = int64_t(groups) * groups * slices, most = degree2_paths_per_launch(per_path);
        if (slices > 1)
            hipLaunchKernelGGL((zero_kernel<T>), dim3(grid_for(batch * s.stride)), dim3(kBlock), 0, stream, out,
                               int64_t(batch * s.stride));
        MainKernelTimer timer(stream, sizeof(T) == 8 ? "degree2_fwd_f64_waves" : "degree2_fwd_f32_waves");
        auto go = [&](auto tiles, auto same) {
            constexpr int TN = decltype(tiles)::value;
            auto run = [&](auto whole_pieces) {
                for (int64_t first = 0; first < int64_t(batch); first += most)
                    hipLaunchKernelGGL((degree2_fwd_waves_kernel<T, TN, decltype(same)::value, decltype(whole_pieces)::value>),
                                       dim3(unsigned(std::min(most, int64_t(batch) - first) * per_path)), dim3(kBlock), 0, stream,
                                       path + first * int64_t(length) * d, out + first * int64_t(s.stride), int64_t(length), d, int64_t(s.stride),
                                       sc, groups, int(slices), slice_len, slices > 1 ? nullptr : flag);
            };
            if (d % TN == 0) run(std::true_type{});
            else run(std::false_type{});
        };
        auto pick = [&](auto same) {
            if (tn == 1) go(IntC<1>{}, same);
            else if (tn == 2) go(IntC<2>{}, same);
            else if (tn == 3) go(IntC<3>{}, same);
            else go(IntC<4>{}, same);
        };
        if (groups == 1) pick(std::true_type{});
        else if (tn <= 3) go(IntC<3>{}, std::false_type{});
        else go(IntC<4>{}, std::false_type{});
        timer.stop();
        if (slices > 1 && flag)
            hipLaunchKernelGGL((finite_rows_kernel<T>), dim3(grid_for(batch * s.stride)), dim3(kBlock), 0, stream, out,
                               int64_t(batch * s.stride), flag);
    } else if (use_degree2(false, s.d_aug, degree, batch)) {
        const int d = int(s.d_aug);
        const int tiles = (d + 15) / 16, col_groups = (tiles + kDeg2Cols - 1) / kDeg2Cols;
        const int64_t waves = int64_t(batch) * tiles * col_groups;
        // A wave walks its time range four steps per iteration, each iteration waiting for its loads: long ranges are
        // cut into slices that add into the output with atomics (d^2 atomics per slice against slice_len * d^2
        // products).  Few paths: enough slices for two waves per SIMD; otherwise slices of 256 steps.
        int64_t slices = waves * 2 <= simd_count() ? std::min<int64_t>(2 * simd_count() / waves, int64_t(s.L) / 64)
                                                   : int64_t(s.L) / 256;
        slices = std::max<int64_t>(slices, 1);
        const int64_t slice_len = ((int64_t(s.L) + slices - 1) / slices + 3) / 4 * 4;
        slices = (int64_t(s.L) + slice_len - 1) / slice_len;
        if (slices > 1)
            hipLaunchKernelGGL((zero_kernel<T>), dim3(grid_for(batch * s.stride)), dim3(kBlock), 0, stream, out,
                               int64_t(batch * s.stride));
        const T time_step = end_time / T(s.len_aug - 1);
        // points staged through LDS: slabs of 4 * rq + 1 points by 64 channels, rq odd, at most 43 KB a slab; chunks of
        // equal length
        const size_t row_bytes = size_t(kDeg2SlabStride) * sizeof(T);
        const bool two_slabs = tiles > kWavesPerBlock;      // row and column channels of a block can differ
        const int rq_max = (sizeof(T) == 8 ? 15 : 33) / (two_slabs ? 2 : 1) | 1;
        const int64_t n_chunks = (slice_len + 4 * rq_max - 1) / (4 * rq_max);
        int rq = int((slice_len + 4 * n_chunks - 1) / (4 * n_chunks));
        rq = std::min(rq | 1, rq_max);
        const bool vec = !time_aug && !lead_lag && dimension % (16 / sizeof(T)) == 0 && reinterpret_cast<uintptr_t>(path) % 16 == 0 &&
                         4 * rq + 1 <= deg2_prefetch_rows<T>();
        // with fewer than four row tiles some of a block's waves would idle and its slabs be mostly padding (measured:
        // d = 64..256 1.4-1.5x faster staged, d <= 32 up to 3x slower)
        const bool staged = g_degree2_staged != 0 && tiles >= kWavesPerBlock;
        MainKernelTimer timer(stream, sizeof(T) == 8 ? (staged ? "degree2_fwd_f64_lds" : "degree2_fwd_f64")
                                                     : (staged ? "degree2_fwd_f32_lds" : "degree2_fwd_f32"));
        if (staged) {
            const int64_t row_groups = (tiles + kWavesPerBlock - 1) / kWavesPerBlock;
            const int64_t blocks = int64_t(batch) * row_groups * col_groups * slices;
            if (blocks > 2147483647LL) throw std::runtime_error("signature_cuda: launch too large");
            auto go = [&](auto mode) {
                hipLaunchKernelGGL((degree2_fwd_staged_kernel<T, decltype(mode)::value>), dim3(unsigned(blocks)), dim3(kBlock),
                                   size_t(4 * rq + 1) * row_bytes * (two_slabs ? 2 : 1), stream, path, out,
                                   int64_t(batch), int64_t(length), int(dimension), int(time_aug), int(lead_lag), time_step,
                                   int64_t(s.stride), sc, tiles, col_groups, int(slices), slice_len, rq,
                                   slices > 1 ? nullptr : flag);
            };
            if (vec) go(std::integral_constant<int, 2>());
            else if (!time_aug && !lead_lag) go(std::integral_constant<int, 1>());
            else go(std::integral_constant<int, 0>());
        } else {
            const int64_t total = waves * slices;
            const int64_t blocks = (total + kWavesPerBlock - 1) / kWavesPerBlock;
            if (blocks > 2147483647LL) throw std::runtime_error("signature_cuda: launch too large");
            hipLaunchKernelGGL((degree2_fwd_kernel<T>), dim3(unsigned(blocks)), dim3(kBlock), 0, stream, path, out, int64_t(batch),
                               int64_t(length), int(dimension), int(time_aug), int(lead_lag), time_step, int64_t(s.stride), sc,
                               tiles, col_groups, int(slices), slice_len, slices > 1 ? nullptr : flag);
        }
        timer.stop();
        if (slices > 1 && flag)
            hipLaunchKernelGGL((finite_rows_kernel<T>), dim3(grid_for(batch * s.stride)), dim3(kBlock), 0, stream, out,
                               int64_t(batch * s.stride), flag);
    } else if (use_deep(s.d_aug, degree)) {
        if (!deep_fits(s.d_aug, degree, batch)) throw std::runtime_error("signature_cuda: launch too large");
        const uint64_t inc_elems = checked_mul(checked_mul(batch, s.L + 2, "increments"), s.d_aug, "increments");
        T* inc = static_cast<T*>(workspace(0, checked_mul(inc_elems, sizeof(T), "increments")));
        compute_increments(path, inc, batch, dimension, length, time_aug, lead_lag, end_time, s, stream);
        FwdParams p;
        p.inc = inc; p.out = out; p.batch = int64_t(batch); p.L = int64_t(s.L); p.d = int(s.d_aug); p.out_stride = int64_t(s.stride);
        p.scalar = sc; p.stream = stream; p.nseg = 1; p.lseg = int64_t(s.L); p.nonfinite = flag;
        tl_last_segments = 1;
        MainKernelTimer timer(stream, sizeof(T) == 8 ? "deep_fwd_f64" : "deep_fwd_f32");
        SIG_HIP(launch_deep_fwd<T>(p, int(degree)));
        timer.stop();
    } else {
        const KernelEntry* e = choose_entry(false, sizeof(T) == 8, s.d_aug, degree, batch, s.L);
        if (!e)
            throw std::runtime_error("signature_cuda: no kernel for dimension " + std::to_string(s.d_aug) +
                                     ", degree " + std::to_string(degree) + " in this build");
        // Few paths cannot fill the chip with whole-path sweeps: split every path into time segments,
        // sweep all (path, segment) pairs concurrently and fold the pieces with Chen's identity.
        // lead-lag sweeps that skip the letters a step cannot move take the step's parity from its position in the
        // segment: segments start on even steps
        const bool sparse_ll = lead_lag && g_lead_lag_sparse != 0;
        // many channels: the by-row sweep, whole paths only.  Without a compiled instance always: in double precision
        // 1.0-1.46x faster than the general run-time kernels (16 / 32 letters per lane) at 33 .. 96 channels, degrees 4 to 6;
        // in single precision, on the matrix units and bit for bit the same (16 paths of 200 steps, 64 channels, degree 4:
        // 2.60 -> 1.27 ms; 5 x 64, 70: 0.89 -> 0.48; 2 x 50, 33, degree 5: 0.69 -> 0.43).  In place of an instance in single
        // precision, where its tiles of 32 x 32 are filled well enough (256 x 256, 64 channels, degree 3: 0.94 -> 0.39 ms;
        // 300 x 200, 96: 2.05 -> 1.39; 8 x 100, 48, degree 4: 0.28 -> 0.22; but 64 x 200, 40, degree 4, 39 % filled:
        // 1.20 -> 1.83) and, at degree 3, the estimates say so (at degree 4 it won at every size tried: one path of 8000 steps,
        // 48 channels 2.40 -> 2.11, two 4.37 -> 3.48).  Lead-lag paths of that many channels have no instance that skips the
        // letters a step cannot move (those end at 40), so the same holds for them (degree 3, 200 paths of 129 points, 60
        // channels, 120 augmented: 8.72 -> 2.11 ms, 4.42 as library products; 100 x 129 x 64: 2.90 -> 1.14, 2.41).
        int64_t instance_waves = total_waves(geom_of(e, int(s.d_aug)), int64_t(batch));
        auto split = [&]() -> SplitPlan {
            if (g_force_segments > 0) return {int(std::min<uint64_t>(uint64_t(g_force_segments), s.L)), 0.0, 0.0};
            return choose_segments(instance_waves, int64_t(s.L), resident_waves(e), batch * (s.full_len - 1) * sizeof(T),
                                   [&](int g) {
                                       const double c = lane_step_cost(int(s.d_aug), e->N, e->tail, e->k) * 2.4e-9;
                                       const bool ring = pick_variant(false, e, instance_waves * g, sparse_ll)->staged;
                                       return ring ? c : std::max(c, 240e-9);
                                   },
                                   sizeof(T) == 8);
        };
        const uint64_t tile = (s.d_aug + 31) / 32 * 32;
        const int rows_mode = g_rows_forward;
        bool by_rows = rows_mode != 0 && g_force_tail == 0 && rows_fwd_supported(sizeof(T), s.d_aug, degree) &&
                       rows_fits(sizeof(T), s.d_aug, degree, batch);
        if (rows_mode == 1 && e->D > 0) by_rows = by_rows && sizeof(T) == 4 && g_force_segments == 0 && 16 * s.d_aug * s.d_aug >= 9 * tile * tile;
        SplitPlan plan{1, 0.0, 0.0};
        const bool compare = by_rows && rows_mode == 1 && e->D > 0 && degree == 3;
        if (!by_rows || compare) plan = split();
        if (compare) {
            const KernelEntry* run = pick_variant(false, e, instance_waves * plan.pieces, sparse_ll);
            by_rows = rows_fwd_seconds(s.d_aug, batch, s.L) < instance_fwd_seconds(run, plan, instance_waves, s.d_aug, s.L);
        }
        const uint64_t n_coef = s.full_len - 1;
        auto finer = [&]() {
            return with_fine(e, pick_variant(false, e, instance_waves * plan.pieces, sparse_ll), plan, false, s.d_aug, degree, batch, s.L,
                             batch * n_coef * sizeof(T), sparse_ll, g_force_segments);
        };
        if (!by_rows) {
            plan = finer();
            if (const KernelEntry* spec = instance_after_all(e, false, s.d_aug, degree, batch, s.L)) {
                e = spec;
                instance_waves = total_waves(geom_of(e, int(s.d_aug)), int64_t(batch));
                const int before = plan.pieces;
                plan = split();
                plan = finer();
                tl_fine_more_pieces = tl_fine_more_pieces || plan.pieces > before;
            }
        }
        const HeadsEntry* heads = sizeof(T) == 8 && !by_rows ? heads_entry(s.d_aug, degree) : nullptr;
        if (heads) {
            const KernelEntry* run = pick_variant(false, e, total_waves(geom_of(e, int(s.d_aug)), int64_t(batch) * plan.pieces), sparse_ll);
            const int pieces = heads_pieces(heads, run, plan, s.d_aug, batch, s.L, batch * n_coef * sizeof(T), sparse_ll);
            if (pieces > 0) {
                plan = SplitPlan{pieces, 0.0, 0.0};
                tl_fine_more_pieces = true;         // needs memory that the tree kernels do not
            } else {
                heads = nullptr;
            }
        }
        int nseg = by_rows ? 1 : plan.pieces;
        FwdParams p;
        p.batch = int64_t(batch) * nseg; p.L = int64_t(s.L); p.d = int(s.d_aug); p.stream = stream;
        p.lseg = (int64_t(s.L) + nseg - 1) / nseg;
        if (sparse_ll) p.lseg += p.lseg & 1;
        nseg = int((int64_t(s.L) + p.lseg - 1) / p.lseg);      // drop segments the rounding left empty
        p.nseg = nseg;
        tl_last_segments = nseg;
        p.batch = int64_t(batch) * nseg;
        T* segs = nullptr;
        T* folds = nullptr;
        if (nseg == 1) {
            p.out = out; p.out_stride = int64_t(s.stride); p.scalar = sc; p.nonfinite = flag;
        } else {
            const uint64_t row_elems = checked_mul(batch, n_coef, "segment signatures");
            const uint64_t bytes = checked_mul(checked_mul(row_elems, uint64_t(nseg), "segment signatures"), sizeof(T), "segment signatures");
            segs = static_cast<T*>(workspace(2, bytes));
            // every halving step's rows, one step after the other: at most nseg + log2(nseg) rows per path
            if (nseg > 2)
                folds = static_cast<T*>(workspace(3, checked_mul(checked_mul(row_elems, uint64_t(nseg) + 32, "segment signatures"),
                                                                 sizeof(T), "segment signatures")));
            p.out = segs; p.out_stride = int64_t(n_coef); p.scalar = 0;
        }
        e = pick_variant(false, e, total_waves(geom_of(e, int(s.d_aug)), p.batch), sparse_ll);
        // staged sweeps of plain narrow paths form the increments themselves while staging the points
        if (!by_rows && !heads && e->staged && !time_aug && !lead_lag && e->D > 0 && e->D <= kPointFedMaxDim && g_point_fed) {
            p.inc = path;
            p.from_points = 1;
        } else {
            const uint64_t inc_elems = checked_mul(checked_mul(batch, s.L + 2, "increments"), s.d_aug, "increments");
            const uint64_t pad = uint64_t(kStageSteps + 2) * s.d_aug;    // staged sweeps read whole chunks past either end
            T* inc = static_cast<T*>(workspace(0, checked_mul(inc_elems + 2 * pad, sizeof(T), "increments"))) + pad;
            compute_increments(path, inc, batch, dimension, length, time_aug, lead_lag, end_time, s, stream);
            p.inc = inc;
        }
        const bool use_ll = !by_rows && !heads && sparse_ll && e->staged && e->fwd_lead_lag && !p.from_points;
        const std::string shown = heads ? "heads_fwd_f64_d" + std::to_string(heads->D) + "_n" + std::to_string(degree)
                                  : by_rows ? std::string(sizeof(T) == 8 ? "rows_fwd_f64_n" : "rows_fwd_f32_n") + std::to_string(degree)
                                  : use_ll ? std::string(e->name) + "_ll" : std::string(e->name);
        MainKernelTimer timer(stream, shown.c_str());
        tl_matrix_form = by_rows && sizeof(T) == 4;
        if (heads) {
            const uint64_t path_bytes = s.L * uint64_t(heads->row) * sizeof(T);
            const uint64_t launch = uint64_t(heads->most_blocks) / (uint64_t(heads->blocks) * uint64_t(p.nseg));      // the memory ends sooner
            const uint64_t chunk = std::min({batch, heads_chunk(heads, s.L), launch});
            HeadsParams hp;
            hp.table = workspace(kHeadsSlot, chunk * path_bytes + uint64_t(heads->row) * sizeof(T));
            hp.L = p.L; hp.out_stride = p.out_stride; hp.scalar = p.scalar; hp.nseg = p.nseg; hp.lseg = p.lseg; hp.nonfinite = p.nonfinite;
            hp.stream = stream;
            for (uint64_t first = 0; first < batch; first += chunk) {
                hp.inc = static_cast<const T*>(p.inc) + first * (s.L + 2) * s.d_aug;
                hp.out = static_cast<T*>(p.out) + first * uint64_t(p.nseg) * uint64_t(p.out_stride);
                hp.paths = int64_t(std::min<uint64_t>(chunk, batch - first));
                SIG_HIP(heads->launch(hp));
            }
        } else if (by_rows) SIG_HIP(sizeof(T) == 4 ? launch_rows_fwd_mfma(p, int(degree)) : launch_rows_fwd_f64(p, int(degree)));
        else SIG_HIP(use_ll ? e->fwd_lead_lag(p) : e->fwd(p));
        timer.stop(/*defer=*/true);
        if (nseg > 1) {
            // ordered product of the segment signatures by pairwise halving: ceil(log2(nseg)) launches.  An unpaired last
            // row stays where it is and joins the next step as its last row (`carry`).
            const T* src = segs;
            int src_rows = nseg;
            const T* carry = nullptr;
            int64_t carry_stride = 0;
            T* next = folds;
            for (int m = nseg; m > 1;) {
                const bool last = m == 2;
                const int pairs = m / 2;
                T* dst = last ? out : next;
                with_chen_fan(s.d_aug, [&](auto fan) {
                    constexpr int FAN = decltype(fan)::value;
                    const uint64_t items = chen_items(s.d_aug, degree, FAN);
                    launch_indexed(n_coef, items, batch * uint64_t(pairs), [&](auto ix, dim3 grid) {
                        using I = decltype(ix);
                        hipLaunchKernelGGL((chen_fold_step_kernel<T, I, FAN>), grid, dim3(kBlock), 0, stream, src, src_rows, carry,
                                           carry_stride, dst, int64_t(batch), m, last ? int64_t(s.stride) : int64_t(n_coef) * pairs,
                                           last ? sc : 0, DivBy<I>(s.d_aug), I(n_coef), I(items), last ? flag : nullptr);
                    });
                });
                SIG_HIP(hipGetLastError());
                if (m & 1) {
                    if (!carry) {       // the last row of this step's source becomes the carry
                        carry = src + uint64_t(m - 1) * n_coef;
                        carry_stride = int64_t(src_rows) * int64_t(n_coef);
                    }
                } else {
                    carry = nullptr;    // paired in this step, if there was one
                }
                src = dst;
                src_rows = pairs;
                next += batch * n_coef * uint64_t(pairs);
                m = pairs + (carry ? 1 : 0);
            }
        }
        exit_sync(stream);
        timer.read();
        if (flag) tl_sig_nonfinite = *g_flag_host;
        return;
    }
    SIG_HIP(hipGetLastError());
    exit_sync(stream);
    if (flag) tl_sig_nonfinite = *g_flag_host;
}

// ---------------------------------------------------------------------------
// backward  (siglib/cpsig/cp_signature.h:909-1019, siglib/cusig/cu_signature.cu:3417-3488)
// ---------------------------------------------------------------------------
// increment gradient -> raw path gradient; plain paths with a channel count that allows it take 16 bytes per lane
template <typename T, typename Z = T>
static void launch_path_grad(const Z* dzinc, T* out, uint64_t batch, uint64_t length, uint64_t dimension, bool time_aug,
                             bool lead_lag, hipStream_t stream, Z* clear = nullptr, uint64_t clear_count = 0)
{
    constexpr int V = int(16 / sizeof(T));
    if (!time_aug && !lead_lag && dimension % V == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
        reinterpret_cast<uintptr_t>(dzinc) % sizeof(VecOf<Z, V>) == 0) {
        const uint64_t per = length * (dimension / V);
        launch_indexed(per, per, batch, [&](auto ix, dim3 grid) {
            using I = decltype(ix);
            hipLaunchKernelGGL((path_grad_vec_kernel<T, Z, I, V>), grid, dim3(kBlock), 0, stream, dzinc, out, int64_t(batch),
                               int64_t(length), DivBy<I>(dimension / V), clear, int64_t(clear_count));
        });
        return;
    }
    launch_indexed(length * dimension, (length * dimension + 1) / 2, batch, [&](auto ix, dim3 grid) {
        using I = decltype(ix);
        hipLaunchKernelGGL((path_grad_kernel<T, Z, I>), grid, dim3(kBlock), 0, stream, dzinc, out, int64_t(batch),
                           int64_t(length), int(time_aug), int(lead_lag), DivBy<I>(dimension), clear, int64_t(clear_count));
    });
}

// A caller-independent block of device memory that a call carves its buffers out of instead of the workspace pool
// (the entry point that must not allocate).  With an arena the call only enqueues on `stream`: no waits, no events,
// whole-path sweeps only (a time split would need buffers of several signature sets).
struct Arena {
    char* base = nullptr;
    size_t bytes = 0, used = 0;
    hipStream_t stream = nullptr;
    void* take(size_t n)
    {
        const size_t off = (used + 255) & ~size_t(255);
        if (off > bytes || n > bytes - off)
            throw std::invalid_argument("this shape needs more than the " + std::to_string(bytes >> 20) +
                                        " MiB of built-in scratch memory; use sig_backprop_cuda_d");
        used = off + n;
        return base + off;
    }
};

template <typename T>
static void sig_backprop_impl(const T* path, T* out, const T* sig_derivs, const T* sig, uint64_t batch,
                              uint64_t dimension, uint64_t length, uint64_t degree, bool time_aug,
                              bool lead_lag, T end_time, bool scalar_term, const T* correction,
                              uint64_t correction_len, Arena* arena = nullptr)
{
    if (dimension == 0) throw std::invalid_argument("sig_backprop_cuda received path of dimension 0");
    validate_correction(correction, correction_len, dimension, degree, lead_lag);
    if (batch == 0) return;
    if (dimension > 0x3fffffff || degree > 0x7fffffff || length > (uint64_t(1) << 40))
        throw std::invalid_argument("sig_backprop_cuda: shape out of range");
    const Shape s = make_shape(dimension, length, degree, time_aug, lead_lag, scalar_term);
    check_degree_limit(s.d_aug, degree, "sig_backprop on this GPU build");
    const uint64_t out_elems = checked_mul(checked_mul(batch, length, "path gradient"), dimension, "path gradient");
    hipStream_t stream = arena ? arena->stream : nullptr;
    if (!arena) entry_sync();
    const int sc = scalar_term ? 1 : 0;
    // library buffers: the grow-only pool (under its mutex), or the caller-independent arena
    auto buffer = [&](int slot, uint64_t bytes) -> void* { return arena ? arena->take(bytes) : workspace(slot, bytes); };
    auto finish = [&] { if (!arena) exit_sync(stream); };
    std::unique_lock<std::mutex> lk(g_ws_mutex, std::defer_lock);
    auto lock_pool = [&] { if (!arena && !lk.owns_lock()) lk.lock(); };
    tl_matrix_form = 0;
    Degree3Buffers<T> d3;
    if (!arena && s.len_aug > 1 && want_degree3_gemm(s.d_aug, degree, s.L, batch, sizeof(T) == 8, true)) {
        lock_pool();
        if (rocblas_ready()) d3.acquire(batch, s, stream, true);
    }
    const bool degree3 = d3.ok;

    if (s.len_aug <= 1 || degree == 0) {
        if (out_elems)
            hipLaunchKernelGGL((zero_kernel<T>), dim3(grid_for(out_elems)), dim3(kBlock), 0, stream, out,
                               int64_t(out_elems));
    } else if (degree == 1) {
        hipLaunchKernelGGL((degree_one_bwd_kernel<T>), dim3(grid_for(out_elems)), dim3(kBlock), 0, stream,
                           sig_derivs, out, int64_t(batch), int64_t(length), int(dimension), int(time_aug),
                           int(lead_lag), sc);
    } else if (degree3) {
        const int d = int(s.d_aug);
        const int64_t L = int64_t(s.L);
        const uint64_t dz_elems = checked_mul(checked_mul(batch, s.L, "increments"), s.d_aug, "increments");
        const uint64_t chunk = d3.chunk;
        T* inc = d3.inc;
        T* dzinc = d3.dzinc;
        T* r1 = d3.r1;
        T* rows = d3.rows;
        compute_increments(path, inc, batch, dimension, length, time_aug, lead_lag, end_time, s, stream, dzinc, dz_elems);
        hipLaunchKernelGGL((zero_kernel<T>), dim3(grid_for(dz_elems)), dim3(kBlock), 0, stream, r1, int64_t(dz_elems));
        RocBlas::Handle h = d3.handle;
        MainKernelTimer timer(stream, sizeof(T) == 8 ? "degree3_bwd_gemm_f64" : "degree3_bwd_gemm_f32", true);
        const int64_t dd = int64_t(d) * d;
        const int groups = (d + kDeg3RowsPerThread - 1) / kDeg3RowsPerThread;
        for (uint64_t first = 0; first < batch; first += chunk) {
            const int nb = int(std::min<uint64_t>(chunk, batch - first));
            const T* g3 = sig_derivs + first * s.stride + sc + d + dd;
            // Y = Z G3^T
            gemm_row_major<T>(h, true, int(L), int(dd), d, inc + (first * (s.L + 2) + 1) * s.d_aug, d, (L + 2) * d, g3, d,
                              int64_t(s.stride), T(0), rows, int(dd), L * dd, nb);
            const dim3 sgrid(unsigned((d + kWave - 1) / kWave), unsigned(nb), unsigned((groups + kWavesPerBlock - 1) / kWavesPerBlock));
            hipLaunchKernelGGL((degree3_scan_kernel<T>), sgrid, dim3(kBlock), 0, stream, (const T*)inc, sig, sig_derivs, rows, dzinc, r1,
                               L, d, int64_t(s.stride), sc, int64_t(first));
            // dz += V G3
            gemm_row_major<T>(h, false, int(L), d, int(dd), (const T*)rows, int(dd), L * dd, g3, d, int64_t(s.stride), T(1),
                              dzinc + first * s.L * s.d_aug, d, L * d, nb);
        }
        hipLaunchKernelGGL((degree3_level1_kernel<T>), dim3(grid_for(batch * s.d_aug)), dim3(kBlock), 0, stream, sig_derivs, (const T*)r1,
                           dzinc, int64_t(batch), L, d, int64_t(s.stride), sc);
        timer.stop();
        launch_path_grad<T>(dzinc, out, batch, length, dimension, time_aug, lead_lag, stream);
        SIG_HIP(hipGetLastError());
        finish();
        return;
    } else if (!arena && use_degree2(true, s.d_aug, degree, batch) &&
               degree2_by_waves(true, s.d_aug, s.L, batch, sizeof(T), time_aug || lead_lag)) {
        lock_pool();        // (the timer's events)
        const int d = int(s.d_aug), tn = (d + 15) / 16;
        // two blocks per CU at least, of 64 rows (four waves of 16) and more each
        const int64_t chunks = (int64_t(length) + 63) / 64;
        int64_t parts = std::min<int64_t>(chunks, std::max<int64_t>(1, (simd_count() / 2 + int64_t(batch) - 1) / int64_t(batch)));
        const int64_t part_rows = (chunks + parts - 1) / parts * 64;
        parts = (int64_t(length) + part_rows - 1) / part_rows;
        const int64_t most = degree2_paths_per_launch(parts);
        MainKernelTimer timer(stream, sizeof(T) == 8 ? "degree2_bwd_f64_waves" : "degree2_bwd_f32_waves");
        auto go = [&](auto tiles) {
            auto run = [&](auto whole_pieces) {
                for (int64_t first = 0; first < int64_t(batch); first += most)
                    hipLaunchKernelGGL((degree2_bwd_waves_kernel<T, decltype(tiles)::value, decltype(whole_pieces)::value>),
                                       dim3(unsigned(std::min(most, int64_t(batch) - first) * parts)), dim3(kBlock), 0, stream,
                                       path + first * int64_t(length) * d, sig_derivs + first * int64_t(s.stride), out + first * int64_t(length) * d,
                                       int64_t(length), d, int64_t(s.stride), sc, int(parts), part_rows);
            };
            if (d % 4 == 0) run(std::true_type{});
            else run(std::false_type{});
        };
        if (tn == 1) go(IntC<1>{});
        else if (tn == 2) go(IntC<2>{});
        else go(IntC<3>{});
        timer.stop();
    } else if (use_degree2(true, s.d_aug, degree, batch)) {
        lock_pool();
        const int d = int(s.d_aug);
        const uint64_t dz_elems = checked_mul(checked_mul(batch, s.L, "increments"), s.d_aug, "increments");
        T* dzinc = static_cast<T*>(buffer(1, checked_mul(dz_elems, sizeof(T), "increments")));
        T* h = static_cast<T*>(buffer(12, checked_mul(checked_mul(batch, s.d_aug, "increments"), sizeof(T), "increments")));
        const int tiles = (d + 15) / 16, col_groups = (tiles + kDeg2Cols - 1) / kDeg2Cols;
        // operands staged through LDS when a block's four waves all have 16 steps to work on and the channels fill the
        // 64-wide slabs (measured: d = 64, 256 1.6-1.75x faster staged, d = 100 equal, d <= 32 up to 2.5x slower)
        const bool staged = g_degree2_staged != 0 && tiles >= kWavesPerBlock && s.L >= 48;
        T* anti = staged ? static_cast<T*>(buffer(13, checked_mul(checked_mul(batch, s.d_aug * s.d_aug, "level-2 gradient"), sizeof(T),
                                                                  "level-2 gradient")))
                         : nullptr;
        const T time_step = end_time / T(s.len_aug - 1);
        if (g_degree2_staged != 0 && tiles >= 3 && tiles <= kDeg2Cols && s.L >= 1) {
            // at most 64 channels: one launch, the level-2 gradient's fragments in registers; plain paths receive
            // their gradient directly
            const bool plain = !time_aug && !lead_lag;
            const bool vec = plain && dimension % (16 / sizeof(T)) == 0 && reinterpret_cast<uintptr_t>(path) % 16 == 0;
            const int64_t out_rows = plain ? int64_t(s.L) + 1 : int64_t(s.L);
            const int64_t chunks = (out_rows + kDeg2BwdRows - 1) / kDeg2BwdRows;
            int64_t parts = std::min<int64_t>(chunks, std::max<int64_t>(1, (2 * int64_t(simd_count()) / 4 + int64_t(batch) - 1) / int64_t(batch)));
            const int64_t part_rows = (chunks + parts - 1) / parts * kDeg2BwdRows;
            parts = (out_rows + part_rows - 1) / part_rows;
            const int64_t blocks = int64_t(batch) * parts;
            if (blocks > 2147483647LL) throw std::runtime_error("sig_backprop_cuda: launch too large");
            MainKernelTimer timer(stream, sizeof(T) == 8 ? "degree2_bwd_f64_rows" : "degree2_bwd_f32_rows", !arena);
            auto go = [&](auto mode) {
                constexpr int MODE = decltype(mode)::value;
                if (deg2_bwd_lds_bytes<T>() > 64 * 1024)       // above the default limit of dynamic LDS
                    SIG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&degree2_bwd_rows_kernel<T, MODE>),
                                                hipFuncAttributeMaxDynamicSharedMemorySize, int(deg2_bwd_lds_bytes<T>())));
                hipLaunchKernelGGL((degree2_bwd_rows_kernel<T, MODE>), dim3(unsigned(blocks)), dim3(kBlock), deg2_bwd_lds_bytes<T>(),
                                   stream, path, sig_derivs, MODE ? out : dzinc, int64_t(batch), int64_t(length), int(dimension),
                                   int(time_aug), int(lead_lag), time_step, int64_t(s.stride), sc, int(parts), part_rows);
            };
            if (vec) go(std::integral_constant<int, 2>());
            else if (plain) go(std::integral_constant<int, 1>());
            else go(std::integral_constant<int, 0>());
            timer.stop();
            if (!plain) launch_path_grad<T>(dzinc, out, batch, length, dimension, time_aug, lead_lag, stream);
            SIG_HIP(hipGetLastError());
            finish();
            return;
        }
        hipLaunchKernelGGL((degree2_h_kernel<T>), dim3(grid_for(batch * s.d_aug, kWavesPerBlock)), dim3(kBlock), 0, stream, path, sig_derivs, h,
                           int64_t(batch), int64_t(length), int(dimension), int(time_aug), int(lead_lag), time_step,
                           int64_t(s.stride), sc);
        if (staged && s.L >= 1 && !time_aug && !lead_lag) {
            // more than 64 channels, plain paths: accumulators of a run of rows in registers, channels walked 64 at a
            // time (with augmentation the per-element evaluation of the points makes it slower than the kernel below)
            const bool plain = true;
            const bool vec = plain && dimension % (16 / sizeof(T)) == 0 && reinterpret_cast<uintptr_t>(path) % 16 == 0;
            const int64_t out_rows = plain ? int64_t(s.L) + 1 : int64_t(s.L);
            const int64_t run = int64_t(deg2_wide_chunks<T>()) * kDeg2BwdRows;
            const int64_t parts = (out_rows + run - 1) / run;
            const int64_t blocks = int64_t(batch) * parts * col_groups;
            if (blocks > 2147483647LL) throw std::runtime_error("sig_backprop_cuda: launch too large");
            MainKernelTimer timer(stream, sizeof(T) == 8 ? "degree2_bwd_f64_wide" : "degree2_bwd_f32_wide", !arena);
            auto go = [&](auto mode) {
                constexpr int MODE = decltype(mode)::value;
                if (deg2_bwd_lds_bytes<T>() > 64 * 1024)
                    SIG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&degree2_bwd_wide_kernel<T, MODE>),
                                                hipFuncAttributeMaxDynamicSharedMemorySize, int(deg2_bwd_lds_bytes<T>())));
                hipLaunchKernelGGL((degree2_bwd_wide_kernel<T, MODE>), dim3(unsigned(blocks)), dim3(kBlock), deg2_bwd_lds_bytes<T>(),
                                   stream, path, sig_derivs, (const T*)h, MODE ? out : dzinc, int64_t(batch), int64_t(length),
                                   int(dimension), int(time_aug), int(lead_lag), time_step, int64_t(s.stride), sc, int(parts),
                                   col_groups);
            };
            if (vec) go(std::integral_constant<int, 2>());
            else if (plain) go(std::integral_constant<int, 1>());
            else go(std::integral_constant<int, 0>());
            timer.stop();
            if (!plain) launch_path_grad<T>(dzinc, out, batch, length, dimension, time_aug, lead_lag, stream);
            SIG_HIP(hipGetLastError());
            finish();
            return;
        }
        MainKernelTimer timer(stream, sizeof(T) == 8 ? (staged ? "degree2_bwd_f64_lds" : "degree2_bwd_f64")
                                                     : (staged ? "degree2_bwd_f32_lds" : "degree2_bwd_f32"), !arena);
        if (staged) {
            hipLaunchKernelGGL((degree2_anti_kernel<T>), dim3(grid_for(batch * s.d_aug * s.d_aug)), dim3(kBlock), 0, stream,
                               sig_derivs, anti, int64_t(batch), d, int64_t(s.stride), sc);
            const int64_t time_groups = (int64_t(s.L) + kDeg2Slab - 1) / kDeg2Slab;
            const int64_t blocks = int64_t(batch) * time_groups * col_groups;
            if (blocks > 2147483647LL) throw std::runtime_error("sig_backprop_cuda: launch too large");
            const size_t lds = (size_t(kDeg2Slab) * (sizeof(T) == 8 ? 65 : 66) + size_t(kDeg2Slab) * kDeg2SlabStride) * sizeof(T);
            hipLaunchKernelGGL((degree2_bwd_staged_kernel<T>), dim3(unsigned(blocks)), dim3(kBlock), lds, stream, path,
                               (const T*)anti, (const T*)h, dzinc, int64_t(batch), int64_t(length), int(dimension), int(time_aug),
                               int(lead_lag), time_step, time_groups, col_groups);
        } else {
            const int64_t time_tiles = (int64_t(s.L) + 15) / 16;
            const int64_t total = int64_t(batch) * time_tiles * col_groups;
            const int64_t blocks = (total + kWavesPerBlock - 1) / kWavesPerBlock;
            if (blocks > 2147483647LL) throw std::runtime_error("sig_backprop_cuda: launch too large");
            hipLaunchKernelGGL((degree2_bwd_kernel<T>), dim3(unsigned(blocks)), dim3(kBlock), 0, stream, path, sig_derivs, h, dzinc,
                               int64_t(batch), int64_t(length), int(dimension), int(time_aug), int(lead_lag), time_step,
                               int64_t(s.stride), sc, time_tiles, col_groups);
        }
        timer.stop();
        launch_path_grad<T>(dzinc, out, batch, length, dimension, time_aug, lead_lag, stream);
        SIG_HIP(hipGetLastError());
        finish();      // the workspaces stay locked until the kernels are done
        return;
    } else if (use_deep(s.d_aug, degree)) {
        if (!deep_fits(s.d_aug, degree, batch)) throw std::runtime_error("sig_backprop_cuda: launch too large");
        lock_pool();
        const uint64_t inc_elems = checked_mul(checked_mul(batch, s.L + 2, "increments"), s.d_aug, "increments");
        const uint64_t dz_elems = checked_mul(checked_mul(batch, s.L, "increments"), s.d_aug, "increments");
        T* inc = static_cast<T*>(buffer(0, checked_mul(inc_elems, sizeof(T), "increments")));
        T* dzinc = static_cast<T*>(buffer(1, checked_mul(dz_elems, sizeof(T), "increments")));
        compute_increments(path, inc, batch, dimension, length, time_aug, lead_lag, end_time, s, stream, dzinc, dz_elems);
        BwdParams p;
        p.inc = inc; p.sig = sig; p.gsig = sig_derivs; p.dzinc = dzinc; p.batch = int64_t(batch);
        p.L = int64_t(s.L); p.d = int(s.d_aug); p.sig_stride = int64_t(s.stride); p.scalar = sc; p.stream = stream;
        MainKernelTimer timer(stream, sizeof(T) == 8 ? "deep_bwd_f64" : "deep_bwd_f32", !arena);
        SIG_HIP(launch_deep_bwd<T>(p, int(degree)));
        timer.stop();
        launch_path_grad<T>(dzinc, out, batch, length, dimension, time_aug, lead_lag, stream);
        SIG_HIP(hipGetLastError());
        finish();
        return;
    } else {
        const KernelEntry* e = choose_entry(true, sizeof(T) == 8, s.d_aug, degree, batch, s.L);
        if (!e)
            throw std::runtime_error("sig_backprop_cuda: no kernel for dimension " + std::to_string(s.d_aug) +
                                     ", degree " + std::to_string(degree) + " in this build");
        lock_pool();
        const uint64_t inc_elems = checked_mul(checked_mul(batch, s.L + 2, "increments"), s.d_aug, "increments");
        const uint64_t dz_elems = checked_mul(checked_mul(batch, s.L, "increments"), s.d_aug, "increments");
        const uint64_t dz_bytes = checked_mul(dz_elems, sizeof(T), "increments");
        const uint64_t pad = uint64_t(kStageSteps + 2) * s.d_aug;
        BwdParams p;
        p.sig = sig; p.gsig = sig_derivs; p.batch = int64_t(batch);
        p.L = int64_t(s.L); p.d = int(s.d_aug); p.sig_stride = int64_t(s.stride); p.scalar = sc; p.stream = stream;
        const uint64_t n_coef = s.full_len - 1;
        const KernelEntry* ef = choose_entry(false, sizeof(T) == 8, s.d_aug, degree, batch, s.L);
        // lead-lag sweeps that skip the letters a step cannot move read a step's parity off its position in the
        // segment: segments start on even steps (a lead-lag path has an even number of steps)
        const bool sparse_ll = lead_lag && g_lead_lag_sparse != 0;
        // many channels beyond the compiled table: the by-row sweep, whole paths only (its launches fill the chip)
        // (also where an instance would lose: measured at 48 .. 128 channels, degrees 3 and 4, the by-row sweep runs
        // 1.1-4x faster than compiled single-precision instances and 1-12x faster than double-precision ones; the
        // instance table leaves these backward shapes out).  Below 48 channels an instance exists up to degree 4; at degree 3
        // the matrix form of single precision competes with it, the estimates decide (64 paths of 200 steps, 40 channels
        // 0.328 -> 0.234 ms, 16 x 200, 36: 0.340 -> 0.121); at degree 4 and 40 channels its tiles are 39 % filled: 4.6 -> 6.0
        // ms.  Lead-lag paths are left to the instances that skip their still letters.
        int64_t instance_waves = total_waves(geom_of(e, int(s.d_aug)), int64_t(batch));
        auto split = [&]() -> SplitPlan {
            if (arena || !ef || degree > uint64_t(kCombMaxLevels)) return {1, 0.0, 0.0};
            if (g_force_bwd_segments > 0) return {int(std::min<uint64_t>(uint64_t(g_force_bwd_segments), s.L)), 0.0, 0.0};
            return choose_bwd_segments(instance_waves, int64_t(s.L), resident_waves(e), batch * n_coef * sizeof(T),
                                       [&](int g) {
                                           // a backward step issues about 3.2 times the forward's instructions
                                           const double c = lane_step_cost(int(s.d_aug), e->N, e->tail, e->k) * 7.7e-9;
                                           const bool ring = pick_variant(true, e, instance_waves * g, sparse_ll)->staged;
                                           return ring ? c : std::max(c, 700e-9);
                                       },
                                       sizeof(T) == 8);
        };
        const int rows_mode = g_rows_backward;
        bool by_rows = !arena && rows_mode != 0 && g_force_tail == 0 && rows_bwd_supported(sizeof(T), s.d_aug, degree) &&
                       rows_fits(sizeof(T), s.d_aug, degree, batch);
        const bool compare = by_rows && rows_mode == 1 && e->D > 0 && s.d_aug < 48;
        if (compare) by_rows = sizeof(T) == 4 && degree == 3 && !lead_lag && g_force_bwd_segments == 0;
        SplitPlan plan{1, 0.0, 0.0};
        if (!by_rows || compare) plan = split();
        if (compare && by_rows) by_rows = rows_bwd_seconds(s.d_aug, batch, s.L) < instance_bwd_seconds(plan, s.d_aug);
        auto finer = [&]() {
            return with_fine(e, pick_variant(true, e, instance_waves * plan.pieces, sparse_ll), plan, true, s.d_aug, degree, batch, s.L,
                             batch * n_coef * sizeof(T), sparse_ll, g_force_bwd_segments, !ef || degree > uint64_t(kCombMaxLevels));
        };
        if (!by_rows && !arena) {
            plan = finer();
            if (const KernelEntry* spec = instance_after_all(e, true, s.d_aug, degree, batch, s.L)) {
                e = spec;
                instance_waves = total_waves(geom_of(e, int(s.d_aug)), int64_t(batch));
                const int before = plan.pieces;
                plan = split();
                plan = finer();
                tl_fine_more_pieces = tl_fine_more_pieces || plan.pieces > before;
            }
        }
        int nseg = by_rows ? 1 : plan.pieces;
        int64_t lseg = int64_t(s.L);
        if (nseg > 1) {
            lseg = (int64_t(s.L) + nseg - 1) / nseg;
            if (sparse_ll) lseg += lseg & 1;
            nseg = int((int64_t(s.L) + lseg - 1) / lseg);
        }
        // Whole-path staged sweeps of plain narrow paths form the increments themselves while staging the points: no
        // pre-pass launch, so the accumulator comes from the pair that takes turns (cleared by the previous call).
        const KernelEntry* e_run = pick_variant(true, e, total_waves(geom_of(e, int(s.d_aug)), int64_t(batch) * nseg), sparse_ll);
        const bool point_fed = !arena && !by_rows && nseg == 1 && e_run->staged && !time_aug && !lead_lag && e_run->D > 0 &&
                               e_run->D <= kPointFedMaxDim && g_point_fed != 0;
        // by rows in single precision: the increment gradient is summed in double precision, and rounded where the path
        // gradient is formed from it
        const bool wide = by_rows && sizeof(T) == 4;
        const bool on_matrix_units = by_rows && sizeof(T) == 4 && rows_mode != 3 && rows_bwd_mfma_supported(s.d_aug) &&
                                     (rows_mode == 2 || rows_bwd_mfma_wins(s.d_aug, degree, batch, s.L));
        T* inc = nullptr;
        T* dzinc = nullptr;
        double* wide_dz = nullptr;
        DzPair* turn = nullptr;
        int mine = 0;
        if (point_fed) {
            int dev = 0;
            SIG_HIP(hipGetDevice(&dev));
            turn = &g_dz[dev];
            mine = turn->next;
            dzinc = static_cast<T*>(dz_pair_buffer(*turn, mine, dz_bytes));
            if (turn->dirty[mine]) {        // first use, or a call that failed half-way: clear it here
                const uint64_t n = (turn->dirty[mine] + sizeof(T) - 1) / sizeof(T);
                hipLaunchKernelGGL((zero_kernel<T>), dim3(grid_for(n)), dim3(kBlock), 0, stream, dzinc, int64_t(n));
                SIG_HIP(hipGetLastError());
                turn->dirty[mine] = 0;
            }
            p.inc = path;
            p.from_points = 1;
        } else {
            inc = static_cast<T*>(buffer(0, checked_mul(inc_elems + 2 * pad, sizeof(T), "increments"))) + pad;
            // one launch writes the increments and clears the increment-gradient accumulator (dz_elems <= increment elements)
            if (wide) {
                wide_dz = static_cast<double*>(buffer(1, checked_mul(dz_elems, sizeof(double), "increments")));
                compute_increments(path, inc, batch, dimension, length, time_aug, lead_lag, end_time, s, stream, wide_dz, dz_elems);
            } else {
                dzinc = static_cast<T*>(buffer(1, dz_bytes));
                compute_increments(path, inc, batch, dimension, length, time_aug, lead_lag, end_time, s, stream, dzinc, dz_elems);
            }
            p.inc = inc;
        }
        p.dzinc = wide_dz ? static_cast<void*>(wide_dz) : dzinc;
        if (nseg > 1) {
            // (path, segment) rows, scalar-free: segment signatures, their running products from the left (the state
            // at each segment's end), from the right (what follows each segment), and the adjoints of the states
            const uint64_t rows = checked_mul(batch, uint64_t(nseg), "segment signatures");
            const uint64_t bytes = checked_mul(checked_mul(rows, n_coef, "segment signatures"), sizeof(T), "segment signatures");
            T* segs = static_cast<T*>(buffer(2, bytes));
            T* left = static_cast<T*>(buffer(8, bytes));
            T* right = static_cast<T*>(buffer(9, bytes));
            T* adj = static_cast<T*>(buffer(10, bytes));
            const int64_t n = int64_t(n_coef);
            FwdParams f;
            f.inc = inc; f.batch = int64_t(rows); f.L = int64_t(s.L); f.d = int(s.d_aug); f.stream = stream;
            f.lseg = lseg; f.nseg = nseg; f.out = segs; f.out_stride = n; f.scalar = 0;
            const KernelEntry* ef_now = pick_variant(false, ef, total_waves(geom_of(ef, int(s.d_aug)), f.batch), sparse_ll);
            with_fine(ef, ef_now, SplitPlan{1, 0.0, 0.0}, false, s.d_aug, degree, rows, uint64_t(lseg), 0, sparse_ll, 0, /*whole_only=*/true);
            ef = pick_variant(false, ef, total_waves(geom_of(ef, int(s.d_aug)), f.batch), sparse_ll);
            SIG_HIP((sparse_ll && ef->staged && ef->fwd_lead_lag) ? ef->fwd_lead_lag(f) : ef->fwd(f));
            // both scans by doubling: ceil(log2(nseg)) launches, ping-ponging between two scratch copies
            int steps = 0;
            while ((1 << steps) < nseg) ++steps;
            T* scratch = steps > 1 ? static_cast<T*>(buffer(11, checked_mul(bytes, steps > 2 ? 4 : 2, "segment signatures")))
                                   : nullptr;
            const uint64_t buf = rows * n_coef;
            const T* xsrc = segs;
            const T* zsrc = segs;
            for (int k = 0; k < steps; ++k) {
                const bool last = k == steps - 1;
                T* xdst = last ? left : scratch + uint64_t(k & 1) * 2 * buf;
                T* zdst = last ? right : scratch + (uint64_t(k & 1) * 2 + 1) * buf;
                with_chen_fan(s.d_aug, [&](auto fan) {
                    constexpr int FAN = decltype(fan)::value;
                    const uint64_t items = chen_items(s.d_aug, degree, FAN);
                    launch_indexed(n_coef, items, 2 * rows, [&](auto ix, dim3 grid) {
                        using I = decltype(ix);
                        hipLaunchKernelGGL((chen_scan_step_kernel<T, I, FAN>), grid, dim3(kBlock), 0, stream, xsrc, zsrc, xdst,
                                           zdst, int64_t(batch), nseg, 1 << k, k == 0 ? 1 : 0, DivBy<I>(s.d_aug), I(n_coef),
                                           I(items));
                    });
                });
                xsrc = xdst;
                zsrc = zdst;
            }
            SIG_HIP(hipGetLastError());
            SigShape rs;
            rs.n_coef = n_coef; rs.stride = n_coef; rs.off = 0;
            SharedRows up;
            up.share = nseg; up.stride = int64_t(s.stride); up.off = sc;
            launch_combine_bwd<T>(sig_derivs, adj, nullptr, nullptr, right, rows, s.d_aug, degree, rs, stream, 1, up, 1);
            SIG_HIP(hipGetLastError());
            p.sig = left; p.gsig = adj; p.sig_stride = n; p.scalar = 0;
            p.batch = int64_t(rows); p.nseg = nseg; p.lseg = lseg;
        }
        e = e_run;
        const bool use_ll = !by_rows && sparse_ll && e->bwd_lead_lag && (s.L & 1) == 0;
        const std::string shown = by_rows ? std::string(sizeof(T) == 8 ? "rows_bwd_f64_n" : "rows_bwd_f32_n") + std::to_string(degree)
                                  : use_ll ? std::string(e->name) + "_ll" : std::string(e->name);
        MainKernelTimer timer(stream, shown.c_str(), !arena);
        if (turn) turn->dirty[mine] = dz_bytes;        // from here on the accumulator holds sums
        tl_matrix_form = on_matrix_units;
        if (by_rows) {
            if (on_matrix_units) SIG_HIP(launch_rows_bwd_mfma(p, int(degree)));
            else SIG_HIP(launch_rows_bwd<T>(p, int(degree)));
        } else {
            SIG_HIP(use_ll ? e->bwd_lead_lag(p) : e->bwd(p));
        }
        timer.stop();
        if (turn) {
            // the same launch clears what the other accumulator still holds: it is the next call's
            const int other = 1 - mine;
            T* clear = turn->dirty[other] ? static_cast<T*>(turn->ptr[other]) : nullptr;
            launch_path_grad<T>(dzinc, out, batch, length, dimension, time_aug, lead_lag, stream, clear,
                                (turn->dirty[other] + sizeof(T) - 1) / sizeof(T));
            SIG_HIP(hipGetLastError());
            turn->dirty[other] = 0;
            turn->next = other;
        } else if (wide_dz) {
            launch_path_grad<T>(wide_dz, out, batch, length, dimension, time_aug, lead_lag, stream);
            SIG_HIP(hipGetLastError());
        } else {
            launch_path_grad<T>(dzinc, out, batch, length, dimension, time_aug, lead_lag, stream);
            SIG_HIP(hipGetLastError());
        }
        finish();
        return;
    }
    SIG_HIP(hipGetLastError());
    finish();
}

// ---------------------------------------------------------------------------
// built-in scratch memory of the entry point that allocates nothing
// ---------------------------------------------------------------------------
constexpr size_t kScratchBytes = size_t(32) << 20;
}  // namespace sigamd

// Every GPU the library runs on holds its own copy of this array (at its own address) until the process ends.  In
// host code the name is only a handle for hipGetSymbolAddress; kernels are given the address that call returns.
static __device__ __align__(256) unsigned char scratch[sigamd::kScratchBytes];

namespace sigamd {

static std::mutex g_scratch_mutex;
static std::map<int, void*> g_scratch_ptr;      // device -> address of that device's copy of `scratch`

static void* scratch_of_current_device()
{
    int dev = 0;
    SIG_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_scratch_mutex);
    auto it = g_scratch_ptr.find(dev);
    if (it != g_scratch_ptr.end()) return it->second;
    void* ptr = nullptr;
    SIG_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) throw std::runtime_error("built-in scratch memory has no device address");
    g_scratch_ptr[dev] = ptr;
    return ptr;
}

void note_alloc_retry() noexcept { ++g_alloc_retries; }

}  // namespace sigamd

using namespace sigamd;

// signature_cuda_* with the batch taken in halves when the device cannot hold the workspace of the whole call
template <typename T>
static void signature_entry(const T* path, T* out, uint64_t batch, uint64_t dimension, uint64_t length, uint64_t degree,
                            bool time_aug, bool lead_lag, T end_time, bool horner, bool scalar_term, const T* correction,
                            uint64_t correction_len)
{
    int nonfinite = 0;
    split_on_bad_alloc(batch, "signature", [&](uint64_t first, uint64_t count) {
        uint64_t stride = 0;
        if (first) stride = make_shape(dimension, length, degree, time_aug, lead_lag, scalar_term).stride;
        fine_if_it_fits([&] {
            signature_impl<T>(path + first * length * dimension, out + first * stride, count, dimension, length, degree, time_aug,
                              lead_lag, end_time, horner, scalar_term, correction, correction_len);
        });
        const int f = tl_sig_nonfinite;
        nonfinite = (nonfinite < 0 || f < 0) ? -1 : (nonfinite | f);
    });
    if (batch) tl_sig_nonfinite = nonfinite;
}

template <typename T>
static void sig_backprop_entry(const T* path, T* out, const T* sig_derivs, const T* sig, uint64_t batch, uint64_t dimension,
                               uint64_t length, uint64_t degree, bool time_aug, bool lead_lag, T end_time, bool scalar_term,
                               const T* correction, uint64_t correction_len)
{
    split_on_bad_alloc(batch, "sig_backprop", [&](uint64_t first, uint64_t count) {
        uint64_t stride = 0;
        if (first) stride = make_shape(dimension, length, degree, time_aug, lead_lag, scalar_term).stride;
        fine_if_it_fits([&] {
            sig_backprop_impl<T>(path + first * length * dimension, out + first * length * dimension, sig_derivs + first * stride,
                                 sig + first * stride, count, dimension, length, degree, time_aug, lead_lag, end_time, scalar_term,
                                 correction, correction_len);
        });
    });
}

extern "C" {

CUSIG_AMD_API int signature_cuda_f(const float* path, float* out, uint64_t batch_size, uint64_t dimension,
                                   uint64_t length, uint64_t degree, bool time_aug, bool lead_lag, float end_time,
                                   bool horner, bool scalar_term, const float* correction,
                                   uint64_t correction_len, uint64_t, uint64_t) noexcept
{
    return guarded([&] {
        signature_entry<float>(path, out, batch_size, dimension, length, degree, time_aug, lead_lag, end_time,
                               horner, scalar_term, correction, correction_len);
    });
}

CUSIG_AMD_API int signature_cuda_d(const double* path, double* out, uint64_t batch_size, uint64_t dimension,
                                   uint64_t length, uint64_t degree, bool time_aug, bool lead_lag,
                                   double end_time, bool horner, bool scalar_term, const double* correction,
                                   uint64_t correction_len, uint64_t, uint64_t) noexcept
{
    return guarded([&] {
        signature_entry<double>(path, out, batch_size, dimension, length, degree, time_aug, lead_lag, end_time,
                                horner, scalar_term, correction, correction_len);
    });
}

CUSIG_AMD_API int sig_backprop_cuda_f(const float* path, float* out, const float* sig_derivs, const float* sig,
                                      uint64_t batch_size, uint64_t dimension, uint64_t length, uint64_t degree,
                                      bool time_aug, bool lead_lag, float end_time, bool scalar_term,
                                      const float* correction, uint64_t correction_len, uint64_t,
                                      uint64_t) noexcept
{
    return guarded([&] {
        sig_backprop_entry<float>(path, out, sig_derivs, sig, batch_size, dimension, length, degree, time_aug,
                                  lead_lag, end_time, scalar_term, correction, correction_len);
    });
}

CUSIG_AMD_API int sig_backprop_cuda_d(const double* path, double* out, const double* sig_derivs,
                                      const double* sig, uint64_t batch_size, uint64_t dimension,
                                      uint64_t length, uint64_t degree, bool time_aug, bool lead_lag,
                                      double end_time, bool scalar_term, const double* correction,
                                      uint64_t correction_len, uint64_t, uint64_t) noexcept
{
    return guarded([&] {
        sig_backprop_entry<double>(path, out, sig_derivs, sig, batch_size, dimension, length, degree, time_aug,
                                   lead_lag, end_time, scalar_term, correction, correction_len);
    });
}

CUSIG_AMD_API int cusig_amd_sig_backprop_noalloc_d(const double* path, double* out, const double* sig_derivs,
                                                   const double* sig, uint64_t batch_size, uint64_t dimension,
                                                   uint64_t length, uint64_t degree, bool time_aug, bool lead_lag,
                                                   double end_time, bool scalar_term, void* stream) noexcept
{
    return guarded([&] {
        Arena arena;
        arena.base = static_cast<char*>(scratch_of_current_device());
        arena.bytes = kScratchBytes;
        arena.stream = static_cast<hipStream_t>(stream);
        sig_backprop_impl<double>(path, out, sig_derivs, sig, batch_size, dimension, length, degree, time_aug, lead_lag,
                                  end_time, scalar_term, nullptr, 0, &arena);
    });
}

CUSIG_AMD_API uint64_t cusig_amd_noalloc_scratch_bytes(void) noexcept { return kScratchBytes; }

CUSIG_AMD_API const char* cusig_last_error_message(void) noexcept { return g_last_error; }

CUSIG_AMD_API void cusig_shutdown(void) noexcept
{
    release_workspaces();
    clear_lyndon_tables();
}

CUSIG_AMD_API uint64_t cusig_amd_sig_length(uint64_t dimension, uint64_t degree) noexcept
{
    return sig_length_u64(dimension, degree);
}

CUSIG_AMD_API void cusig_amd_set_profiling(int enabled) noexcept { g_profile = enabled != 0; }

CUSIG_AMD_API float cusig_amd_last_kernel_ms(void) noexcept { return g_last_ms; }

CUSIG_AMD_API const char* cusig_amd_last_kernel_name(void) noexcept
{
    static thread_local char name[sizeof g_last_name];
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    std::memcpy(name, g_last_name, sizeof name);
    return name;
}

CUSIG_AMD_API void cusig_amd_force_segments(int segments) noexcept { if (g_test_hooks) g_force_segments = segments; }
CUSIG_AMD_API int cusig_amd_last_segments(void) noexcept { return tl_last_segments; }
CUSIG_AMD_API void cusig_amd_set_point_fed(int on) noexcept { if (g_test_hooks) g_point_fed = on; }
CUSIG_AMD_API void cusig_amd_set_lead_lag_sparse(int on) noexcept { if (g_test_hooks) g_lead_lag_sparse = on; }

CUSIG_AMD_API void cusig_amd_force_bwd_segments(int segments) noexcept { if (g_test_hooks) g_force_bwd_segments = segments; }

CUSIG_AMD_API void cusig_amd_set_fine(int mode) noexcept { if (g_test_hooks) g_fine = mode; }
CUSIG_AMD_API int cusig_amd_last_sweep_on_matrix_units(void) noexcept { return tl_matrix_form; }
CUSIG_AMD_API void cusig_amd_set_rows_backward(int mode) noexcept { if (g_test_hooks) g_rows_backward = mode; }
CUSIG_AMD_API void cusig_amd_set_heads_forward(int mode) noexcept { if (g_test_hooks) g_heads = mode; }
CUSIG_AMD_API void cusig_amd_set_heads_table_limit(uint64_t bytes) noexcept { if (g_test_hooks) g_heads_table = bytes ? bytes : kHeadsTableBytes; }
CUSIG_AMD_API void cusig_amd_set_rows_forward(int mode) noexcept { if (g_test_hooks) g_rows_forward = mode; }

CUSIG_AMD_API void cusig_amd_force_staged(int mode) noexcept { if (g_test_hooks) g_force_staged = mode; }

CUSIG_AMD_API void cusig_amd_force_wide_index(int enabled) noexcept { if (g_test_hooks) g_force_wide_index = enabled; }
CUSIG_AMD_API void cusig_amd_force_chen_adjoint(int mode) noexcept { if (g_test_hooks) g_chen_adjoint_mode = mode; }
CUSIG_AMD_API void cusig_amd_set_chen_low_levels(int enabled) noexcept { if (g_test_hooks) g_chen_low_levels = enabled; }

CUSIG_AMD_API void cusig_amd_set_row_forms(int mode) noexcept { if (g_test_hooks) g_row_forms = mode; }
CUSIG_AMD_API int cusig_amd_last_row_form(void) noexcept { return tl_row_form; }
CUSIG_AMD_API int cusig_amd_last_chen_both(void) noexcept { return tl_chen_both; }

CUSIG_AMD_API void cusig_amd_set_stream_ordered(int enabled) noexcept { g_stream_ordered = enabled; }

CUSIG_AMD_API int cusig_amd_last_sig_nonfinite(void) noexcept { return tl_sig_nonfinite; }

CUSIG_AMD_API void cusig_amd_force_degree2(int mode) noexcept { if (g_test_hooks) g_force_degree2 = mode; }
CUSIG_AMD_API void cusig_amd_force_degree3(int mode) noexcept { if (g_test_hooks) g_force_degree3 = mode; }

CUSIG_AMD_API void cusig_amd_force_deep(int enabled) noexcept { if (g_test_hooks) g_force_deep = enabled; }

CUSIG_AMD_API void cusig_amd_set_degree2_staged(int enabled) noexcept { if (g_test_hooks) g_degree2_staged = enabled; }

CUSIG_AMD_API void cusig_amd_ignore_instance_table(int on) noexcept { if (g_test_hooks) g_ignore_table = on; }
CUSIG_AMD_API void cusig_amd_force_run_time_wide(int enabled) noexcept { if (g_test_hooks) g_force_run_time_wide = enabled; }

CUSIG_AMD_API void cusig_amd_force_partition(int tail, int k) noexcept
{
    if (!g_test_hooks) return;
    g_force_tail = tail;
    g_force_k = k;
}

CUSIG_AMD_API void cusig_amd_enable_test_hooks(int enabled) noexcept
{
    g_test_hooks = enabled != 0;
    if (enabled) return;
    // back to the defaults
    g_force_segments = 0;
    g_point_fed = 1;
    g_lead_lag_sparse = 1;
    g_force_bwd_segments = 0;
    g_fine = 1;
    g_rows_backward = 1;
    g_rows_forward = 1;
    g_heads = 1;
    g_heads_table = kHeadsTableBytes;
    g_force_staged = -1;
    g_force_wide_index = 0;
    g_chen_adjoint_mode = 0;
    g_chen_low_levels = 1;
    g_row_forms = 1;
    g_force_degree2 = -1;
    g_force_degree3 = -1;
    g_force_deep = 0;
    g_degree2_staged = 1;
    g_force_run_time_wide = 0;
    g_ignore_table = 0;
    g_force_tail = 0;
    g_force_k = 0;
    g_alloc_limit = 0;
    g_pool_limit = 0;
}

CUSIG_AMD_API uint64_t cusig_amd_workspace_bytes(void) noexcept
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    return pool_bytes(dev);
}

CUSIG_AMD_API void cusig_amd_set_alloc_limit(uint64_t bytes) noexcept { if (g_test_hooks) g_alloc_limit = bytes; }
CUSIG_AMD_API void cusig_amd_set_pool_limit(uint64_t bytes) noexcept { if (g_test_hooks) g_pool_limit = bytes; }
CUSIG_AMD_API int cusig_amd_alloc_retries(void) noexcept { return g_alloc_retries; }

CUSIG_AMD_API int cusig_amd_kernel_choice(int backward, int is_f64, uint64_t dimension, uint64_t degree,
                                          int* tail, int* k, int* specialised) noexcept
{
    const KernelEntry* e = find_entry(backward != 0, is_f64 != 0, dimension, degree);
    if (!e) return 0;
    if (tail) *tail = e->tail;
    if (k) *k = e->k;
    if (specialised) *specialised = e->D > 0;
    return 1;
}

}  // extern "C"
