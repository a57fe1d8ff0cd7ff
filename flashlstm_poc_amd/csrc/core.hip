// Plan object and orchestration of the device-resident LSTM forward / BPTT core.
//
// Forward  = [convert x] -> MFMA GEMM  G = X * W_ih^T  (hoisted input projection, the chunked
//            "projchunksz" GEMM of src/lstm.cu:1204-1239) -> persistent recurrence kernel that turns G
//            in place into the fp16 gate cache and fills the h / c state arrays -> [unpad outputs].
// Backward = persistent BPTT kernel (reads gate cache + c states, writes dG) -> dX = dG * W_ih
//            -> dW = dG^T * [X ; H_prev] as one split-K GEMM -> reductions into caller layout.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <cmath>
#include <initializer_list>
#include <mutex>
#include <new>
#include <vector>

#include "../../include/flashlstm/lstm_core.h"
#include "core_internal.h"
#include "gemm.h"
#include "pack.h"
#include "recurrent.h"

using namespace flstm_hip;

// Scratch memory of flstm_core_forward_static: what that entry point's kernels need beyond the caller's tensors and what a
// plan has anyway (packed weights, status block, ring of the whole passes): converted x rows, x-projection / gate rows, state
// rows, exchange ring.  One array per device, owned by the code object; host code reaches it only through the address
// hipGetSymbolAddress returns for the device that is current (static_scratch()).
static constexpr size_t kStaticScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
static constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[kMaxDevices] = {};

// address of `scratch` on the current device (looked up once per device)
static int static_scratch(int dev, void** out) {
    if (dev < 0 || dev >= kMaxDevices) return FLSTM_E_INVALID;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return int(e);
        if (!ptr) return int(hipErrorInvalidSymbol);
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

namespace {

struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    bool borrowed = false;   // a view of memory owned elsewhere: never grown, never freed
    // grows (never shrinks); contents are lost on growth
    hipError_t reserve(size_t need) {
        if (need <= bytes) return hipSuccess;
        if (borrowed) return hipErrorOutOfMemory;
        if (p) { hipError_t e = hipFree(p); p = nullptr; bytes = 0; if (e != hipSuccess) return e; }
        hipError_t e = hipMalloc(&p, need);
        if (e == hipSuccess) bytes = need;
        return e;
    }
    void release() { if (p && !borrowed) (void)hipFree(p); p = nullptr; bytes = 0; borrowed = false; }
    template <typename T> T* as() const { return static_cast<T*>(p); }
    static DevBuf view(void* ptr, size_t n) { DevBuf b; b.p = ptr; b.bytes = n; b.borrowed = true; return b; }
};

}  // namespace

constexpr int kFirstHold = 8, kMaxHold = 1024;

// Factors of a backward pass: on dY and on the incoming state gradients as they are read, on dx and on the parameter and
// initial-state gradients as they are written.
struct BwdScales {
    float dy = 1.f, state = 1.f, dx = 1.f, grads = 1.f;
    static BwdScales loss_scale(float S) { return BwdScales{S, S, 1.f / S, 1.f / S}; }
};

// The plan's status block on the device: word 0 the status, words 1 and 2 the delay hints of the two recurrences, the
// time stamps of a pass, and sets of seat counters: every recurrence launch needs eight zeroed ones, so a pass that
// launches several (ranges of steps, windows of rows) takes the sets its setup has zeroed one after the other.
constexpr size_t kStampsOffset = 64, kSeatsOffset = 256;
constexpr int kSeatSets = 64;
constexpr int kSeatWords = 32;   // eight seat counters, the ticket counters of BesideCopies (one) and, from word 16 on, ProjectBeside (eight)
constexpr size_t kStatusBytes = kSeatsOffset + size_t(kSeatSets) * kSeatWords * sizeof(unsigned);
static_assert(kStampsOffset + kStampCount * sizeof(long long) <= kSeatsOffset, "stamps fit in front of the seats");

struct flstm_core_plan {
    int device = 0;
    int num_cus = 0;
    int clock_khz = 0;   // maximum engine clock the runtime reports
    Dims d{};
    RecLayout Lf{}, Lb{};
    // options
    int opt_stepwise = 0, opt_spin_limit = 1 << 30, opt_spin_ms = 250, opt_dw_splits = 0, opt_accumulate = 0;
    // A persistent launch that gave up (its workgroups were not all running at once, or not spread over the XCDs
    // as expected) demotes that direction to step-wise launches for `hold` passes; then the persistent kernel is
    // tried again.  Every further give-up doubles the hold (at most kMaxHold passes).
    int hold_fwd = 0, hold_bwd = 0, backoff_fwd = kFirstHold, backoff_bwd = kFirstHold;
    long fallbacks = 0, demotions_fwd = 0, demotions_bwd = 0;
    // A cooperative launch refused because the grid cannot be co-resident: that direction runs step-wise from then on.
    bool refused_fwd = false, refused_bwd = false;
    long coop_refusals = 0;
    bool static_call = false;   // flstm_core_forward_static in force: nothing may allocate (no graph capture either)
    // Tuned launch choices per sequence length (flstm_core_tune): 16- or 32-row blocks and persistent or step-wise
    // launches per direction, split-K count of the weight-gradient GEMM.  eff_* hold the entry in force for the
    // sequence length of the current pass (0 = no tuned value: the rules of thumb decide); explicit options win.
    struct Tuned { size_t T; int mt_f, mt_b, step_f, step_b, dw_splits, two_d; float ms_f, ms_b, ms_dw, pass_f, products; };   // two_d: -1 = not tuned, else the bwd_two_d option
    std::vector<Tuned> tuned;
    int opt_mt_f = 0, opt_mt_b = 0;
    int eff_mt_f = 0, eff_mt_b = 0, eff_step_f = 0, eff_step_b = 0, eff_dw = 0, eff_two_d = -1;
    bool two_d_explicit = false;   // option "bwd_two_d" (or its environment variable) was given: a tuned value does not replace it
    size_t eff_T = 0;
    int opt_cooperative = 0;
    StepGraphCache graphs_f, graphs_b;   // captured step-wise launches (only used where the persistent kernels are not)
    int opt_graphs = 1;
    int opt_two_d = 1;   // backward recurrence for 2048 hidden units, two-way split: 0 never, 1 where it is faster, 2 wherever it can run
    int opt_waves_f = 0;   // wavefronts per workgroup of the forward recurrence: 0 = by size, 4, 8 (one-way kernels, whose weights are packed for it)
    HostStatus* status_host = nullptr;   // pinned: the last launch of a pass leaves the status word and the stamps here
    int seat_sets_left = 0;              // zeroed sets of seat counters in the status block
    int inject_stall = 0;         // test hook: treat the next N passes as if their launches had given up
    // weights
    DevBuf wih_p, wih_t, wfrag[kFragKinds], bias_p;
    bool weights_packed = false, bias_packed = false;
    bool frag_there[2] = {false, false};   // kFragFwd, kFragFwdSplit (one that is not is made from the other: forward_fragments)
    bool many_steps = false;   // of the pass that use_tuned was told of (many_steps())
    // forward state / caches
    DevBuf X16, G, Y, C, status, xch_f, xch_b;
    // ring of the whole passes that are one launch (forward_whole): its own, because it stays ready from one to the next
    DevBuf ring;
    bool ring_ready = false;   // all slots but ring_base hold the 'unwritten' pattern
    int ring_base = 0;
    size_t T_cache = 0;
    bool have_cache = false;
    // pass in progress (begin / steps / end)
    struct { size_t T = 0; const void* x = nullptr; flstm_dtype x_dtype = FLSTM_F16; bool open = false;
             half_t* y_direct = nullptr;   // the recurrence writes the caller's y itself
             bool whole = false;           // one launch (forward_whole)
             int few = 0;                  // RecLayout::few that the exchange ring is laid out for
             int begin = kStampFwdBegin;   // the stamp that begins the pass
             bool begin_on_device = false;   // ... it and kStampFwdStart are not among the published ones (forward_whole)
             int projection = 0;           // where the x-projection is formed: 0 in front of the recurrence, 1 beside it, 2 inside its launch
             bool behind = false;          // the caller's final states are written by a launch of their own behind the recurrence ...
             bool rows_behind = false; } fw;   // ... and y with them
    struct { size_t T = 0; const half_t* dYk = nullptr; const void* dY = nullptr; flstm_dtype dy_dtype = FLSTM_F16;
             RecLayout L{};   // of the whole pass: the ring and the groups of the bias gradient are laid out for it, whatever options change meanwhile
             BwdScales k; float dy_scale = 1.f; void* dx = nullptr; flstm_dtype dx_dtype = FLSTM_F16; bool open = false;
             bool shared = false; } bw;   // dX and the weight gradients in one launch
    DevBuf tile_words;         // ProjectBeside::ready
    unsigned tile_mark = 0;    // ... of the last launch
    ProjectBeside project;     // for the next forward recurrence launch
    BesideCopies beside_f, beside_b;   // for the next recurrence launch of a pass fed in ranges (core_copy_beside)
    // backward scratch
    DevBuf dYp, dG, dHn, dC, dH0, db_part, dw_part, prof, part_b;
    int opt_profile = 0, wall_khz = 100000;
    long long prof_f[8] = {}, prof_b[8] = {};
    float ms_fwd[3] = {-1, -1, -1}, ms_bwd[4] = {-1, -1, -1, -1};
};

namespace {

#define FL_TRY(expr)                                  \
    do {                                              \
        hipError_t _e = (expr);                       \
        if (_e != hipSuccess) return int(_e);         \
    } while (0)

void replan(flstm_core_plan* p) {
    p->Lf = plan_rec_fwd(p->d.B, p->d.Hp, p->num_cus, p->opt_stepwise || p->hold_fwd > 0 || p->eff_step_f || p->refused_fwd,
                         p->opt_mt_f ? p->opt_mt_f : p->eff_mt_f, p->opt_waves_f, p->many_steps);
    p->Lb = plan_rec_bwd(p->d.B, p->d.Hp, p->num_cus, p->opt_stepwise || p->hold_bwd > 0 || p->eff_step_b || p->refused_bwd,
                         p->opt_mt_b ? p->opt_mt_b : p->eff_mt_b,
                         (!p->two_d_explicit && p->eff_two_d >= 0) ? p->eff_two_d : p->opt_two_d);
    p->Lf.cooperative = p->Lb.cooperative = p->opt_cooperative;
}

bool many_steps(const flstm_core_plan* p, size_t T);

// Puts the tuned entry for sequence length T in force: the entry tuned at exactly T, else the nearest one within a
// factor of two, else none; and the forward layout for as many steps.
void use_tuned(flstm_core_plan* p, size_t T) {
    const flstm_core_plan::Tuned* best = nullptr;
    double best_d = 1.0;   // |log2(T / T')| <= 1
    for (const auto& t : p->tuned) {
        const double dist = std::fabs(std::log2(double(T) / double(t.T)));
        if (dist <= best_d && (!best || dist < best_d)) { best = &t; best_d = dist; }
    }
    const int mt_f = best ? best->mt_f : 0, mt_b = best ? best->mt_b : 0, sf = best ? best->step_f : 0,
              sb = best ? best->step_b : 0, td = best ? best->two_d : -1;
    p->eff_dw = best ? best->dw_splits : 0;
    p->eff_T = best ? best->T : 0;
    const bool many = many_steps(p, T);
    if (many != p->many_steps || mt_f != p->eff_mt_f || mt_b != p->eff_mt_b || sf != p->eff_step_f || sb != p->eff_step_b || td != p->eff_two_d) {
        p->many_steps = many;
        p->eff_mt_f = mt_f; p->eff_mt_b = mt_b; p->eff_step_f = sf; p->eff_step_b = sb; p->eff_two_d = td;
        replan(p);
    }
}

long long* stamps_of(const flstm_core_plan* p) { return reinterpret_cast<long long*>(p->status.as<char>() + kStampsOffset); }

// The last launch of a pass: it leaves the status word of the recurrence kernels and the stamps in pinned host memory,
// so the wait that ends the pass anyway is also the one that makes them readable: no second round trip to the device.
int publish_with(flstm_core_plan* p, OpList& last, int stamp, hipStream_t s) {
    last.status = p->status.as<int>();
    last.stamps = stamps_of(p);
    last.stamp = stamp;
    last.publish = p->status_host;
    if (last.only_if_ok && p->inject_stall > 0) FL_TRY(fill_words(p->status.p, sizeof(int), 1u, s));   // (take_status would be too late)
    FL_TRY(run_ops(last, s));
    return 0;
}
int wait_stream(hipStream_t s) {
    FL_TRY(wait_for_persistent(s));
    return 0;
}
// after the stream has been waited for: the status of the pass; a non-zero one is cleared on the device
int take_status(flstm_core_plan* p, hipStream_t s, int* out) {
    *out = *static_cast<volatile int*>(&p->status_host->status);
    if (*out != 0) FL_TRY(fill_zero(p->status.p, sizeof(int), s));
    if (p->inject_stall > 0) {   // (2 in a row: the step-wise repeat of a pass fails too, i.e. the call does)
        p->inject_stall--;
        if (*out == 0) *out = 1;
    }
    return 0;
}
// a status nobody will look at (the pass is repeated because of another plan's) does not stay behind
int clear_status(flstm_core_plan* p, hipStream_t s) {
    if (*static_cast<volatile int*>(&p->status_host->status) != 0) FL_TRY(fill_zero(p->status.p, sizeof(int), s));
    return 0;
}
int wait_status(flstm_core_plan* p, OpList& last, int stamp, hipStream_t s, int* out) {
    int rc = publish_with(p, last, stamp, s);
    if (rc) return rc;
    rc = wait_stream(s);
    if (rc) return rc;
    return take_status(p, s, out);
}

// Eight zeroed seat counters for the next recurrence launch.
int next_seats(flstm_core_plan* p, unsigned** out, hipStream_t s) {
    char* const first = p->status.as<char>() + kSeatsOffset;
    if (p->seat_sets_left <= 0) {
        FL_TRY(fill_zero(first, size_t(kSeatSets) * kSeatWords * sizeof(unsigned), s));
        p->seat_sets_left = kSeatSets;
    }
    *out = reinterpret_cast<unsigned*>(first) + size_t(--p->seat_sets_left) * kSeatWords;
    return 0;
}

// A persistent launch gave up: step-wise launches for the next `hold` passes of that direction.
void demote(flstm_core_plan* p, bool fwd) {
    int& hold = fwd ? p->hold_fwd : p->hold_bwd;
    int& backoff = fwd ? p->backoff_fwd : p->backoff_bwd;
    hold = backoff;
    backoff = backoff * 2 > kMaxHold ? kMaxHold : backoff * 2;
    (fwd ? p->demotions_fwd : p->demotions_bwd)++;
    p->fallbacks++;
    replan(p);
}
// A pass of a demoted direction went through: one pass less to hold; at zero the persistent kernel is back.
void pass_done(flstm_core_plan* p, bool fwd) {
    int& hold = fwd ? p->hold_fwd : p->hold_bwd;
    if (hold > 0 && --hold == 0) replan(p);
}

// milliseconds between two stamps of the pass that has just been waited for (-1: not both there)
float elapsed(const flstm_core_plan* p, int from, int to) {
    const long long a = p->status_host->stamps[from], b = p->status_host->stamps[to];
    return (a > 0 && b >= a) ? float(double(b - a) / p->wall_khz) : -1.f;
}

// the phases of a forward pass that begin in front of its recurrence
void from_the_beginning(flstm_core_plan* p) {
    p->ms_fwd[0] = p->fw.projection == 0 ? elapsed(p, kStampFwdStart, kStampFwdRec) : -1.f;
    p->ms_fwd[2] = elapsed(p, p->fw.begin, kStampFwdEnd);
}

}  // namespace

extern "C" int flstm_core_create(size_t batch, size_t input_size, size_t hidden_size, flstm_core_plan** out) {
    if (!out) return FLSTM_E_INVALID;
    *out = nullptr;
    if (batch == 0 || input_size == 0 || hidden_size == 0) return FLSTM_E_INVALID;
    if (batch > (1u << 20) || input_size > (1u << 20) || hidden_size > (1u << 18)) return FLSTM_E_INVALID;
    auto* p = new (std::nothrow) flstm_core_plan();
    if (!p) return int(hipErrorOutOfMemory);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&p->num_cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess && hipDeviceGetAttribute(&p->clock_khz, hipDeviceAttributeClockRate, dev) != hipSuccess)
        p->clock_khz = 0;
    if (e == hipSuccess && (hipDeviceGetAttribute(&p->wall_khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess ||
                            p->wall_khz <= 0))
        p->wall_khz = 100000;
    if (e != hipSuccess) { delete p; return int(e); }
    p->device = dev;
    {   // this device's copy of the static scratch array: looked up now, while its device is current
        void* sp = nullptr;
        const int rc = static_scratch(dev, &sp);
        if (rc) { delete p; return rc; }
    }
    p->d.B = int(batch);
    p->d.I = int(input_size);
    p->d.H = int(hidden_size);
    p->d.Ip = int(round_up(input_size, 64));
    p->d.Hp = int(round_up(hidden_size, hidden_size > 2048 ? 64 : 32));   // (the wide backward kernel has 64-column slices)
    // Persistent launches go through the gate of launch_persistent; FLASHLSTM_COOPERATIVE_LAUNCH=1 or the option
    // "cooperative" sends them through hipLaunchCooperativeKernel instead (not for use under a rocprofiler-sdk tool: with
    // rocprofv3 attached, a process that has made a cooperative launch takes a segmentation fault inside the tool when it exits).
    {
        if (const char* v = getenv("FLASHLSTM_COOPERATIVE_LAUNCH")) p->opt_cooperative = atoi(v) != 0;
        if (const char* v = getenv("FLASHLSTM_STEP_GRAPHS")) p->opt_graphs = atoi(v) != 0;
        if (const char* v = getenv("FLASHLSTM_BWD_TWO_D")) { p->opt_two_d = atoi(v) < 0 ? 0 : (atoi(v) > 2 ? 2 : atoi(v)); p->two_d_explicit = true; }
        if (const char* v = getenv("FLASHLSTM_WAVES_FWD")) p->opt_waves_f = (atoi(v) == 4 || atoi(v) == 8) ? atoi(v) : 0;
    }
    replan(p);
    e = p->status.reserve(kStatusBytes + kAbsmaxBlocks * sizeof(unsigned));
    if (e == hipSuccess) e = hipMemset(p->status.p, 0, kStatusBytes);
    if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void**>(&p->status_host), sizeof(HostStatus), hipHostMallocDefault);
    if (e == hipSuccess) memset(p->status_host, 0, sizeof(HostStatus));
    if (e != hipSuccess) { flstm_core_destroy(p); return int(e); }
    *out = p;
    return 0;
}

extern "C" int flstm_core_destroy(flstm_core_plan* p) {
    if (!p) return FLSTM_E_INVALID;
    for (DevBuf& b : p->wfrag) b.release();
    for (DevBuf* b : {&p->wih_p, &p->wih_t, &p->part_b, &p->bias_p, &p->ring, &p->tile_words, &p->X16, &p->G, &p->Y, &p->C,
                      &p->status, &p->xch_f, &p->xch_b, &p->dYp, &p->dG, &p->dHn, &p->dC,
                      &p->dH0, &p->db_part, &p->dw_part, &p->prof})
        b->release();
    if (p->status_host) (void)hipHostFree(p->status_host);
    delete p;
    return 0;
}

extern "C" int flstm_core_set_option(flstm_core_plan* p, const char* name, long value) {
    if (!p || !name) return FLSTM_E_INVALID;
    if (!strcmp(name, "stepwise")) { p->opt_stepwise = value != 0; replan(p); return 0; }
    if (!strcmp(name, "proj_chunk")) return 0;   // (accepted; the projection is one product: forward_project)
    if (!strcmp(name, "spin_limit")) { if (value < 0) return FLSTM_E_INVALID; p->opt_spin_limit = int(value); return 0; }
    if (!strcmp(name, "spin_ms")) { if (value < 1 || value > 60000) return FLSTM_E_INVALID; p->opt_spin_ms = int(value); return 0; }
    if (!strcmp(name, "profile")) {
        p->opt_profile = value != 0;
        if (p->opt_profile) {
            FL_TRY(p->prof.reserve(16 * sizeof(long long)));
        }
        return 0;
    }
    if (!strcmp(name, "row_tiles_fwd") || !strcmp(name, "row_tiles_bwd")) {
        if (value < 0 || value > 2) return FLSTM_E_INVALID;
        (name[10] == 'f' ? p->opt_mt_f : p->opt_mt_b) = int(value);
        replan(p);
        return 0;
    }
    if (!strcmp(name, "clear_tuned")) { p->tuned.clear(); use_tuned(p, 1); return 0; }
    if (!strcmp(name, "cooperative")) { p->opt_cooperative = value != 0; replan(p); return 0; }
    if (!strcmp(name, "step_graphs")) { p->opt_graphs = value != 0; return 0; }
    if (!strcmp(name, "bwd_two_d")) { if (value < 0 || value > 2) return FLSTM_E_INVALID; p->opt_two_d = int(value); p->two_d_explicit = true; replan(p); return 0; }
    if (!strcmp(name, "waves_fwd")) {
        // wavefronts per workgroup of the forward recurrence: the one-way kernels' weight fragments are packed for 4 or 8
        // of them, so a change from one to the other un-packs them
        if (value != 0 && value != 4 && value != 8) return FLSTM_E_INVALID;
        const int before = p->Lf.nw;
        p->opt_waves_f = int(value);
        replan(p);
        if (p->Lf.nw != before) p->weights_packed = false;
        return 0;
    }
    if (!strcmp(name, "inject_stall")) { if (value < 0) return FLSTM_E_INVALID; p->inject_stall = int(value); return 0; }
    if (!strcmp(name, "dw_splits")) { if (value < 0) return FLSTM_E_INVALID; p->opt_dw_splits = int(value); return 0; }
    if (!strcmp(name, "accumulate_grads")) { p->opt_accumulate = value != 0; return 0; }
    return FLSTM_E_INVALID;
}

extern "C" long flstm_core_get_info(const flstm_core_plan* p, const char* name) {
    if (!p || !name) return -1;
    if (!strcmp(name, "persistent_fwd")) return p->Lf.persistent;
    if (!strcmp(name, "persistent_bwd")) return p->Lb.persistent;
    if (!strcmp(name, "xcd_local_fwd")) return p->Lf.xcd_local;
    if (!strcmp(name, "xcd_local_bwd")) return p->Lb.xcd_local;
    if (!strcmp(name, "resident_fwd")) return p->Lf.resident;
    if (!strcmp(name, "resident_bwd")) return p->Lb.resident;
    if (!strcmp(name, "row_tiles")) return p->Lf.mt;
    if (!strcmp(name, "row_tiles_fwd")) return p->Lf.mt;
    if (!strcmp(name, "row_tiles_bwd")) return p->Lb.mt;
    if (!strcmp(name, "cooperative")) return p->opt_cooperative;
    if (!strcmp(name, "bwd_two_d")) return p->Lb.two_d;
    if (!strcmp(name, "waves_fwd")) return rec_threads(p->Lf) / kWave;
    if (!strcmp(name, "graph_captures")) return p->graphs_f.captures + p->graphs_b.captures;
    if (!strcmp(name, "graph_replays")) return p->graphs_f.replays + p->graphs_b.replays;
    if (!strcmp(name, "graphs_disabled")) return (p->graphs_f.disabled ? 1 : 0) + (p->graphs_b.disabled ? 2 : 0);
    if (!strcmp(name, "tuned_entries")) return long(p->tuned.size());
    if (!strcmp(name, "tuned_T")) return long(p->eff_T);
    if (!strcmp(name, "tuned_row_tiles_fwd")) return p->eff_mt_f;
    if (!strcmp(name, "tuned_row_tiles_bwd")) return p->eff_mt_b;
    if (!strcmp(name, "tuned_stepwise_fwd")) return p->eff_step_f;
    if (!strcmp(name, "tuned_stepwise_bwd")) return p->eff_step_b;
    if (!strcmp(name, "tuned_dw_splits")) return p->eff_dw;
    if (!strcmp(name, "tuned_bwd_two_d")) return p->eff_two_d;
    if (!strcmp(name, "device_bytes")) {
        size_t sum = 0;
        for (const DevBuf& b : p->wfrag) sum += b.bytes;
        for (const DevBuf* b : {&p->wih_p, &p->wih_t, &p->part_b, &p->bias_p, &p->ring, &p->tile_words, &p->X16, &p->G, &p->Y, &p->C,
                                &p->status, &p->xch_f, &p->xch_b, &p->dYp, &p->dG, &p->dHn, &p->dC, &p->dH0, &p->db_part,
                                &p->dw_part, &p->prof})
            sum += b->bytes;
        return long(sum);
    }
    if (!strcmp(name, "whole_fwd")) return p->fw.whole;
    if (!strcmp(name, "projection_fwd")) return p->fw.projection;
    if (!strcmp(name, "products_shared")) return p->bw.shared;
    if (!strcmp(name, "outputs_behind")) return p->fw.behind;
    if (!strcmp(name, "rows_behind")) return p->fw.rows_behind;
    if (!strcmp(name, "slice_fwd")) return p->Lf.jb;
    if (!strcmp(name, "slice_bwd")) return p->Lb.jb;
    if (!strcmp(name, "groups_fwd")) return p->Lf.ng;
    if (!strcmp(name, "groups_bwd")) return p->Lb.ng;
    if (!strcmp(name, "few_rows_fwd")) return p->Lf.few;
    if (!strcmp(name, "few_rows_bwd")) return p->Lb.few;
    if (!strcmp(name, "fallbacks")) return p->fallbacks;
    if (!strcmp(name, "demotions_fwd")) return p->demotions_fwd;
    if (!strcmp(name, "demotions_bwd")) return p->demotions_bwd;
    if (!strcmp(name, "cooperative_refusals")) return p->coop_refusals;
    if (!strcmp(name, "hold_fwd")) return p->hold_fwd;
    if (!strcmp(name, "hold_bwd")) return p->hold_bwd;
    if (!strcmp(name, "static_scratch_bytes")) return long(kStaticScratchBytes);
    if (!strcmp(name, "num_cus")) return p->num_cus;
    if (!strcmp(name, "clock_khz")) return p->clock_khz;
    if (!strcmp(name, "hidden_padded")) return p->d.Hp;
    if (!strcmp(name, "input_padded")) return p->d.Ip;
    return -1;
}

extern "C" int flstm_core_pack_weights(flstm_core_plan* p, const float* w_ih, const float* w_hh, void* stream) {
    const int rc = core_pack_weights_async(p, w_ih, w_hh, static_cast<hipStream_t>(stream));
    if (rc) return rc;
    FL_TRY(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
    return 0;
}

int flstm_hip::core_pack_weights_async(flstm_core_plan* p, const float* w_ih, const float* w_hh, hipStream_t s) {
    if (!p || !w_ih || !w_hh) return FLSTM_E_INVALID;
    const Dims& d = p->d;
    FL_TRY(p->wih_p.reserve(size_t(4) * d.Hp * d.Ip * sizeof(half_t)));
    FL_TRY(p->wih_t.reserve(size_t(4) * d.Hp * d.Ip * sizeof(half_t)));
    // Fragments for every kernel that the options can choose for these sizes, whichever the current ones do: options and
    // tuned entries change after the weights are packed.  (The one-way kernels have theirs wherever 32-row blocks can be
    // asked for; those for short contractions, up to 512 units, add at most 2 MiB, those for few rows, up to 1024, 8 MiB.  Of these
    // last and the one-way kernel's, those that the rule reads are packed, and the others wait for a pass that needs them: packed
    // with them each time they took 8 us of the 70 of a packing of 1024 units, and a training step packs its weights.)
    FragLayout frag[kFragKinds];
    auto want = [&](int kind, const RecLayout& L, int ks, size_t fragments) -> hipError_t {
        FragLayout& f = frag[kind];
        const hipError_t e = p->wfrag[kind].reserve(fragments * kWave * sizeof(half8));
        f.out = p->wfrag[kind].as<half8>(); f.fragments = fragments; f.ks = ks;
        f.nt = L.nt; f.rot_div = L.rot_div; f.nw = L.nw; f.unit_major = L.unit_major;
        return e;
    };
    const RecLayout fwd = plan_rec_fwd(d.B, d.Hp, p->num_cus, false, 2, p->opt_waves_f), split = plan_rec_fwd(d.B, d.Hp, p->num_cus, false, 0, 0, true);
    const bool few_by_rule = plan_rec_fwd(d.B, d.Hp, p->num_cus, false).few != 0;
    const RecLayout bwd = plan_rec_bwd(d.B, d.Hp, p->num_cus, false, 2, 0), broad = plan_rec_bwd(d.B, d.Hp, p->num_cus, false, 0, 0);
    FL_TRY(want(kFragFwd, fwd, rec_fwd_ks(fwd, d.Hp), rec_fwd_fragments(fwd, d.Hp)));
    frag[kFragFwd].wide = fwd.wide;
    if (split.split || split.broad || (split.few && fwd.nw == 4)) {
        FL_TRY(want(kFragFwdSplit, split, rec_fwd_ks(split, d.Hp), rec_fwd_fragments(split, d.Hp)));
        frag[kFragFwdSplit].split = split.split;
        // (the rings here: flstm_core_forward_static allocates nothing)
        if (split.split) FL_TRY(p->ring.reserve(4 * exchange_slot_halfs(d.B, d.Hp) * sizeof(half_t)));
        if (few_by_rule) FL_TRY(p->xch_f.reserve(4 * rec_fwd_slot_halfs(split, d.B, d.Hp) * sizeof(half_t)));
    }
    p->frag_there[kFragFwd] = p->frag_there[kFragFwdSplit] = true;
    if (split.few && fwd.nw == 4) {   // (the memory is there: flstm_core_forward_static allocates nothing)
        const int later = few_by_rule ? kFragFwd : kFragFwdSplit;
        frag[later].fragments = 0;
        p->frag_there[later] = false;
    }
    FL_TRY(want(kFragBwd, bwd, rec_bwd_ks(bwd, d.Hp), rec_bwd_fragments(bwd, d.Hp)));
    if (broad.broad) FL_TRY(want(kFragBwdBroad, broad, rec_bwd_ks(broad, d.Hp), rec_bwd_fragments(broad, d.Hp)));
    if (rec_bwd_two_d_possible(d.Hp, p->num_cus)) {
        FragLayout& f = frag[kFragBwdTwoD];
        f.kq = rec_bwd_two_d_kq(d.B, d.Hp);
        f.wide = d.Hp > 2048;
        f.ks = f.wide ? rec_wide_ks(d.Hp) : d.Hp / (32 * f.kq);
        f.fragments = size_t(d.Hp / 64) * f.kq * 4 * f.ks * 4;
        FL_TRY(p->wfrag[kFragBwdTwoD].reserve(f.fragments * kWave * sizeof(half8)));
        f.out = p->wfrag[kFragBwdTwoD].as<half8>();
    }
    FL_TRY(pack_weights(d, w_ih, w_hh, p->wih_p.as<half_t>(), p->wih_t.as<half_t>(), frag, s));
    p->weights_packed = true;
    return 0;
}

extern "C" int flstm_core_pack_bias(flstm_core_plan* p, const float* b_ih, const float* b_hh, void* stream) {
    if (!p) return FLSTM_E_INVALID;
    hipStream_t s = static_cast<hipStream_t>(stream);
    FL_TRY(p->bias_p.reserve(size_t(4) * p->d.Hp * sizeof(float)));
    if (!b_ih || !b_hh) {
        // zeros for a missing vector: pack against a zeroed scratch vector
        FL_TRY(p->db_part.reserve(size_t(4) * p->d.Hp * sizeof(float)));
        FL_TRY(fill_zero(p->db_part.p, size_t(4) * p->d.Hp * sizeof(float), s));
        const float* z = p->db_part.as<float>();
        FL_TRY(pack_bias(p->d, b_ih ? b_ih : z, b_hh ? b_hh : z, p->bias_p.as<float>(), s));
    } else {
        FL_TRY(pack_bias(p->d, b_ih, b_hh, p->bias_p.as<float>(), s));
    }
    p->bias_packed = true;
    return 0;
}

namespace {

// A tensor as the bytes it covers (a null pointer: none).
struct Bytes { uintptr_t from = 0, to = 0; };
Bytes bytes_of(const void* t, size_t elements, flstm_dtype type) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(t);
    return t ? Bytes{at, at + elements * (type == FLSTM_F32 ? 4 : 2)} : Bytes{};
}
bool overlap(std::initializer_list<Bytes> some, std::initializer_list<Bytes> others) {
    for (const Bytes& a : some)
        for (const Bytes& b : others)
            if (a.from < b.to && b.from < a.to) return true;
    return false;
}

// Forward pass in three parts so that a caller can feed it in ranges of steps: setup (state rows, exchange
// ring), any number of step ranges in order (x rows -> projection -> recurrence), and the status check.
bool x_in_place(const flstm_core_plan* p, flstm_dtype x_dtype) { return x_dtype == FLSTM_F16 && p->d.I == p->d.Ip; }

// (whole_x: the operand of all steps is made here; a pass fed in ranges has not got x yet)
int forward_setup(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype, const void* h0,
                  const void* c0, flstm_dtype state_dtype, bool whole_x, hipStream_t s) {
    const Dims& d = p->d;
    const size_t TB = T * size_t(d.B);
    p->fw.T = T; p->fw.x = x; p->fw.x_dtype = x_dtype; p->fw.open = true; p->fw.whole = false; p->fw.few = p->Lf.few;
    p->fw.begin = kStampFwdBegin;
    p->fw.begin_on_device = false;
    p->beside_f.count = 0;
    if (!x_in_place(p, x_dtype)) FL_TRY(p->X16.reserve(TB * d.Ip * sizeof(half_t)));
    FL_TRY(p->G.reserve(TB * 4 * d.Hp * sizeof(half_t)));
    FL_TRY(p->Y.reserve((TB + d.B) * d.Hp * sizeof(half_t)));
    FL_TRY(p->C.reserve((TB + d.B) * d.Hp * sizeof(float)));
    const size_t xslot = rec_fwd_slot_halfs(p->Lf, d.B, d.Hp);
    FL_TRY(p->xch_f.reserve(4 * xslot * sizeof(half_t)));
    // One launch: the initial state rows (a null h0 / c0 reads as zeros), the exchange ring -- slot 0 holds h0 (rows past B
    // zero), slots 1 to 3 the 'unwritten' pattern --, the seat and phase counters, and (whole passes) the fp16 operand
    // made of x.
    OpList prep;
    const int f32 = state_dtype == FLSTM_F32;
    prep.to_half(h0, f32, size_t(d.B), d.H, size_t(d.H), 1.f, p->Y.as<half_t>(), size_t(d.B), size_t(d.Hp));
    prep.to_float(c0, f32, size_t(d.B), d.H, 1.f, p->C.as<float>(), size_t(d.Hp));
    prep.to_exchange(h0, f32, size_t(d.B), d.H, d.Hp, p->xch_f.as<half_t>(), p->Lf.few);
    prep.fill(p->xch_f.as<half_t>() + xslot, 3 * xslot * sizeof(half_t), 0xFFFFFFFFu);
    prep.fill(p->status.as<char>() + kSeatsOffset, kStatusBytes - kSeatsOffset, 0u);
    if (p->opt_profile) prep.fill(p->prof.p, 8 * sizeof(long long), 0u);
    if (whole_x && !x_in_place(p, x_dtype))
        prep.to_half(x, x_dtype == FLSTM_F32, TB, d.I, size_t(d.I), 1.f, p->X16.as<half_t>(), TB, size_t(d.Ip));
    prep.stamps = stamps_of(p);
    prep.begin = kStampFwdBegin;
    prep.stamp = kStampFwdStart;
    FL_TRY(run_ops(prep, s));
    p->seat_sets_left = kSeatSets;
    return 0;
}

// x rows of steps [t0, t0+n) as the projection's fp16 operand
int forward_operand(flstm_core_plan* p, size_t t0, size_t n, bool converted, hipStream_t s, const half_t** A, size_t* lda) {
    const Dims& d = p->d;
    if (x_in_place(p, p->fw.x_dtype)) {
        *A = static_cast<const half_t*>(p->fw.x) + t0 * d.B * d.I;
        *lda = size_t(d.I);
        return 0;
    }
    const size_t esz = p->fw.x_dtype == FLSTM_F32 ? 4 : 2;
    const char* src = static_cast<const char*>(p->fw.x) + t0 * d.B * d.I * esz;
    half_t* dst = p->X16.as<half_t>() + t0 * d.B * d.Ip;
    if (!converted) {
        OpList conv;
        conv.to_half(src, p->fw.x_dtype == FLSTM_F32, n * d.B, d.I, size_t(d.I), 1.f, dst, n * d.B, size_t(d.Ip));
        FL_TRY(run_ops(conv, s));
    }
    *A = dst;
    *lda = size_t(d.Ip);
    return 0;
}

// Whether the projection of n steps is formed beside their recurrence (ProjectBeside) by the workgroups without a seat there:
// estimated microseconds of both ways.  Where these set the pace a tile of 128 x 128 takes one of them 4.6 us and 0.52 per 64
// features (1 / 2 / 8 / 16 / 32 slabs 5.1 / 5.7 / 8.8 / 12.8 / 21.2 us, with 16 to 96 of them at work); the recurrence starts a tile
// later, for which the first ones, with memory to themselves, take 2.5 and 0.65.  In front of it the product takes what
// gemm_nt_cost says, a launch and a gap.  A step takes 1.65 us (to 768 units; few rows 1.5), 1.8 (to 1024; few rows 1.7) or 2.4 for every row
// block that a workgroup has in it; behind the last tile there are the steps of its 128 rows left.
// Measured, us a forward pass, in front / beside: 512 steps of 64 rows, 1024 features and units 1275 / 990, of 16 rows of 2048
// 1443 / 1208, of 64 rows of 640 units and 2048 features 1316 / 956; 128 steps of the first 347 / 292, 32 steps 130 / 116; 200 steps of
// 100 rows of 1536 units and 32 features, two turns a step 1036 / 946; the other side of the line: 256 steps of 200 rows of 512 units,
// 32 features and 48 workgroups to form it 509 / 704, 128 features 513 / 786; 32 steps of 32 rows of 1536 units, 1024 features 128 / 138 (512 steps
// 1439 / 1280); 211 steps of 256 rows of 384 units and 32 features 389 / 438.  Of 570 combinations measured both ways the choice is on
// average 0.15 % off the faster one, at most 3 us or 2 % where it is beside.  Fewer than 16 workgroups are not tried: where 241 and more have seats a step takes
// 8 tiles or more (17 rows of 2048 units, 113 of 1024), which so few do not keep up with.
bool beside_pays(const Dims& d, const RecLayout& L, size_t n) {
    const int helpers = rec_projecting_workgroups(L);
    if (helpers < 16) return false;
    const double slabs = d.Ip / 64, tile = slabs * 0.52 + 4.6, first = slabs * 0.65 + 2.5;
    const double rounds = double(ceil_div(ceil_div(n * d.B, 128) * (4 * d.Hp / 128), size_t(helpers)));
    const double one = d.Hp <= 768 ? (L.few == 8 ? 1.5 : 1.65) : d.Hp <= 1024 ? (L.few == 8 ? 1.7 : 1.8) : 2.4;
    const double step = one * double(ceil_div(size_t(L.nrb), size_t(L.ng)));
    const double recurrence = step * double(n), last = step * std::fmin(double(n), 128.0 / d.B);
    const double in_front = recurrence + gemm_nt_cost(int(n * d.B), 4 * d.Hp, d.Ip) + 5.0;
    return std::fmax(recurrence + 1.5 * first + 2.0, 1.05 * rounds * tile + last + 4.0) < in_front;
}
bool projects_beside(const flstm_core_plan* p, size_t n, const half_t* A) {
    return !p->opt_profile && reinterpret_cast<uintptr_t>(A) % 16 == 0 && beside_pays(p->d, p->Lf, n);
}

// Whether the 16-row blocks of a pass run in rec_fwd_few_kernel (plan_rec_fwd; 65 to 128 rows of 769 to 1024 units): from 512 steps on with the
// projection in front, from 2048 on with it beside.  That kernel's step is the shorter one once the clock has fallen under the load; at the clock
// that a short pass runs at, its stores of four bytes cost more than it gains.  Time with it over that with rec_fwd_kernel, 66 to 128 rows,
// 800 to 1024 units, 64 to 1024 features, forward alone / forward of a training step: in front 2048 steps 0.83-0.94 / 0.87-0.93, 1024 steps 0.83-0.95 /
// 0.89-0.98, 512 steps 0.86-1.00 / 0.89-1.03, 256 steps 0.98-1.05 / 0.97-1.04, 128 steps 0.99-1.08 / 1.01-1.07; beside 2048 steps 0.85-1.00 / 0.92-1.07,
// 1024 steps 0.92-1.08 / 0.99-1.13, 512 steps 0.99-1.08 / 0.99-1.09, 16 steps 0.99-1.04.  (The bits are the same either way.)
bool many_steps(const flstm_core_plan* p, size_t T) {
    const Dims& d = p->d;
    if (T < 512 || plan_rec_fwd(d.B, d.Hp, p->num_cus, false, 0, 0, true).few != 16) return false;
    return T >= 2048 || !beside_pays(d, plan_rec_fwd(d.B, d.Hp, p->num_cus, false), T);
}

// x rows of steps [t0, t0+n) -> fp16 operand -> x-projection (+ bias) in G, or left to the recurrence's launch
// (`stamp`: where the product leaves its start, if anywhere)
int forward_project(flstm_core_plan* p, size_t t0, size_t n, bool converted, bool may_leave_it, hipStream_t s, long long* stamp = nullptr) {
    const Dims& d = p->d;
    GemmNT g{};
    int rc = forward_operand(p, t0, n, converted, s, &g.A, &g.lda);
    if (rc) return rc;
    // The hoisted input projection, one product over all steps.  Cutting it into chunks of time steps (the reference's
    // projchunksz, option "proj_chunk") saves no memory here, where the gate rows of the whole pass are kept, and changes
    // no result; chunks of 64 steps of 32 rows at 1024 units took 32 launches of 24.5 us where one product takes 410 us.
    g.B = p->wih_p.as<half_t>(); g.ldb = size_t(d.Ip);
    g.M = int(n * d.B); g.N = 4 * d.Hp; g.K = d.Ip;
    g.C16 = p->G.as<half_t>() + t0 * d.B * 4 * d.Hp; g.C32 = nullptr; g.ldc = size_t(4) * d.Hp;
    g.alpha = 1.f; g.splits = 1; g.split_stride = 0;
    g.bias = p->bias_p.as<float>();   // b_ih + b_hh, packed gate order: the recurrence reads x-projection + bias
    g.stamp = stamp;
    p->project = ProjectBeside{};
    p->fw.projection = 0;
    if (may_leave_it && projects_beside(p, n, g.A)) {
        const size_t words = ceil_div(size_t(g.M), 128) * (g.N / 128) * sizeof(unsigned);
        if (words <= p->tile_words.bytes || !p->static_call) {
            if (words > p->tile_words.bytes || p->tile_mark == ~0u) {
                FL_TRY(p->tile_words.reserve(words));
                FL_TRY(fill_zero(p->tile_words.p, p->tile_words.bytes, s));
                p->tile_mark = 0;
            }
            p->project.A = g.A; p->project.lda = g.lda; p->project.B = g.B; p->project.bias = g.bias; p->project.C = g.C16;
            p->project.M = g.M; p->project.N = g.N; p->project.K = g.K;
            p->project.ready = p->tile_words.as<unsigned>();
            p->project.mark = ++p->tile_mark;
            rec_share_columns(p->Lf, p->project);
            p->fw.projection = 1;
            return 0;
        }
    }
    FL_TRY(launch_gemm_nt(g, s));
    return 0;
}

// the copies waiting for the next recurrence launch become that launch's
template <typename Args>
void take_beside(BesideCopies& waiting, Args& a) {
    if (waiting.count > 0) { a.beside = waiting; a.beside.ticket = a.seats + 8; }
    else a.beside.count = 0;   // (a later window of batch rows: the first one has made them)
    waiting.count = 0;
}

// The fragments of the forward layout; those that packing left out are made here the first time that a pass needs them.
int forward_fragments(flstm_core_plan* p, const half8** fragments, hipStream_t s) {
    const int kind = p->Lf.split || p->Lf.broad || p->Lf.few ? kFragFwdSplit : kFragFwd;
    if (!p->frag_there[kind]) {
        const int other = kind == kFragFwd ? kFragFwdSplit : kFragFwd;
        FL_TRY(reorder_fragments(p->wfrag[other].as<half8>(), p->wfrag[kind].as<half8>(), rec_fwd_fragments(p->Lf, p->d.Hp), kind == kFragFwd, s));
        p->frag_there[kind] = true;
    }
    *fragments = p->wfrag[kind].as<half8>();
    return 0;
}

// The exchange ring as the steps from t0 on expect it, for a layout that came into force during the pass: h of the last step from its
// state rows, the other slots 'unwritten'.
int forward_ring_again(flstm_core_plan* p, size_t t0, hipStream_t s) {
    const Dims& d = p->d;
    const size_t xslot = rec_fwd_slot_halfs(p->Lf, d.B, d.Hp);
    FL_TRY(p->xch_f.reserve(4 * xslot * sizeof(half_t)));
    OpList ring;
    for (size_t k = 0; k < 4; ++k) {
        half_t* const slot = p->xch_f.as<half_t>() + k * xslot;
        if (k == (t0 & 3)) ring.to_exchange(p->Y.as<half_t>() + t0 * d.B * d.Hp, 0, size_t(d.B), d.Hp, d.Hp, slot, p->Lf.few);
        else ring.fill(slot, xslot * sizeof(half_t), 0xFFFFFFFFu);
    }
    p->fw.few = p->Lf.few;
    FL_TRY(run_ops(ring, s));
    return 0;
}

int forward_recur(flstm_core_plan* p, size_t t0, size_t n, hipStream_t s) {
    const Dims& d = p->d;
    if (p->fw.few != p->Lf.few) {
        const int changed = forward_ring_again(p, t0, s);
        if (changed) return changed;
    }
    RecFwdArgs a;
    memset(static_cast<void*>(&a), 0, sizeof(a));   // (padding too: the arguments are the key of a captured graph)
    int rc = forward_fragments(p, &a.wfrag, s);
    if (rc) return rc;
    a.Y = p->Y.as<half_t>(); a.G = p->G.as<half_t>(); a.C = p->C.as<float>();
    a.y_out = p->fw.y_direct;
    a.X = p->xch_f.as<half_t>(); a.x_slot = rec_fwd_slot_halfs(p->Lf, d.B, d.Hp);
    a.status = p->status.as<int>();
    a.delay_hint = p->status.as<int>() + 1;
    a.stamps = stamps_of(p) + kStampFwdRec;
    rc = next_seats(p, &a.seats, s);
    if (rc) return rc;
    take_beside(p->beside_f, a);
    if (p->project.M != 0) {   // (else all of it stays zero: an assigned struct brings padding of its own into a graph's key)
        a.project = p->project;
        a.project.ticket = a.seats + 16;
        p->project = ProjectBeside{};
    }
    a.B = d.B; a.Hp = d.Hp; a.T = int(p->fw.T); a.t0 = int(t0); a.t1 = int(t0 + n);
    a.spin_limit = p->opt_spin_limit;
    a.spin_ticks = (long long)p->opt_spin_ms * p->wall_khz;
    a.prof = p->opt_profile ? p->prof.as<long long>() : nullptr;
    // Step-wise launches are replayed from a captured graph only for whole passes: a sequence fed in ranges has a new
    // range (a new graph) every call, each used once.  Never inside flstm_core_forward_static (a capture allocates).
    const bool whole = (t0 == 0 && n == p->fw.T);
    hipError_t e = launch_rec_fwd(p->Lf, a, s, (p->opt_graphs && whole && !p->static_call) ? &p->graphs_f : nullptr);
    if (e == hipErrorCooperativeLaunchTooLarge && p->Lf.persistent) {
        // the grid cannot be co-resident: this direction runs step-wise from now on, starting with these steps
        p->refused_fwd = true;
        p->coop_refusals++;
        replan(p);
        OpList copies;   // step-wise launches have no workgroups to spare
        for (int i = 0; i < a.beside.count; ++i) copies.op[copies.count++] = a.beside.op[i];
        a.beside.count = 0;
        FL_TRY(run_ops(copies, s));
        if (a.project.M != 0) {
            rc = forward_project(p, t0, n, true, false, s);
            if (rc) return rc;
            a.project = ProjectBeside{};
        }
        e = launch_rec_fwd(p->Lf, a, s, nullptr);   // (a plan's blocks are the same step-wise: the ring and the fragments stand)
    }
    FL_TRY(e);
    return 0;
}

int forward_once(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype, const void* h0,
                 const void* c0, flstm_dtype state_dtype, hipStream_t s) {
    int rc = forward_setup(p, T, x, x_dtype, h0, c0, state_dtype, true, s);
    if (rc) return rc;
    rc = forward_project(p, 0, T, true, true, s);
    if (rc) return rc;
    return forward_recur(p, 0, T, s);
}

void final_states(const flstm_core_plan* p, size_t TB, void* hy, void* cy, flstm_dtype dtype, OpList& out) {
    const Dims& d = p->d;
    out.unpad(p->Y.as<half_t>() + TB * d.Hp, 0, size_t(d.Hp), size_t(d.B), d.H, 1.f, hy, dtype == FLSTM_F32);
    out.unpad(p->C.as<float>() + TB * d.Hp, 1, size_t(d.Hp), size_t(d.B), d.H, 1.f, cy, dtype == FLSTM_F32);
}

// Whether a pass can be one launch (rec_fwd_whole_kernel): the layout is the one for short contractions.
bool whole_possible(const flstm_core_plan* p) { return !p->opt_profile && p->ring.p && rec_whole_possible(p->Lf); }
// Microseconds a step that the projection takes inside it (fp16 rows of up to 128 features): what the exchange does not hide.
// Measured over 64 to 1024 steps, in front / inside, us a pass: 32 units and one row 523 / 627 over 1024 steps; 256 units, 64 rows and 64
// features 874 / 867, 128 features 871 / 882, with caches 891 / 917; 200 rows (two waves a workgroup) 1207 / 967; 384 units, 64
// features, one row 973 / 1033, 64 rows 1088 / 1024; 512 units, 16 rows, 128 features and 256 steps 19 / 2 less than separate launches.
double inside_step(const flstm_core_plan* p, bool save) {
    const Dims& d = p->d;
    const bool long_rows = d.Ip > 64;
    if (d.Hp > 256) return long_rows ? (save ? 0.1 : 0.05) : d.B >= 4 || d.Hp > 384 ? 0.0 : 0.06;
    if (p->Lf.split > 1) return 0.0;
    const double short_rows = d.Hp > 128 ? (save ? 0.05 : 0.022) : d.Hp < 128 || save ? 0.1 : 0.06;
    return short_rows + (long_rows ? (d.Hp > 128 ? 0.03 : 0.035) : 0.0);
}
// ... and whether that launch forms the projection itself: the input rows are short enough for a wave to hold its part of W_ih,
// fp16 rows used in place are aligned, and it is the faster way: it saves the product, a launch and a gap.  Up to 32 steps always;
// rows of more than 128 features cost 0.3 us a step.  (Two and four waves a workgroup with 65 to 128 features: up to 192 units only
// for 64 steps, 192 units and 200 rows 613 / 630 us over 512 with caches.)
bool whole_projects(const flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype, bool save) {
    const Dims& d = p->d;
    if (d.Ip > kRecWholeInput || (x_in_place(p, x_dtype) && reinterpret_cast<uintptr_t>(x) % 16 != 0)) return false;
    if (T <= 32) return true;
    if (d.Ip > 128 || (p->Lf.split > 1 && d.Hp <= 192 && d.Ip > 64 && T > 64)) return false;
    return double(T) * inside_step(p, save) < gemm_nt_cost(int(T * size_t(d.B)), 4 * d.Hp, d.Ip) + 3.0;
}
// ... and whether one launch is the faster way at all.  It saves two launches and their gaps, 8 us.  With one wave a workgroup and up
// to 256 units its steps are longer for what they write (caches, the caller's y) between h and the next request, 0.03 us with
// caches, 0.015 without at 64 to 128 units, 16 to 256 rows and up to 128 features.  Separate / one launch, us: 16 rows of 64 units, 32
// features, with caches 108 / 103 over 128 steps, 180 / 184 over 256, 601 / 628 over 1024; without 601 / 614; 133 rows of 120 units and 1799
// features over 1292 steps, without, 1930 / 1869.  Two and more waves and more units gain throughout
// (512 rows of 256 units 2669 -> 998 us over 1024 steps).
bool whole_pays(const flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype, bool save) {
    const Dims& d = p->d;
    if (p->Lf.split > 1 || d.Hp > 256 || T <= 32) return true;
    double loss = double(T) * (save ? 0.03 : d.Hp >= 64 && d.Hp <= 128 && d.Ip <= 128 && d.B >= 16 && d.B <= 256 ? 0.015 : 0.0);
    if (whole_projects(p, T, x, x_dtype, save))
        loss += double(T) * inside_step(p, save) - gemm_nt_cost(int(T * size_t(d.B)), 4 * d.Hp, d.Ip) - 3.0;
    return loss <= 8.0;
}

int forward_whole(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype, const void* h0, const void* c0,
                  flstm_dtype state_dtype, void* y, flstm_dtype y_dtype, void* hy, void* cy, flstm_dtype out_state_dtype,
                  bool save, hipStream_t s) {
    const Dims& d = p->d;
    const size_t TB = T * size_t(d.B), xslot = exchange_slot_halfs(d.B, d.Hp);
    const int f32 = state_dtype == FLSTM_F32;
    p->fw.T = T; p->fw.x = x; p->fw.x_dtype = x_dtype; p->fw.open = true; p->fw.whole = true;
    RecWholeArgs a{};
    OpList prep;   // what there is to do in front of it: converted rows, a ring that is not ready, an h0 no 16-byte load fits
    const bool projects = whole_projects(p, T, x, x_dtype, save);
    if (x_in_place(p, x_dtype)) {
        a.x = static_cast<const half_t*>(x);
        a.ldx = d.I;
    } else {
        FL_TRY(p->X16.reserve(TB * d.Ip * sizeof(half_t)));
        prep.to_half(x, x_dtype == FLSTM_F32, TB, d.I, size_t(d.I), 1.f, p->X16.as<half_t>(), TB, size_t(d.Ip));
        a.x = p->X16.as<half_t>();
        a.ldx = d.Ip;
    }
    if (!p->ring_ready) {
        p->ring_base = 0;
        prep.fill(p->ring.as<half_t>() + xslot, 3 * xslot * sizeof(half_t), 0xFFFFFFFFu);
    }
    a.base = p->ring_base;
    a.h0_in_ring = h0 && (d.H % 8 != 0 || reinterpret_cast<uintptr_t>(h0) % 16 != 0);
    if (a.h0_in_ring) prep.to_exchange(h0, f32, size_t(d.B), d.H, d.Hp, p->ring.as<half_t>() + size_t(a.base) * xslot);
    p->ring_ready = false;   // (until the pass is known to have gone through)
    if (save || !projects) FL_TRY(p->G.reserve(TB * 4 * d.Hp * sizeof(half_t)));
    if (save) {
        FL_TRY(p->Y.reserve((TB + d.B) * d.Hp * sizeof(half_t)));
        FL_TRY(p->C.reserve((TB + d.B) * d.Hp * sizeof(float)));
        a.Y = p->Y.as<half_t>(); a.C = p->C.as<float>();
    }
    a.G = p->G.as<half_t>();
    a.status = p->fw.behind ? p->status.as<int>() : &p->status_host->status;   // (behind: published by the outputs' launch)
    a.stamps = p->fw.behind ? stamps_of(p) : p->status_host->stamps;
    // What comes in front leaves its stamps in the status block, where flstm_core_last_ms fetches them: written to host memory they
    // made each such launch 1.5 us longer (16 steps of 16 rows of 64 units and 32 features 39.3 -> 42.1).
    p->fw.begin = prep.count > 0 ? kStampFwdBegin : projects ? kStampFwdRec : kStampFwdStart;   // (of whichever launch comes first)
    p->fw.begin_on_device = p->fw.begin != kStampFwdRec && !p->fw.behind;
    if (prep.count > 0) {
        prep.stamps = stamps_of(p);
        prep.begin = kStampFwdBegin;
        prep.stamp = kStampFwdStart;
        FL_TRY(run_ops(prep, s));
    }
    p->fw.projection = 2;
    if (!projects) {
        a.x = nullptr;
        const int rc = forward_project(p, 0, T, true, false, s, prep.count > 0 ? nullptr : stamps_of(p) + kStampFwdStart);
        if (rc) return rc;
    }
    a.wfrag = p->wfrag[kFragFwdSplit].as<half8>();
    a.wih = p->wih_p.as<half_t>(); a.bias = p->bias_p.as<float>(); a.Ip = d.Ip;
    a.h0 = h0; a.c0 = c0; a.state_f32 = f32;
    a.ring = p->ring.as<half_t>(); a.x_slot = xslot;
    a.y = y; a.hy = hy; a.cy = cy;
    a.y_f32 = y_dtype == FLSTM_F32; a.out_f32 = out_state_dtype == FLSTM_F32;
    auto pairs = [&](const void* t, int is_f32) { return d.H % 2 == 0 && reinterpret_cast<uintptr_t>(t) % (is_f32 ? 8 : 4) == 0; };
    a.y_pairs = pairs(y, a.y_f32); a.hy_pairs = pairs(hy, a.out_f32); a.cy_pairs = pairs(cy, a.out_f32);
    int rc = next_seats(p, &a.seats, s);
    if (rc) return rc;
    p->status_host->status = 0;   // (nothing of this plan is running: every pass is waited for)
    a.B = d.B; a.H = d.H; a.Hp = d.Hp; a.T = int(T);
    a.spin_limit = p->opt_spin_limit;
    a.spin_ticks = (long long)p->opt_spin_ms * p->wall_khz;
    FL_TRY(launch_rec_fwd_whole(p->Lf, a, s));
    return 0;
}

// Outputs and final states out of the plan's own arrays, one launch; the last of a pass.
int forward_outputs(flstm_core_plan* p, size_t TB, void* y, flstm_dtype y_dtype, void* hy, void* cy, flstm_dtype out_state_dtype,
                    hipStream_t s) {
    const Dims& d = p->d;
    OpList out;
    out.only_if_ok = p->fw.behind;
    out.unpad(p->Y.as<half_t>() + size_t(d.B) * d.Hp, 0, size_t(d.Hp), TB, d.H, 1.f, y, y_dtype == FLSTM_F32);
    final_states(p, TB, hy, cy, out_state_dtype, out);
    return publish_with(p, out, kStampFwdEnd, s);
}

// One whole forward pass, enqueued: projection, recurrence, outputs, status.  The outputs are written behind the
// recurrence without waiting for its status: if the persistent launch gave up, the whole pass is repeated step-wise
// and overwrites them -- unless one of them lies in an input, which the repeat will read: then the launch that writes them looks
// at the status first.
// A caller may hand over outputs that lie in inputs: the state carried in place (hy is h0, cy is c0), y over x.  Within the
// recurrence's launch nothing orders one workgroup's outputs behind another's reads of h0 (a single step has no exchange) or of
// x (rows read by the projection's tiles, or a step ahead), so such a pass writes only the plan's own arrays there, as one that
// saves its caches does, and the caller's tensors are written by a launch behind it: one step of a row of 256 units takes 27.8 us
// with its state in place, 21.5 with outputs of its own, 37 as separate launches throughout.  A recurrence of separate launches,
// whose states leave in a launch behind it anyway, goes on writing a y that lies in no input (512 steps of 64 rows of 1024 units
// with the state in place 976 -> 955 us).  A whole pass does not: 64 steps of 64 rows of 256 units take 84 us with y copied, 88
// with y and the caches both written from within.
int forward_enqueue(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype, const void* h0, const void* c0,
                    flstm_dtype state_dtype, void* y, flstm_dtype y_dtype, void* hy, void* cy,
                    flstm_dtype out_state_dtype, bool save, hipStream_t s) {
    const Dims& d = p->d;
    const size_t TB = T * size_t(d.B);
    use_tuned(p, T);
    p->fw.whole = false;
    const size_t BH = size_t(d.B) * d.H;
    const auto inputs = {bytes_of(x, TB * d.I, x_dtype), bytes_of(h0, BH, state_dtype), bytes_of(c0, BH, state_dtype)};
    const bool rows_behind = overlap({bytes_of(y, TB * d.H, y_dtype)}, inputs);
    const bool behind = rows_behind || overlap({bytes_of(hy, BH, out_state_dtype), bytes_of(cy, BH, out_state_dtype)}, inputs);
    p->fw.behind = behind;
    if (whole_possible(p) && whole_pays(p, T, x, x_dtype, save || behind)) {
        p->fw.rows_behind = behind;
        const int rc = behind ? forward_whole(p, T, x, x_dtype, h0, c0, state_dtype, nullptr, y_dtype, nullptr, nullptr, out_state_dtype, true, s)
                              : forward_whole(p, T, x, x_dtype, h0, c0, state_dtype, y, y_dtype, hy, cy, out_state_dtype, save, s);
        if (rc == 0 && behind) return forward_outputs(p, TB, y, y_dtype, hy, cy, out_state_dtype, s);
        if (rc != int(hipErrorCooperativeLaunchTooLarge)) return rc;
        p->refused_fwd = true;   // (as in forward_recur)
        p->coop_refusals++;
        p->fw.whole = false;
        replan(p);
    }
    // An fp16 output whose rows are the state rows is written by the persistent recurrence itself (no copy afterwards).
    // Step-wise launches leave it to the copy: every argument of theirs is then plan-owned, and the graph they were
    // captured into can be replayed on the next pass.
    half_t* const y_direct =
        (y && y_dtype == FLSTM_F16 && d.H == d.Hp && p->Lf.persistent && !rows_behind) ? static_cast<half_t*>(y) : nullptr;
    p->fw.y_direct = y_direct;
    p->fw.rows_behind = behind && y && !y_direct;
    int rc = forward_once(p, T, x, x_dtype, h0, c0, state_dtype, s);
    p->fw.y_direct = nullptr;
    if (rc) return rc;
    return forward_outputs(p, TB, y_direct ? nullptr : y, y_dtype, hy, cy, out_state_dtype, s);
}
// ... once the stream has been waited for: FLSTM_E_STALLED if it has to be repeated (demoted if it was persistent)
int forward_conclude(flstm_core_plan* p, hipStream_t s) {
    int st = 0;
    int rc = take_status(p, s, &st);
    if (rc) return rc;
    if (p->fw.whole && st == 0) {
        p->ring_base = int((size_t(p->ring_base) + p->fw.T - 1) & 3);
        p->ring_ready = true;
    }
    if (st != 0) {
        p->fw.begin_on_device = false;   // (there are no times of a pass that gave up)
        if (p->Lf.persistent) demote(p, true);   // workgroups not co-resident or not where expected: next time with one launch per step
        return FLSTM_E_STALLED;
    }
    pass_done(p, true);
    if (p->opt_profile) FL_TRY(hipMemcpy(p->prof_f, p->prof.p, sizeof(p->prof_f), hipMemcpyDeviceToHost));
    p->ms_fwd[1] = elapsed(p, kStampFwdRec, kStampFwdRecEnd);
    if (!p->fw.begin_on_device) from_the_beginning(p);
    p->fw.open = false;
    return 0;
}

int forward_pass(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype, const void* h0, const void* c0,
                 flstm_dtype state_dtype, void* y, flstm_dtype y_dtype, void* hy, void* cy,
                 flstm_dtype out_state_dtype, bool save, hipStream_t s) {
    for (int attempt = 0;; ++attempt) {
        int rc = forward_enqueue(p, T, x, x_dtype, h0, c0, state_dtype, y, y_dtype, hy, cy, out_state_dtype, save, s);
        if (rc) return rc;
        rc = wait_stream(s);
        if (rc) return rc;
        const bool persistent = p->Lf.persistent != 0;
        rc = forward_conclude(p, s);
        if (rc != FLSTM_E_STALLED || !persistent || attempt > 0) return rc;
    }
}

}  // namespace

extern "C" int flstm_core_forward(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype,
                                  const void* h0, const void* c0, flstm_dtype state_dtype, void* y,
                                  flstm_dtype y_dtype, void* hy, void* cy, flstm_dtype out_state_dtype,
                                  int save_for_backward, void* stream) {
    if (!p) return FLSTM_E_INVALID;
    if (!p->weights_packed || !p->bias_packed) return FLSTM_E_NOT_PACKED;
    if (T == 0) return 0;
    if (!x || T > (size_t(1) << 24)) return FLSTM_E_INVALID;
    p->have_cache = false;
    int rc = forward_pass(p, T, x, x_dtype, h0, c0, state_dtype, y, y_dtype, hy, cy, out_state_dtype,
                          save_for_backward != 0, static_cast<hipStream_t>(stream));
    p->fw.open = false;   // (also when the pass failed: no range of steps may follow it)
    if (rc) return rc;
    if (save_for_backward) { p->have_cache = true; p->T_cache = T; }
    return 0;
}

namespace {

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

}  // namespace

extern "C" int flstm_core_forward_static(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype,
                                         const void* h0, const void* c0, flstm_dtype state_dtype, void* y,
                                         flstm_dtype y_dtype, void* hy, void* cy, flstm_dtype out_state_dtype,
                                         void* stream) {
    if (!p) return FLSTM_E_INVALID;
    if (!p->weights_packed || !p->bias_packed) return FLSTM_E_NOT_PACKED;
    if (T == 0) return 0;
    if (!x || T > (size_t(1) << 24) || p->fw.open || p->bw.open) return FLSTM_E_INVALID;
    int dev = -1;
    FL_TRY(hipGetDevice(&dev));
    if (dev != p->device) return FLSTM_E_INVALID;
    void* base = nullptr;
    int rc = static_scratch(dev, &base);
    if (rc) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Dims& d = p->d;
    const size_t TB = T * size_t(d.B);
    // the same buffers forward_setup() sizes, carved out of the static array instead of allocated
    const size_t need[5] = {x_in_place(p, x_dtype) ? 0 : TB * d.Ip * sizeof(half_t),
                            TB * 4 * d.Hp * sizeof(half_t),
                            (TB + d.B) * d.Hp * sizeof(half_t),
                            (TB + d.B) * d.Hp * sizeof(float),
                            4 * exchange_slot_halfs(d.B, d.Hp) * sizeof(half_t)};
    size_t off[5], total = align256(kStatusBytes);   // (the limit counts a status block; the plan's own is used)
    for (int i = 0; i < 5; ++i) { off[i] = total; total += align256(need[i]); }
    if (total > kStaticScratchBytes) return FLSTM_E_TOO_LARGE;
    char* b = static_cast<char*>(base);
    DevBuf* slot[5] = {&p->X16, &p->G, &p->Y, &p->C, &p->xch_f};
    // (the ring of RecLayout::few may be larger than the one that the limit counts: where the rule takes that layout, packing has reserved
    // it in the plan, and the pass sums in the order of flstm_core_forward up to the limit)
    const int carved = plan_rec_fwd(d.B, d.Hp, p->num_cus, false).few ? 4 : 5;
    DevBuf saved[5];
    for (int i = 0; i < carved; ++i) { saved[i] = *slot[i]; *slot[i] = DevBuf::view(b + off[i], need[i]); }
    const bool had_cache = p->have_cache;
    p->have_cache = false;   // (the plan's own caches are untouched, but no pass may use the borrowed ones later)
    // (step-wise launches, if the pass comes to them, are plain launches: a graph capture allocates)
    p->static_call = true;
    rc = forward_pass(p, T, x, x_dtype, h0, c0, state_dtype, y, y_dtype, hy, cy, out_state_dtype, false, s);
    p->static_call = false;
    p->fw.open = false;   // (also when the pass failed: the next call must not find a pass in progress)
    for (int i = 0; i < carved; ++i) *slot[i] = saved[i];
    p->have_cache = had_cache;
    return rc;
}

namespace {

// Backward recurrence in parts, like the forward pass: setup, step ranges from the end of the sequence towards
// its start (dY rows -> BPTT steps -> dX rows), and the weight-gradient GEMMs over the whole sequence.
int backward_setup(flstm_core_plan* p, size_t T, const void* dY, flstm_dtype dy_dtype, const void* d_hn,
                   const void* d_cn, flstm_dtype dstate_dtype, const BwdScales& k, void* dx, flstm_dtype dx_dtype,
                   bool whole_dy, hipStream_t s) {
    const Dims& d = p->d;
    const size_t TB = T * size_t(d.B);
    p->bw.T = T; p->bw.dY = dY; p->bw.dy_dtype = dy_dtype; p->bw.k = k; p->bw.dx = dx; p->bw.dx_dtype = dx_dtype;
    p->bw.open = true;
    const RecLayout& L = p->bw.L = p->Lb;
    p->beside_b.count = 0;
    // (step-wise launches always read a plan-owned copy, so that their captured graph can be replayed)
    if (dy_dtype == FLSTM_F16 && d.H == d.Hp && L.persistent) {
        p->bw.dYk = static_cast<const half_t*>(dY);
        p->bw.dy_scale = k.dy;
    } else {
        FL_TRY(p->dYp.reserve(TB * d.Hp * sizeof(half_t)));
        p->bw.dYk = p->dYp.as<half_t>();
        p->bw.dy_scale = 1.f;   // the scale is applied while the rows are converted
    }
    const size_t st_bytes = size_t(d.B) * d.Hp * sizeof(float);
    FL_TRY(p->dHn.reserve(st_bytes));
    FL_TRY(p->dC.reserve(st_bytes));
    FL_TRY(p->dH0.reserve(st_bytes));
    FL_TRY(p->dG.reserve(TB * 4 * d.Hp * sizeof(half_t)));
    FL_TRY(p->db_part.reserve(size_t(L.ng) * 4 * d.Hp * sizeof(float)));
    const size_t xslot = rec_bwd_slot_halfs(L, d.B, d.Hp);
    const size_t dg_slots = size_t(rec_bwd_dg_slots(L));
    FL_TRY(p->xch_b.reserve(dg_slots * xslot * sizeof(half_t)));
    // One launch (see forward_setup): the dG ring 'unwritten', the ring of partial sums in its starting parities, the
    // scaled state gradients, the bias-gradient partials, the seat counters, the phase counters.
    static_assert(kRecBwdPartSlots + 7 <= kMaxOps, "what an OpList holds");
    OpList prep;
    prep.fill(p->xch_b.p, dg_slots * xslot * sizeof(half_t), 0xFFFFFFFFu);
    if (L.two_d) {
        const size_t pslot = rec_bwd_part_slot_floats(L) * sizeof(float);
        FL_TRY(p->part_b.reserve(kRecBwdPartSlots * pslot));
        for (int i = 0; i < kRecBwdPartSlots; ++i)
            prep.fill(static_cast<char*>(p->part_b.p) + size_t(i) * pslot, pslot, rec_bwd_part_fill(L, i, int(T)));
    }
    prep.to_float(d_hn, dstate_dtype == FLSTM_F32, size_t(d.B), d.H, k.state, p->dHn.as<float>(), size_t(d.Hp));
    prep.to_float(d_cn, dstate_dtype == FLSTM_F32, size_t(d.B), d.H, k.state, p->dC.as<float>(), size_t(d.Hp));
    prep.fill(p->db_part.p, size_t(L.ng) * 4 * d.Hp * sizeof(float), 0u);
    prep.fill(p->status.as<char>() + kSeatsOffset, kStatusBytes - kSeatsOffset, 0u);
    if (p->opt_profile) prep.fill(p->prof.as<long long>() + 8, 8 * sizeof(long long), 0u);
    if (whole_dy && p->bw.dYk != dY)
        prep.to_half(dY, dy_dtype == FLSTM_F32, TB, d.H, size_t(d.H), k.dy, p->dYp.as<half_t>(), TB, size_t(d.Hp));
    prep.stamps = stamps_of(p);
    prep.begin = kStampBwdBegin;
    prep.stamp = kStampBwdStart;
    FL_TRY(run_ops(prep, s));
    p->seat_sets_left = kSeatSets;
    return 0;
}

// steps t_hi .. t_lo (t_lo = -1 includes the closing dh0 product); dY rows of these steps are converted first
// when the caller's dY cannot be used in place
int backward_recur(flstm_core_plan* p, long t_hi, long t_lo, bool converted, hipStream_t s) {
    const Dims& d = p->d;
    const RecLayout& L = p->bw.L;
    const long lo = t_lo < 0 ? 0 : t_lo;
    if (!converted && p->bw.dYk != p->bw.dY && t_hi >= lo) {
        const size_t esz = p->bw.dy_dtype == FLSTM_F32 ? 4 : 2;
        const size_t rows = size_t(t_hi - lo + 1) * d.B;
        const char* src = static_cast<const char*>(p->bw.dY) + size_t(lo) * d.B * d.H * esz;
        half_t* dst = p->dYp.as<half_t>() + size_t(lo) * d.B * d.Hp;
        OpList conv;
        conv.to_half(src, p->bw.dy_dtype == FLSTM_F32, rows, d.H, size_t(d.H), p->bw.k.dy, dst, rows, size_t(d.Hp));
        FL_TRY(run_ops(conv, s));
    }
    RecBwdArgs a;
    memset(static_cast<void*>(&a), 0, sizeof(a));   // (as in forward_recur)
    a.wfrag = p->wfrag[L.broad ? kFragBwdBroad : kFragBwd].as<half8>();
    a.G = p->G.as<half_t>(); a.C = p->C.as<float>(); a.dY = p->bw.dYk; a.dG = p->dG.as<half_t>();
    a.dHn = p->dHn.as<float>(); a.dC = p->dC.as<float>(); a.dH0 = p->dH0.as<float>();
    a.X = p->xch_b.as<half_t>(); a.x_slot = rec_bwd_slot_halfs(L, d.B, d.Hp);
    if (L.two_d) {
        a.wfrag2 = p->wfrag[kFragBwdTwoD].as<half8>();
        a.P = p->part_b.as<float>();
        a.p_slot = rec_bwd_part_slot_floats(L);
    }
    a.db_part = p->db_part.as<float>();
    a.status = p->status.as<int>();
    a.delay_hint = p->status.as<int>() + 2;
    a.stamp_end = stamps_of(p) + kStampBwdRecEnd;
    a.B = d.B; a.Hp = d.Hp; a.T = int(p->bw.T); a.dy_scale = p->bw.dy_scale;
    a.t_hi = int(t_hi); a.t_lo = int(t_lo);
    a.spin_limit = p->opt_spin_limit;
    a.spin_ticks = (long long)p->opt_spin_ms * p->wall_khz;
    a.prof = p->opt_profile ? p->prof.as<long long>() + 8 : nullptr;
    // One launch, or one per window of batch rows (RecLayout::win_rows).  The windows share the ring of partial sums,
    // so every launch of a windowed pass starts from a ring prepared for ITS first product step (a single window's
    // launches continue each other's parities instead).
    const int win = (L.two_d && L.win_rows) ? L.win_rows : d.B;
    for (int b_lo = 0; b_lo < d.B; b_lo += win) {
        a.b_lo = b_lo;
        a.b_hi = b_lo + win < d.B ? b_lo + win : d.B;
        int rc = next_seats(p, &a.seats, s);
        if (rc) return rc;
        take_beside(p->beside_b, a);
        if (win < d.B) {
            const size_t pslot = a.p_slot * sizeof(float);
            const int first_T = t_hi >= long(p->bw.T) - 1 ? int(p->bw.T) : int(t_hi) + 2;   // (its first product step is first_T - 2)
            for (int k = 0; k < kRecBwdPartSlots; ++k)
                FL_TRY(fill_words(static_cast<char*>(p->part_b.p) + size_t(k) * pslot, pslot, rec_bwd_part_fill(L, k, first_T), s));
        }
        const bool whole = (t_hi == long(p->bw.T) - 1 && t_lo == -1);   // (graphs for whole passes only: see forward_recur)
        hipError_t e = launch_rec_bwd(L, a, s, (p->opt_graphs && whole) ? &p->graphs_b : nullptr);
        if (e == hipErrorCooperativeLaunchTooLarge && L.persistent) return int(e);   // (handled by the caller: the layout changes)
        FL_TRY(e);
    }
    return 0;
}

// dX rows of steps [t_lo, t_hi] = dG * W_ih  (contraction over the packed gate columns)
GemmNT dx_product(flstm_core_plan* p, long t_hi, long t_lo) {
    const Dims& d = p->d;
    const size_t row0 = size_t(t_lo) * d.B, rows = size_t(t_hi - t_lo + 1) * d.B;
    GemmNT g{};
    g.A = p->dG.as<half_t>() + row0 * 4 * d.Hp; g.lda = size_t(4) * d.Hp;
    g.B = p->wih_t.as<half_t>(); g.ldb = size_t(4) * d.Hp;
    g.M = int(rows); g.N = d.I; g.K = 4 * d.Hp;
    if (p->bw.dx_dtype == FLSTM_F32) g.C32 = static_cast<float*>(p->bw.dx) + row0 * d.I;
    else g.C16 = static_cast<half_t*>(p->bw.dx) + row0 * d.I;
    g.ldc = size_t(d.I); g.alpha = p->bw.k.dx; g.splits = 1; g.split_stride = 0;
    return g;
}
int backward_dx(flstm_core_plan* p, long t_hi, long t_lo, hipStream_t s) {
    if (!p->bw.dx || t_hi < t_lo) return 0;
    FL_TRY(launch_gemm_nt(dx_product(p, t_hi, t_lo), s));
    return 0;
}

int backward_rec_once(flstm_core_plan* p, size_t T, const void* dY, flstm_dtype dy_dtype, const void* d_hn,
                      const void* d_cn, flstm_dtype dstate_dtype, const BwdScales& k, void* dx, flstm_dtype dx_dtype,
                      hipStream_t s) {
    int rc = backward_setup(p, T, dY, dy_dtype, d_hn, d_cn, dstate_dtype, k, dx, dx_dtype, true, s);
    if (rc) return rc;
    return backward_recur(p, long(T) - 1, -1, true, s);
}

// dW_ih = dG^T * X and dW_hh = dG^T * H_prev over the whole sequence, bias gradient and state gradients (enqueued; the
// last launch of a pass).  `with_dx`: a whole pass, whose dX is formed here as well, in the same launch where both products are
// small (launch_gemm_tn_and_nt).
int backward_finish(flstm_core_plan* p, const void* x, flstm_dtype x_dtype, bool with_dx, float* dW_ih, float* dW_hh,
                    float* db_ih, float* db_hh, float* dh0, float* dc0, hipStream_t s) {
    const Dims& d = p->d;
    const size_t TB = p->bw.T * size_t(d.B);
    const float invS = p->bw.k.grads;
    // k-major operands exactly as the recurrence left them (H_prev of step t is row block t of the state array,
    // row block 0 = h0), split over K, fp32 partials.  Both gradients come out of ONE launch, dG^T * [X | H_prev]:
    // dG (the large operand) is read once, and the tiles of both products fill the machine together.
    const bool direct = (x_dtype == FLSTM_F16 && d.I == d.Ip);
    const half_t* Xop = direct ? static_cast<const half_t*>(x) : p->X16.as<half_t>();
    const half_t* Hop = p->Y.as<half_t>();
    const int n_ih = dW_ih ? d.Ip : 0, n_hh = dW_hh ? d.Hp : 0, ncols = n_ih + n_hh;
    const bool accumulate = p->opt_accumulate != 0;
    OpList out;   // gradients into the caller's layout, one launch
    with_dx = with_dx && p->bw.dx;
    p->bw.shared = false;
    if (with_dx && ncols == 0) FL_TRY(launch_gemm_nt(dx_product(p, long(p->bw.T) - 1, 0), s));
    if (ncols > 0) {
        // automatic: what the kernels' schedules make fastest (gemm_tn_plan_splits), at least two 64-row slabs per split
        int want = p->opt_dw_splits > 0 ? p->opt_dw_splits : p->eff_dw;
        if (want <= 0) {
            const size_t cap = TB / 128 < 64 ? TB / 128 : 64;
            want = gemm_tn_plan_splits(4 * d.Hp, n_ih ? n_ih : n_hh, n_ih ? n_hh : 0, int(TB), cap < 1 ? 1 : int(cap));
        }
        if (want > 64) want = 64;
        const int splits = gemm_effective_splits(int(TB), want);
        const size_t per = size_t(4) * d.Hp * ncols;
        FL_TRY(p->dw_part.reserve(per * splits * sizeof(float)));
        GemmNT g{};
        g.A = p->dG.as<half_t>(); g.lda = size_t(4) * d.Hp;
        g.M = 4 * d.Hp; g.N = ncols; g.K = int(TB);
        if (n_ih && n_hh) {
            g.B = Xop; g.ldb = size_t(d.Ip); g.N1 = n_ih;
            g.B2 = Hop; g.ldb2 = size_t(d.Hp);
        } else {
            g.B = n_ih ? Xop : Hop; g.ldb = size_t(n_ih ? d.Ip : d.Hp);
        }
        g.C16 = nullptr; g.C32 = p->dw_part.as<float>(); g.ldc = size_t(ncols);
        g.alpha = 1.f; g.splits = splits; g.split_stride = per;
        g.stamp = stamps_of(p) + kStampBwdDw;
        if (with_dx) FL_TRY(launch_gemm_tn_and_nt(g, dx_product(p, long(p->bw.T) - 1, 0), s, &p->bw.shared));
        else FL_TRY(launch_gemm_tn(g, s));
        out.reduce_dw(d, p->dw_part.as<float>(), splits, size_t(ncols), 0, d.I, invS, accumulate, dW_ih);
        out.reduce_dw(d, p->dw_part.as<float>(), splits, size_t(ncols), n_ih, d.H, invS, accumulate, dW_hh);
    }
    out.reduce_db(d, p->db_part.as<float>(), p->bw.L.ng, invS, accumulate, db_ih, db_hh);
    out.unpad(p->dH0.as<float>(), 1, size_t(d.Hp), size_t(d.B), d.H, invS, dh0, 1);
    out.unpad(p->dC.as<float>(), 1, size_t(d.Hp), size_t(d.B), d.H, invS, dc0, 1);
    return publish_with(p, out, kStampBwdEnd, s);
}

// One whole backward pass, enqueued.  dX and the weight gradients follow the recurrence without waiting for its status
// (one wait per pass); a persistent launch that gave up is found at the end and the pass repeated step-wise over the
// same outputs.  Only when the caller's gradients are added to (accumulate_grads), or an output lies in an input of the
// recurrence (dh0 in d_hn's place, dx in dY's), the status is checked first (FLSTM_E_STALLED).
int backward_enqueue(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype, const void* dY, flstm_dtype dy_dtype,
                     const void* d_hn, const void* d_cn, flstm_dtype dstate_dtype, const BwdScales& k, void* dx,
                     flstm_dtype dx_dtype, float* dW_ih, float* dW_hh, float* db_ih, float* db_hh, float* dh0, float* dc0,
                     hipStream_t s) {
    use_tuned(p, T);
    int rc = backward_rec_once(p, T, dY, dy_dtype, d_hn, d_cn, dstate_dtype, k, dx, dx_dtype, s);
    if (rc == int(hipErrorCooperativeLaunchTooLarge) && p->Lb.persistent && !p->refused_bwd) {
        // the grid cannot be co-resident: nothing was launched; this direction runs step-wise from now on
        p->refused_bwd = true;
        p->coop_refusals++;
        replan(p);
        rc = backward_rec_once(p, T, dY, dy_dtype, d_hn, d_cn, dstate_dtype, k, dx, dx_dtype, s);
    }
    if (rc) return rc;
    const Dims& d = p->d;
    const size_t TB = T * size_t(d.B), BH = size_t(d.B) * d.H;
    if (p->opt_accumulate || overlap({bytes_of(dx, TB * d.I, dx_dtype), bytes_of(dh0, BH, FLSTM_F32), bytes_of(dc0, BH, FLSTM_F32)},
                                     {bytes_of(dY, TB * d.H, dy_dtype), bytes_of(d_hn, BH, dstate_dtype), bytes_of(d_cn, BH, dstate_dtype)})) {
        int st = 0;
        OpList nothing;
        rc = wait_status(p, nothing, -1, s, &st);
        if (rc) return rc;
        if (st != 0) return FLSTM_E_STALLED;
    }
    return backward_finish(p, x, x_dtype, true, dW_ih, dW_hh, db_ih, db_hh, dh0, dc0, s);
}
// ... once the stream has been waited for (as forward_conclude)
int backward_conclude(flstm_core_plan* p, bool weight_gradients, hipStream_t s) {
    p->bw.open = false;
    int st = 0;
    int rc = take_status(p, s, &st);
    if (rc) return rc;
    if (st != 0) {
        if (p->bw.L.persistent) demote(p, false);
        return FLSTM_E_STALLED;
    }
    pass_done(p, false);
    if (p->opt_profile)
        FL_TRY(hipMemcpy(p->prof_b, p->prof.as<long long>() + 8, sizeof(p->prof_b), hipMemcpyDeviceToHost));
    const int dw_start = weight_gradients ? kStampBwdDw : kStampBwdEnd;   // (without that product the dX one ends with the pass; where they share a launch bwd_dw is both)
    p->ms_bwd[0] = elapsed(p, kStampBwdStart, kStampBwdRecEnd);
    p->ms_bwd[1] = elapsed(p, kStampBwdRecEnd, dw_start);
    p->ms_bwd[2] = elapsed(p, dw_start, kStampBwdEnd);
    p->ms_bwd[3] = elapsed(p, kStampBwdBegin, kStampBwdEnd);
    return 0;
}

int backward_pass(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype, const void* dY, flstm_dtype dy_dtype,
                  const void* d_hn, const void* d_cn, flstm_dtype dstate_dtype, const BwdScales& k, void* dx,
                  flstm_dtype dx_dtype, float* dW_ih, float* dW_hh, float* db_ih, float* db_hh, float* dh0, float* dc0,
                  hipStream_t s) {
    for (int attempt = 0;; ++attempt) {
        int rc = backward_enqueue(p, T, x, x_dtype, dY, dy_dtype, d_hn, d_cn, dstate_dtype, k, dx, dx_dtype, dW_ih, dW_hh, db_ih,
                                  db_hh, dh0, dc0, s);
        if (rc == 0) rc = wait_stream(s);
        const bool persistent = p->bw.L.persistent != 0;
        if (rc == 0) rc = backward_conclude(p, dW_ih || dW_hh, s);
        else if (rc == FLSTM_E_STALLED && persistent) demote(p, false);   // (the check ahead of accumulation)
        p->bw.open = false;
        if (rc != FLSTM_E_STALLED || !persistent || attempt > 0) return rc;
    }
}

}  // namespace

extern "C" int flstm_core_backward(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype,
                                   const void* dY, flstm_dtype dy_dtype, const void* d_hn, const void* d_cn,
                                   flstm_dtype dstate_dtype, float grad_scale, void* dx, flstm_dtype dx_dtype,
                                   float* dW_ih, float* dW_hh, float* db_ih, float* db_hh, float* dh0,
                                   float* dc0, void* stream) {
    if (!p) return FLSTM_E_INVALID;
    if (T == 0) return 0;
    if (!p->have_cache || p->T_cache != T) return FLSTM_E_NO_CACHE;
    if (!dY) return FLSTM_E_INVALID;
    if (dW_ih && !x) return FLSTM_E_INVALID;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const BwdScales k = BwdScales::loss_scale(grad_scale > 0.f ? grad_scale : 1.f);
    return backward_pass(p, T, x, x_dtype, dY, dy_dtype, d_hn, d_cn, dstate_dtype, k, dx, dx_dtype, dW_ih, dW_hh, db_ih, db_hh, dh0, dc0, s);
}

// ---- stacks of layers: the same passes, layer behind layer on one stream with ONE wait at the end

extern "C" int flstm_core_pack(flstm_core_plan* p, const float* w_ih, const float* w_hh, const float* b_ih, const float* b_hh,
                               void* stream) {
    int rc = core_pack_weights_async(p, w_ih, w_hh, static_cast<hipStream_t>(stream));
    if (rc) return rc;
    return flstm_core_pack_bias(p, b_ih, b_hh, stream);
}

extern "C" int flstm_stack_forward(flstm_core_plan* const* plans, int layers, size_t T, const void* x, flstm_dtype x_dtype,
                                   const void* h0, const void* c0, flstm_dtype state_dtype, void* const* ys, flstm_dtype y_dtype,
                                   void* hy, void* cy, void* stream) {
    if (!plans || layers < 1 || !ys) return FLSTM_E_INVALID;
    if (T == 0) return 0;
    if (!x || T > (size_t(1) << 24)) return FLSTM_E_INVALID;
    hipStream_t s = static_cast<hipStream_t>(stream);
    for (int l = 0; l < layers; ++l) {
        const flstm_core_plan* p = plans[l];
        if (!p || !ys[l] || p->d.B != plans[0]->d.B || p->d.H != plans[0]->d.H || (l > 0 && p->d.I != p->d.H)) return FLSTM_E_INVALID;
        if (!p->weights_packed || !p->bias_packed) return FLSTM_E_NOT_PACKED;
    }
    const size_t TB = T * size_t(plans[0]->d.B), BH = size_t(plans[0]->d.B) * plans[0]->d.H;
    const size_t state_in = BH * (state_dtype == FLSTM_F32 ? 4 : 2), state_out = BH * (y_dtype == FLSTM_F32 ? 4 : 2);
    auto at = [](const void* base, size_t off) -> const void* { return base ? static_cast<const char*>(base) + off : nullptr; };
    auto layer = [&](int l, auto&& pass) -> int {
        return pass(plans[l], T, l == 0 ? x : ys[l - 1], l == 0 ? x_dtype : y_dtype, at(h0, l * state_in), at(c0, l * state_in),
                    state_dtype, ys[l], y_dtype, const_cast<void*>(at(hy, l * state_out)), const_cast<void*>(at(cy, l * state_out)), y_dtype, true, s);
    };
    int rc = 0;
    // Where an output lies in what a layer reads -- the states carried in place, one layer's rows over another's --, a layer that
    // gave up could not be repeated once the layers above it have run: each is waited for then.  So it is where a plan stands for
    // several layers (weights that they share): what a plan knows of its pass -- the status, the ring's slot -- is that of one pass.
    bool in_place = overlap({bytes_of(hy, layers * BH, y_dtype), bytes_of(cy, layers * BH, y_dtype)},
                            {bytes_of(x, TB * plans[0]->d.I, x_dtype), bytes_of(h0, layers * BH, state_dtype), bytes_of(c0, layers * BH, state_dtype)});
    for (int l = 0; l < layers; ++l) {
        const Bytes rows = bytes_of(ys[l], TB * plans[0]->d.H, y_dtype);
        in_place = in_place || overlap({rows}, {bytes_of(x, TB * plans[0]->d.I, x_dtype), bytes_of(h0, layers * BH, state_dtype), bytes_of(c0, layers * BH, state_dtype)});
        for (int m = 0; m < l; ++m) in_place = in_place || plans[m] == plans[l] || overlap({rows}, {bytes_of(ys[m], TB * plans[0]->d.H, y_dtype)});
    }
    for (int l = 0; l < layers && rc == 0; ++l) {
        plans[l]->have_cache = false;
        rc = in_place ? layer(l, forward_pass) : layer(l, forward_enqueue);
    }
    if (in_place) {
        for (int l = 0; l < layers; ++l) {
            plans[l]->fw.open = false;
            if (rc == 0) { plans[l]->have_cache = true; plans[l]->T_cache = T; }
        }
        return rc;
    }
    const int waited = wait_stream(s);
    if (rc == 0) rc = waited;
    for (int l = 0; l < layers && rc == 0; ++l) {
        const bool persistent = plans[l]->Lf.persistent != 0;
        rc = forward_conclude(plans[l], s);
        if (rc == FLSTM_E_STALLED && persistent) {   // this layer again, and with it everything that has read its outputs
            rc = 0;
            for (int m = l + 1; m < layers && rc == 0; ++m) rc = clear_status(plans[m], s);
            for (int m = l; m < layers && rc == 0; ++m) {
                rc = layer(m, forward_pass);
                if (rc == 0) { plans[m]->have_cache = true; plans[m]->T_cache = T; }
            }
            break;
        }
        if (rc == 0) { plans[l]->have_cache = true; plans[l]->T_cache = T; }
    }
    for (int l = 0; l < layers; ++l) plans[l]->fw.open = false;
    return rc;
}

extern "C" int flstm_stack_backward(flstm_core_plan* const* plans, int layers, size_t T, const void* const* xs, flstm_dtype x_dtype,
                                    const void* dY, flstm_dtype dy_dtype, float dy_scale, const void* const* d_hn,
                                    const void* const* d_cn, flstm_dtype dstate_dtype, float loss_scale, void* const* dxs,
                                    flstm_dtype dx_dtype, float* const* dW_ih, float* const* dW_hh, float* const* db_ih,
                                    float* const* db_hh, float* const* dh0, float* const* dc0, void* stream) {
    if (!plans || layers < 1 || !xs || !dY || !dxs || !dW_ih || !dW_hh || !db_ih || !dh0 || !dc0) return FLSTM_E_INVALID;
    if (T == 0) return 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    for (int l = 0; l < layers; ++l) {
        if (!plans[l] || !xs[l] || (l > 0 && !dxs[l])) return FLSTM_E_INVALID;
        if (!plans[l]->have_cache || plans[l]->T_cache != T) return FLSTM_E_NO_CACHE;
        if (plans[l]->opt_accumulate) return FLSTM_E_INVALID;
    }
    // from layer to layer gradients stay fp16 with the loss scale on them; it is divided out of everything returned
    const float S = loss_scale > 0.f ? loss_scale : 1.f;
    auto layer = [&](int l, auto&& pass) -> int {
        const bool top = l == layers - 1;
        const BwdScales k{top ? dy_scale : 1.f, S, l == 0 ? 1.f / S : 1.f, 1.f / S};
        return pass(plans[l], T, xs[l], l == 0 ? x_dtype : FLSTM_F16, top ? dY : dxs[l + 1], top ? dy_dtype : FLSTM_F16,
                                d_hn ? d_hn[l] : nullptr, d_cn ? d_cn[l] : nullptr, dstate_dtype, k, dxs[l], l == 0 ? dx_dtype : FLSTM_F16,
                                dW_ih[l], dW_hh[l], db_ih[l], db_hh ? db_hh[l] : nullptr, dh0[l], dc0[l], s);
    };
    int rc = 0, from = layers - 1;
    // (as forward: gradients over gradients that a layer above has yet to be repeated from, one buffer for the dxs of several layers)
    bool in_place = false;
    for (int l = 0; l < layers && !in_place; ++l) {
        const Dims& d = plans[l]->d;
        const size_t TB = T * size_t(d.B), BH = size_t(d.B) * d.H;
        auto dx_of = [&](int m) { return bytes_of(dxs[m], TB * plans[m]->d.I, m == 0 ? dx_dtype : FLSTM_F16); };
        for (int m = 0; m < layers && !in_place; ++m) {
            in_place = overlap({dx_of(l), bytes_of(dh0[l], BH, FLSTM_F32), bytes_of(dc0[l], BH, FLSTM_F32)},
                               {bytes_of(dY, TB * d.H, dy_dtype), bytes_of(xs[m], TB * plans[m]->d.I, m == 0 ? x_dtype : FLSTM_F16), bytes_of(d_hn ? d_hn[m] : nullptr, BH, dstate_dtype),
                                bytes_of(d_cn ? d_cn[m] : nullptr, BH, dstate_dtype)}) ||
                       (m < l && overlap({dx_of(l)}, {dx_of(m)}));
        }
    }
    if (in_place) {
        for (int l = from; l >= 0 && rc == 0; --l) rc = layer(l, backward_pass);
        return rc;
    }
    for (int attempt = 0;; ++attempt) {   // a layer that gave up is repeated step-wise, and every layer below it with it
        for (int l = from; l >= 0 && rc == 0; --l) rc = layer(l, backward_enqueue);
        const int waited = wait_stream(s);
        if (rc == 0) rc = waited;
        bool again = false;
        for (int l = from; l >= 0 && rc == 0; --l) {
            const bool persistent = plans[l]->bw.L.persistent != 0;
            rc = backward_conclude(plans[l], true, s);
            if (rc == FLSTM_E_STALLED && persistent && attempt < layers) {
                from = l;
                again = true;
                for (int m = l - 1; m >= 0; --m) {
                    const int cleared = clear_status(plans[m], s);
                    if (cleared) return cleared;
                }
            }
        }
        for (int l = 0; l < layers; ++l) plans[l]->bw.open = false;
        if (!again) return rc;
        rc = 0;
    }
}

// The largest |value| of a device tensor (NaN if there is one), on the host: what an automatic loss scale is chosen from.
extern "C" int flstm_core_absmax(flstm_core_plan* p, const void* t, flstm_dtype dtype, size_t n, float* out, void* stream) {
    if (!p || !out || (n > 0 && !t)) return FLSTM_E_INVALID;
    hipStream_t s = static_cast<hipStream_t>(stream);
    *out = 0.f;
    if (n == 0) return 0;
    FL_TRY(absmax(t, dtype == FLSTM_F32, n, p->status.as<unsigned>() + kStatusBytes / 4, &p->status_host->absmax, s));
    FL_TRY(hipStreamSynchronize(s));
    *out = *static_cast<volatile float*>(&p->status_host->absmax);
    return 0;
}

// ---- the same passes fed in ranges of steps (for callers that stream the sequence through the device)

extern "C" int flstm_core_forward_begin(flstm_core_plan* p, size_t T, const void* x, flstm_dtype x_dtype,
                                        const void* h0, const void* c0, flstm_dtype state_dtype, void* stream) {
    if (!p) return FLSTM_E_INVALID;
    if (!p->weights_packed || !p->bias_packed) return FLSTM_E_NOT_PACKED;
    if (T == 0 || !x || T > (size_t(1) << 24)) return FLSTM_E_INVALID;
    p->have_cache = false;
    for (float& m : p->ms_fwd) m = -1.f;
    use_tuned(p, T);
    p->fw.behind = true;   // (flstm_core_forward_end; the rows are the caller's to fetch)
    p->fw.rows_behind = false;
    return forward_setup(p, T, x, x_dtype, h0, c0, state_dtype, false, static_cast<hipStream_t>(stream));
}

extern "C" int flstm_core_forward_steps(flstm_core_plan* p, size_t t0, size_t nsteps, void* stream) {
    if (!p || !p->fw.open || t0 + nsteps > p->fw.T) return FLSTM_E_INVALID;
    if (nsteps == 0) return 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    int rc = forward_project(p, t0, nsteps, false, false, s);
    if (rc) return rc;
    return forward_recur(p, t0, nsteps, s);
}

extern "C" int flstm_core_forward_end(flstm_core_plan* p, void* hy, void* cy, flstm_dtype out_state_dtype,
                                      int save_for_backward, void* stream) {
    if (!p || !p->fw.open) return FLSTM_E_INVALID;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Dims& d = p->d;
    const size_t TB = p->fw.T * size_t(d.B);
    p->fw.open = false;
    OpList out;
    out.only_if_ok = true;   // (a window's state may be carried in place, and the repeat reads it)
    final_states(p, TB, hy, cy, out_state_dtype, out);
    int st = 0;
    int rc = wait_status(p, out, kStampFwdEnd, s, &st);
    if (rc) return rc;
    if (st != 0) {   // a persistent launch gave up: the caller repeats the pass through flstm_core_forward
        if (p->Lf.persistent) demote(p, true);
        return FLSTM_E_STALLED;
    }
    pass_done(p, true);
    if (save_for_backward) { p->have_cache = true; p->T_cache = p->fw.T; }
    return 0;
}

extern "C" int flstm_core_backward_begin(flstm_core_plan* p, size_t T, const void* dY, flstm_dtype dy_dtype,
                                         const void* d_hn, const void* d_cn, flstm_dtype dstate_dtype,
                                         float grad_scale, void* dx, flstm_dtype dx_dtype, void* stream) {
    if (!p || !dY || T == 0) return FLSTM_E_INVALID;
    if (!p->have_cache || p->T_cache != T) return FLSTM_E_NO_CACHE;
    for (float& m : p->ms_bwd) m = -1.f;
    const float S = grad_scale > 0.f ? grad_scale : 1.f;
    use_tuned(p, T);
    return backward_setup(p, T, dY, dy_dtype, d_hn, d_cn, dstate_dtype, BwdScales::loss_scale(S), dx, dx_dtype, false, static_cast<hipStream_t>(stream));
}

extern "C" int flstm_core_backward_steps(flstm_core_plan* p, size_t t_hi, size_t nsteps, void* stream) {
    if (!p || !p->bw.open || t_hi >= p->bw.T || nsteps == 0 || nsteps > t_hi + 1) return FLSTM_E_INVALID;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const long lo = long(t_hi) - long(nsteps) + 1;
    // the range that reaches step 0 also runs the closing product for dh0
    int rc = backward_recur(p, long(t_hi), lo == 0 ? -1 : lo, false, s);
    if (rc == int(hipErrorCooperativeLaunchTooLarge) && p->bw.L.persistent && !p->refused_bwd) {
        // the grid cannot be co-resident: step-wise from now on; the rings of this pass were laid out for the persistent
        // kernel, so the caller repeats the pass (as after a launch that gave up)
        p->refused_bwd = true;
        p->coop_refusals++;
        p->bw.open = false;
        replan(p);
        return FLSTM_E_STALLED;
    }
    if (rc) return rc;
    return backward_dx(p, long(t_hi), lo, s);
}

extern "C" int flstm_core_backward_end(flstm_core_plan* p, const void* x, flstm_dtype x_dtype, float* dW_ih,
                                       float* dW_hh, float* db_ih, float* db_hh, float* dh0, float* dc0,
                                       void* stream) {
    if (!p || !p->bw.open) return FLSTM_E_INVALID;
    if (dW_ih && !x) return FLSTM_E_INVALID;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // the caller's gradients may be accumulated into: the status of the recurrence is checked before they are touched
    int st = 0;
    OpList nothing;
    int rc = wait_status(p, nothing, -1, s, &st);
    if (rc) return rc;
    if (st != 0) {   // the caller repeats the pass through flstm_core_backward
        p->bw.open = false;
        if (p->bw.L.persistent) demote(p, false);
        return FLSTM_E_STALLED;
    }
    rc = backward_finish(p, x, x_dtype, false, dW_ih, dW_hh, db_ih, db_hh, dh0, dc0, s);
    if (rc) return rc;
    rc = wait_stream(s);
    if (rc) return rc;
    p->bw.open = false;
    pass_done(p, false);
    return 0;
}

bool flstm_hip::core_copy_beside(flstm_core_plan* p, bool forward, const OpList& copies) {
    // 48 workgroups of 256 threads with one 16-byte load in flight each keep a PCIe link of 57 GB/s busy.  What counts is the
    // threads: the kernels for short contractions have workgroups of 64, 128 and 256 of them.
    constexpr int kFewest = 16 * 256, kThreads = 48 * 256;
    const RecLayout& L = forward ? p->Lf : p->bw.L;
    const int idle = rec_idle_workgroups(L), threads = rec_threads(L), enough = kThreads / threads;
    if (idle * threads < kFewest || copies.count < 1 || copies.count > BesideCopies::kMost) return false;
    BesideCopies& b = forward ? p->beside_f : p->beside_b;
    for (int i = 0; i < copies.count; ++i) {
        if (copies.op[i].kind != LayoutOp::kUnpad) return false;
        b.op[i] = copies.op[i];
    }
    b.count = copies.count;
    b.helpers = idle < enough ? idle : enough;
    return true;
}

extern "C" int flstm_core_cache_ptr(const flstm_core_plan* p, int which, const void** ptr, size_t* ld) {
    if (!p || !ptr || !ld || !(p->have_cache || p->fw.open)) return FLSTM_E_INVALID;
    switch (which) {
        case 0: *ptr = p->Y.p; *ld = size_t(p->d.Hp); return 0;
        case 1: *ptr = p->C.p; *ld = size_t(p->d.Hp); return 0;
        case 2: *ptr = p->G.p; *ld = size_t(4) * p->d.Hp; return 0;
    }
    return FLSTM_E_INVALID;
}

extern "C" double flstm_core_last_ms(const flstm_core_plan* p, const char* phase) {
    if (!p || !phase) return -1.0;
    if (p->fw.begin_on_device && !p->fw.open && (!strcmp(phase, "fwd_proj") || !strcmp(phase, "fwd_total"))) {
        flstm_core_plan* const q = const_cast<flstm_core_plan*>(p);   // (what is fetched is kept until the next pass)
        static_assert(kStampFwdBegin == 0 && kStampFwdStart == 1, "the two that are fetched");
        if (hipMemcpy(q->status_host->stamps, stamps_of(p), 2 * sizeof(long long), hipMemcpyDeviceToHost) != hipSuccess) {
            (void)hipGetLastError();
            return -1.0;
        }
        from_the_beginning(q);
        q->fw.begin_on_device = false;
    }
    if (!strcmp(phase, "fwd_proj")) return p->ms_fwd[0];
    if (!strcmp(phase, "fwd_rec")) return p->ms_fwd[1];
    if (!strcmp(phase, "fwd_total")) return p->ms_fwd[2];
    if (!strcmp(phase, "bwd_rec")) return p->ms_bwd[0];
    if (!strcmp(phase, "bwd_dx")) return p->ms_bwd[1];
    if (!strcmp(phase, "bwd_dw")) return p->ms_bwd[2];
    if (!strcmp(phase, "bwd_total")) return p->ms_bwd[3];
    // counters of workgroup 0 (option "profile"), in milliseconds of the constant-rate clock: 0..4 wait, product, partials,
    // pointwise, publish; 6 the whole launch; 5 the launch in shader-engine clocks / the constant clock's rate, so that
    // clk5 / clk6 x that rate is the engine clock the kernel ran at
    if (!strncmp(phase, "fwd_clk", 7) && phase[7] >= '0' && phase[7] <= '7')
        return double(p->prof_f[phase[7] - '0']) / p->wall_khz;
    if (!strncmp(phase, "bwd_clk", 7) && phase[7] >= '0' && phase[7] <= '7')
        return double(p->prof_b[phase[7] - '0']) / p->wall_khz;
    return -1.0;
}

// ---- the GEMMs the passes are built from, callable on their own

extern "C" int flstm_gemm_nt(const void* A, size_t lda, const void* B, size_t ldb, size_t M, size_t N, size_t K,
                             void* C, flstm_dtype c_dtype, size_t ldc, float alpha, const float* bias, void* stream) {
    if (!A || !B || !C || M > (1u << 30) || N > (1u << 30) || K > (1u << 30)) return FLSTM_E_INVALID;
    GemmNT g{};
    g.A = static_cast<const half_t*>(A); g.lda = lda;
    g.B = static_cast<const half_t*>(B); g.ldb = ldb;
    g.M = int(M); g.N = int(N); g.K = int(K);
    if (c_dtype == FLSTM_F32) g.C32 = static_cast<float*>(C);
    else g.C16 = static_cast<half_t*>(C);
    g.ldc = ldc; g.alpha = alpha; g.splits = 1; g.split_stride = 0; g.bias = bias;
    if (lda < K || ldb < K || ldc < N) return FLSTM_E_INVALID;
    FL_TRY(launch_gemm_nt(g, static_cast<hipStream_t>(stream)));
    return 0;
}

extern "C" size_t flstm_gemm_tn_workspace_bytes(size_t M, size_t N, size_t K, int splits) {
    if (splits <= 1 || K == 0 || K > (1u << 30)) return 0;
    const int eff = gemm_effective_splits(int(K), splits);
    return eff <= 1 ? 0 : size_t(eff) * M * N * sizeof(float);
}

extern "C" int flstm_gemm_tn_auto_splits(size_t M, size_t N, size_t K, int max_splits) {
    if (M == 0 || N == 0 || K == 0 || M > (1u << 30) || N > (1u << 30) || K > (1u << 30)) return 1;
    return gemm_tn_auto_splits(int(M), int(N), 0, int(K), max_splits < 1 ? 1 : (max_splits > 64 ? 64 : max_splits));
}

extern "C" int flstm_gemm_tn(const void* A, size_t lda, const void* B, size_t ldb, size_t M, size_t N, size_t K,
                             float* C, size_t ldc, float alpha, int splits, void* workspace, void* stream) {
    if (!A || !B || !C || M > (1u << 30) || N > (1u << 30) || K > (1u << 30)) return FLSTM_E_INVALID;
    if (lda < M || ldb < N || ldc < N) return FLSTM_E_INVALID;
    if (M == 0 || N == 0 || K == 0) return 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int eff = gemm_effective_splits(int(K), splits < 1 ? 1 : splits);
    GemmNT g{};
    g.A = static_cast<const half_t*>(A); g.lda = lda;
    g.B = static_cast<const half_t*>(B); g.ldb = ldb;
    g.M = int(M); g.N = int(N); g.K = int(K);
    g.alpha = alpha; g.bias = nullptr;
    if (eff <= 1) {
        g.C32 = C; g.ldc = ldc; g.splits = 1; g.split_stride = 0;
        FL_TRY(launch_gemm_tn(g, s));
        return 0;
    }
    if (!workspace) return FLSTM_E_INVALID;
    g.C32 = static_cast<float*>(workspace); g.ldc = N; g.splits = eff; g.split_stride = M * N;
    FL_TRY(launch_gemm_tn(g, s));
    FL_TRY(reduce_partials(static_cast<const float*>(workspace), eff, M * N, int(M), int(N), ldc, C, s));
    return 0;
}

// ---- tuner

extern "C" int flstm_core_tune(flstm_core_plan* p, size_t T, int repeats, int try_stepwise, void* stream) {
    if (!p || T == 0 || T > (size_t(1) << 24) || p->fw.open || p->bw.open) return FLSTM_E_INVALID;
    if (!p->weights_packed || !p->bias_packed) return FLSTM_E_NOT_PACKED;
    if (repeats < 1) repeats = 1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Dims& d = p->d;
    const size_t TB = T * size_t(d.B);
    // synthetic inputs: varied values (the matrix cores draw more power on them than on constants, and the GEMMs run
    // about a fifth slower: candidates are compared under the clock they will run at)
    DevBuf x, dy, dwi, dwh, y, dx;
    int rc = 0;
    auto fail = [&](int code) { x.release(); dy.release(); dwi.release(); dwh.release(); y.release(); dx.release(); return code; };
    if (x.reserve(TB * d.I * sizeof(half_t)) != hipSuccess || dy.reserve(TB * d.H * sizeof(half_t)) != hipSuccess ||
        dwi.reserve(size_t(4) * d.H * d.I * sizeof(float)) != hipSuccess ||
        dwh.reserve(size_t(4) * d.H * d.H * sizeof(float)) != hipSuccess)
        return fail(int(hipErrorOutOfMemory));
    if (fill_noise(x.as<half_t>(), TB * d.I, 0x1234567u, 1.7f, s) != hipSuccess ||
        fill_noise(dy.as<half_t>(), TB * d.H, 0x89ABCDEu, 1.7f, s) != hipSuccess)
        return fail(int(hipErrorUnknown));
    // y and dx as passes in use write them (without memory for them, passes that leave them out are compared)
    if (y.reserve(TB * d.H * sizeof(half_t)) != hipSuccess || dx.reserve(TB * d.I * sizeof(half_t)) != hipSuccess) {
        (void)hipGetLastError();
        y.release();
        dx.release();
    }
    // the plan's explicit options and tuned state are set aside while candidates run
    const int keep_step = p->opt_stepwise, keep_mtf = p->opt_mt_f, keep_mtb = p->opt_mt_b, keep_dw = p->opt_dw_splits,
              keep_acc = p->opt_accumulate, keep_two_d = p->opt_two_d;
    const bool keep_two_d_explicit = p->two_d_explicit;
    const bool keep_cache = p->have_cache;
    const std::vector<flstm_core_plan::Tuned> keep_tuned = p->tuned;
    p->tuned.clear();
    use_tuned(p, T);
    p->opt_accumulate = 0;
    auto restore = [&]() {
        p->opt_stepwise = keep_step; p->opt_mt_f = keep_mtf; p->opt_mt_b = keep_mtb; p->opt_dw_splits = keep_dw;
        p->opt_accumulate = keep_acc; p->opt_two_d = keep_two_d; p->two_d_explicit = keep_two_d_explicit;
        p->tuned = keep_tuned;
        p->have_cache = false;   // the caches now hold the synthetic sequence
        (void)keep_cache;
        use_tuned(p, T);
        replan(p);
    };
    flstm_core_plan::Tuned best{};
    best.T = T; best.ms_f = best.ms_b = best.ms_dw = best.pass_f = best.products = -1.f; best.two_d = -1;
    // A forward candidate is judged by the whole call: whether its projection and outputs have launches of their own or are part
    // of the recurrence's depends on the candidate, so the phases do not hold the same work.  A split count by all products, of
    // which dX may share the launch.
    struct Times { float pass_f, f, b, products, dw; } ms;
    auto run = [&]() -> int {
        ms = Times{1e30f, 1e30f, 1e30f, 1e30f, 1e30f};
        auto least = [](float& to, float v) { if (v > 0 && v < to) to = v; };
        for (int r = 0; r <= repeats; ++r) {   // first pass is a warm-up
            const auto before = std::chrono::steady_clock::now();
            int e = flstm_core_forward(p, T, x.p, FLSTM_F16, nullptr, nullptr, FLSTM_F16, y.p, FLSTM_F16, nullptr, nullptr,
                                       FLSTM_F16, 1, s);
            if (e) return e;
            const float whole = std::chrono::duration<float, std::milli>(std::chrono::steady_clock::now() - before).count();
            e = flstm_core_backward(p, T, x.p, FLSTM_F16, dy.p, FLSTM_F16, nullptr, nullptr, FLSTM_F16, 1.f, dx.p, FLSTM_F16,
                                    dwi.as<float>(), dwh.as<float>(), nullptr, nullptr, nullptr, nullptr, s);
            if (e) return e;
            if (r == 0) continue;
            least(ms.pass_f, whole);
            least(ms.f, p->ms_fwd[1]);
            least(ms.b, p->ms_bwd[0]);
            least(ms.products, p->ms_bwd[1] + p->ms_bwd[2]);
            least(ms.dw, p->ms_bwd[2]);
        }
        return 0;
    };
    // 1) row-block height and launch mode of the two recurrences (independent of each other and of the GEMMs)
    p->opt_dw_splits = 0;
    for (int step = 0; step <= (try_stepwise ? 1 : 0); ++step) {
        bool rule_f = false, rule_b = false;   // whether the rule is neither
        for (int mt : {1, 2, 0}) {
            p->opt_stepwise = step; p->opt_mt_f = mt; p->opt_mt_b = mt;
            replan(p);
            const bool f_is = mt ? p->Lf.mt == mt : rule_f && p->Lf.few, b_is = mt ? p->Lb.mt == mt : rule_b && p->Lb.few;   // 16-row blocks may not fit
            if (mt == 1) { rule_f = !p->Lf.few; rule_b = !p->Lb.few; }
            if (!f_is && !b_is) continue;
            rc = run();
            if (rc) { restore(); return fail(rc); }
            if (f_is && (best.pass_f < 0 || ms.pass_f < best.pass_f)) { best.pass_f = ms.pass_f; best.ms_f = ms.f; best.mt_f = mt; best.step_f = step; }
            if (b_is && (best.ms_b < 0 || ms.b < best.ms_b)) { best.ms_b = ms.b; best.mt_b = mt; best.step_b = step; }
        }
    }
    // 1b) the layout of the backward recurrence where the two-way split can run (2048 and 1024 hidden units): off /
    // where the rule of thumb has it / wherever it fits, with the row-block height the rule picks for each
    if (rec_bwd_two_d_possible(d.Hp, p->num_cus) && !keep_two_d_explicit) {
        p->opt_stepwise = 0; p->opt_mt_f = best.mt_f; p->opt_mt_b = 0;
        p->two_d_explicit = true;
        float best_td_ms = -1.f;
        for (int td = 0; td <= 2; ++td) {
            p->opt_two_d = td;
            replan(p);
            if (!p->Lb.persistent) continue;
            if (td == 2 && !p->Lb.two_d) continue;   // (nothing new: the split does not fit this batch)
            rc = run();
            if (rc) { restore(); return fail(rc); }
            if (best_td_ms < 0 || ms.b < best_td_ms) { best_td_ms = ms.b; best.two_d = td; }
        }
        // (the entry keeps the better of: the best row-block height under the plan's own setting, the best setting)
        if (best_td_ms >= 0 && best_td_ms < best.ms_b) { best.ms_b = best_td_ms; best.mt_b = 0; best.step_b = 0; }
        else best.two_d = -1;
        p->opt_two_d = keep_two_d; p->two_d_explicit = keep_two_d_explicit;
    }
    // 2) split-K count of the weight-gradient GEMM around what the schedule model picks
    p->opt_stepwise = best.step_f && best.step_b; p->opt_mt_f = best.mt_f; p->opt_mt_b = best.mt_b;
    replan(p);
    const size_t cap = TB / 128 < 64 ? TB / 128 : 64;
    const int rule = gemm_tn_plan_splits(4 * d.Hp, d.Ip, d.Hp, int(TB), cap < 1 ? 1 : int(cap));
    int last_eff = -1;
    for (int cand : {rule / 2, rule, rule + 1, rule * 2, rule * 4}) {
        if (cand < 1 || cand > 64) continue;
        const int eff = gemm_effective_splits(int(TB), cand);
        if (eff == last_eff) continue;
        last_eff = eff;
        p->opt_dw_splits = cand;
        rc = run();
        if (rc) { restore(); return fail(rc); }
        if (best.products < 0 || ms.products < best.products) { best.products = ms.products; best.ms_dw = ms.dw; best.dw_splits = cand; }
    }
    restore();
    for (auto it = p->tuned.begin(); it != p->tuned.end();)
        it = (it->T == T) ? p->tuned.erase(it) : it + 1;
    p->tuned.push_back(best);
    use_tuned(p, T);
    return fail(0);
}

// A tuned entry written into / read out of a plan: what a tuning run found, kept by the caller between processes.
extern "C" int flstm_core_set_tuned(flstm_core_plan* p, size_t T, int row_tiles_fwd, int row_tiles_bwd, int stepwise_fwd,
                                    int stepwise_bwd, int dw_splits, int bwd_two_d) {
    if (!p || T == 0 || T > (size_t(1) << 24) || row_tiles_fwd < 0 || row_tiles_fwd > 2 || row_tiles_bwd < 0 ||
        row_tiles_bwd > 2 || dw_splits < 0 || dw_splits > 64 || bwd_two_d < -1 || bwd_two_d > 2)
        return FLSTM_E_INVALID;
    flstm_core_plan::Tuned t{};
    t.T = T; t.mt_f = row_tiles_fwd; t.mt_b = row_tiles_bwd; t.step_f = stepwise_fwd != 0; t.step_b = stepwise_bwd != 0;
    t.dw_splits = dw_splits; t.two_d = bwd_two_d; t.ms_f = t.ms_b = t.ms_dw = t.pass_f = t.products = -1.f;
    for (auto it = p->tuned.begin(); it != p->tuned.end();)
        it = (it->T == T) ? p->tuned.erase(it) : it + 1;
    p->tuned.push_back(t);
    use_tuned(p, T);
    return 0;
}

extern "C" int flstm_core_get_tuned(const flstm_core_plan* p, size_t index, size_t* T, int* row_tiles_fwd, int* row_tiles_bwd,
                                    int* stepwise_fwd, int* stepwise_bwd, int* dw_splits, int* bwd_two_d) {
    if (!p || index >= p->tuned.size()) return FLSTM_E_INVALID;
    const auto& t = p->tuned[index];
    if (T) *T = t.T;
    if (row_tiles_fwd) *row_tiles_fwd = t.mt_f;
    if (row_tiles_bwd) *row_tiles_bwd = t.mt_b;
    if (stepwise_fwd) *stepwise_fwd = t.step_f;
    if (stepwise_bwd) *stepwise_bwd = t.step_b;
    if (dw_splits) *dw_splits = t.dw_splits;
    if (bwd_two_d) *bwd_two_d = t.two_d;
    return 0;
}

extern "C" double flstm_core_tuned_ms(const flstm_core_plan* p, size_t T, const char* phase) {
    if (!p || !phase) return -1.0;
    for (const auto& t : p->tuned)
        if (t.T == T) {
            if (!strcmp(phase, "fwd_pass")) return t.pass_f;
            if (!strcmp(phase, "bwd_products")) return t.products;
            if (!strcmp(phase, "fwd_rec")) return t.ms_f;
            if (!strcmp(phase, "bwd_rec")) return t.ms_b;
            if (!strcmp(phase, "bwd_dw")) return t.ms_dw;
        }
    return -1.0;
}
