// RRSPH_HIP: C-ABI implementation (host side) of the MI355X WCSPH step.
//
// The context owns the device buffers, one HIP stream at default priority
// and (optionally) a captured hipGraph of one step.  Every entry point is
// declared in include/rrsph_hip.h with the reference interface it replaces.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <optional>
#include <string>
#include <vector>

#include "../../include/rrsph_hip.h"
#include "device_common.hpp"
#include "diagnostics.hpp"
#include "radix_sort.hpp"
#include "resort.hpp"
#include "adjoint.hpp"
#include "adjoint3.hpp"
#include "step_kernels.hpp"
#include "step3d.hpp"
#include "pair_tile.hpp"
#include "list_step.hpp"
#include "list_step3.hpp"

using namespace rrsph;

namespace {

enum KernelClass : uint32_t {
    K_PROLOGUE = 0,
    K_UPSWEEP,
    K_SCAN,
    K_DOWNSWEEP,
    K_REORDER,
    K_DENSITY_SUM,
    K_PAIR,
    K_INTEGRATE,
    K_RESORT_SORT,
    K_RESORT_SCATTER,
    K_LIST_BUILD,
    K_NUM_CLASSES
};
const char* const kClassNames[K_NUM_CLASSES] = {"step_prologue", "radix_upsweep", "radix_scan", "radix_downsweep",
                                                "reorder_kernel", "density_sum_kernel", "pair_kernel",
                                                "integrate_kernel", "resort_sort_small", "resort_scatter",
                                                "list_build_kernel"};

struct Profiler {
    std::vector<std::pair<uint32_t, std::pair<hipEvent_t, hipEvent_t>>> rec;
};

template <class T> T* dalloc(size_t n, hipError_t& err) {
    void* p = nullptr;
    if (err == hipSuccess) err = hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(T));
    return (T*)p;
}

// Host copies of the smoothing-kernel W (SmoothingKernel.h:14-242) for constants.
double host_w(const rrsph_params_c& p, double dist, int skf) {
    const double h = p.hsml, pi = p.pi, q = dist / h;
    switch (skf) {
    case 2: return 1 / (pi * h * h) * std::exp(-q * q);
    case 3: {
        if (q > 2) return 0;
        double t = 1 - 0.5 * q;
        return 7 / (4 * pi * h * h) * (t * t * t * t) * (2 * q + 1);
    }
    case 4: return q <= 2 ? 5 / (16 * pi * h * h) * (2 - q) * (2 - q) * (2 - q) : 0;
    default: {
        double f = double(15) / (double(7) * pi * (h * h));
        if (q <= 1) return f * (double(2) / double(3) - q * q + q * q * q * 0.5);
        if (q <= 2) return f * (double(1) / double(6) * ((2 - q) * (2 - q) * (2 - q)));
        return 0;
    }
    }
}

}  // namespace

// Device scratch of rrsph_hip_smooth_gauges_noalloc: the block partial sums
// of every gauge (2 kMaxGauges kGaugeBlocks doubles), then eta, sum w e and
// sum w of every gauge (3 kMaxGauges).  1.03 MiB per device, held until the
// process ends.  Host code never uses this name as an address: the device's
// own address comes from hipGetSymbolAddress (scratch_address below).
constexpr size_t kScratchDoubles = 2 * (size_t)kMaxGauges * kGaugeBlocks + 3 * (size_t)kMaxGauges;
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {
std::mutex g_scratch_mu;
std::vector<double*> g_scratch;  // per device ordinal: the address of `scratch` on that device

// Address of `scratch` on the current device, looked up once per device (at
// context creation, with the context's device current).
hipError_t scratch_address(int device, double** out) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (device < 0) return hipErrorInvalidDevice;
    if ((size_t)device >= g_scratch.size()) g_scratch.resize(device + 1, nullptr);
    if (!g_scratch[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch[device] = (double*)p;
    }
    *out = g_scratch[device];
    return hipSuccess;
}
}  // namespace

// Checkpoints and per-step records of a differentiable run (FP64 only).
struct AdjTape {
    bool valid = false;
    bool allocated = false;              // every buffer below is there: a forward of the same shape reuses them
    bool segments = false;               // RRSPH_HIP_ADJ_STORE=segments when they were allocated
    uint32_t nsteps = 0, every = 0;
    GaugeSpec3 spec{};
    size_t blob = 0;                     // bytes of one saved state
    std::vector<void*> ck;               // checkpoint before step k * every; last entry: final state
    void* seg = nullptr;                 // states of one replayed segment (every blobs), or of every step
    bool seg_last = false;               // seg holds the last segment's states (kept by the forward)
    // seg holds the state before every step of the run (and the sorts):
    // the forward keeps them all when they fit in half the free device
    // memory (with list steps: together with their lists, see tape_fits), and
    // the reverse pass replays
    // nothing (943,906-particle basin, 12 steps in two segments: 23.6 -> 20.2 ms)
    bool keep_all = false;
    // the cell sort each step of seg ran with (keys, permutation): the reverse
    // step reorders its state with them instead of sorting it again
    uint32_t *seg_keys = nullptr, *seg_perm = nullptr;
    std::vector<uint8_t> seg_sorted;     // per seg slot: keys / perm hold that step's sort
    AdjStep* rec = nullptr;              // per step (device)
    Ctrl* uctrl = nullptr;               // per step: the control block its reverse step sorts and reorders with
                                         // (cur_dt = the step's dt_pred, nothing halted)
    std::vector<AdjStep> hrec;           // per step (host copy)
    double *eta = nullptr, *zs = nullptr, *ws = nullptr;  // nsteps x kMaxGauges
    double *eta_bar = nullptr, *partials = nullptr, *piston_sum = nullptr;
    double *lam[2] = {nullptr, nullptr}, *direct = nullptr, *drho_adj = nullptr;
    double4* out_adj = nullptr;          // 2D: out_a (n), or with lists the AdjRec2 records; 3D: the AdjRec3 records
    uint32_t* flag = nullptr;
    // With neighbour lists the tape runs list steps.  The forward builds
    // at every checkpoint step and records which steps built; a replay
    // repeats that schedule, so it repeats its steps exactly.  The segment
    // in hand (with keep_all the run) keeps the lists (and sorted cell keys)
    // of each of its builds; the reverse step of a list step reads its state
    // in the slot order of its build and that build's lists.
    bool lists = false;
    bool may_list = false;               // tape_lists when the buffers were allocated
    bool no_room = false;                // a kept tape could not allocate a build's lists
    size_t max_lists = 0;                // ... or may not: the builds whose lists fit (tape_memory)
    std::vector<uint8_t> builds;         // per step: the step built lists
    struct Lists {
        uint32_t *nbl = nullptr, *nbc = nullptr, *keys = nullptr;
    };
    std::vector<Lists> seg_lists;        // lists of the segment's builds (allocated on demand, reused)
    uint32_t nseg_lists = 0;             // builds of the segment in hand
    std::vector<int32_t> seg_build;      // per seg slot: the build (index in seg_lists) its step read
    float4* nearf = nullptr;             // FP32 step: near records of the reverse step's state (n)
    uint64_t force_build = ~0ull;        // tape step that must build (after a stale-list halt)
    // the forward's sorted step with the incremental re-sort, its record and
    // its gauges in one graph (rows from the control block's step count
    // - tbase); captured on the forward's first such step
    hipGraph_t tgraph = nullptr;
    hipGraphExec_t texec = nullptr;
    uint64_t tbase = 0;
    // list steps with every state kept: the records and gauges of all steps
    // are taken from the kept states in a few launches behind the last step
    bool batched() const { return lists && keep_all; }
};

// Captured steps with neighbour lists: a build step, and runs of 1, 2, 4 and
// 8 list steps.  Between two graphs the stream idles for 3 us or more (8 us
// where a profiler looks on), between the kernels of one for about 1.
constexpr uint32_t kListRunMax = 8;
constexpr uint64_t kFirstChunk = 16;
struct ListGraphs {
    hipGraph_t graph[5] = {};
    hipGraphExec_t exec[5] = {};
};

struct rrsph_ctx {
    rrsph_params_c prm{};
    StepParams P{};
    std::string err;
    int device = 0;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    bool fp32 = true;
    bool fused = true;
    bool export_fields = false;
    bool use_graph = true;
    bool uploaded = false;
    bool stepped = false;
    bool fields_valid = false;  // der (list steps: adA) / xs hold the last step's fields in A's slot order
    bool list_fields = false;   // the last step was a list or build step
    bool pres_in_order = true;  // false: pres is in the slot order of a step that failed
    uint32_t passes = 0;
    uint32_t ntiles = 0;
    // buffers
    double2 *posA = nullptr, *posB = nullptr;
    void *vaA = nullptr, *vaB = nullptr, *adA = nullptr, *pred = nullptr, *der = nullptr, *xs = nullptr,
         *pred_scratch = nullptr, *pres = nullptr, *pres_scratch = nullptr;
    void *pw = nullptr, *pw_scratch = nullptr;  // 3D: p / rho^2 (2D keeps it in pred.w)
    void* adB = nullptr;  // A.ad of the step's input, kept only if a fused step may be undone
    bool fast_pair = false;
    int pair_impl = 1;  // 0 general, 1 two-phase walk with LDS hit lists, 2 LDS tiles, 3 single-phase walk
    uint32_t *oidA = nullptr, *oidB = nullptr;
    uint32_t *key_next = nullptr, *kbuf[2] = {nullptr, nullptr}, *vbuf[2] = {nullptr, nullptr};
    uint32_t* hist = nullptr;
    uint32_t* digit_total = nullptr;
    unsigned long long* maxslots = nullptr;
    uint32_t* LB = nullptr;
    Ctrl* ctrl = nullptr;
    Ctrl* ctrl_cur = nullptr;   // list steps: the snapshot of the step in flight (list_step.hpp)
    Ctrl* util_ctrl = nullptr;
    Ctrl* host_ctrl = nullptr;  // pinned mirror
    double* scratch = nullptr;  // this device's `scratch` (rrsph_hip_smooth_gauges_noalloc)
    double* host_eta = nullptr; // pinned, kMaxGauges doubles: gauge results on their way to the caller
    double* red = nullptr;      // diagnostics partials
    // staging for up/download (device)
    double *st_r = nullptr, *st_v = nullptr, *st_rho = nullptr, *st_p = nullptr, *st_a = nullptr,
           *st_drho = nullptr, *st_av = nullptr, *st_mu = nullptr;
    int32_t* st_itype = nullptr;
    uint32_t* st_u32 = nullptr;
    hipGraph_t graph = nullptr;        // step with the incremental re-sort
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph_full = nullptr;   // step with the full radix sort
    hipGraphExec_t gexec_full = nullptr;
    const uint32_t* sorted_keys = nullptr;
    const uint32_t* sorted_perm = nullptr;
    const uint32_t* last_keys = nullptr;  // the cell sort of the last launched step
    const uint32_t* last_perm = nullptr;
    // incremental re-sort
    uint32_t* skeyA = nullptr;          // key each slot of A was sorted by
    unsigned long long* chg = nullptr;       // changed slots as (key << 32 | slot)
    unsigned long long* chg_mask = nullptr;  // per wavefront of slots: ballot of the changed ones
    uint32_t* wpre = nullptr;                // per wavefront: changed slots in the wavefronts before
    uint32_t resort_cap = kResortCap;
    uint32_t resort_stage = kBlock;     // changed composites a scatter block stages in LDS (more: binary search)
    bool incremental = true;            // false: every step runs the full radix sort
    bool need_full = true;              // skeyA does not describe A (after upload)
    uint64_t launched = 0;              // steps launched by this context
    uint64_t full_until = 0;            // after repeated re-sort overflows: full sorts until this launch count
    uint64_t last_fallback = ~0ull;     // step index of the last re-sort overflow
    uint64_t full_run_end = 0;          // step index where the last run of full sorts ended
    uint64_t full_run = 0;              // length of the last run of full sorts
    uint64_t n_incremental = 0, n_full = 0, n_fallback = 0;
    // neighbour-list steps: lists built every
    // list_interval steps (host schedule, adapted to the measured
    // displacement rate); the device halts a step whose lists may be stale
    bool list_mode = false;
    bool all_terms = false;             // artificial viscosity, XSPH and the wall force are all on
    int lanes = 1;                      // lanes per particle of the 2D list passes
    bool list_suspended = false;        // 2D tapes without lists, and their replays
    uint32_t no_keep_steps = 0, no_keep_every = 0;  // the shape of the last tape if its lists ran out of room when it kept them all
    size_t tape_lists_max = ~(size_t)0; // the most builds whose lists a kept tape allocates (RRSPH_HIP_TAPE_LISTS)
    uint32_t *nbl = nullptr, *nbc = nullptr;
    void* rec = nullptr;                // records of the list pass (ListRec per slot)
    void* dens = nullptr;               // 3D: records of the summation density pass (real4 per slot)
    uint32_t* home = nullptr;           // each slot's cell at the last build
    unsigned long long* dslots = nullptr;  // list steps: largest displacement (block maxima; 2 sets by step index, 4 where steps fuse)
    unsigned long long* dtslots = nullptr; // list steps: dt maxima (2 sets by step index)
    uint32_t* cell_count = nullptr;         // builds with the counting sort: cell counts (zero between builds), scan sums
    float4* cand = nullptr;                 // 3D builds: candidate records (FP32 home-relative position, z cell)
    ListGraphs list_graphs;             // of plain runs
    bool taping = false;                // ctx->P holds the taped runs' skin
    bool fuse = false;                  // list steps may run in fused pairs (fused_step_begin)
    void* rec1 = nullptr;               // fused steps: the second array of records
    Ctrl* ctrl_alt = nullptr;           // ... and, with continuity, control block
    uint64_t build_at = 0;              // step index of the last build launched
    double tape_skin = 0;               // skin of taped runs (fraction of the cut-off)
    uint64_t list_interval = 8;         // steps between builds
    uint64_t list_chunk = kFirstChunk;  // steps between looks at the control block
    uint64_t n_list = 0, n_build = 0, n_list_halts = 0;
    // where list and build steps leave the state (pos null: in place)
    struct Out {
        double2* pos = nullptr;
        void *va = nullptr, *ad = nullptr, *pres = nullptr;
        uint32_t* oid = nullptr;
        Ctrl* keep = nullptr;           // the control block after the step, for the tape
    } out;
    AdjTape adj;
};

namespace {

rrsph_status fail(rrsph_ctx* c, rrsph_status st, const std::string& msg) {
    if (c) c->err = msg;
    return st;
}

#define HIP_TRY(expr)                                                                                 \
    do {                                                                                              \
        hipError_t e_ = (expr);                                                                       \
        if (e_ != hipSuccess)                                                                         \
            return fail(ctx, RRSPH_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));        \
    } while (0)

template <class R> StateA<R> stateA(rrsph_ctx* c) {
    return StateA<R>{c->posA, (real4<R>*)c->vaA, (real4<R>*)c->adA, c->oidA};
}
template <class R> StateB<R> stateB(rrsph_ctx* c, void* pred, void* pres) {
    return StateB<R>{c->posB, (real4<R>*)c->vaB, (real4<R>*)pred, c->oidB, (R*)pres, nullptr};
}
// the state a list or build step leaves
template <class R> StateA<R> stateOut(rrsph_ctx* c) {
    return c->out.pos ? StateA<R>{c->out.pos, (real4<R>*)c->out.va, (real4<R>*)c->out.ad, c->out.oid} : stateA<R>(c);
}
void* pres_out(const rrsph_ctx* c) { return c->out.pos ? c->out.pres : c->pres; }
// the step's B copy; keeps A.ad too when the fused pass may have to be undone
template <class R> StateB<R> stepB(rrsph_ctx* c) {
    return StateB<R>{c->posB, (real4<R>*)c->vaB, (real4<R>*)c->pred, c->oidB, (R*)c->pres, (real4<R>*)c->adB};
}
// 3D: the position buffers hold double4 (two double2 slots per particle)
template <class R> StateA3<R> stateA3(rrsph_ctx* c) {
    return StateA3<R>{(double4*)c->posA, (real4<R>*)c->vaA, (real4<R>*)c->adA, c->oidA};
}
template <class R> StateA3<R> stateOut3(rrsph_ctx* c) {
    const StateA<R> o = stateOut<R>(c);
    return StateA3<R>{(double4*)o.pos, o.va, o.ad, o.oid};
}
template <class R> StateB3<R> stateB3(rrsph_ctx* c, void* pred, void* pw, void* pres) {
    return StateB3<R>{(double4*)c->posB, (real4<R>*)c->vaB, (real4<R>*)pred, (R*)pw, (R*)pres, c->oidB, nullptr};
}
template <class R> StateB3<R> stepB3(rrsph_ctx* c) {
    return StateB3<R>{(double4*)c->posB, (real4<R>*)c->vaB, (real4<R>*)c->pred, (R*)c->pw, (R*)c->pres, c->oidB,
                      (real4<R>*)c->adB};
}

uint32_t grid_blocks(uint32_t n, uint32_t bs) { return (n + bs - 1) / bs; }

// After two incremental re-sort overflows within kFallbackWindow steps of
// each other, the next kFullSortRun steps use the full radix sort; an
// overflow soon after such a run ends doubles the run (up to kFullSortRunMax).
constexpr uint64_t kFullSortRun = 64;
constexpr uint64_t kFullSortRunMax = 4096;
constexpr uint64_t kFallbackWindow = 8;

// The reach and the skin of the neighbour lists from the skin's fraction of
// the cut-off.
void set_skin(StepParams& P, double skin_frac) {
    P.list_reach = P.cell * (1.0 + skin_frac);
    P.list_r2 = P.list_reach * P.list_reach * (1.0 + 1e-12);
    P.skin_half = 0.5 * P.cell * skin_frac * (1.0 - 1e-9);
}

// Launch helper that optionally records HIP events around the launch.
struct Launcher {
    rrsph_ctx* c;
    Profiler* prof;
    template <class F> void operator()(uint32_t cls, F&& launch) {
        if (prof) {
            hipEvent_t a, b;
            (void)hipEventCreate(&a);
            (void)hipEventCreate(&b);
            (void)hipEventRecord(a, c->stream);
            launch();
            (void)hipEventRecord(b, c->stream);
            prof->rec.push_back({cls, {a, b}});
        } else {
            launch();
        }
    }
};

// Sort key_next (values = index) into kbuf/vbuf; returns final buffers.
void enqueue_sort(rrsph_ctx* c, Ctrl* ctrl, Launcher& L) {
    const uint32_t n = c->P.n;
    const uint32_t* src_k = c->key_next;
    const uint32_t* src_v = nullptr;
    for (uint32_t p = 0; p < c->passes; ++p) {
        uint32_t* dk = c->kbuf[p & 1];
        uint32_t* dv = c->vbuf[p & 1];
        const uint32_t shift = p * kRadixBits;
        const uint32_t nt = c->ntiles;
        L(K_UPSWEEP, [&] { radix_upsweep<<<nt, kBlock, 0, c->stream>>>(src_k, n, shift, c->hist, nt, ctrl); });
        L(K_SCAN, [&] { radix_scan_digits<<<kRadix, kScanBlock, 0, c->stream>>>(c->hist, nt, c->digit_total, ctrl); });
        L(K_DOWNSWEEP, [&] {
            radix_downsweep<<<nt, kBlock, 0, c->stream>>>(src_k, src_v, dk, dv, n, shift, c->hist, nt, c->digit_total,
                                                          ctrl);
        });
        src_k = dk;
        src_v = dv;
    }
    c->sorted_keys = src_k;
    c->sorted_perm = src_v;
}

// The sort of a list build: the counting sort, whose reorder puts the slots
// of a cell in order (the permutation then lies in cell_sort_perm), or the
// radix sort where most cells of the grid are empty.
uint32_t* cell_sort_perm(const rrsph_ctx* c) { return c->vbuf[(c->passes - 1) & 1u]; }
void enqueue_build_sort(rrsph_ctx* c, Ctrl* ctrl, Launcher& L) {
    if (!c->cell_count) {
        enqueue_sort(c, ctrl, L);
        return;
    }
    const StepParams& P = c->P;
    const uint32_t fb = (c->passes - 1) & 1u, nb = P.blocks_per_xcd * kNumXcd, sb = scan_blocks(P.ncells);
    uint32_t *skey = c->kbuf[fb], *place = c->kbuf[1 - fb], *slots = c->vbuf[1 - fb];
    uint32_t* sums = c->cell_count + (size_t)sb * kScanCells;
    L(K_UPSWEEP, [&] { cell_count_kernel<<<nb, kBlock, 0, c->stream>>>(P, c->key_next, place, c->cell_count, ctrl); });
    L(K_SCAN, [&] {
        cell_sums_kernel<<<sb, kBlock, 0, c->stream>>>(c->cell_count, sums, ctrl);
        cell_starts_kernel<<<sb, kBlock, 0, c->stream>>>(P.ncells, c->cell_count, sums, c->LB, ctrl);
    });
    L(K_DOWNSWEEP, [&] {
        cell_scatter_kernel<<<nb, kBlock, 0, c->stream>>>(P, c->key_next, place, c->LB, skey, slots, ctrl);
    });
    c->sorted_keys = skey;
    c->sorted_perm = slots;
}

// Incremental re-sort of key_next against skeyA into kbuf[0] / vbuf[0]; its
// first kernel also runs the step prologue.
void enqueue_resort(rrsph_ctx* c, Launcher& L) {
    const uint32_t n = c->P.n;
    const uint32_t nb = grid_blocks(n, kBlock);
    L(K_RESORT_SORT, [&] {
        resort_sort_small<<<1, kResortBlock, 0, c->stream>>>(c->P, c->key_next, c->resort_cap, c->chg, c->wpre,
                                                             c->ctrl);
    });
    L(K_RESORT_SCATTER, [&] {
        resort_scatter<<<nb, kBlock, 0, c->stream>>>(c->skeyA, c->chg, c->chg_mask, c->wpre, n, c->kbuf[0],
                                                     c->vbuf[0], c->ctrl, c->resort_stage);
    });
    c->sorted_keys = c->kbuf[0];
    c->sorted_perm = c->vbuf[0];
}

template <class R> void enqueue_step_t(rrsph_ctx* c, Profiler* prof, bool full_sort) {
    Launcher L{c, prof};
    const StepParams& P = c->P;
    const uint32_t nb = grid_blocks(P.n, kBlock);
    const uint32_t nb_xcd = P.blocks_per_xcd * kNumXcd;
    if (full_sort) {
        L(K_PROLOGUE, [&] { step_prologue<<<1, kWave, 0, c->stream>>>(P, c->ctrl); });
        enqueue_sort(c, c->ctrl, L);
    } else {
        enqueue_resort(c, L);
    }
    StateA<R> A = stateA<R>(c);
    StateB<R> B = stepB<R>(c);
    L(K_REORDER, [&] {
        reorder_kernel<R><<<nb, kBlock, 0, c->stream>>>(P, c->ctrl, c->sorted_keys, c->sorted_perm, A, B, c->LB,
                                                        c->maxslots, c->skeyA);
    });
    if (P.density_treatment == 0) {
        L(K_DENSITY_SUM, [&] {
            density_sum_kernel<R><<<nb_xcd, kBlock, 0, c->stream>>>(P, c->ctrl, B, c->sorted_keys, c->LB);
        });
    }
    real4<R>* der = (real4<R>*)c->der;
    real4<R>* xs = (real4<R>*)c->xs;
    const uint32_t nt_xcd = P.tile_blocks_per_xcd * kNumXcd;
    const int impl = c->fast_pair ? c->pair_impl : 0;
    auto pair = [&](auto kernel) {
        const uint32_t grid = impl == 2 ? nt_xcd : nb_xcd;
        const uint32_t block = impl == 2 ? kTile * kTilesPerBlock : kBlock;
        L(K_PAIR, [&] {
            kernel<<<grid, block, 0, c->stream>>>(P, c->ctrl, B, c->sorted_keys, c->LB, A, c->key_next, der, xs,
                                                  c->maxslots);
        });
    };
    auto choose = [&](auto general, auto fast, auto tile, auto walk) {
        if (impl == 3) pair(walk);
        else if (impl == 2) pair(tile);
        else if (impl == 1) pair(fast);
        else pair(general);
    };
    if (c->fused) {
        if (c->export_fields)
            choose(pair_kernel<R, true, true>, pair_fast_kernel<R, true, true>, pair_tile_kernel<R, true, true>,
                   pair_fast_kernel<R, true, true, false>);
        else
            choose(pair_kernel<R, true, false>, pair_fast_kernel<R, true, false>, pair_tile_kernel<R, true, false>,
                   pair_fast_kernel<R, true, false, false>);
    } else {
        choose(pair_kernel<R, false, true>, pair_fast_kernel<R, false, true>, pair_tile_kernel<R, false, true>,
               pair_fast_kernel<R, false, true, false>);
        L(K_INTEGRATE, [&] {
            integrate_kernel<R><<<nb, kBlock, 0, c->stream>>>(P, c->ctrl, B, der, xs, A, c->key_next, c->maxslots,
                                                              c->sorted_keys);
        });
    }
}

template <class R> void enqueue_step3_t(rrsph_ctx* c, Profiler* prof, bool full_sort) {
    Launcher L{c, prof};
    const StepParams& P = c->P;
    const uint32_t nb = grid_blocks(P.n, kBlock);
    const uint32_t nb_xcd = P.blocks_per_xcd * kNumXcd;
    if (full_sort) {
        L(K_PROLOGUE, [&] { step_prologue<<<1, kWave, 0, c->stream>>>(P, c->ctrl); });
        enqueue_sort(c, c->ctrl, L);
    } else {
        enqueue_resort(c, L);
    }
    StateA3<R> A = stateA3<R>(c);
    StateB3<R> B = stepB3<R>(c);
    L(K_REORDER, [&] {
        reorder3_kernel<R><<<nb, kBlock, 0, c->stream>>>(P, c->ctrl, c->sorted_keys, c->sorted_perm, A, B, c->LB,
                                                         c->maxslots, c->skeyA);
    });
    if (P.density_treatment == 0) {
        L(K_DENSITY_SUM, [&] {
            density_sum3_kernel<R><<<nb_xcd, kBlock, 0, c->stream>>>(P, c->ctrl, B, c->sorted_keys, c->LB);
        });
    }
    real4<R>* der = (real4<R>*)c->der;
    real4<R>* xs = (real4<R>*)c->xs;
    auto pair = [&](auto kernel) {
        L(K_PAIR, [&] {
            kernel<<<nb_xcd, kBlock, 0, c->stream>>>(P, c->ctrl, B, c->sorted_keys, c->LB, A, c->key_next, der, xs,
                                                     c->maxslots);
        });
    };
    if (c->fused) {
        if (c->export_fields) pair(pair3_kernel<R, true, true>);
        else pair(pair3_kernel<R, true, false>);
    } else {
        pair(pair3_kernel<R, false, true>);
        L(K_INTEGRATE, [&] {
            integrate3_kernel<R><<<nb, kBlock, 0, c->stream>>>(P, c->ctrl, B, der, xs, A, c->key_next, c->maxslots,
                                                               c->sorted_keys);
        });
    }
}

// A list step's kind: a build, a list step, or the first or second of a pair
// of fused ones (fused_step_begin in list_step.hpp).
enum ListStep { kBuildStep, kPlainStep, kFusedFirst, kFusedSecond };

// The arrays between which fused steps go back and forth: the records, and in
// FP32 the positions.
void fused_arrays(rrsph_ctx* c, ListStep kind, void*& rec, void*& rec_out, double2*& pos, double2*& pos_out) {
    const bool second = kind == kFusedSecond;
    rec = second ? c->rec1 : c->rec;
    rec_out = second ? c->rec : c->rec1;
    pos = second && c->fp32 ? c->posB : c->posA;
    pos_out = !second && c->fp32 ? c->posB : c->posA;
}

// The summation and pair passes of a 2D neighbour-list step, LPP lanes per particle.
template <class R, int LPP, bool ALL>
void enqueue_list_passes(rrsph_ctx* c, Launcher& L, ListState<R> X, ListStep kind) {
    const StepParams& P = c->P;
    const uint32_t nb = group_blocks_per_xcd<LPP>(P.n) * kNumXcd;
    ListRec<R>* rec = (ListRec<R>*)c->rec;
    Ctrl *next = c->ctrl, *cur = c->ctrl_cur;
    ListOut<R> O{};
    const bool fused = kind == kFusedFirst || kind == kFusedSecond;
    if (fused) {
        void *r, *ro;
        double2 *p, *po;
        fused_arrays(c, kind, r, ro, p, po);
        rec = (ListRec<R>*)r;
        X.pos = p;
        O = ListOut<R>{po, (real4<R>*)c->vaA, (ListRec<R>*)ro, c->home, c->key_next, c->ctrl, kind == kFusedSecond};
    }
    bool first = kind != kBuildStep;
    if (P.density_treatment == 0) {
        auto density = [&](auto kernel) {
            L(K_DENSITY_SUM, [&] {
                kernel<<<nb, kBlock, 0, c->stream>>>(P, next, cur, X, rec, (R*)pres_out(c), c->nbl, c->nbc, c->dslots);
            });
        };
        if (first) density(density_sum_list<R, true, LPP>);
        else density(density_sum_list<R, false, LPP>);
        first = false;
    } else if (fused) {  // the step's only kernel reads the control block here and publishes there
        next = kind == kFusedSecond ? c->ctrl_alt : c->ctrl;
        cur = kind == kFusedSecond ? c->ctrl : c->ctrl_alt;
    }
    auto pair = [&](auto kernel) {
        L(K_PAIR, [&] {
            kernel<<<nb, kBlock, 0, c->stream>>>(P, next, cur, X, rec, (R*)pres_out(c), c->nbl, c->nbc,
                                                 stateOut<R>(c).ad, (real2<R>*)c->xs, c->dtslots, c->dslots, O);
        });
    };
    auto general = [&](auto kernel) {
        L(K_PAIR, [&] {
            kernel<<<nb, kBlock, 0, c->stream>>>(P, next, cur, X, rec, (R*)pres_out(c), c->nbl, c->nbc,
                                                 stateOut<R>(c).ad, (real2<R>*)c->xs, c->dtslots, c->dslots);
        });
    };
    if constexpr (ALL) {
        if (fused) {
            if (P.density_treatment == 0) pair(pair_list_kernel<R, false, LPP, false, true, true>);
            else pair(pair_list_kernel<R, true, LPP, true, true, true>);
            return;
        }
    }
    if (c->fast_pair) {
        if (P.density_treatment == 0) pair(pair_list_kernel<R, false, LPP, false, ALL, false>);
        else if (first) pair(pair_list_kernel<R, true, LPP, true, ALL, false>);
        else pair(pair_list_kernel<R, false, LPP, true, ALL, false>);
    } else if (first) {
        general(pair_list_general_kernel<R, true, LPP>);
    } else {
        general(pair_list_general_kernel<R, false, LPP>);
    }
}

// One neighbour-list step (a build: sort, reorder and new lists first).
template <class R> void enqueue_list_step_t(rrsph_ctx* c, Profiler* prof, ListStep kind) {
    Launcher L{c, prof};
    const StepParams& P = c->P;
    const uint32_t nb = grid_blocks(P.n, kBlock);
    const uint32_t nb_xcd = P.blocks_per_xcd * kNumXcd;
    ListState<R> X{c->posA, (const real4<R>*)c->vaA, c->oidA};
    ListRec<R>* rec = (ListRec<R>*)c->rec;
    if (kind == kBuildStep) {
        L(K_PROLOGUE, [&] {
            list_prologue<<<1, kBlock, 0, c->stream>>>(P, c->ctrl, c->ctrl_cur, c->dslots, c->dtslots);
        });
        enqueue_build_sort(c, c->ctrl_cur, L);
        StateA<R> A = stateA<R>(c);
        StateB<R> B = stateB<R>(c, c->pred, pres_out(c));
        L(K_REORDER, [&] {
            auto reorder = [&](auto kernel) {
                kernel<<<nb, kBlock, 0, c->stream>>>(P, c->ctrl_cur, c->sorted_keys, c->sorted_perm, A, B, rec, c->home,
                                                     c->LB, cell_sort_perm(c));
            };
            if (c->cell_count) reorder(reorder_list_kernel<R, true>);
            else reorder(reorder_list_kernel<R, false>);
        });
        L(K_LIST_BUILD, [&] {
            list_build_kernel<R><<<nb_xcd, kBlock, 0, c->stream>>>(P, c->ctrl, c->ctrl_cur, c->posB, (const real4<R>*)c->vaB,
                                                                   c->sorted_keys, c->LB, c->nbl, c->nbc);
        });
        X = ListState<R>{c->posB, (const real4<R>*)c->vaB, c->oidB};
    }
    // the first kernel of a list step makes its prologue
    if (!c->all_terms && c->fast_pair) enqueue_list_passes<R, 1, false>(c, L, X, kind);
    else if (c->lanes == 8) enqueue_list_passes<R, 8, true>(c, L, X, kind);
    else if (c->lanes == 2) enqueue_list_passes<R, 2, true>(c, L, X, kind);
    else enqueue_list_passes<R, 1, true>(c, L, X, kind);
    if (kind == kFusedFirst || kind == kFusedSecond) return;
    L(K_INTEGRATE, [&] {
        integrate_list_kernel<R><<<nb, kBlock, 0, c->stream>>>(P, c->ctrl, c->ctrl_cur, X, (const real2<R>*)c->xs, rec, c->home, stateOut<R>(c),
                                                               c->key_next, c->dtslots, c->dslots, c->out.keep);
    });
}

// One 3D neighbour-list step (build: sort, reorder and new lists first).
template <class R> void enqueue_list_step3_t(rrsph_ctx* c, Profiler* prof, ListStep kind) {
    Launcher L{c, prof};
    const StepParams& P = c->P;
    const uint32_t nb = grid_blocks(P.n, kBlock);
    const uint32_t nb_xcd = P.blocks_per_xcd * kNumXcd;
    ListState3<R> X{(const double4*)c->posA, (const real4<R>*)c->vaA, c->oidA};
    ListRec<R>* rec = (ListRec<R>*)c->rec;
    real4<R>* dens = (real4<R>*)c->dens;
    const bool build = kind == kBuildStep, fused = kind == kFusedFirst || kind == kFusedSecond;
    ListOut3<R> O{};
    if (fused) {
        void *r, *ro;
        double2 *p, *po;
        fused_arrays(c, kind, r, ro, p, po);
        rec = (ListRec<R>*)r;
        X.pos = (const double4*)p;
        O = ListOut3<R>{(double4*)po,    (real4<R>*)c->vaA, (ListRec<R>*)ro,      dens,
                        c->home, c->key_next,       c->ctrl, kind == kFusedSecond};
    }
    if (build) {
        L(K_PROLOGUE, [&] {
            list_prologue<<<1, kBlock, 0, c->stream>>>(P, c->ctrl, c->ctrl_cur, c->dslots, c->dtslots);
        });
        enqueue_build_sort(c, c->ctrl_cur, L);
        StateA3<R> A = stateA3<R>(c);
        StateB3<R> B = stateB3<R>(c, c->pred, c->pw, pres_out(c));
        L(K_REORDER, [&] {
            auto reorder = [&](auto kernel) {
                kernel<<<nb, kBlock, 0, c->stream>>>(P, c->ctrl_cur, c->sorted_keys, c->sorted_perm, A, B, rec, dens,
                                                     c->home, c->cand, c->LB, cell_sort_perm(c));
            };
            if (c->cell_count) reorder(reorder_list3_kernel<R, true>);
            else reorder(reorder_list3_kernel<R, false>);
        });
        L(K_LIST_BUILD, [&] {
            list_build3_kernel<<<nb_xcd, kBlock, 0, c->stream>>>(P, c->ctrl, c->ctrl_cur, (const double4*)c->posB, c->cand,
                                                                 c->sorted_keys, c->LB, c->nbl, c->nbc);
        });
        X = ListState3<R>{(const double4*)c->posB, (const real4<R>*)c->vaB, c->oidB};
    }
    bool first = !build;
    if (P.density_treatment == 0) {
        auto density = [&](auto kernel) {
            L(K_DENSITY_SUM, [&] {
                kernel<<<nb_xcd, kBlock, 0, c->stream>>>(P, c->ctrl, c->ctrl_cur, X, dens, rec, (R*)pres_out(c), c->nbl,
                                                         c->nbc, c->dslots);
            });
        };
        if (first) density(density_sum_list3<R, true>);
        else density(density_sum_list3<R, false>);
        first = false;
    }
    auto pair = [&](auto kernel) {
        L(K_PAIR, [&] {
            kernel<<<nb_xcd, kBlock, 0, c->stream>>>(P, c->ctrl, c->ctrl_cur, X, rec, (R*)pres_out(c), c->nbl, c->nbc,
                                                     stateOut<R>(c).ad, (real4<R>*)c->xs, c->dtslots, c->dslots, O);
        });
    };
    auto choose = [&](auto summed, auto first_kernel, auto kernel) {
        if (P.density_treatment == 0) pair(summed);
        else if (first) pair(first_kernel);
        else pair(kernel);
    };
    if (fused) {
        pair(pair_list3_kernel<R, false, false, true, true>);
        return;
    }
    if (c->all_terms)
        choose(pair_list3_kernel<R, false, false, true, false>, pair_list3_kernel<R, true, true, true, false>,
               pair_list3_kernel<R, false, true, true, false>);
    else
        choose(pair_list3_kernel<R, false, false, false, false>, pair_list3_kernel<R, true, true, false, false>,
               pair_list3_kernel<R, false, true, false, false>);
    L(K_INTEGRATE, [&] {
        integrate_list3_kernel<R><<<nb, kBlock, 0, c->stream>>>(P, c->ctrl, c->ctrl_cur, X,
                                                                (const real4<R>*)c->xs, rec, dens, c->home,
                                                                stateOut3<R>(c), c->key_next, c->dtslots, c->dslots,
                                                                c->out.keep);
    });
}

void enqueue_list_step(rrsph_ctx* c, Profiler* prof, ListStep kind) {
    if (c->P.dim == 3) {
        if (c->fp32) enqueue_list_step3_t<float>(c, prof, kind);
        else enqueue_list_step3_t<double>(c, prof, kind);
        return;
    }
    if (c->fp32) enqueue_list_step_t<float>(c, prof, kind);
    else enqueue_list_step_t<double>(c, prof, kind);
}

bool list_active(const rrsph_ctx* c) { return c->list_mode && !c->list_suspended; }

void enqueue_step(rrsph_ctx* c, Profiler* prof, bool full_sort) {
    if (c->P.dim == 3) {
        if (c->fp32) enqueue_step3_t<float>(c, prof, full_sort);
        else enqueue_step3_t<double>(c, prof, full_sort);
        return;
    }
    if (c->fp32) enqueue_step_t<float>(c, prof, full_sort);
    else enqueue_step_t<double>(c, prof, full_sort);
}

void drop_list_graphs(rrsph_ctx* c) {
    for (auto e : c->list_graphs.exec)
        if (e) (void)hipGraphExecDestroy(e);
    for (auto g : c->list_graphs.graph)
        if (g) (void)hipGraphDestroy(g);
    c->list_graphs = ListGraphs{};
}

void drop_graph(rrsph_ctx* c) {
    hipGraphExec_t* ex[] = {&c->gexec, &c->gexec_full};
    hipGraph_t* gr[] = {&c->graph, &c->graph_full};
    for (auto* e : ex) {
        if (*e) (void)hipGraphExecDestroy(*e);
        *e = nullptr;
    }
    for (auto* g : gr) {
        if (*g) (void)hipGraphDestroy(*g);
        *g = nullptr;
    }
    drop_list_graphs(c);
}

// Capture one step with the incremental re-sort and one with the full sort.
rrsph_status build_graph(rrsph_ctx* ctx) {
    drop_graph(ctx);
    HIP_TRY(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    enqueue_step(ctx, nullptr, false);
    HIP_TRY(hipStreamEndCapture(ctx->stream, &ctx->graph));
    HIP_TRY(hipGraphInstantiate(&ctx->gexec, ctx->graph, nullptr, nullptr, 0));
    HIP_TRY(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    enqueue_step(ctx, nullptr, true);
    HIP_TRY(hipStreamEndCapture(ctx->stream, &ctx->graph_full));
    HIP_TRY(hipGraphInstantiate(&ctx->gexec_full, ctx->graph_full, nullptr, nullptr, 0));
    return RRSPH_OK;
}

// Launch a build step (build) or `steps` list steps (a power of two up to
// kListRunMax) through the captured graphs, or directly.
rrsph_status launch_list_run(rrsph_ctx* ctx, bool build, uint32_t steps) {
    auto enqueue = [&]() {
        for (uint32_t k = 0; k < steps; ++k) {
            const ListStep kind = build ? kBuildStep
                                  : ctx->fuse && !ctx->taping && steps > 1 ? (k & 1 ? kFusedSecond : kFusedFirst)
                                                                           : kPlainStep;
            enqueue_list_step(ctx, nullptr, kind);
        }
    };
    // a taped step reads and leaves its state at addresses of its own, and every
    // run sets new piston coefficients, which a graph would hold
    if (!ctx->use_graph || ctx->taping) {
        enqueue();
        return RRSPH_OK;
    }
    ListGraphs& G = ctx->list_graphs;
    const uint32_t i = build ? 0 : 1 + (uint32_t)__builtin_ctz(steps);
    if (!G.exec[i]) {
        HIP_TRY(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        enqueue();
        HIP_TRY(hipStreamEndCapture(ctx->stream, &G.graph[i]));
        HIP_TRY(hipGraphInstantiate(&G.exec[i], G.graph[i], nullptr, nullptr, 0));
    }
    HIP_TRY(hipGraphLaunch(G.exec[i], ctx->stream));
    return RRSPH_OK;
}

// Sort + reorder of the current state into B (with a scratch pred) for the
// utility queries, using a control block that is never halted.
// The arrays of a state saved in an adjoint blob (pos | va | ad | oid | ...),
// read in place by the reverse steps.
struct StateView {
    void *pos, *va, *ad;
    uint32_t* oid;
};
template <class R> void enqueue_util_reorder(rrsph_ctx* c, const StateView* src = nullptr, Ctrl* uc = nullptr);
template <class R> void enqueue_util_sort(rrsph_ctx* c, Ctrl* uc = nullptr) {
    Launcher L{c, nullptr};
    enqueue_sort(c, uc ? uc : c->util_ctrl, L);
    enqueue_util_reorder<R>(c, nullptr, uc);
}

// Reorder of the current state (or of the saved state src) by sorted_keys /
// sorted_perm into B (scratch pred) and the cell-start table, for the
// utility queries; with the control block uc (its cur_dt predicts) instead
// of the context's utility one.
template <class R> void enqueue_util_reorder(rrsph_ctx* c, const StateView* src, Ctrl* uc) {
    const uint32_t nb = grid_blocks(c->P.n, kBlock);
    const Ctrl* ctrl = uc ? uc : c->util_ctrl;
    if (c->P.dim == 3) {
        StateA3<R> A = stateA3<R>(c);
        if (src) A = StateA3<R>{(double4*)src->pos, (real4<R>*)src->va, (real4<R>*)src->ad, src->oid};
        reorder3_kernel<R><<<nb, kBlock, 0, c->stream>>>(c->P, ctrl, c->sorted_keys, c->sorted_perm, A,
                                                         stateB3<R>(c, c->pred_scratch, c->pw_scratch, c->pres_scratch),
                                                         c->LB, c->maxslots + 2 * kMaxSlots, nullptr);
        return;
    }
    StateA<R> A = stateA<R>(c);
    if (src) A = StateA<R>{(double2*)src->pos, (real4<R>*)src->va, (real4<R>*)src->ad, src->oid};
    StateB<R> B = stateB<R>(c, c->pred_scratch, c->pres_scratch);
    reorder_kernel<R><<<nb, kBlock, 0, c->stream>>>(c->P, ctrl, c->sorted_keys, c->sorted_perm, A, B, c->LB,
                                                    c->maxslots + 2 * kMaxSlots, nullptr);
}

// Up to kCopyRanges device-to-device copies in one launch (the saved-state
// blobs of the adjoint move five arrays at a time; separate copies cost a
// launch each, which dominates at tens of thousands of particles).  Lengths
// are in 4-byte words; a range moves 16 bytes per access when both ends are
// 16-byte aligned.
constexpr int kCopyRanges = 8;
struct CopyRange {
    const uint32_t* src;
    uint32_t* dst;
    size_t words;
};
struct CopyPlan {
    CopyRange r[kCopyRanges];
    int n = 0;
    void add(const void* src, void* dst, size_t bytes) { r[n++] = {(const uint32_t*)src, (uint32_t*)dst, bytes / 4}; }
};
__global__ void __launch_bounds__(kBlock) copy_ranges_kernel(CopyPlan plan) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
    for (int k = 0; k < plan.n; ++k) {
        const CopyRange c = plan.r[k];
        size_t done = 0;
        if (((reinterpret_cast<uintptr_t>(c.src) | reinterpret_cast<uintptr_t>(c.dst)) & 15u) == 0) {
            const size_t n4 = c.words / 4;
            const uint4* __restrict__ s = (const uint4*)c.src;
            uint4* __restrict__ d = (uint4*)c.dst;
            for (size_t i = t; i < n4; i += stride) d[i] = s[i];
            done = n4 * 4;
        }
        for (size_t i = done + t; i < c.words; i += stride) c.dst[i] = c.src[i];
    }
}
rrsph_status enqueue_copies(rrsph_ctx* ctx, const CopyPlan& plan) {
    size_t units = 0;
    for (int k = 0; k < plan.n; ++k) units = std::max(units, plan.r[k].words / 4 + 1);
    const uint32_t blocks = (uint32_t)std::min<size_t>(2048, (units + kBlock - 1) / kBlock);
    copy_ranges_kernel<<<std::max(blocks, 1u), kBlock, 0, ctx->stream>>>(plan);
    HIP_TRY(hipGetLastError());
    return RRSPH_OK;
}

std::string status_message(uint32_t st) {
    switch (st) {
    case RRSPH_ERR_TOO_MANY_NEIGHBOURS: return "making neighbours grid: error occured";
    case RRSPH_ERR_NEVER_ENDING: return "never ending simulation";
    case RRSPH_ERR_OUTSIDE_BOUNDARIES: return "Encounter particle outside boundaries";
    default: return "";
    }
}

void enqueue_state_keys(rrsph_ctx* ctx);

// A fused step whose neighbour lists overflowed under the consistency check
// was integrated in its pair pass; the prologue after it refused to commit
// it.  Put back the state the step started from: its sorted copy B (pos, va,
// oid) and the copy of A.ad the reorder kept, then the cell keys of that
// state for the next sort.
rrsph_status rollback_fused_step(rrsph_ctx* ctx) {
    const size_t n = ctx->P.n, pb = ctx->P.dim == 3 ? 32 : 16, vb = ctx->fp32 ? 16 : 32;
    if (!ctx->adB) return fail(ctx, RRSPH_ERR_HIP, "RRSPH_HIP: no copy of the step's input to restore");
    CopyPlan plan;
    plan.add(ctx->posB, ctx->posA, pb * n);
    plan.add(ctx->vaB, ctx->vaA, vb * n);
    plan.add(ctx->adB, ctx->adA, vb * n);
    plan.add(ctx->oidB, ctx->oidA, 4 * n);
    if (const rrsph_status st = enqueue_copies(ctx, plan); st != RRSPH_OK) return st;
    enqueue_state_keys(ctx);
    ctx->need_full = true;
    ctx->host_ctrl->rollback = 0;
    HIP_TRY(hipMemcpyAsync(ctx->ctrl, ctx->host_ctrl, sizeof(Ctrl), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return RRSPH_OK;
}

// A halt that the host answers by running the halted step again (resume_halt), none of rrsph_status.
bool rerun_status(uint32_t status) {
    return status == kStatusResort || status == kStatusRebuild || status == kStatusListOverflow ||
           status == kStatusUnfused;
}

// Read the control block after the stream drained and turn it into a status.
rrsph_status sync_status(rrsph_ctx* ctx) {
    HIP_TRY(hipMemcpyAsync(ctx->host_ctrl, ctx->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    const Ctrl& c = *ctx->host_ctrl;
    if (c.halted && c.status != 0 && !rerun_status(c.status)) {
        if (c.rollback) {
            if (const rrsph_status st = rollback_fused_step(ctx); st != RRSPH_OK) return st;
        } else if (c.status == RRSPH_ERR_TOO_MANY_NEIGHBOURS || c.status == RRSPH_ERR_NEVER_ENDING) {
            // the step has left its fields (with lists A.ad, which the next step
            // would have started from) and pressures in the slot order that it
            // sorted into, and the state in the one before; a list step (some
            // displacement counted since its build) sorted nothing
            ctx->pres_in_order = ctx->list_fields && c.disp_acc > 0.0;
            ctx->fields_valid = ctx->fields_valid && ctx->pres_in_order;
        }
        return fail(ctx, (rrsph_status)c.status, status_message(c.status));
    }
    if (c.pending) {
        if (ctx->P.consistency_check && c.nbr_overflow) {
            // the last launched step was a fused one that overflowed: no
            // prologue ran after it, so do what it would have done (leave the
            // step uncommitted, put its input back, stay halted)
            Ctrl& h = *ctx->host_ctrl;
            h.pending = 0;
            h.halted = 1;
            h.status = RRSPH_ERR_TOO_MANY_NEIGHBOURS;
            if (h.wall_disappear) h.nwm_done = 0;
            if (const rrsph_status st = rollback_fused_step(ctx); st != RRSPH_OK) return st;
            return fail(ctx, RRSPH_ERR_TOO_MANY_NEIGHBOURS, status_message(RRSPH_ERR_TOO_MANY_NEIGHBOURS));
        }
        if (ctx->P.consistency_check && ctrl_outside(c) > 0 && ctx->P.consistency_treatment == 1)
            return fail(ctx, RRSPH_ERR_OUTSIDE_BOUNDARIES, status_message(RRSPH_ERR_OUTSIDE_BOUNDARIES));
    }
    return RRSPH_OK;
}

rrsph_status setup_params(rrsph_ctx* ctx, const rrsph_params_c& p) {
    StepParams& P = ctx->P;
    P = StepParams{};
    if (p.dim != 2 && p.dim != 3) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: dim must be 2 or 3");
    const bool d3 = p.dim == 3;
    if (p.ntotal == 0 || p.max_neighbours < 2 || !(p.hsml > 0) || !(p.cell_scale_k > 0))
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: invalid sizes");
    if (p.nfluid > p.ntotal) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: nfluid > ntotal");
    P.n = p.ntotal;
    P.nfluid = p.nfluid;
    P.max_nbr = p.max_neighbours;
    P.dim = p.dim;
    P.cell = p.cell_scale_k * p.hsml;
    // Input.cpp:45-70: at most 2^16 cells per axis in 2D, 2^10 in 3D
    const double tx = (p.x_maxgeom - p.x_mingeom) / P.cell, ty = (p.y_maxgeom - p.y_mingeom) / P.cell;
    const double tz = d3 ? (p.z_maxgeom - p.z_mingeom) / P.cell : 0.0;
    const double max_id = d3 ? 1024.0 : 65536.0;
    if (!(tx >= 0) || !(ty >= 0) || !(tz >= 0) || tx > max_id || ty > max_id || (d3 && tz >= max_id))
        return fail(ctx, RRSPH_ERR_TOO_MANY_CELLS, "can't make grid with so many cells");
    P.ncx = (int32_t)(uint64_t)tx + 1;
    P.ncy = (int32_t)(uint64_t)ty + 1;
    P.ncz = d3 ? (int32_t)(uint64_t)tz + 1 : 1;
    const uint64_t ncells = (uint64_t)P.ncx * (uint64_t)P.ncy * (uint64_t)P.ncz;
    if (ncells + 2 >= (1ull << 31)) return fail(ctx, RRSPH_ERR_TOO_MANY_CELLS, "can't make grid with so many cells");
    P.ncells = (uint32_t)ncells;
    P.xmin = p.x_mingeom;
    P.ymin = p.y_mingeom;
    P.zmin = p.z_mingeom;
    P.xmax = p.x_maxgeom;
    P.ymax = p.y_maxgeom;
    P.zmax = p.z_maxgeom;
    P.cut2 = P.cell * P.cell;
    P.h = p.hsml;
    P.mass = p.mass;
    P.rho0 = p.rho0;
    P.g = p.g;
    const double h = p.hsml, pi = p.pi;
    // SmoothingKernel.h:22-23, 93-94, 136-137, 194-195
    P.f_cubic = d3 ? double(3) / (double(2) * pi * (h * h * h)) : double(15) / (double(7) * pi * (h * h));
    P.f_gauss = d3 ? 1 / (pi * std::sqrt(pi) * (h * h * h)) : 1 / (pi * (h * h));
    P.f_wend = d3 ? 21 / (16 * pi * (h * h * h)) : 7 / (4 * pi * (h * h));
    P.f_desb = d3 ? 15 / (pi * (4 * h) * (4 * h) * (4 * h)) : 5 / (16 * pi * (h * h));
    P.inv_h = 1.0 / h;
    P.c_q1 = P.f_cubic / (h * h);
    P.c_q2 = 0.5 * P.f_cubic / h;
    P.w_q2 = P.f_cubic / 6.0;
    P.g_gauss = -2.0 / (h * h);
    P.g_wend = (double)(-5.0L * P.f_wend / ((long double)h * h));
    P.g_desb = (double)(-3.0L * P.f_desb / ((long double)h * h));
    P.lp_a2 = 2.0 * h * (p.artificial_shear_visc * p.eos_sound_vel);
    P.lp_b2 = 2.0 * h * h * p.artificial_bulk_visc;
    P.lp_mF = -2.0 * P.f_cubic * p.mass / (h * h * h);
    P.lp_mW = 2.0 * p.average_velocity_coef * p.mass * P.f_cubic / (h * h * h);
    P.skf_density = p.density_skf;
    P.skf_intf = p.intf_skf;
    P.skf_av = p.artificial_viscosity_skf;
    P.skf_xsph = p.average_velocity_skf;
    P.skf_ap = p.artificial_pressure_skf;
    P.eos_B = p.eos_c_sqr * p.rho0 / 7;
    P.density_treatment = p.density_treatment;
    if (p.density_normalization && p.density_treatment != 0)
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: density_normalization needs density_treatment 0");
    P.renorm = p.density_normalization ? 1 : 0;
    P.renorm_every = p.density_normalization_every ? p.density_normalization_every : 1u;
    P.dhc = p.density_delta_sph_coef * p.hsml * p.eos_c;
    P.intf_approx = p.intf_sph_approximation;
    P.art_pressure = p.artificial_pressure;
    P.ap_coef = p.artificial_pressure_coef;
    P.ap_index = p.artificial_pressure_index;
    P.ap_wdelta = host_w(p, p.delta, p.artificial_pressure_skf);
    P.av_on = p.artificial_viscosity;
    P.av_alpha = p.artificial_shear_visc;
    P.av_beta = p.artificial_bulk_visc;
    P.av_c = p.eos_sound_vel;
    const double etq = (double)0.1f;  // ArtificialViscosity.h:22 (a float literal)
    P.av_eta2 = (p.hsml * etq) * (p.hsml * etq);
    P.xsph_on = p.average_velocity;
    P.xsph_eps = p.average_velocity_coef;
    P.lj_on = p.boundary_treatment == 1;
    P.lj_r0 = 2 * p.hsml;
    P.lj_D = 5 * p.g * p.depth;
    P.dt_method = p.dt_correction_method;
    P.dt_dynamic_mode = p.dt_dynamic_mode;
    P.dt0 = p.dt;
    P.cfl = p.CFL_coef;
    P.c0 = p.eos_c;
    P.never_ending = (p.hsml / p.eos_c) * 1.E-6;
    P.consistency_check = p.consistency_check;
    P.consistency_treatment = p.consistency_treatment;
    P.boundary_motion = p.boundary_motion;
    P.nwm = p.nwm;
    P.nwm_axis = -1;
    if (p.nwm == 2 || p.nwm == 3 || p.nwm == 6) {
        if (p.nwm_direction == 1) P.nwm_axis = 0;
        else if (p.nwm_direction == 2) P.nwm_axis = 1;
        else if (p.nwm_direction == 3 && d3) P.nwm_axis = 2;
        else if (p.nwm_direction == 4 && d3 && p.boundary_motion)
            return fail(ctx, RRSPH_ERR_NOT_IMPLEMENTED, "RRSPH_HIP: radial wave makers are not implemented");
    } else if (p.nwm == 5) {
        P.nwm_axis = 0;
    }
    bool range_ok = !(p.nwm_particles_start < p.nfluid || p.nwm_particles_end < p.nfluid ||
                      p.nwm_particles_end < p.nwm_particles_start || p.nwm_particles_end > p.ntotal);
    if (!range_ok) P.nwm = 0;  // CLTimeIntegration.cpp:375-385: wrong range -> no wave maker
    P.nwm_start = p.nwm_particles_start;
    P.nwm_end = p.nwm_particles_end;
    P.nwm_time_start = p.nwm_time_start;
    P.nwm_freq = p.nwm_freq;
    P.nwm_delta = p.nwm_phase - p.nwm_freq * p.nwm_time_start;
    {
        const double kd = p.nwm_wave_number * p.depth, H = p.nwm_wave_magnitude;
        const double sh = std::sinh(kd), ch = std::cosh(kd);
        const double m1 = 2 * sh * sh / (sh * ch + kd);
        P.nwm_S0 = m1 != 0 ? H / m1 : 0;
        P.nwm_e2 = (m1 != 0 && sh != 0) ? (H * H / (32 * p.depth)) * (3 * ch / (sh * sh * sh) - 2 / m1) : 0;
        const double Hs = p.nwm_wave_magnitude, hd = p.depth;
        P.sol_H = Hs;
        P.sol_h = hd;
        P.sol_k = std::sqrt(3 * Hs / (4 * hd * hd * (Hs + hd)));
        P.sol_c = std::sqrt(p.g * (Hs + hd));
        P.sol_Tf = 2 / (P.sol_k * P.sol_c) * (3.8 + Hs / hd);
    }
    const int32_t segs = p.piston_segments > 1 ? p.piston_segments : 1;
    if (p.piston_nharm < 0 || segs > kMaxSegments || (int64_t)p.piston_nharm * segs > 32)
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT,
                    "RRSPH_HIP: piston_nharm * piston_segments must be at most 32, piston_segments at most 8");
    if (segs > 1 && (!d3 || p.nwm != 6 || !(p.piston_seg_zmax > p.piston_seg_zmin)))
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT,
                    "RRSPH_HIP: a segmented piston needs dim 3, nwm 6 and piston_seg_zmax > piston_seg_zmin");
    P.piston_nharm = p.piston_nharm;
    P.piston_segments = segs;
    P.piston_seg_z0 = segs > 1 ? p.piston_seg_zmin : 0.0;
    P.piston_seg_inv_w = segs > 1 ? segs / (p.piston_seg_zmax - p.piston_seg_zmin) : 0.0;
    P.piston_omega = p.piston_omega;
    for (int k = 0; k < 32; ++k) {
        P.piston_a[k] = p.piston_a[k];
        P.piston_b[k] = p.piston_b[k];
    }
    P.nblocks = grid_blocks(P.n, kBlock);
    P.blocks_per_xcd = (P.nblocks + kNumXcd - 1) / kNumXcd;
    P.ntiles = grid_blocks(P.n, kTile);
    P.tile_blocks_per_xcd = (grid_blocks(P.ntiles, kTilesPerBlock) + kNumXcd - 1) / kNumXcd;
    // radix passes over the key bits (dead key = ncells must fit)
    uint32_t bits = 0;
    while ((1ull << bits) <= (uint64_t)P.ncells) ++bits;
    ctx->passes = (bits + kRadixBits - 1) / kRadixBits;
    if (ctx->passes == 0) ctx->passes = 1;
    ctx->ntiles = grid_blocks(P.n, kSortTile);
    ctx->fp32 = p.precision == RRSPH_FP32;
    if (const char* e = std::getenv("RRSPH_HIP_SORT")) ctx->incremental = std::strcmp(e, "full") != 0;
    if (const char* e = std::getenv("RRSPH_HIP_RESORT_CAP")) {
        const long v = std::strtol(e, nullptr, 10);
        if (v >= 0 && v < (long)kResortCap) ctx->resort_cap = (uint32_t)v;
    }
    if (const char* e = std::getenv("RRSPH_HIP_RESORT_STAGE")) {  // test hook: force the binary-search placement
        const long v = std::strtol(e, nullptr, 10);
        if (v >= 0 && v <= (long)kBlock) ctx->resort_stage = (uint32_t)v;
    }
    ctx->fused = !(p.dt_correction_method == 2 && p.dt_dynamic_mode == 1);
    if (const char* e = std::getenv("RRSPH_HIP_PAIR_KERNEL")) {
        if (!std::strcmp(e, "general")) ctx->pair_impl = 0;
        else if (!std::strcmp(e, "tile")) ctx->pair_impl = 2;
        else if (!std::strcmp(e, "walk")) ctx->pair_impl = 3;
        else ctx->pair_impl = 1;
    }
    ctx->fast_pair = p.density_skf == 1 && p.intf_skf == 1 && p.artificial_viscosity_skf == 1 &&
                     p.average_velocity_skf == 1 && p.intf_sph_approximation == 2 && !p.artificial_pressure &&
                     (p.density_treatment == 0 || p.density_treatment == 1) && std::fabs(p.cell_scale_k - 2.0) == 0.0;
    // neighbour-list steps: every 2D configuration and the cubic one in 3D
    // (187,530 particles with Wendland kernels, delta-SPH and artificial
    // pressure, FP64: 81 us a step with lists, 205 us sorted); an entry holds
    // a slot in kSlotBits bits in 2D, kSlotBits3 in 3D.  The skin, a fraction
    // of the cut-off: a wider one makes builds rarer and lists longer, and in
    // 3D the lists grow faster.  Per 50 steps of 1,020,263 particles (FP32): 5250
    // us at 0.125, 5050 at 0.15, 5380 at 0.18; below 25,000 particles, where a
    // pass is bound by latency, 0.23 (a step at 0.15, 0.23 and 0.27, FP64: dam
    // breaks of 2,213 particles 9.0, 8.9 and 9.0 us, of 6,923 10.1, 9.5 and 9.6, of
    // 14,813 12.3, 11.5 and 11.1; flumes of 11,842 18.5, 17.2 and 17.0, of 20,400
    // 20.7, 19.0 and 18.4, of 27,229 20.7, 20.3 and 19.8, of 46,894 23.8, 24.1
    // and 24.7); 3D, per 25 steps of 555,686 (FP64):
    // 11110 at 0.06, 11100 at 0.08, 11520 at 0.1, 11630 at 0.125
    double skin_frac = d3 ? 0.08 : P.n < 25000 ? 0.23 : 0.15;
    if (const char* e = std::getenv("RRSPH_HIP_LIST_SKIN")) skin_frac = std::strtod(e, nullptr);
    ctx->list_mode = (ctx->fast_pair || !d3) && skin_frac > 0.0 && skin_frac < 0.9 && P.n <= (d3 ? kSlotMask3 : kSlotMask);
    if (const char* e = std::getenv("RRSPH_HIP_LIST")) ctx->list_mode = ctx->list_mode && std::strcmp(e, "0") != 0;
    ctx->all_terms = P.av_on && P.xsph_on && P.lj_on;
    // lanes per particle of the 2D list passes (LaneGroup), from event-timed
    // passes with 1, 2 and 8 lanes: 8 below 25,000 particles, where the chip
    // is not filled (continuity, 6,432 particles FP64 14.8 / 11.9 / 10.8 us,
    // 22,662 15.2 / 12.5 / 12.1, 54,200 15.7 / 14.0 / 20.0); 2 above (413,242
    // FP64 44.3 / 44.6 / -, 1,020,263 108.5 / 104.7 / -; summation density
    // 519,203 FP32 36.1 / 32.9 / 57.4; general pair pass 413,242 FP32 52.6 /
    // 42.0 / 76.1), but for the FP32 continuity pass, which has the least to
    // do per entry, at large n (188,656 particles 18.3 / 19.4 / 31.4,
    // 1,020,263 61.4 / 61.6 / 146.7)
    ctx->lanes = P.n < 25000 ? 8 : 2;
    if (P.n >= 150000 && ctx->fast_pair && ctx->fp32 && P.density_treatment != 0) ctx->lanes = 1;
    // fused pairs of list steps: the cubic configuration with a constant dt
    // and no wave maker (in 3D with a summation pass: its continuity pass
    // gathers the neighbours' state)
    ctx->fuse = ctx->fast_pair && ctx->all_terms && P.dt_method != 2 && !P.boundary_motion &&
                (!d3 || P.density_treatment == 0);
    P.dset_mask = ctx->fuse && P.density_treatment != 0 ? 3 : 1;
    // a taped run keeps every build's lists, so that its builds cost more: 12
    // steps and their gradients, 943,906 particles (3D FP32), 30.6 ms at 0.08,
    // 25.3 at 0.1, 23.1 at 0.125, 23.6 at 0.15
    ctx->tape_skin = d3 && !std::getenv("RRSPH_HIP_LIST_SKIN") ? 0.125 : skin_frac;
    set_skin(P, skin_frac);
    const double grow = std::pow(1.0 + std::max(skin_frac, ctx->tape_skin), d3 ? 3 : 2);
    P.list_cap = (uint32_t)std::ceil(p.max_neighbours * grow) + 8;
    // the list pass addresses the lists (list_cap + kListPad rows) with
    // 32-bit byte offsets: fewer rows where n is large (a build that finds
    // more entries for a particle runs its step without lists)
    const uint64_t rows_max = 0xffffffffull / (4ull * P.n);
    if (P.list_cap + kListPad > rows_max) {
        if (rows_max >= (uint64_t)p.max_neighbours + kListPad) P.list_cap = (uint32_t)(rows_max - kListPad);
        else ctx->list_mode = false;
    }
    if (d3 && !ctx->fast_pair)
        return fail(ctx, RRSPH_ERR_NOT_IMPLEMENTED,
                    "RRSPH_HIP: 3D supports cubic kernels for every term, approximation 2, no artificial pressure, "
                    "summation or continuity density");
    return RRSPH_OK;
}

void drop_tape_graph(AdjTape& T) {
    if (T.texec) (void)hipGraphExecDestroy(T.texec);
    if (T.tgraph) (void)hipGraphDestroy(T.tgraph);
    T.texec = nullptr;
    T.tgraph = nullptr;
}

void free_tape(AdjTape& T) {
    drop_tape_graph(T);
    for (void* p : T.ck)
        if (p) (void)hipFree(p);
    T.ck.clear();
    for (auto& L : T.seg_lists) {
        void* lp[] = {L.nbl, L.nbc, L.keys};
        for (void* p : lp)
            if (p) (void)hipFree(p);
    }
    T.seg_lists.clear();
    if (T.nearf) (void)hipFree(T.nearf);
    void* ptrs[] = {T.seg, T.eta, T.zs, T.ws, T.eta_bar, T.partials, T.piston_sum, T.lam[0], T.lam[1], T.direct,
                    T.drho_adj, T.out_adj, T.flag, T.rec, T.uctrl, T.seg_keys, T.seg_perm};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    T = AdjTape{};
}

void free_all(rrsph_ctx* c) {
    drop_graph(c);
    free_tape(c->adj);
    void* ptrs[] = {c->posA, c->posB, c->vaA, c->vaB, c->adA, c->pred, c->der, c->xs, c->pred_scratch, c->pres,
                    c->pres_scratch, c->oidA,
                    c->oidB, c->key_next, c->kbuf[0], c->kbuf[1], c->vbuf[0], c->vbuf[1], c->hist, c->digit_total,
                    c->maxslots, c->LB, c->ctrl, c->ctrl_cur,
                    c->util_ctrl, c->red, c->st_r, c->st_v, c->st_rho, c->st_p, c->st_a, c->st_drho, c->st_av,
                    c->st_mu, c->st_itype, c->st_u32, c->skeyA, c->chg, c->chg_mask, c->wpre, c->pw,
                    c->pw_scratch, c->adB, c->nbl, c->nbc, c->rec, c->dens, c->home, c->dslots, c->dtslots, c->cand, c->rec1, c->ctrl_alt,
                    c->cell_count};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    if (c->host_ctrl) (void)hipHostFree(c->host_ctrl);
    if (c->host_eta) (void)hipHostFree(c->host_eta);
    if (c->stream && c->own_stream) (void)hipStreamDestroy(c->stream);
}

// Cell keys of state A for the next step's sort.
void enqueue_state_keys(rrsph_ctx* ctx) {
    const uint32_t nb = grid_blocks(ctx->P.n, kBlock);
    if (ctx->P.dim == 3)
        state_keys3_kernel<<<nb, kBlock, 0, ctx->stream>>>(ctx->P, (const double4*)ctx->posA, ctx->key_next);
    else if (ctx->fp32)
        state_keys_kernel<float><<<nb, kBlock, 0, ctx->stream>>>(ctx->P, ctx->posA, (const float4*)ctx->vaA,
                                                                 ctx->key_next);
    else
        state_keys_kernel<double><<<nb, kBlock, 0, ctx->stream>>>(ctx->P, ctx->posA, (const double4*)ctx->vaA,
                                                                  ctx->key_next);
}

}  // namespace

// The reverse of one step on its re-sorted state (state precision R, adjoint
// arithmetic FP64): whole_step reverse, then the pair gather.  In 2D over
// lists the step's saved state src is read in place, through perm if the step
// was a build (else null; in 3D only then), and the gradient of the gauges of
// that state comes with the pair gather (eta_bar, zs, ws: their row, or null).  8 lanes a
// particle below 25,000, where the list passes take them (setup_params).
constexpr uint32_t kAdjLanes8 = 25000;
template <class R>
static void enqueue_reverse_step(rrsph_ctx* ctx, const AdjStep& S, Ctrl* uc, const double* lam_in, double* lam_out,
                                 double* psum, const uint32_t* keys, const uint32_t* perm,
                                 const AdjTape::Lists* lists, const StateView* src, const double* eta_bar,
                                 const double* zs, const double* ws) {
    AdjTape& T = ctx->adj;
    const StepParams& P = ctx->P;
    const size_t n = P.n;
    const uint32_t nb = grid_blocks(P.n, kBlock);
    const uint32_t nb_xcd = P.blocks_per_xcd * kNumXcd;  // the pair gathers map blocks to XCDs
    if (P.dim == 2 && lists) {
        AdjRec2* rec = (AdjRec2*)T.out_adj;
        const StateA<R> A{(double2*)src->pos, (real4<R>*)src->va, (real4<R>*)src->ad, src->oid};
        adj_prep_list<R><<<nb, kBlock, 0, ctx->stream>>>(P, S, A, perm, lam_in, rec, psum);
        auto pair = [&](auto kernel, uint32_t blocks) {
            kernel<<<blocks * kNumXcd, kBlock, 0, ctx->stream>>>(P, S, rec, lists->nbl, lists->nbc, lam_in, lam_out,
                                                                 T.flag, T.spec.g, eta_bar, zs, ws);
        };
        if (P.n < kAdjLanes8) pair(adj_pair_list<8>, group_blocks_per_xcd<8>(P.n));
        else pair(adj_pair_list<2>, group_blocks_per_xcd<2>(P.n));
        return;
    }
    const bool in_order = lists && !perm;  // (3D) src is in the slot order of its build
    if (!in_order && keys) {  // the sort step k ran with, saved by the replay: reorder only
        ctx->sorted_keys = keys;
        ctx->sorted_perm = perm;
        enqueue_util_reorder<R>(ctx, src, uc);
    } else if (!in_order) {
        enqueue_util_sort<R>(ctx, uc);
    }
    if (P.dim == 3) {
        StateB3<R> B = stateB3<R>(ctx, ctx->pred_scratch, ctx->pw_scratch, ctx->pres_scratch);
        if (in_order) {
            B.pos = (double4*)src->pos;
            B.va = (real4<R>*)src->va;
            B.oid = src->oid;
        }
        AdjRec3<R>* rec = (AdjRec3<R>*)T.out_adj;
        // FP32 step over lists: near records relative to the home cells of
        // the build (its sorted keys) for the pair adjoint's walk
        float4* nearf = lists && sizeof(R) == 4 ? T.nearf : nullptr;
        auto prep = [&](auto kernel) {
            kernel<<<nb, kBlock, 0, ctx->stream>>>(P, S, B, in_order ? (const real4<R>*)src->ad : nullptr, lam_in, rec,
                                                   T.direct, psum, nearf ? lists->keys : nullptr, nearf);
        };
        if (in_order) prep(adj_prep3<R, true>);
        else prep(adj_prep3<R, false>);
        if (lists)
            adj_pair3<R, true><<<nb_xcd, kBlock, 0, ctx->stream>>>(P, S, B, ctx->sorted_keys, ctx->LB, lists->nbl,
                                                                   lists->nbc, rec, T.direct, lam_out, T.flag,
                                                                   nearf, T.spec, eta_bar, zs, ws);
        else
            adj_pair3<R, false><<<nb_xcd, kBlock, 0, ctx->stream>>>(P, S, B, ctx->sorted_keys, ctx->LB, nullptr,
                                                                    nullptr, rec, T.direct, lam_out, T.flag,
                                                                    nullptr, GaugeSpec3{}, nullptr, nullptr, nullptr);
    } else {
        StateB<R> B = stateB<R>(ctx, ctx->pred_scratch, ctx->pres_scratch);
        adj_prep<R><<<nb, kBlock, 0, ctx->stream>>>(P, S, B, lam_in, T.out_adj, T.drho_adj, T.direct, psum);
        adj_pair<R><<<nb_xcd, kBlock, 0, ctx->stream>>>(P, S, B, ctx->sorted_keys, ctx->LB, T.out_adj, T.drho_adj,
                                                    T.direct, lam_out, T.flag);
    }
}

extern "C" {

rrsph_status rrsph_hip_create(const rrsph_params_c* params, rrsph_ctx** out) {
    if (!params || !out) return RRSPH_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    rrsph_ctx* ctx = new rrsph_ctx();
    if (params->struct_size != sizeof(rrsph_params_c)) {
        ctx->err = "RRSPH_HIP: rrsph_params_c size mismatch";
        *out = ctx;
        return RRSPH_ERR_INVALID_ARGUMENT;
    }
    ctx->prm = *params;
    *out = ctx;
    // parameters are validated on the host before any device is touched
    rrsph_status st = setup_params(ctx, *params);
    if (st != RRSPH_OK) return st;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return fail(ctx, RRSPH_ERR_NO_DEVICE, "RRSPH_HIP: no HIP device");
    HIP_TRY(hipGetDevice(&ctx->device));
    HIP_TRY(hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking));
    ctx->own_stream = true;
    const size_t n = ctx->P.n;
    const size_t r4 = ctx->fp32 ? sizeof(float4) : sizeof(double4);
    hipError_t e = hipSuccess;
    const size_t dim = ctx->P.dim;
    ctx->posA = dalloc<double2>(n * (dim == 3 ? 2 : 1), e);  // 3D: one double4 per particle
    ctx->posB = dalloc<double2>(n * (dim == 3 ? 2 : 1), e);
    ctx->vaA = dalloc<char>(n * r4, e);
    ctx->vaB = dalloc<char>(n * r4, e);
    ctx->adA = dalloc<char>(n * r4, e);
    ctx->pred = dalloc<char>(n * r4, e);
    ctx->der = dalloc<char>(n * r4, e);
    ctx->xs = dalloc<char>(n * r4, e);
    ctx->pred_scratch = dalloc<char>(n * r4, e);
    ctx->pres = dalloc<char>(n * (r4 / 4), e);
    ctx->pres_scratch = dalloc<char>(n * (r4 / 4), e);
    if (dim == 3) {
        ctx->pw = dalloc<char>(n * (r4 / 4), e);
        ctx->pw_scratch = dalloc<char>(n * (r4 / 4), e);
    }
    // the fused pair pass integrates in the same launch; with the consistency
    // check a neighbour overflow undoes the step from B and this copy of A.ad
    if (ctx->fused && ctx->P.consistency_check) ctx->adB = dalloc<char>(n * r4, e);
    ctx->oidA = dalloc<uint32_t>(n, e);
    ctx->oidB = dalloc<uint32_t>(n, e);
    ctx->key_next = dalloc<uint32_t>(n, e);
    ctx->kbuf[0] = dalloc<uint32_t>(n, e);
    ctx->kbuf[1] = dalloc<uint32_t>(n, e);
    ctx->vbuf[0] = dalloc<uint32_t>(n, e);
    ctx->vbuf[1] = dalloc<uint32_t>(n, e);
    ctx->hist = dalloc<uint32_t>((size_t)kRadix * ctx->ntiles, e);
    ctx->digit_total = dalloc<uint32_t>(kRadix, e);
    ctx->maxslots = dalloc<unsigned long long>(4 * kMaxSlots, e);  // second half: utility sorts
    ctx->LB = dalloc<uint32_t>((size_t)ctx->P.ncells + 2, e);
    ctx->ctrl = dalloc<Ctrl>(1, e);
    ctx->ctrl_cur = dalloc<Ctrl>(1, e);
    ctx->util_ctrl = dalloc<Ctrl>(1, e);
    ctx->red = dalloc<double>(kDiagSlots * (size_t)kDiagMaxBlocks + 64, e);
    ctx->skeyA = dalloc<uint32_t>(n, e);
    ctx->chg = dalloc<unsigned long long>(kResortCap, e);
    ctx->chg_mask = dalloc<unsigned long long>(n / kWave + 1, e);
    ctx->wpre = dalloc<uint32_t>(n / kWave + 1, e);
    ctx->P.chg_mask = ctx->chg_mask;
    if (ctx->list_mode) {
        ctx->nbl = dalloc<uint32_t>((size_t)(ctx->P.list_cap + kListPad) * n, e);
        ctx->nbc = dalloc<uint32_t>(n, e);
        ctx->rec = dalloc<ListRec<double>>(n, e);
        if (dim == 3) ctx->dens = dalloc<double4>(n, e);
        if (dim == 3) ctx->cand = dalloc<float4>(n, e);
        ctx->home = dalloc<uint32_t>(n, e);
        ctx->dslots = dalloc<unsigned long long>(4 * kSlotSet, e);
        if (ctx->fuse) {
            ctx->rec1 = dalloc<char>(2 * r4 * n, e);
            ctx->ctrl_alt = dalloc<Ctrl>(1, e);
        }
        ctx->dtslots = dalloc<unsigned long long>(2 * kDtSet, e);
        // the counting sort's scan passes over every cell of the grid (16 bytes a
        // cell: read twice, cleared, the start written), which the radix sort does
        // not; sparser grids keep that one.  Steps that all build, counting and
        // radix, us: 1,020,263 particles 222 and 250 with 2 cells a particle, 235
        // and 256 with 4, 266 and 269 with 8, 326 and 306 with 16; 187,530
        // particles 76 and 112 with 4, 148 and 153 with 64; the line is where
        // the largest still gains
        if (const char* e2 = std::getenv("RRSPH_HIP_TAPE_LISTS")) ctx->tape_lists_max = std::strtoull(e2, nullptr, 10);
        const char* sort = std::getenv("RRSPH_HIP_BUILD_SORT");
        if ((uint64_t)ctx->P.ncells <= 4ull * n && !(sort && std::strcmp(sort, "radix") == 0)) {
            const size_t blocks = scan_blocks(ctx->P.ncells);
            ctx->cell_count = dalloc<uint32_t>(blocks * (kScanCells + 1), e);
        }
    }
    if (e != hipSuccess) return fail(ctx, RRSPH_ERR_HIP, std::string("hipMalloc: ") + hipGetErrorString(e));
    if (ctx->dslots) HIP_TRY(hipMemset(ctx->dslots, 0, 4 * kSlotSet * sizeof(unsigned long long)));
    if (ctx->cell_count)
        HIP_TRY(hipMemset(ctx->cell_count, 0, (size_t)scan_blocks(ctx->P.ncells) * kScanCells * sizeof(uint32_t)));
    if (ctx->nbl) HIP_TRY(hipMemset(ctx->nbl, 0, (size_t)(ctx->P.list_cap + kListPad) * n * sizeof(uint32_t)));
    HIP_TRY(hipHostMalloc((void**)&ctx->host_ctrl, sizeof(Ctrl), hipHostMallocDefault));
    HIP_TRY(hipHostMalloc((void**)&ctx->host_eta, kMaxGauges * sizeof(double), hipHostMallocDefault));
    HIP_TRY(scratch_address(ctx->device, &ctx->scratch));
    std::memset(ctx->host_ctrl, 0, sizeof(Ctrl));
    HIP_TRY(hipMemcpy(ctx->util_ctrl, ctx->host_ctrl, sizeof(Ctrl), hipMemcpyHostToDevice));
    return RRSPH_OK;
}

void rrsph_hip_destroy(rrsph_ctx* ctx) {
    if (!ctx) return;
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    free_all(ctx);
    delete ctx;
}

const char* rrsph_hip_last_error(const rrsph_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

static rrsph_status ensure_staging(rrsph_ctx* ctx) {
    if (ctx->st_r) return RRSPH_OK;
    const size_t n = ctx->P.n;
    hipError_t e = hipSuccess;
    const size_t dim = ctx->P.dim;
    ctx->st_r = dalloc<double>(dim * n, e);
    ctx->st_v = dalloc<double>(dim * n, e);
    ctx->st_rho = dalloc<double>(n, e);
    ctx->st_p = dalloc<double>(n, e);
    ctx->st_a = dalloc<double>(dim * n, e);
    ctx->st_drho = dalloc<double>(n, e);
    ctx->st_av = dalloc<double>(dim * n, e);
    ctx->st_mu = dalloc<double>(n, e);
    ctx->st_itype = dalloc<int32_t>(n, e);
    ctx->st_u32 = dalloc<uint32_t>(n, e);
    if (e != hipSuccess) return fail(ctx, RRSPH_ERR_HIP, std::string("hipMalloc: ") + hipGetErrorString(e));
    return RRSPH_OK;
}

rrsph_status rrsph_hip_upload(rrsph_ctx* ctx, const double* r, const double* v, const double* rho,
                              const int32_t* itype, uint32_t ntotal) {
    if (!ctx || !ctx->stream) return RRSPH_ERR_INVALID_ARGUMENT;
    if (!r || !v || !rho || !itype || ntotal != ctx->P.n)
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "dump corrupted: dump ntotal doesn't match params.ntotal!");
    rrsph_status st = ensure_staging(ctx);
    if (st != RRSPH_OK) return st;
    const size_t n = ctx->P.n;
    const size_t dim = ctx->P.dim;
    HIP_TRY(hipMemcpyAsync(ctx->st_r, r, dim * n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipMemcpyAsync(ctx->st_v, v, dim * n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipMemcpyAsync(ctx->st_rho, rho, n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipMemcpyAsync(ctx->st_itype, itype, n * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream));
    Ctrl c{};
    c.time = ctx->prm.start_time;
    c.dt = ctx->prm.dt;
    c.t_end = INFINITY;
    *ctx->host_ctrl = c;
    HIP_TRY(hipMemcpyAsync(ctx->ctrl, ctx->host_ctrl, sizeof(Ctrl), hipMemcpyHostToDevice, ctx->stream));
    const uint32_t nb = grid_blocks(ctx->P.n, kBlock);
    if (dim == 3) {
        if (ctx->fp32)
            init3_kernel<float><<<nb, kBlock, 0, ctx->stream>>>(ctx->P, ctx->st_r, ctx->st_v, ctx->st_rho,
                                                                ctx->st_itype, stateA3<float>(ctx), ctx->key_next,
                                                                ctx->ctrl);
        else
            init3_kernel<double><<<nb, kBlock, 0, ctx->stream>>>(ctx->P, ctx->st_r, ctx->st_v, ctx->st_rho,
                                                                 ctx->st_itype, stateA3<double>(ctx), ctx->key_next,
                                                                 ctx->ctrl);
    } else if (ctx->fp32) {
        init_kernel<float><<<nb, kBlock, 0, ctx->stream>>>(ctx->P, ctx->st_r, ctx->st_v, ctx->st_rho, ctx->st_itype,
                                                           stateA<float>(ctx), ctx->key_next, ctx->ctrl);
    } else {
        init_kernel<double><<<nb, kBlock, 0, ctx->stream>>>(ctx->P, ctx->st_r, ctx->st_v, ctx->st_rho,
                                                            ctx->st_itype, stateA<double>(ctx), ctx->key_next,
                                                            ctx->ctrl);
    }
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    ctx->uploaded = true;
    ctx->stepped = false;
    ctx->fields_valid = false;
    ctx->pres_in_order = true;
    ctx->need_full = true;
    // step indices restart: forget the overflow history
    ctx->full_until = ctx->launched;
    ctx->last_fallback = ~0ull;
    ctx->full_run = ctx->full_run_end = 0;
    return RRSPH_OK;
}

// Enqueue nsteps steps: the first after an upload (or a re-sort overflow)
// with the full radix sort, the others with the incremental re-sort.
static uint64_t committed_steps(const Ctrl& c);

// Whether the next list step is a build: after an upload, a restore or a
// run without lists, and every list_interval steps.
static bool next_is_build(const rrsph_ctx* ctx, uint64_t step) {
    return ctx->need_full || step - ctx->build_at >= ctx->list_interval;
}

static rrsph_status launch_steps(rrsph_ctx* ctx, uint32_t nsteps) {
    if (list_active(ctx)) {
        // step indices from the committed count of the last synchronisation
        const uint64_t base = committed_steps(*ctx->host_ctrl);
        for (uint32_t k = 0; k < nsteps;) {
            const bool build = next_is_build(ctx, base + k);
            uint32_t run = 1;  // list steps to the next build, in powers of two
            if (!build) {
                const uint64_t left = std::min<uint64_t>(nsteps - k, ctx->build_at + ctx->list_interval - (base + k));
                while (run < kListRunMax && 2 * run <= left) run *= 2;
            }
            const rrsph_status st = launch_list_run(ctx, build, run);
            if (st != RRSPH_OK) return st;
            if (build) {
                ctx->build_at = base + k;
                ++ctx->n_build;
                ++ctx->n_full;
            } else {
                ctx->n_list += run;
            }
            ctx->launched += run;
            ctx->need_full = false;
            k += run;
        }
        HIP_TRY(hipGetLastError());
        if (nsteps) {
            ctx->stepped = true;
            ctx->fields_valid = true;
            ctx->list_fields = true;
        }
        return RRSPH_OK;
    }
    if (ctx->use_graph && !ctx->gexec) {
        rrsph_status st = build_graph(ctx);
        if (st != RRSPH_OK) return st;
    }
    for (uint32_t k = 0; k < nsteps; ++k) {
        const bool full = ctx->need_full || !ctx->incremental || ctx->launched < ctx->full_until;
        if (ctx->use_graph) HIP_TRY(hipGraphLaunch(full ? ctx->gexec_full : ctx->gexec, ctx->stream));
        else enqueue_step(ctx, nullptr, full);
        // where this step's sort lands: the last radix pass's buffers, or the re-sort's
        const uint32_t fb = (ctx->passes - 1) & 1u;
        ctx->last_keys = full ? ctx->kbuf[fb] : ctx->kbuf[0];
        ctx->last_perm = full ? ctx->vbuf[fb] : ctx->vbuf[0];
        ++(full ? ctx->n_full : ctx->n_incremental);
        ++ctx->launched;
        ctx->need_full = false;
    }
    HIP_TRY(hipGetLastError());
    if (nsteps) {
        ctx->stepped = true;
        ctx->fields_valid = true;
        ctx->list_fields = false;
    }
    return RRSPH_OK;
}

static uint64_t committed_steps(const Ctrl& c) { return c.step + (c.pending ? 1 : 0); }

// One list step with the build decided by the caller (the adjoint's tapes
// follow their own schedule); `abs_step` is its step index since the upload.
// A build's sort lands in kbuf / vbuf of the last radix pass.
static rrsph_status launch_list_step(rrsph_ctx* ctx, bool build, uint64_t abs_step) {
    const rrsph_status st = launch_list_run(ctx, build, 1);
    if (st != RRSPH_OK) return st;
    HIP_TRY(hipGetLastError());
    if (build) {
        const uint32_t fb = (ctx->passes - 1) & 1u;
        ctx->last_keys = ctx->kbuf[fb];
        ctx->last_perm = ctx->vbuf[fb];
        ctx->build_at = abs_step;
        ++ctx->n_build;
        ++ctx->n_full;
    } else {
        ++ctx->n_list;
    }
    ++ctx->launched;
    ctx->need_full = false;
    ctx->stepped = true;
    ctx->fields_valid = true;
    ctx->list_fields = true;
    return RRSPH_OK;
}

// A step overflowed the incremental re-sort at step index `at`.  Overflows
// in close succession mean many particles change cell every step: keep to
// the full sort for a while instead of paying a host round trip (and the
// no-op tail of the launched batch) per step, then try again.  A lone
// overflow, e.g. the first step after an upload, costs one round trip.
// Distances are in committed steps, not launches: a halted batch still
// counts its no-op launches.
static void note_resort_overflow(rrsph_ctx* ctx, uint64_t at) {
    ++ctx->n_fallback;
    if (ctx->last_fallback != ~0ull && at - ctx->last_fallback <= kFallbackWindow) {
        const bool again = ctx->full_run && at - ctx->full_run_end <= kFallbackWindow;
        ctx->full_run = again ? std::min(2 * ctx->full_run, kFullSortRunMax) : kFullSortRun;
        ctx->full_until = ctx->launched + ctx->full_run;
        ctx->full_run_end = at + ctx->full_run;
    }
    ctx->last_fallback = at;
    ctx->need_full = true;  // the overflowing step itself runs with the full sort
}

// A list step found its lists possibly stale at step index `at` (the
// displacements since the build reached half the skin): build every
// 0.8 x that many steps from now on, until the measured rate says more.
static void note_list_stale(rrsph_ctx* ctx, uint64_t at) {
    ++ctx->n_list_halts;
    const uint64_t age = at > ctx->build_at ? at - ctx->build_at : 1;
    ctx->list_interval = std::max<uint64_t>(1, age * 4 / 5);
    ctx->need_full = true;  // the halted step runs as a build
}

// After a clean batch: the interval between builds from the displacement
// per step (80% of the steps that use up half the skin), the larger of the
// mean since the last build and the last step's.
static void adapt_list_interval(rrsph_ctx* ctx) {
    const Ctrl& c = *ctx->host_ctrl;
    const uint64_t now = committed_steps(c);
    // disp_acc covers the steps after the build up to the one before the last
    const uint64_t counted = now > ctx->build_at + 1 ? now - ctx->build_at - 1 : 0;
    double rate = c.disp_last;
    if (counted > 0) rate = std::max(rate, c.disp_acc / (double)counted);
    const double k = rate > 0.0 ? 0.8 * ctx->P.skin_half / rate : 1e9;
    ctx->list_interval = (uint64_t)std::min(2048.0, std::max(1.0, std::floor(k)));
}

// After a synchronised launch: a step that halted for a reason the host
// handles (more changed cells than the incremental re-sort takes; lists
// possibly stale; a list out of room) did so before touching the state;
// clear the halt and set up the re-run of that step.
static rrsph_status resume_halt(rrsph_ctx* ctx, bool* resumed) {
    Ctrl& c = *ctx->host_ctrl;
    *resumed = false;
    if (!c.halted || !rerun_status(c.status)) return RRSPH_OK;
    const uint64_t at = committed_steps(c);  // the step that halted
    if (c.status == kStatusResort) {
        note_resort_overflow(ctx, at);
    } else if (c.status == kStatusRebuild) {
        note_list_stale(ctx, at);
    } else if (c.status == kStatusUnfused) {
        ctx->fuse = false;
        drop_list_graphs(ctx);  // (the stream is idle)
        ctx->need_full = true;
    } else {                     // kStatusListOverflow
        ctx->list_mode = false;  // more candidates than a list holds: sort every step from here
        ctx->need_full = true;
    }
    c.halted = 0;
    c.status = 0;
    c.list_overflow = 0;
    HIP_TRY(hipMemcpyAsync(ctx->ctrl, ctx->host_ctrl, sizeof(Ctrl), hipMemcpyHostToDevice, ctx->stream));
    *resumed = true;
    return RRSPH_OK;
}

// Run nsteps steps to completion (or to a halt) and report the status.
// List steps go in batches: kFirstChunk steps in a fresh context, about twice the
// build interval and at least 32 in a steady flow (a look at the control
// block idles the stream for 25 us), few after a halt, when the interval is
// still falling and the launches behind the next halt do nothing.
static rrsph_status run_steps(rrsph_ctx* ctx, uint32_t nsteps) {
    const uint64_t target = committed_steps(*ctx->host_ctrl) + nsteps;
    while (true) {
        const uint64_t now = committed_steps(*ctx->host_ctrl);
        if (now >= target) return RRSPH_OK;
        uint64_t chunk = target - now;
        if (list_active(ctx)) chunk = std::min(chunk, ctx->list_chunk);
        rrsph_status st = launch_steps(ctx, (uint32_t)chunk);
        if (st != RRSPH_OK) return st;
        st = sync_status(ctx);
        if (st != RRSPH_OK) return st;
        bool resumed = false;
        st = resume_halt(ctx, &resumed);
        if (st != RRSPH_OK) return st;
        if (!resumed && ctx->host_ctrl->halted) return RRSPH_OK;  // stopped at t_end
        if (!list_active(ctx)) continue;
        if (!resumed) adapt_list_interval(ctx);
        const uint64_t two = 2 * ctx->list_interval;
        ctx->list_chunk = resumed ? std::max<uint64_t>(4, std::min(kFirstChunk, two))
                                  : std::min<uint64_t>(2 * ctx->list_chunk, std::min<uint64_t>(256, std::max<uint64_t>(32, two)));
    }
}

rrsph_status rrsph_hip_step(rrsph_ctx* ctx, uint32_t nsteps) {
    if (!ctx || !ctx->uploaded) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: no state uploaded");
    return run_steps(ctx, nsteps);
}

rrsph_status rrsph_hip_run_until(rrsph_ctx* ctx, double t_end, uint64_t max_steps, uint64_t* steps_taken) {
    if (!ctx || !ctx->uploaded) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: no state uploaded");
    // set t_end on the device (the prologue halts with status 0 past it)
    HIP_TRY(hipMemcpyAsync(ctx->host_ctrl, ctx->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    const uint64_t step0 = ctx->host_ctrl->step + (ctx->host_ctrl->pending ? 1 : 0);
    if (ctx->host_ctrl->halted && ctx->host_ctrl->status == 0) ctx->host_ctrl->halted = 0;
    ctx->host_ctrl->t_end = t_end;
    HIP_TRY(hipMemcpyAsync(ctx->ctrl, ctx->host_ctrl, sizeof(Ctrl), hipMemcpyHostToDevice, ctx->stream));
    uint64_t done = 0;
    rrsph_status st = RRSPH_OK;
    while (done < max_steps) {
        const uint32_t chunk = (uint32_t)std::min<uint64_t>(max_steps - done, 256);
        st = run_steps(ctx, chunk);
        done += chunk;
        if (st != RRSPH_OK || ctx->host_ctrl->halted) break;
    }
    const uint64_t step1 = ctx->host_ctrl->step + (ctx->host_ctrl->pending ? 1 : 0);
    if (steps_taken) *steps_taken = step1 - step0;
    if (list_active(ctx)) ctx->need_full = true;  // a list build launched after the stop did not run
    // clear the stop so later calls run
    ctx->host_ctrl->t_end = INFINITY;
    if (ctx->host_ctrl->halted && ctx->host_ctrl->status == 0) ctx->host_ctrl->halted = 0;
    HIP_TRY(hipMemcpyAsync(ctx->ctrl, ctx->host_ctrl, sizeof(Ctrl), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return st;
}

rrsph_status rrsph_hip_get_time(rrsph_ctx* ctx, double* time, double* dt, uint64_t* step) {
    if (!ctx) return RRSPH_ERR_INVALID_ARGUMENT;
    HIP_TRY(hipMemcpyAsync(ctx->host_ctrl, ctx->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    const Ctrl& c = *ctx->host_ctrl;
    if (time) *time = c.pending ? c.time + c.dt_new : c.time;
    if (dt) *dt = c.pending ? c.dt_new : c.dt;
    if (step) *step = c.step + (c.pending ? 1 : 0);
    return RRSPH_OK;
}

// The current state in original particle order into the device staging
// arrays st_r, st_v, st_rho, st_p, st_itype (what rrsph_hip_download copies).
static rrsph_status enqueue_unpack(rrsph_ctx* ctx) {
    const size_t dim = ctx->P.dim;
    const uint32_t nb = grid_blocks(ctx->P.n, kBlock);
    const void* pres = ctx->stepped && ctx->pres_in_order ? ctx->pres : nullptr;  // null: the equation of state's of rho
    if (dim == 3) {
        if (ctx->fp32)
            download3_kernel<float><<<nb, kBlock, 0, ctx->stream>>>(
                ctx->P, stateA3<float>(ctx), (const float*)pres, ctx->st_r, ctx->st_v,
                ctx->st_rho, ctx->st_p, ctx->st_itype);
        else
            download3_kernel<double><<<nb, kBlock, 0, ctx->stream>>>(
                ctx->P, stateA3<double>(ctx), (const double*)pres, ctx->st_r,
                ctx->st_v, ctx->st_rho, ctx->st_p, ctx->st_itype);
    } else if (ctx->fp32) {
        download_kernel<float><<<nb, kBlock, 0, ctx->stream>>>(
            ctx->P, stateA<float>(ctx), (const float*)pres, ctx->st_r, ctx->st_v,
            ctx->st_rho, ctx->st_p, ctx->st_itype);
    } else {
        download_kernel<double><<<nb, kBlock, 0, ctx->stream>>>(
            ctx->P, stateA<double>(ctx), (const double*)pres, ctx->st_r, ctx->st_v,
            ctx->st_rho, ctx->st_p, ctx->st_itype);
    }
    HIP_TRY(hipGetLastError());
    return RRSPH_OK;
}

rrsph_status rrsph_hip_download(rrsph_ctx* ctx, uint32_t fields, double* r, double* v, double* rho, double* p,
                                int32_t* itype) {
    if (!ctx || !ctx->uploaded) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: no state uploaded");
    const size_t n = ctx->P.n, dim = ctx->P.dim;
    if (const rrsph_status st = enqueue_unpack(ctx); st != RRSPH_OK) return st;
    if ((fields & RRSPH_FIELD_R) && r)
        HIP_TRY(hipMemcpyAsync(r, ctx->st_r, dim * n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if ((fields & RRSPH_FIELD_V) && v)
        HIP_TRY(hipMemcpyAsync(v, ctx->st_v, dim * n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if ((fields & RRSPH_FIELD_RHO) && rho)
        HIP_TRY(hipMemcpyAsync(rho, ctx->st_rho, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if ((fields & RRSPH_FIELD_P) && p)
        HIP_TRY(hipMemcpyAsync(p, ctx->st_p, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if ((fields & RRSPH_FIELD_ITYPE) && itype)
        HIP_TRY(hipMemcpyAsync(itype, ctx->st_itype, n * sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return RRSPH_OK;
}

rrsph_status rrsph_hip_set_export_fields(rrsph_ctx* ctx, int32_t enable) {
    if (!ctx) return RRSPH_ERR_INVALID_ARGUMENT;
    if ((bool)enable != ctx->export_fields) {
        ctx->export_fields = enable != 0;
        drop_graph(ctx);
    }
    return RRSPH_OK;
}

rrsph_status rrsph_hip_fields(rrsph_ctx* ctx, double* a, double* drho, double* av, double* arvmu) {
    if (!ctx || !ctx->stepped) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: no step taken yet");
    if (!ctx->fields_valid)
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: no fields of the current state (it was restored, or the last step failed)");
    if (ctx->fused && !ctx->export_fields)
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: enable rrsph_hip_set_export_fields before stepping");
    const size_t n = ctx->P.n, dim = ctx->P.dim;
    const uint32_t nb = grid_blocks(ctx->P.n, kBlock);
    const void* der = ctx->list_fields ? ctx->adA : ctx->der;
    if (dim == 3 && ctx->fp32)
        fields3_kernel<float><<<nb, kBlock, 0, ctx->stream>>>(ctx->P.n, ctx->oidA, (const float4*)der,
                                                              (const float4*)ctx->xs, ctx->st_a, ctx->st_drho,
                                                              ctx->st_av, ctx->st_mu);
    else if (dim == 3)
        fields3_kernel<double><<<nb, kBlock, 0, ctx->stream>>>(ctx->P.n, ctx->oidA, (const double4*)der,
                                                               (const double4*)ctx->xs, ctx->st_a, ctx->st_drho,
                                                               ctx->st_av, ctx->st_mu);
    else if (ctx->fp32)
        fields_kernel<float><<<nb, kBlock, 0, ctx->stream>>>(ctx->P.n, ctx->oidA, (const float4*)der,
                                                             (const float4*)ctx->xs, ctx->st_a, ctx->st_drho,
                                                             ctx->st_av, ctx->st_mu);
    else
        fields_kernel<double><<<nb, kBlock, 0, ctx->stream>>>(ctx->P.n, ctx->oidA, (const double4*)der,
                                                              (const double4*)ctx->xs, ctx->st_a, ctx->st_drho,
                                                              ctx->st_av, ctx->st_mu);
    HIP_TRY(hipGetLastError());
    if (a) HIP_TRY(hipMemcpyAsync(a, ctx->st_a, dim * n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if (drho) HIP_TRY(hipMemcpyAsync(drho, ctx->st_drho, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if (av) HIP_TRY(hipMemcpyAsync(av, ctx->st_av, dim * n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if (arvmu) HIP_TRY(hipMemcpyAsync(arvmu, ctx->st_mu, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return RRSPH_OK;
}

rrsph_status rrsph_hip_cell_keys(rrsph_ctx* ctx, uint32_t* keys) {
    if (!ctx || !ctx->uploaded || !keys) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad arguments");
    const uint32_t nb = grid_blocks(ctx->P.n, kBlock);
    if (ctx->P.dim == 3)
        morton3_kernel<<<nb, kBlock, 0, ctx->stream>>>(ctx->P, (const double4*)ctx->posA, ctx->oidA, ctx->st_u32);
    else
        morton_kernel<<<nb, kBlock, 0, ctx->stream>>>(ctx->P, ctx->posA, ctx->oidA, ctx->st_u32);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(keys, ctx->st_u32, ctx->P.n * sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return RRSPH_OK;
}

rrsph_status rrsph_hip_neighbours(rrsph_ctx* ctx, uint32_t* out, uint32_t max_nbr) {
    if (!ctx || !ctx->uploaded || !out || max_nbr < 2)
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad arguments");
    const size_t n = ctx->P.n;
    uint32_t* dout = nullptr;
    HIP_TRY(hipMalloc((void**)&dout, n * (size_t)max_nbr * sizeof(uint32_t)));
    Ctrl zero{};
    HIP_TRY(hipMemcpyAsync(ctx->util_ctrl, &zero, sizeof(Ctrl), hipMemcpyHostToDevice, ctx->stream));
    const uint32_t nb = grid_blocks(ctx->P.n, kBlock);
    if (ctx->P.dim == 3 && ctx->fp32) {
        enqueue_util_sort<float>(ctx);
        neighbours3_kernel<float><<<nb, kBlock, 0, ctx->stream>>>(
            ctx->P, stateB3<float>(ctx, ctx->pred_scratch, ctx->pw_scratch, ctx->pres_scratch), ctx->sorted_keys,
            ctx->LB, dout, max_nbr, ctx->util_ctrl);
    } else if (ctx->P.dim == 3) {
        enqueue_util_sort<double>(ctx);
        neighbours3_kernel<double><<<nb, kBlock, 0, ctx->stream>>>(
            ctx->P, stateB3<double>(ctx, ctx->pred_scratch, ctx->pw_scratch, ctx->pres_scratch), ctx->sorted_keys,
            ctx->LB, dout, max_nbr, ctx->util_ctrl);
    } else if (ctx->fp32) {
        enqueue_util_sort<float>(ctx);
        neighbours_kernel<float><<<nb, kBlock, 0, ctx->stream>>>(ctx->P, stateB<float>(ctx, ctx->pred_scratch, ctx->pres_scratch),
                                                                 ctx->sorted_keys, ctx->LB, dout, max_nbr,
                                                                 ctx->util_ctrl);
    } else {
        enqueue_util_sort<double>(ctx);
        neighbours_kernel<double><<<nb, kBlock, 0, ctx->stream>>>(ctx->P, stateB<double>(ctx, ctx->pred_scratch, ctx->pres_scratch),
                                                                  ctx->sorted_keys, ctx->LB, dout, max_nbr,
                                                                  ctx->util_ctrl);
    }
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(out, dout, n * (size_t)max_nbr * sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipMemcpyAsync(ctx->host_ctrl, ctx->util_ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    HIP_TRY(hipFree(dout));
    const uint32_t overflow = ctx->host_ctrl->nbr_overflow;
    // restore the main control block mirror
    HIP_TRY(hipMemcpy(ctx->host_ctrl, ctx->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost));
    if (overflow && ctx->P.consistency_check)
        return fail(ctx, RRSPH_ERR_TOO_MANY_NEIGHBOURS, status_message(RRSPH_ERR_TOO_MANY_NEIGHBOURS));
    return RRSPH_OK;
}

rrsph_status rrsph_hip_diagnostics(rrsph_ctx* ctx, rrsph_diagnostics* out) {
    if (!ctx || !ctx->uploaded || !out) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad arguments");
    const uint32_t nblk = std::min<uint32_t>(kDiagMaxBlocks, grid_blocks(ctx->P.n, kBlock));
    if (ctx->P.dim == 3 && ctx->fp32)
        diag_partials3<float><<<nblk, kBlock, 0, ctx->stream>>>(ctx->P, stateA3<float>(ctx), ctx->red);
    else if (ctx->P.dim == 3)
        diag_partials3<double><<<nblk, kBlock, 0, ctx->stream>>>(ctx->P, stateA3<double>(ctx), ctx->red);
    else if (ctx->fp32)
        diag_partials<float><<<nblk, kBlock, 0, ctx->stream>>>(ctx->P, stateA<float>(ctx), ctx->red);
    else
        diag_partials<double><<<nblk, kBlock, 0, ctx->stream>>>(ctx->P, stateA<double>(ctx), ctx->red);
    diag_final<<<1, kBlock, 0, ctx->stream>>>(ctx->red, nblk);
    HIP_TRY(hipGetLastError());
    double h[kDiagSlots];
    HIP_TRY(hipMemcpyAsync(h, ctx->red + (size_t)kDiagSlots * kDiagMaxBlocks, sizeof(h), hipMemcpyDeviceToHost,
                           ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    double t, dt;
    uint64_t step;
    rrsph_status st = rrsph_hip_get_time(ctx, &t, &dt, &step);
    if (st != RRSPH_OK) return st;
    out->time = t;
    out->dt = dt;
    out->step = step;
    out->n_fluid_alive = (uint32_t)h[0];
    out->n_outside = (uint32_t)h[1];
    out->mass_fluid = h[0] * ctx->P.mass;
    out->kinetic_energy = h[2];
    out->potential_energy = h[3];
    out->internal_energy = h[4];
    out->max_speed = h[5];
    out->rho_min = -h[6];
    out->rho_max = h[7];
    return RRSPH_OK;
}

rrsph_status rrsph_hip_gauges(rrsph_ctx* ctx, const double* x_gauges, uint32_t ngauges, double search_n,
                              int32_t ptype, double* out) {
    if (!ctx || !ctx->uploaded || (!x_gauges && ngauges) || (!out && ngauges))
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad arguments");
    if (ngauges == 0) return RRSPH_OK;
    if (ngauges > 4096) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: at most 4096 gauges");
    if (ctx->P.dim == 3) return fail(ctx, RRSPH_ERR_NOT_IMPLEMENTED, "RRSPH_HIP: gauges are 2D (x-y layers)");
    double* dx = ctx->red;  // ngauges inputs followed by ngauges results
    HIP_TRY(hipMemcpyAsync(dx, x_gauges, ngauges * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipMemsetAsync(dx + ngauges, 0, ngauges * sizeof(double), ctx->stream));
    const double radius = search_n * ctx->P.h;
    const uint32_t nblk = std::min<uint32_t>(1024, grid_blocks(ctx->P.n, kBlock));
    dim3 grid(nblk, ngauges);
    if (ctx->fp32)
        gauge_kernel<float><<<grid, kBlock, 0, ctx->stream>>>(ctx->P.n, stateA<float>(ctx), dx, radius, ptype,
                                                              (unsigned long long*)(dx + ngauges));
    else
        gauge_kernel<double><<<grid, kBlock, 0, ctx->stream>>>(ctx->P.n, stateA<double>(ctx), dx, radius, ptype,
                                                               (unsigned long long*)(dx + ngauges));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(out, dx + ngauges, ngauges * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return RRSPH_OK;
}

rrsph_status rrsph_hip_probe(rrsph_ctx* ctx, const double* points, uint32_t npoints, uint32_t field,
                             double* out) {
    if (!ctx || !ctx->uploaded || (npoints && (!points || !out)))
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad arguments");
    const StepParams& P = ctx->P;
    const uint32_t dim = (uint32_t)P.dim;
    // fatp.cpp:92-119 (check_input): a field the layer holds, a point in the geometry box
    if (field > RRSPH_PROBE_RHO || (field == RRSPH_PROBE_VZ && dim != 3))
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "wrong target value");
    if (npoints == 0) return RRSPH_OK;
    if (npoints > RRSPH_MAX_PROBES) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: too many probe points");
    const double lo[3] = {P.xmin, P.ymin, P.zmin}, hi[3] = {P.xmax, P.ymax, P.zmax};
    for (uint32_t g = 0; g < npoints; ++g)
        for (uint32_t d = 0; d < dim; ++d) {
            const double x = points[(size_t)g * dim + d];
            if (!(lo[d] <= x && lo[d] + (hi[d] - lo[d]) >= x))
                return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "point is outside bounds");
        }
    // the field as a dump layer holds it
    if (const rrsph_status st = enqueue_unpack(ctx); st != RRSPH_OK) return st;
    const double* fld = field == RRSPH_PROBE_P ? ctx->st_p : field == RRSPH_PROBE_RHO ? ctx->st_rho : ctx->st_v;
    const uint32_t stride = field <= RRSPH_PROBE_VZ ? dim : 1u, comp = field <= RRSPH_PROBE_VZ ? field : 0u;
    // summation density of the current positions on the sorted copy (never halted)
    Ctrl zero{};
    HIP_TRY(hipMemcpyAsync(ctx->util_ctrl, &zero, sizeof(Ctrl), hipMemcpyHostToDevice, ctx->stream));
    double* dpts = ctx->red;  // dim * npoints points, then npoints results
    double* dout = dpts + (size_t)dim * npoints;
    HIP_TRY(hipMemcpyAsync(dpts, points, (size_t)dim * npoints * sizeof(double), hipMemcpyHostToDevice,
                           ctx->stream));
    const uint32_t nb_xcd = P.blocks_per_xcd * kNumXcd, pb = grid_blocks(npoints, kWave);
    auto run = [&](auto tag) {
        using R = decltype(tag);
        enqueue_util_sort<R>(ctx);
        if (dim == 3) {
            StateB3<R> B = stateB3<R>(ctx, ctx->pred_scratch, ctx->pw_scratch, ctx->pres_scratch);
            density_sum3_kernel<R><<<nb_xcd, kBlock, 0, ctx->stream>>>(P, ctx->util_ctrl, B, ctx->sorted_keys,
                                                                       ctx->LB);
            probe3_kernel<R><<<pb, kWave, 0, ctx->stream>>>(P, B, ctx->LB, dpts, npoints, fld, stride, comp, dout);
        } else {
            StateB<R> B = stateB<R>(ctx, ctx->pred_scratch, ctx->pres_scratch);
            density_sum_kernel<R><<<nb_xcd, kBlock, 0, ctx->stream>>>(P, ctx->util_ctrl, B, ctx->sorted_keys,
                                                                      ctx->LB);
            probe_kernel<R><<<pb, kWave, 0, ctx->stream>>>(P, B, ctx->LB, dpts, npoints, fld, stride, comp, dout);
        }
    };
    if (ctx->fp32) run(float{});
    else run(double{});
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(out, dout, npoints * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    Ctrl u{};
    HIP_TRY(hipMemcpyAsync(&u, ctx->util_ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    // the layer's find_neighbours (fatp.cpp:136-137) throws on overflow with the check on
    if (u.nbr_overflow && P.consistency_check)
        return fail(ctx, RRSPH_ERR_TOO_MANY_NEIGHBOURS, status_message(RRSPH_ERR_TOO_MANY_NEIGHBOURS));
    return RRSPH_OK;
}

void* rrsph_hip_stream(rrsph_ctx* ctx) { return ctx ? (void*)ctx->stream : nullptr; }

rrsph_status rrsph_hip_set_graph(rrsph_ctx* ctx, int32_t enable) {
    if (!ctx) return RRSPH_ERR_INVALID_ARGUMENT;
    ctx->use_graph = enable != 0;
    if (!ctx->use_graph) drop_graph(ctx);
    return RRSPH_OK;
}

uint32_t rrsph_hip_kernel_class_count(void) { return K_NUM_CLASSES; }
const char* rrsph_hip_kernel_class_name(uint32_t k) { return k < K_NUM_CLASSES ? kClassNames[k] : ""; }

rrsph_status rrsph_hip_profile_steps(rrsph_ctx* ctx, uint32_t nsteps, double* avg_ms, uint32_t n_classes,
                                     double* total_ms) {
    if (!ctx || !ctx->uploaded) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: no state uploaded");
    Profiler prof;
    hipEvent_t t0, t1;
    HIP_TRY(hipEventCreate(&t0));
    HIP_TRY(hipEventCreate(&t1));
    HIP_TRY(hipEventRecord(t0, ctx->stream));
    const uint64_t first = committed_steps(*ctx->host_ctrl);
    bool second = false;  // the second of a fused pair
    for (uint32_t k = 0; k < nsteps; ++k) {
        if (list_active(ctx)) {
            const bool build = next_is_build(ctx, first + k);
            // as launch_steps: two list steps in a row are fused where the context fuses
            const bool pair = !build && !second && ctx->fuse && k + 1 < nsteps &&
                              !next_is_build(ctx, first + k + 1);
            enqueue_list_step(ctx, &prof, build ? kBuildStep : second ? kFusedSecond : pair ? kFusedFirst : kPlainStep);
            second = pair;
            if (build) {
                ctx->build_at = first + k;
                ++ctx->n_build;
                ++ctx->n_full;
            } else {
                ++ctx->n_list;
            }
        } else {
            const bool full = ctx->need_full || !ctx->incremental || ctx->launched < ctx->full_until;
            enqueue_step(ctx, &prof, full);
            ++(full ? ctx->n_full : ctx->n_incremental);
        }
        ++ctx->launched;
        ctx->need_full = false;
    }
    HIP_TRY(hipEventRecord(t1, ctx->stream));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    if (nsteps) {
        ctx->stepped = true;
        ctx->fields_valid = true;
        ctx->list_fields = list_active(ctx);
    }
    std::vector<double> sum(K_NUM_CLASSES, 0.0);
    std::vector<uint32_t> cnt(K_NUM_CLASSES, 0);
    for (auto& r : prof.rec) {
        float ms = 0;
        (void)hipEventElapsedTime(&ms, r.second.first, r.second.second);
        sum[r.first] += ms;
        cnt[r.first] += 1;
        (void)hipEventDestroy(r.second.first);
        (void)hipEventDestroy(r.second.second);
    }
    for (uint32_t k = 0; k < n_classes && k < K_NUM_CLASSES; ++k) avg_ms[k] = cnt[k] ? sum[k] / cnt[k] : 0.0;
    float tot = 0;
    (void)hipEventElapsedTime(&tot, t0, t1);
    if (total_ms) *total_ms = tot;
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    rrsph_status st = sync_status(ctx);
    if (st != RRSPH_OK) return st;
    bool resumed = false;
    st = resume_halt(ctx, &resumed);
    if (st != RRSPH_OK || !resumed) return st;
    // finish the steps after a halted one, unprofiled
    return run_steps(ctx, (uint32_t)(first + nsteps - committed_steps(*ctx->host_ctrl)));
}

rrsph_status rrsph_hip_time_steps(rrsph_ctx* ctx, uint32_t nsteps, double* total_ms) {
    if (!ctx || !ctx->uploaded) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: no state uploaded");
    if (ctx->use_graph && !ctx->gexec) {
        rrsph_status st = build_graph(ctx);
        if (st != RRSPH_OK) return st;
    }
    hipEvent_t t0, t1;
    HIP_TRY(hipEventCreate(&t0));
    HIP_TRY(hipEventCreate(&t1));
    HIP_TRY(hipEventRecord(t0, ctx->stream));
    rrsph_status st = run_steps(ctx, nsteps);
    HIP_TRY(hipEventRecord(t1, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    float ms = 0;
    (void)hipEventElapsedTime(&ms, t0, t1);
    if (total_ms) *total_ms = ms;
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    return st;
}

rrsph_status rrsph_hip_sort_stats(rrsph_ctx* ctx, uint64_t* incremental_steps, uint64_t* full_steps,
                                  uint64_t* fallbacks, uint32_t* last_changed) {
    if (!ctx) return RRSPH_ERR_INVALID_ARGUMENT;
    if (incremental_steps) *incremental_steps = ctx->n_incremental;
    if (full_steps) *full_steps = ctx->n_full;
    if (fallbacks) *fallbacks = ctx->n_fallback;
    if (last_changed) *last_changed = ctx->host_ctrl ? ctx->host_ctrl->resort_count : 0;
    return RRSPH_OK;
}

rrsph_status rrsph_hip_list_stats(rrsph_ctx* ctx, uint64_t* list_steps, uint64_t* builds, uint64_t* stale_halts,
                                  uint32_t* interval) {
    if (!ctx) return RRSPH_ERR_INVALID_ARGUMENT;
    if (list_steps) *list_steps = ctx->n_list;
    if (builds) *builds = ctx->n_build;
    if (stale_halts) *stale_halts = ctx->n_list_halts;
    if (interval) *interval = ctx->list_mode ? (uint32_t)ctx->list_interval : 0u;
    return RRSPH_OK;
}

// ---------------------------------------------------------------- differentiation
static rrsph_status to_gauge_spec(rrsph_ctx* ctx, const rrsph_gauge_spec* in, GaugeSpec3& G) {
    if (!in || in->n > kMaxGauges || !(in->radius > 0) || !(in->tau > 0))
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad gauge spec");
    G = GaugeSpec3{};
    G.g.n = in->n;
    G.g.ptype = in->ptype;
    G.g.radius = in->radius;
    G.g.tau = in->tau;
    G.g.y_ref = in->y_ref;
    for (uint32_t g = 0; g < in->n; ++g) {
        G.g.x[g] = in->x[g];
        G.z[g] = in->z[g];
    }
    return RRSPH_OK;
}

// smooth gauges of state A into eta/zs/ws (device, kMaxGauges entries each)
// (with ctrl: into row ctrl->step - base of tapes of nsteps rows), or with
// `saved` of `rows` states saved `stride` bytes apart, into consecutive rows
static rrsph_status enqueue_smooth_gauges(rrsph_ctx* ctx, const GaugeSpec3& G, double* partials, double* eta,
                                          double* zs, double* ws, const Ctrl* ctrl = nullptr, uint64_t base = 0,
                                          uint32_t nsteps = 0, const StateView* saved = nullptr, uint32_t rows = 1,
                                          size_t stride = 0) {
    const uint32_t nb = gauge_blocks(ctx->P.n);  // partials holds 2 kMaxGauges nb doubles a row
    const void* pos = saved ? saved->pos : (const void*)ctx->posA;
    const void* va = saved ? saved->va : ctx->vaA;
    const dim3 grid(nb, rows);
    if (ctx->P.dim == 3)
        smooth_gauge_partials3<<<grid, kBlock, 0, ctx->stream>>>(ctx->P.n, (const double4*)pos, G, partials, stride);
    else if (ctx->fp32)
        smooth_gauge_partials<float><<<grid, kBlock, 0, ctx->stream>>>(ctx->P.n, (const double2*)pos,
                                                                       (const float4*)va, G.g, partials, stride);
    else
        smooth_gauge_partials<double><<<grid, kBlock, 0, ctx->stream>>>(ctx->P.n, (const double2*)pos,
                                                                        (const double4*)va, G.g, partials, stride);
    smooth_gauge_final<<<dim3(std::max(G.g.n, 1u), rows), kBlock, 0, ctx->stream>>>(nb, G.g, partials, eta, zs, ws,
                                                                                     ctrl, base, nsteps);
    HIP_TRY(hipGetLastError());
    return RRSPH_OK;
}

static rrsph_status adjoint_supported(rrsph_ctx* ctx) {
    const StepParams& P = ctx->P;
    if (!ctx->fast_pair || P.density_treatment != 1)
        return fail(ctx, RRSPH_ERR_NOT_IMPLEMENTED,
                    "RRSPH_HIP: the adjoint needs continuity density, cubic kernels, approximation 2 and no "
                    "artificial pressure");
    if (P.dt_method == 2 && P.dt_dynamic_mode == 1)
        return fail(ctx, RRSPH_ERR_NOT_IMPLEMENTED, "RRSPH_HIP: the adjoint needs dt independent of the state");
    if (P.nwm == 4 || P.nwm == 5)
        return fail(ctx, RRSPH_ERR_NOT_IMPLEMENTED, "RRSPH_HIP: the adjoint supports the piston wave makers only");
    return RRSPH_OK;
}

// bytes per particle of the FP64 position array (2D double2, 3D double4)
// and of one real4 state array (va, ad: FP32 or FP64)
static size_t pos_bytes(const rrsph_ctx* ctx) { return ctx->P.dim == 3 ? 32 : 16; }
static size_t real4_bytes(const rrsph_ctx* ctx) { return ctx->fp32 ? 16 : 32; }
// bytes of one saved state: pos | va | ad | oid | pressure | control block
// (the pressure of the step that produced the state, in its slot order: the
// reference's p array, which download() returns)
// Each array on a 32-byte boundary: steps read and write saved states in place.
constexpr int kStateArrays = 6;
struct StateLayout {
    size_t off[kStateArrays + 1], bytes[kStateArrays];
    explicit StateLayout(const rrsph_ctx* ctx) {
        const size_t n = ctx->P.n, pb = pos_bytes(ctx), vb = real4_bytes(ctx);
        const size_t b[kStateArrays] = {pb * n, vb * n, vb * n, 4 * n, vb / 4 * n, sizeof(Ctrl)};
        off[0] = 0;
        for (int k = 0; k < kStateArrays; ++k) {
            bytes[k] = b[k];
            off[k + 1] = (off[k] + b[k] + 31) / 32 * 32;
        }
    }
};
static size_t state_ctrl_offset(const rrsph_ctx* ctx) { return StateLayout(ctx).off[kStateArrays - 1]; }
static size_t state_bytes(const rrsph_ctx* ctx) { return StateLayout(ctx).off[kStateArrays]; }

// the blob of one saved state: posA | vaA | adA | oidA | pres | ctrl
// (without the control block if !ctrl)
static CopyPlan state_plan(rrsph_ctx* ctx, void* blob, bool save, bool ctrl = true) {
    const StateLayout S(ctx);
    char* d = (char*)blob;
    void* arrays[kStateArrays] = {ctx->posA, ctx->vaA, ctx->adA, ctx->oidA, ctx->pres, ctx->ctrl};
    CopyPlan plan;
    for (int k = 0; k < kStateArrays - (ctrl ? 0 : 1); ++k) {
        if (save) plan.add(arrays[k], d + S.off[k], S.bytes[k]);
        else plan.add(d + S.off[k], arrays[k], S.bytes[k]);
    }
    return plan;
}

static rrsph_status save_state(rrsph_ctx* ctx, void* dst) { return enqueue_copies(ctx, state_plan(ctx, dst, true)); }

// The arrays of the state saved in blob, in place (layout of state_plan).
static StateView state_view(const rrsph_ctx* ctx, void* blob) {
    const StateLayout S(ctx);
    char* d = (char*)blob;
    return StateView{d, d + S.off[1], d + S.off[2], (uint32_t*)(d + S.off[3])};
}

static rrsph_status restore_state(rrsph_ctx* ctx, const void* src, bool keys = true) {
    if (const rrsph_status st = enqueue_copies(ctx, state_plan(ctx, const_cast<void*>(src), false)); st != RRSPH_OK)
        return st;
    ctx->fields_valid = false;  // der / xs belong to whatever step ran last
    ctx->pres_in_order = true;
    // the next step's cell keys from the restored positions, and a full sort
    ctx->need_full = true;
    if (!keys) return RRSPH_OK;  // the caller reorders with a saved sort and launches no step
    enqueue_state_keys(ctx);
    HIP_TRY(hipGetLastError());
    return RRSPH_OK;
}

// restore_state, then bring the host mirror of the control block up to date
static rrsph_status restore_state_sync(rrsph_ctx* ctx, const void* src) {
    rrsph_status st = restore_state(ctx, src);
    if (st != RRSPH_OK) return st;
    HIP_TRY(hipMemcpyAsync(ctx->host_ctrl, ctx->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return RRSPH_OK;
}

// One forward tape step as the graph of a sorted step with the incremental
// re-sort, then its record and gauges (rows of the step index - base),
// when that is what launch_steps would launch; returns false (nothing
// launched) otherwise.  A launch after a kernel launched on its own (the
// record, the gauges) waits several microseconds longer for the stream
// than a kernel inside a graph, so the step costs about 20 us less.
static rrsph_status launch_taped_step(rrsph_ctx* ctx, uint64_t base, bool& launched) {
    AdjTape& T = ctx->adj;
    launched = false;
    if (!ctx->use_graph || ctx->need_full || !ctx->incremental || ctx->launched < ctx->full_until) return RRSPH_OK;
    if (!T.texec || T.tbase != base) {
        drop_tape_graph(T);
        HIP_TRY(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        enqueue_step(ctx, nullptr, false);
        adj_record<<<1, 1, 0, ctx->stream>>>(ctx->ctrl, T.rec, base, T.nsteps);
        const rrsph_status st = enqueue_smooth_gauges(ctx, T.spec, T.partials, T.eta, T.zs, T.ws, ctx->ctrl, base,
                                                      T.nsteps);
        hipGraph_t g = nullptr;
        const hipError_t e = hipStreamEndCapture(ctx->stream, &g);
        if (st != RRSPH_OK || e != hipSuccess) {
            if (g) (void)hipGraphDestroy(g);
            return st != RRSPH_OK ? st : fail(ctx, RRSPH_ERR_HIP, std::string("hipStreamEndCapture: ") +
                                                                      hipGetErrorString(e));
        }
        T.tgraph = g;
        HIP_TRY(hipGraphInstantiate(&T.texec, T.tgraph, nullptr, nullptr, 0));
        T.tbase = base;
    }
    HIP_TRY(hipGraphLaunch(T.texec, ctx->stream));
    // launch_steps' bookkeeping of a step with the incremental re-sort
    ctx->last_keys = ctx->kbuf[0];
    ctx->last_perm = ctx->vbuf[0];
    ++ctx->n_incremental;
    ++ctx->launched;
    ctx->need_full = false;
    ctx->stepped = true;
    ctx->fields_valid = true;
    ctx->list_fields = false;
    launched = true;
    return RRSPH_OK;
}

// The skin of taped runs while they launch steps.  Lists built with either
// skin: a taped range starts with a build, and the wider lists left behind
// serve the narrower skin.
struct TapeSkin {
    StepParams& P;
    const StepParams before;
    bool& taping;
    TapeSkin(rrsph_ctx* ctx) : P(ctx->P), before(ctx->P), taping(ctx->taping) {
        if (!ctx->adj.lists) return;
        set_skin(P, ctx->tape_skin);
        taping = true;
    }
    ~TapeSkin() {
        taping = false;
        P.list_reach = before.list_reach;
        P.list_r2 = before.list_r2;
        P.skin_half = before.skin_half;
    }
};

// While a tape launches steps: the lists go where the tape keeps them, not
// into the context's (copying them took 280 us a build at 943,906 particles
// in 3D, two thirds of the build itself).  A range of list steps starts with
// a build, also where it resumes, and the next step of the context builds.
struct TapeBuildLists {
    rrsph_ctx* c;
    uint32_t *nbl, *nbc;
    explicit TapeBuildLists(rrsph_ctx* ctx) : c(ctx), nbl(ctx->nbl), nbc(ctx->nbc) {}
    ~TapeBuildLists() {
        c->nbl = nbl;
        c->nbc = nbc;
    }
};
// The next build writes the next of the tape's lists (allocated when first needed).
static rrsph_status tape_build_lists(rrsph_ctx* ctx) {
    AdjTape& T = ctx->adj;
    const size_t n = ctx->P.n, rows = ctx->P.list_cap + kListPad;
    if (T.nseg_lists == T.seg_lists.size()) {
        AdjTape::Lists L;
        hipError_t e = T.keep_all && T.nseg_lists >= std::min(T.max_lists, ctx->tape_lists_max) ? hipErrorOutOfMemory
                                                                                                : hipSuccess;
        L.nbl = dalloc<uint32_t>(rows * n, e);
        L.nbc = dalloc<uint32_t>(n, e);
        L.keys = dalloc<uint32_t>(n, e);
        if (e == hipSuccess) e = hipMemsetAsync(L.nbl, 0, rows * n * sizeof(uint32_t), ctx->stream);  // (list_entry)
        if (e != hipSuccess) {
            void* got[] = {L.nbl, L.nbc, L.keys};
            for (void* p : got)
                if (p) (void)hipFree(p);
            (void)hipGetLastError();
            T.no_room = T.keep_all;
            return fail(ctx, RRSPH_ERR_HIP, std::string("hipMalloc (adjoint lists): ") + hipGetErrorString(e));
        }
        T.seg_lists.push_back(L);
    }
    ctx->nbl = T.seg_lists[T.nseg_lists].nbl;
    ctx->nbc = T.seg_lists[T.nseg_lists].nbc;
    ++T.nseg_lists;
    return RRSPH_OK;
}

// While a batched tape launches steps: a step reads the kept state before it
// and leaves the kept state after it, the first from and the last to the
// context's arrays (saving a copy after every step took 6.1 us and a launch
// gap of the 100 of a step of 134,042 particles, 21 at 943,906 in 3D).
struct TapeStates {
    rrsph_ctx* c;
    double2* pos;
    void *va, *ad, *pres;
    uint32_t* oid;
    explicit TapeStates(rrsph_ctx* ctx)
        : c(ctx), pos(ctx->posA), va(ctx->vaA), ad(ctx->adA), pres(ctx->pres), oid(ctx->oidA) {}
    ~TapeStates() { context_arrays(); }
    void context_arrays() {
        c->posA = pos;
        c->vaA = va;
        c->adA = ad;
        c->pres = pres;
        c->oidA = oid;
        c->out = rrsph_ctx::Out{};
    }
    // in, out: saved states, or null for the context's arrays
    void step(char* in, char* out) {
        const StateLayout S(c);
        context_arrays();
        if (out)
            c->out = rrsph_ctx::Out{(double2*)out, out + S.off[1], out + S.off[2], out + S.off[4],
                                    (uint32_t*)(out + S.off[3]), (Ctrl*)(out + S.off[5])};
        else if (in)
            c->out = rrsph_ctx::Out{pos, va, ad, pres, oid, nullptr};
        if (!in) return;
        c->posA = (double2*)in;
        c->vaA = in + S.off[1];
        c->adA = in + S.off[2];
        c->oidA = (uint32_t*)(in + S.off[3]);
        c->pres = in + S.off[4];
    }
};

constexpr uint32_t kHaltCheck = 64;  // tape steps between two looks at the control block

// Launch steps [k0, k1) of the tape, reading the control block back every
// kHaltCheck steps only: every step's record, the checkpoints (forward) or
// segment states (replay; slot k - kslot of seg_base), and the gauges
// (forward).  Returns the status read after the last step (or after the
// look that found a halt).
static rrsph_status adjoint_run(rrsph_ctx* ctx, uint32_t k0, uint32_t k1, bool forward, void* seg_base,
                                uint32_t kslot, uint64_t abs0) {
    AdjTape& T = ctx->adj;
    const TapeSkin skin(ctx);
    const TapeBuildLists own(ctx);
    TapeStates states(ctx);
    const size_t n = ctx->P.n;
    // the forward keeps the states of the last segment (of every step with
    // keep_all): the reverse pass starts there and needs no replay of it
    const uint32_t last0 = T.keep_all ? 0 : (T.nsteps - 1) / T.every * T.every;
    const uint64_t base = abs0 - k0;  // step index of tape step 0
    // the copies after a step (its sort, its build's lists) wait for the
    // state copy before the next step and go in the same launch when the
    // ranges fit one; the next step's sort overwrites them only after that
    if (forward && T.keep_all && T.lists)  // the builds before k0 (those launched after a halt left no lists)
        T.nseg_lists = k0 > 0 ? (uint32_t)(T.seg_build[k0 - 1] + 1) : 0u;
    const bool chained = forward && T.batched();
    // a halt leaves the state before the halted step in the context's arrays
    auto finish = [&](rrsph_status st) -> rrsph_status {
        states.context_arrays();
        if (chained && ctx->host_ctrl->halted) {
            const uint64_t at = committed_steps(*ctx->host_ctrl) - base;
            if (at > k0 && at < k1) {
                const rrsph_status s2 =
                    enqueue_copies(ctx, state_plan(ctx, (char*)seg_base + (size_t)at * T.blob, false, false));
                if (s2 != RRSPH_OK) return s2;
            }
        }
        return st;
    };
    CopyPlan pending;
    auto flush = [&]() -> rrsph_status {
        if (pending.n == 0) return RRSPH_OK;
        const CopyPlan p = pending;
        pending.n = 0;
        return enqueue_copies(ctx, p);
    };
    auto save = [&](void* dst) -> rrsph_status {
        const CopyPlan p = state_plan(ctx, dst, true);
        if (pending.n + p.n > kCopyRanges) {
            if (const rrsph_status s2 = flush(); s2 != RRSPH_OK) return s2;
        }
        for (int i = 0; i < p.n; ++i) pending.r[pending.n++] = p.r[i];
        return flush();
    };
    for (uint32_t k = k0; k < k1; ++k) {
        rrsph_status st = RRSPH_OK;
        // after a halt the rest of the range is launches that do nothing:
        // look every kHaltCheck steps, so that a halt early in a long range
        // costs at most that many (the caller resumes from the halted step)
        if (k > k0 && (k - k0) % kHaltCheck == 0) {
            st = flush();
            if (st != RRSPH_OK) return st;
            HIP_TRY(hipMemcpyAsync(ctx->host_ctrl, ctx->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, ctx->stream));
            HIP_TRY(hipStreamSynchronize(ctx->stream));
            if (ctx->host_ctrl->halted) return finish(sync_status(ctx));
        }
        if (chained)  // (a batched tape keeps state k in slot k)
            states.step(k > k0 ? (char*)seg_base + (size_t)k * T.blob : nullptr,
                        k + 1 < k1 ? (char*)seg_base + (size_t)(k + 1) * T.blob : nullptr);
        if (forward && k % T.every == 0) {
            if (T.lists && k > 0) {  // the build interval from the displacements so far
                HIP_TRY(hipMemcpyAsync(ctx->host_ctrl, ctx->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, ctx->stream));
                HIP_TRY(hipStreamSynchronize(ctx->stream));
                if (!ctx->host_ctrl->halted) adapt_list_interval(ctx);
            }
            st = save(T.ck[k / T.every]);
            if (st != RRSPH_OK) return st;
        }
        const bool keep = forward ? k >= last0 : true;  // seg holds this step's state
        const size_t slot = forward ? k - last0 : k - kslot;
        // a batched tape's steps leave their states where they are kept, and a
        // range that resumes at a halted step has the state before it there
        if (keep) {
            if (!chained || k == 0) st = save((char*)seg_base + slot * T.blob);
            else st = flush();
            if (st != RRSPH_OK) return st;
            if (!forward && k + 1 == k1) {  // the state before the segment's last step is all the adjoint needs
                // that step is not launched: a list step reads the lists of the segment's last build; a
                // step that would build sorts its state in the reverse pass
                if (T.lists) T.seg_build[slot] = T.builds[k] ? -1 : (int32_t)T.nseg_lists - 1;
                break;
            }
        }
        bool build = false, taped = false;
        if (T.lists) {
            const uint64_t abs = abs0 + (k - k0);
            build = forward ? (k % T.every == 0 || k == T.force_build || abs - ctx->build_at >= ctx->list_interval)
                            : T.builds[k] != 0;
            if (forward) T.builds[k] = build ? 1 : 0;
            if (keep && build) {
                if (slot == 0 && !T.keep_all) T.nseg_lists = 0;
                st = tape_build_lists(ctx);
                if (st != RRSPH_OK) return st;
            }
            st = launch_list_step(ctx, build, abs);
        } else {
            st = forward ? launch_taped_step(ctx, base, taped) : RRSPH_OK;
            if (st == RRSPH_OK && !taped) st = launch_steps(ctx, 1);
        }
        if (st != RRSPH_OK) return st;
        if (keep) {
            CopyPlan plan;
            if (!T.lists || build) {  // keep the sort of a step whose state seg holds
                plan.add(ctx->last_keys, T.seg_keys + slot * n, n * sizeof(uint32_t));
                plan.add(ctx->last_perm, T.seg_perm + slot * n, n * sizeof(uint32_t));
                T.seg_sorted[slot] = 1;
            } else {
                T.seg_sorted[slot] = 0;  // its state is in its build's slot order
            }
            if (T.lists && build)  // and its build's sorted keys (the lists are in place)
                plan.add(ctx->last_keys, T.seg_lists[T.nseg_lists - 1].keys, n * sizeof(uint32_t));
            if (T.lists) T.seg_build[slot] = (int32_t)T.nseg_lists - 1;
            pending = plan;  // empty before: the state copy before the step took it
        }
        if (forward && !taped && !T.batched()) {
            adj_record<<<1, 1, 0, ctx->stream>>>(ctx->ctrl, T.rec, base, T.nsteps);
            st = enqueue_smooth_gauges(ctx, T.spec, T.partials, T.eta, T.zs, T.ws, ctx->ctrl, base, T.nsteps);
            if (st != RRSPH_OK) return st;
        }
    }
    if (const rrsph_status st = flush(); st != RRSPH_OK) return st;
    return finish(sync_status(ctx));
}

// adjoint_run with its halts handled: a step that changed more cells than
// the incremental re-sort takes, or (forward, list steps) found its lists
// possibly stale, halts before touching the state, and the launches after
// it do nothing; clear the halt and resume the range from that step, which
// runs with the full sort or as a build (its record, checkpoint, segment
// state and gauges are written again).
static rrsph_status adjoint_run_checked(rrsph_ctx* ctx, uint32_t k0, uint32_t k1, bool forward, void* seg_base) {
    HIP_TRY(hipMemcpyAsync(ctx->host_ctrl, ctx->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    const uint64_t start = committed_steps(*ctx->host_ctrl);
    AdjTape& T = ctx->adj;
    uint32_t from = k0;
    while (true) {
        rrsph_status st = adjoint_run(ctx, from, k1, forward, seg_base, k0, start + (from - k0));
        if (st != RRSPH_OK) return st;
        Ctrl& c = *ctx->host_ctrl;
        if (!c.halted) return RRSPH_OK;
        const bool resort = c.status == kStatusResort;
        const bool stale = c.status == kStatusRebuild && forward && T.lists;
        if (c.status == kStatusListOverflow)
            return fail(ctx, RRSPH_ERR_NOT_IMPLEMENTED,
                        "RRSPH_HIP: a neighbour list ran out of room during the adjoint's tape; run it with "
                        "RRSPH_HIP_LIST=0");
        if (!resort && !stale) return RRSPH_OK;
        const uint32_t at = k0 + (uint32_t)(committed_steps(c) - start);  // the step that halted
        // the resumed step runs with the full sort or builds, so every resume advances
        if (at < from || at >= k1 || (at == from && from != k0))
            return fail(ctx, RRSPH_ERR_HIP, "RRSPH_HIP: halt outside the replayed range");
        if (resort) {
            note_resort_overflow(ctx, committed_steps(c));
        } else {
            note_list_stale(ctx, committed_steps(c));
            T.force_build = at;
        }
        c.halted = 0;
        c.status = 0;
        HIP_TRY(hipMemcpyAsync(ctx->ctrl, ctx->host_ctrl, sizeof(Ctrl), hipMemcpyHostToDevice, ctx->stream));
        from = at;
    }
}

rrsph_status rrsph_hip_smooth_gauges(rrsph_ctx* ctx, const rrsph_gauge_spec* spec, double* eta) {
    if (!ctx || !ctx->uploaded || !eta) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad arguments");
    GaugeSpec3 G;
    rrsph_status st = to_gauge_spec(ctx, spec, G);
    if (st != RRSPH_OK) return st;
    const uint32_t nb = grid_blocks(ctx->P.n, kBlock);
    double* buf = nullptr;
    HIP_TRY(hipMalloc((void**)&buf, (2 * kMaxGauges * (size_t)nb + 3 * kMaxGauges) * sizeof(double)));
    double* out = buf + 2 * kMaxGauges * (size_t)nb;
    st = enqueue_smooth_gauges(ctx, G, buf, out, out + kMaxGauges, out + 2 * kMaxGauges);
    if (st == RRSPH_OK) {
        HIP_TRY(hipMemcpyAsync(eta, out, G.g.n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    HIP_TRY(hipFree(buf));
    return st;
}

rrsph_status rrsph_hip_smooth_gauges_noalloc(rrsph_ctx* ctx, const rrsph_gauge_spec* spec, double* eta) {
    if (!ctx || !ctx->uploaded || !eta || !spec)
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad arguments");
    if (spec->n > kMaxGauges)
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT,
                    "RRSPH_HIP: rrsph_hip_smooth_gauges_noalloc takes at most 64 gauges (its scratch holds 64)");
    GaugeSpec3 G;
    rrsph_status st = to_gauge_spec(ctx, spec, G);
    if (st != RRSPH_OK) return st;
    if (!ctx->scratch || !ctx->host_eta) return fail(ctx, RRSPH_ERR_HIP, "RRSPH_HIP: no scratch on this device");
    // every partial and result slot used below is written before it is read:
    // nothing in the scratch needs clearing
    double* partials = ctx->scratch;
    double* out = ctx->scratch + 2 * (size_t)kMaxGauges * kGaugeBlocks;
    st = enqueue_smooth_gauges(ctx, G, partials, out, out + kMaxGauges, out + 2 * kMaxGauges);
    if (st != RRSPH_OK) return st;
    HIP_TRY(hipMemcpyAsync(ctx->host_eta, out, G.g.n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    std::memcpy(eta, ctx->host_eta, G.g.n * sizeof(double));
    return RRSPH_OK;
}

rrsph_status rrsph_hip_set_piston(rrsph_ctx* ctx, double omega, uint32_t nharm, const double* a, const double* b) {
    if (!ctx) return RRSPH_ERR_INVALID_ARGUMENT;
    const uint32_t total = nharm * (uint32_t)ctx->P.piston_segments;  // paddle-major
    if (nharm > RRSPH_MAX_HARMONICS || total > RRSPH_MAX_HARMONICS || (nharm && (!a || !b)))
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad piston coefficients");
    ctx->prm.piston_omega = omega;
    ctx->prm.piston_nharm = (int32_t)nharm;
    ctx->P.piston_omega = omega;
    ctx->P.piston_nharm = (int32_t)nharm;
    for (uint32_t k = 0; k < RRSPH_MAX_HARMONICS; ++k) {
        const double ak = k < total ? a[k] : 0.0, bk = k < total ? b[k] : 0.0;
        ctx->prm.piston_a[k] = ak;
        ctx->prm.piston_b[k] = bk;
        ctx->P.piston_a[k] = ak;
        ctx->P.piston_b[k] = bk;
    }
    drop_graph(ctx);  // the captured steps hold the old coefficients
    ctx->adj.valid = false;
    return RRSPH_OK;
}

// Whether a tape runs list steps (builds at its checkpoints and by the
// displacements, the schedule recorded for the replays).
// In 2D: 60 steps of 134,042 particles forward and back 10.2 -> 8.2 ms, 40 of
// 18,544 4.1 -> 2.4 and of 5,040 4.0 -> 2.2.  The line is not one of speed (40
// steps of 474 particles would take 1.6 ms instead of 3.5, of 3,649 1.6 instead
// of 3.7): list tapes are tested from 4,237 particles on, and smaller runs keep
// the sorted steps that theirs are tested with.
constexpr uint32_t kTapeListMin2 = 4096;
static bool tape_lists(const rrsph_ctx* ctx) {
    if (!list_active(ctx)) return false;
    return ctx->P.dim == 3 || (ctx->P.n >= kTapeListMin2 && ctx->P.n <= kAdjListMax);
}

// Other 2D tapes and replays run without neighbour lists (a replay must
// repeat its step exactly, whatever the list schedule was).  Entering and
// leaving that state forces a full sort and a list build.
struct ListSuspend {
    rrsph_ctx* c;
    bool was;
    explicit ListSuspend(rrsph_ctx* ctx) : c(ctx), was(ctx->list_suspended) {
        if (c->list_mode && !was) c->need_full = true;
        c->list_suspended = true;
    }
    ~ListSuspend() {
        c->list_suspended = was;
        if (c->list_mode && !was) c->need_full = true;
    }
};

static rrsph_status adjoint_forward_impl(rrsph_ctx* ctx, uint32_t nsteps, uint32_t checkpoint_every,
                                         const rrsph_gauge_spec* spec, double* eta);
static rrsph_status adjoint_backward_impl(rrsph_ctx* ctx, const double* eta_bar, double* grad_a, double* grad_b,
                                          double* grad_r0, double* grad_v0, double* grad_rho0);

rrsph_status rrsph_hip_adjoint_forward(rrsph_ctx* ctx, uint32_t nsteps, uint32_t checkpoint_every,
                                       const rrsph_gauge_spec* spec, double* eta) {
    if (!ctx) return RRSPH_ERR_INVALID_ARGUMENT;
    const rrsph_status st = adjoint_forward_impl(ctx, nsteps, checkpoint_every, spec, eta);
    if (ctx->P.dim == 3 || list_active(ctx)) ctx->need_full = true;  // the next step builds lists of its own
    return st;
}

rrsph_status rrsph_hip_adjoint_backward(rrsph_ctx* ctx, const double* eta_bar, double* grad_a, double* grad_b,
                                        double* grad_r0, double* grad_v0, double* grad_rho0) {
    if (!ctx) return RRSPH_ERR_INVALID_ARGUMENT;
    if (ctx->P.dim == 3 || ctx->adj.lists) {
        rrsph_status st = adjoint_backward_impl(ctx, eta_bar, grad_a, grad_b, grad_r0, grad_v0, grad_rho0);
        ctx->need_full = true;
        return st;
    }
    ListSuspend guard(ctx);
    return adjoint_backward_impl(ctx, eta_bar, grad_a, grad_b, grad_r0, grad_v0, grad_rho0);
}

constexpr uint32_t kGaugeRows = 64;  // steps whose gauges one launch takes

// The records and gauges of every step of a batched tape, from the states
// kept before the next step and the final state.  A record and two gauge
// kernels after each step took 14 us and their launch gaps.
static rrsph_status tape_records_and_gauges(rrsph_ctx* ctx) {
    AdjTape& T = ctx->adj;
    const uint32_t N = T.nsteps;
    char* final_state = (char*)T.ck.back();
    const size_t at = state_ctrl_offset(ctx);
    tape_records_kernel<<<grid_blocks(N, kBlock), kBlock, 0, ctx->stream>>>((const char*)T.seg + T.blob + at, T.blob,
                                                                            final_state + at, T.rec, N);
    HIP_TRY(hipGetLastError());
    for (uint32_t k = 0; k < N;) {
        const bool last = k + 1 == N;
        const uint32_t rows = last ? 1u : std::min(kGaugeRows, N - 1 - k);
        const StateView v = state_view(ctx, last ? final_state : (char*)T.seg + (size_t)(k + 1) * T.blob);
        const size_t o = (size_t)k * kMaxGauges;
        const rrsph_status st = enqueue_smooth_gauges(ctx, T.spec, T.partials, T.eta + o, T.zs + o, T.ws + o, nullptr,
                                                      0, 0, &v, rows, T.blob);
        if (st != RRSPH_OK) return st;
        k += rows;
    }
    return RRSPH_OK;
}

// What a tape that keeps every state may take: half the free memory, or what
// RRSPH_HIP_TAPE_MEMORY says (bytes; a process that shares the device).
static double tape_memory() {
    if (const char* e = std::getenv("RRSPH_HIP_TAPE_MEMORY")) return std::strtod(e, nullptr);
    size_t free_b = 0, total_b = 0;
    return hipMemGetInfo(&free_b, &total_b) == hipSuccess ? 0.5 * (double)free_b : 0.0;
}
// Bytes of every state and sort of the tape, and of one build's lists.
static double tape_state_bytes(const rrsph_ctx* ctx) {
    return (double)ctx->adj.nsteps * ((double)state_bytes(ctx) + 256 + 8.0 * ctx->P.n);
}
static double tape_list_bytes(const rrsph_ctx* ctx) { return 4.0 * ctx->P.n * (double)(ctx->P.list_cap + kListPad + 2); }

// Whether every state and sort of the tape, and with list steps the lists
// of a build in every fourth step and every checkpoint, fit in tape_memory.
// (A kept tape that builds more often than fits (max_lists), or finds no
// memory for a build's lists, starts over: in 3D with one segment's states,
// in 2D on sorted steps if all their states fit.)
static bool tape_fits(const rrsph_ctx* ctx, bool lists) {
    const AdjTape& T = ctx->adj;
    const double builds = lists ? T.nsteps / 4.0 + (double)((T.nsteps + T.every - 1) / T.every) + 1 : 0.0;
    return tape_state_bytes(ctx) + builds * tape_list_bytes(ctx) <= tape_memory();
}

// Whether a tape of this shape has not just run out of room for its lists.
static bool tape_may_keep(const rrsph_ctx* ctx) {
    return ctx->no_keep_steps != ctx->adj.nsteps || ctx->no_keep_every != ctx->adj.every;
}

// The buffers of a tape of T.nsteps steps with a checkpoint every T.every.
static rrsph_status alloc_tape(rrsph_ctx* ctx) {
    AdjTape& T = ctx->adj;
    const uint32_t nsteps = T.nsteps;
    const size_t n = ctx->P.n;
    const bool d3 = ctx->P.dim == 3;
    T.blob = (state_bytes(ctx) + 255) / 256 * 256;
    const uint32_t nck = (nsteps + T.every - 1) / T.every;
    const uint32_t nb = grid_blocks(ctx->P.n, kBlock);
    hipError_t e = hipSuccess;
    T.ck.assign(nck + 1, nullptr);
    for (auto& p : T.ck) p = dalloc<char>(T.blob, e);
    // (RRSPH_HIP_ADJ_STORE=segments keeps one segment's states, and replays)
    T.keep_all = !T.segments && (tape_may_keep(ctx) || !T.lists) && tape_fits(ctx, T.lists);
    if (T.batched()) T.max_lists = (size_t)std::max(0.0, (tape_memory() - tape_state_bytes(ctx)) / tape_list_bytes(ctx));
    uint32_t cap = T.keep_all ? nsteps : T.every;  // states seg holds
    const bool alloc_ok = e == hipSuccess;
    T.seg = dalloc<char>(T.blob * cap, e);
    T.seg_keys = dalloc<uint32_t>(n * cap, e);
    T.seg_perm = dalloc<uint32_t>(n * cap, e);
    if (alloc_ok && e != hipSuccess && T.keep_all) {  // every state did not fit after all: one segment's
        void* got[] = {T.seg, T.seg_keys, T.seg_perm};
        for (void* p : got)
            if (p) (void)hipFree(p);
        (void)hipGetLastError();
        e = hipSuccess;
        T.keep_all = false;
        cap = T.every;
        T.seg = dalloc<char>(T.blob * cap, e);
        T.seg_keys = dalloc<uint32_t>(n * cap, e);
        T.seg_perm = dalloc<uint32_t>(n * cap, e);
    }
    T.seg_sorted.assign(cap, 0);
    T.builds.assign(nsteps, 0);
    T.seg_build.assign(cap, -1);
    if (T.lists && d3 && ctx->fp32) T.nearf = dalloc<float4>(n, e);
    T.eta = dalloc<double>((size_t)nsteps * kMaxGauges, e);
    T.zs = dalloc<double>((size_t)nsteps * kMaxGauges, e);
    T.ws = dalloc<double>((size_t)nsteps * kMaxGauges, e);
    T.eta_bar = dalloc<double>((size_t)nsteps * kMaxGauges, e);
    T.partials = dalloc<double>(2 * kMaxGauges * (T.batched() ? (size_t)gauge_blocks(ctx->P.n) * kGaugeRows : nb), e);
    T.piston_sum = dalloc<double>((size_t)nsteps * kMaxSegments, e);
    T.lam[0] = dalloc<double>((d3 ? kLam3 : 8) * n, e);
    T.lam[1] = dalloc<double>((d3 ? kLam3 : 8) * n, e);
    T.direct = dalloc<double>((d3 ? kDirect3 : 5) * n, e);
    T.drho_adj = dalloc<double>(n, e);
    T.out_adj = dalloc<double4>((d3        ? sizeof(AdjRec3<double>) / sizeof(double4)
                                 : T.lists ? sizeof(AdjRec2) / sizeof(double4)
                                           : 1) * n, e);
    T.flag = dalloc<uint32_t>(1, e);
    if (e != hipSuccess) {
        free_tape(ctx->adj);
        return fail(ctx, RRSPH_ERR_HIP, std::string("hipMalloc (adjoint tape): ") + hipGetErrorString(e));
    }
    T.rec = dalloc<AdjStep>(nsteps, e);
    T.uctrl = dalloc<Ctrl>(nsteps, e);
    if (e != hipSuccess) {
        free_tape(ctx->adj);
        return fail(ctx, RRSPH_ERR_HIP, std::string("hipMalloc (adjoint tape): ") + hipGetErrorString(e));
    }
    T.allocated = true;
    return RRSPH_OK;
}

static rrsph_status adjoint_forward_impl(rrsph_ctx* ctx, uint32_t nsteps, uint32_t checkpoint_every,
                                         const rrsph_gauge_spec* spec, double* eta) {
    if (!ctx || !ctx->uploaded || nsteps == 0 || checkpoint_every == 0 || !eta)
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad arguments");
    rrsph_status st = adjoint_supported(ctx);
    if (st != RRSPH_OK) return st;
    GaugeSpec3 G;
    st = to_gauge_spec(ctx, spec, G);
    if (st != RRSPH_OK) return st;
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    // a forward of the shape of the last one runs on its buffers: a training
    // loop allocates once (the 943,906-particle basin, 12 steps: 32.4 -> 24.3 ms; the tank, 60 steps: 13.0 -> 10.0); another shape frees them first
    const char* store = std::getenv("RRSPH_HIP_ADJ_STORE");
    const bool segments = store && std::strcmp(store, "segments") == 0;
    const bool may_list = tape_lists(ctx);
    AdjTape& T = ctx->adj;
    T.valid = false;
    if (T.allocated && T.nsteps == nsteps && T.every == std::min(checkpoint_every, nsteps) && T.may_list == may_list &&
        T.segments == segments) {
        drop_tape_graph(T);  // captured with the last run's gauges and piston
    } else {
        free_tape(T);
        T.nsteps = nsteps;
        T.every = std::min(checkpoint_every, nsteps);
        T.segments = segments;
        T.may_list = may_list;
        if (tape_may_keep(ctx)) ctx->no_keep_steps = ctx->no_keep_every = 0;
        // in 2D sorted steps whose states can all be kept beat list steps that replay
        T.lists = may_list && (ctx->P.dim == 3 || segments || (tape_may_keep(ctx) && tape_fits(ctx, true)) ||
                               !tape_fits(ctx, false));
        st = alloc_tape(ctx);
        if (st != RRSPH_OK) return st;
    }
    std::optional<ListSuspend> guard;
    if (ctx->P.dim == 2 && !T.lists) guard.emplace(ctx);
    const size_t n = ctx->P.n;
    const uint32_t nck = (uint32_t)T.ck.size() - 1;
    T.spec = G;
    T.seg_last = false;
    std::fill(T.seg_sorted.begin(), T.seg_sorted.end(), (uint8_t)0);
    std::fill(T.builds.begin(), T.builds.end(), (uint8_t)0);
    std::fill(T.seg_build.begin(), T.seg_build.end(), -1);
    T.nseg_lists = 0;
    T.force_build = ~0ull;
    const uint64_t interval = ctx->list_interval;
    st = adjoint_run_checked(ctx, 0, nsteps, true, T.seg);
    const bool overflowed = T.lists && ctx->P.dim == 2 && ctx->host_ctrl->halted &&
                            ctx->host_ctrl->status == kStatusListOverflow;
    if (st != RRSPH_OK && (overflowed || T.no_room)) {
        // a list ran out of room: the run starts over on sorted steps, which
        // the context keeps to from here (as resume_halt has it); no memory for
        // a build's lists: see tape_fits
        st = restore_state_sync(ctx, T.ck[0]);
        if (st != RRSPH_OK) return st;
        if (overflowed) ctx->list_mode = false;
        else ctx->no_keep_steps = T.nsteps, ctx->no_keep_every = T.every;
        ctx->list_interval = interval;  // (the schedule of a run that had not been tried)
        free_tape(T);
        ctx->err.clear();
        return adjoint_forward_impl(ctx, nsteps, checkpoint_every, spec, eta);
    }
    if (st != RRSPH_OK) return st;
    if (ctx->host_ctrl->halted)
        return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: the run halted during the adjoint forward");
    st = save_state(ctx, T.ck[nck]);
    if (st != RRSPH_OK) return st;
    if (T.batched()) {
        st = tape_records_and_gauges(ctx);
        if (st != RRSPH_OK) return st;
    }
    T.seg_last = true;
    std::vector<double> h((size_t)nsteps * kMaxGauges);
    HIP_TRY(hipMemcpyAsync(h.data(), T.eta, h.size() * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    T.hrec.resize(nsteps);
    HIP_TRY(hipMemcpyAsync(T.hrec.data(), T.rec, nsteps * sizeof(AdjStep), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    for (uint32_t k = 0; k < nsteps; ++k)
        for (uint32_t g = 0; g < G.g.n; ++g) eta[(size_t)k * G.g.n + g] = h[(size_t)k * kMaxGauges + g];
    {
        std::vector<Ctrl> uc(nsteps, Ctrl{});
        for (uint32_t k = 0; k < nsteps; ++k) uc[k].cur_dt = T.hrec[k].dt_pred;
        HIP_TRY(hipMemcpyAsync(T.uctrl, uc.data(), nsteps * sizeof(Ctrl), hipMemcpyHostToDevice, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    T.valid = true;
    return RRSPH_OK;
}

// dL/dx of the loss term of the gauges of state A, or of the saved state
// src (lam += ...)
static void enqueue_gauge_grad(rrsph_ctx* ctx, uint32_t k, double* lam, const StateView* src = nullptr) {
    AdjTape& T = ctx->adj;
    const uint32_t nb = grid_blocks(ctx->P.n, kBlock);
    const size_t o = (size_t)k * kMaxGauges;
    const void* pos = src ? src->pos : (const void*)ctx->posA;
    const void* va = src ? src->va : ctx->vaA;
    const uint32_t* oid = src ? src->oid : ctx->oidA;
    if (ctx->P.dim == 3)
        smooth_gauge_grad3<<<nb, kBlock, 0, ctx->stream>>>(ctx->P.n, (const double4*)pos, oid, T.spec,
                                                           T.eta_bar + o, T.zs + o, T.ws + o, lam);
    else if (ctx->fp32)
        smooth_gauge_grad<float><<<nb, kBlock, 0, ctx->stream>>>(ctx->P.n, (const double2*)pos, (const float4*)va,
                                                                 oid, T.spec.g, T.eta_bar + o, T.zs + o,
                                                                 T.ws + o, lam);
    else
        smooth_gauge_grad<double><<<nb, kBlock, 0, ctx->stream>>>(ctx->P.n, (const double2*)pos, (const double4*)va,
                                                                  oid, T.spec.g, T.eta_bar + o, T.zs + o,
                                                                  T.ws + o, lam);
}

static rrsph_status adjoint_backward_impl(rrsph_ctx* ctx, const double* eta_bar, double* grad_a, double* grad_b,
                                          double* grad_r0, double* grad_v0, double* grad_rho0) {
    if (!ctx || !eta_bar) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: bad arguments");
    AdjTape& T = ctx->adj;
    if (!T.valid) return fail(ctx, RRSPH_ERR_INVALID_ARGUMENT, "RRSPH_HIP: run rrsph_hip_adjoint_forward first");
    const StepParams& P = ctx->P;
    const bool d3 = P.dim == 3;
    const size_t n = P.n;
    const uint32_t lw = d3 ? kLam3 : 8;  // doubles of adjoint state per particle
    const uint32_t N = T.nsteps, G = T.spec.g.n;
    const uint32_t nb = grid_blocks(P.n, kBlock);
    {
        std::vector<double> h((size_t)N * kMaxGauges, 0.0);
        for (uint32_t k = 0; k < N; ++k)
            for (uint32_t g = 0; g < G; ++g) h[(size_t)k * kMaxGauges + g] = eta_bar[(size_t)k * G + g];
        HIP_TRY(hipMemcpyAsync(T.eta_bar, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    HIP_TRY(hipMemsetAsync(T.piston_sum, 0, (size_t)N * kMaxSegments * sizeof(double), ctx->stream));
    HIP_TRY(hipMemsetAsync(T.lam[0], 0, lw * n * sizeof(double), ctx->stream));
    HIP_TRY(hipMemsetAsync(T.flag, 0, sizeof(uint32_t), ctx->stream));
    const uint32_t nck = (N + T.every - 1) / T.every;
    // the loss term of the final state
    rrsph_status st = restore_state(ctx, T.ck[nck]);
    if (st != RRSPH_OK) return st;
    enqueue_gauge_grad(ctx, N - 1, T.lam[0]);
    HIP_TRY(hipGetLastError());
    int cur = 0;
    for (int seg = (int)nck - 1; seg >= 0; --seg) {
        const uint32_t n0 = (uint32_t)seg * T.every, n1 = std::min(n0 + T.every, N);
        // replay the segment from its checkpoint, keeping the state before each
        // step (the last segment's states are there already after a forward)
        if (!T.keep_all && !(T.seg_last && seg == (int)nck - 1)) {
            std::fill(T.seg_sorted.begin(), T.seg_sorted.end(), (uint8_t)0);
            std::fill(T.seg_build.begin(), T.seg_build.end(), -1);
            st = restore_state(ctx, T.ck[seg]);
            if (st != RRSPH_OK) return st;
            st = adjoint_run_checked(ctx, n0, n1, false, T.seg);
            if (st != RRSPH_OK) return st;
        }
        T.seg_last = false;
        for (int k = (int)n1 - 1; k >= (int)n0; --k) {
            const size_t slot = (size_t)(T.keep_all ? k : k - (int)n0);
            const bool sorted = T.seg_sorted[slot] != 0;  // the replay launched step k with a sort
            // list steps: the build whose lists step k read, its state in that build's slot order
            const int32_t b = T.lists ? T.seg_build[slot] : -1;
            const AdjTape::Lists* lists = b >= 0 ? &T.seg_lists[(size_t)b] : nullptr;
            // a replay does not launch a segment's last step: one that builds is
            // reversed by the cell walk, in 3D FP32 with FP64 separations where
            // lists have the near records' FP32, and so it is on kept tapes
            if (T.batched() && d3 && ctx->fp32 && T.builds[k] && k + 1 == (int)n1 && n1 < N) lists = nullptr;
            // a step reordered with a saved sort reads its state where it was
            // saved; one that sorts again needs it in A (and its cell keys)
            char* blob = (char*)T.seg + slot * T.blob;
            const bool in_place = sorted || lists;
            const StateView view = state_view(ctx, blob);
            const StateView* src = in_place ? &view : nullptr;
            if (!in_place) {
                st = restore_state(ctx, blob, true);
                if (st != RRSPH_OK) return st;
            }
            // sort and reorder state k exactly as its step did (predict with its dt)
            const uint32_t* sk = sorted ? T.seg_keys + slot * n : (lists ? lists->keys : nullptr);
            const uint32_t* sp = sorted ? T.seg_perm + slot * n : nullptr;
            // the loss term of state k: over lists with the pair gather
            const bool with_gauges = lists && k >= 1;
            const size_t row = k >= 1 ? (size_t)(k - 1) * kMaxGauges : 0;
            const double *eb = with_gauges ? T.eta_bar + row : nullptr, *zs = T.zs + row, *ws = T.ws + row;
            if (ctx->fp32)
                enqueue_reverse_step<float>(ctx, T.hrec[k], T.uctrl + k, T.lam[cur], T.lam[1 - cur],
                                            T.piston_sum + (size_t)k * kMaxSegments, sk, sp, lists, src,
                                            eb, zs, ws);
            else
                enqueue_reverse_step<double>(ctx, T.hrec[k], T.uctrl + k, T.lam[cur], T.lam[1 - cur],
                                             T.piston_sum + (size_t)k * kMaxSegments, sk, sp, lists, src,
                                            eb, zs, ws);
            if (k >= 1 && !with_gauges) enqueue_gauge_grad(ctx, k - 1, T.lam[1 - cur], src);
            HIP_TRY(hipGetLastError());
            cur = 1 - cur;
        }
    }
    // piston coefficients of paddle g: dV_g/da_{g,k} = k w cos(k w t), dV_g/db_{g,k} = -k w sin(k w t)
    std::vector<double> ps((size_t)N * kMaxSegments);
    HIP_TRY(hipMemcpyAsync(ps.data(), T.piston_sum, ps.size() * sizeof(double), hipMemcpyDeviceToHost,
                           ctx->stream));
    if (grad_r0 || grad_v0 || grad_rho0) {
        const size_t D = d3 ? 3 : 2;
        unpack_gradients_kernel<<<nb, kBlock, 0, ctx->stream>>>(P.n, T.lam[cur], lw, (uint32_t)D, ctx->st_r,
                                                                ctx->st_v, ctx->st_rho);
        HIP_TRY(hipGetLastError());
        if (grad_r0)
            HIP_TRY(hipMemcpyAsync(grad_r0, ctx->st_r, D * n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        if (grad_v0)
            HIP_TRY(hipMemcpyAsync(grad_v0, ctx->st_v, D * n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        if (grad_rho0)
            HIP_TRY(hipMemcpyAsync(grad_rho0, ctx->st_rho, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    }
    uint32_t flag = 0;
    HIP_TRY(hipMemcpyAsync(&flag, T.flag, sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    const int nh = P.nwm == 6 ? std::max(P.piston_nharm, 0) : 0;
    for (int g = 0; g < P.piston_segments; ++g) {
        for (int k = 0; k < nh; ++k) {
            double ga = 0, gb = 0;
            const double kw = (k + 1) * P.piston_omega;
            for (uint32_t s = 0; s < N; ++s) {
                const double v = ps[(size_t)s * kMaxSegments + g];
                ga += v * kw * std::cos(kw * T.hrec[s].t);
                gb -= v * kw * std::sin(kw * T.hrec[s].t);
            }
            if (grad_a) grad_a[g * nh + k] = ga;
            if (grad_b) grad_b[g * nh + k] = gb;
        }
    }
    // leave the context as the forward left it (restore_state makes the next
    // step sort, and build when it runs list steps)
    st = restore_state_sync(ctx, T.ck[nck]);
    if (st != RRSPH_OK) return st;
    if (flag) return fail(ctx, RRSPH_ERR_TOO_MANY_NEIGHBOURS, status_message(RRSPH_ERR_TOO_MANY_NEIGHBOURS));
    return RRSPH_OK;
}

uint32_t RRSPH_HIP_GetSpecificVersionMajor(void) { return RRSPH_HIP_VERSION_MAJOR; }
uint32_t RRSPH_HIP_GetSpecificVersionMinor(void) { return RRSPH_HIP_VERSION_MINOR; }
uint32_t RRSPH_HIP_GetSpecificVersionPatch(void) { return RRSPH_HIP_VERSION_PATCH; }
const char* RRSPH_HIP_GetSpecificVersionName(void) { return "RRSPH_HIP"; }

}  // extern "C"
