// Neighbour-list steps (2D): the cell sort and the cell walk once every
// several steps instead of every step.
//
// A build step sorts the particles by cell, reorders the state, and walks
// the cells within reach k h + skin of each particle (list_build_kernel):
// every particle i with |r_i - r_j| < k h + skin goes into j's list, in the
// walk order, k-major (entry k of slot j at nbl[k n + j], count nbc[j]).
// Until the next build the slot order stays as it is, and a step reads the
// lists instead of walking the cells: the pair pass decides each entry with
// the reference's FP64 cut-off test (GridFind.cpp:144-176, |r|^2 < (k h)^2
// with separate roundings), so the neighbour sets are those of the cell
// walk.  A pair closer than k h now was closer than k h + skin at the build
// as long as no particle has moved skin / 2 since: the integrator reduces
// each step's largest displacement, the prologue sums them, and a step
// whose lists may be stale halts before it reads them (status
// kStatusRebuild); the host re-runs it as a build step.  The host schedules
// builds ahead from the measured displacement rate, so such halts are rare.
//
// What the pair pass gathers per entry, one record of two halves per slot
// (32 bytes in FP32, 64 in FP64, so one cache line):
//   near  FP32: (xi_x, xi_y, vx, vy), xi the position relative to the
//         origin of the particle's home cell (its cell at the last build),
//         rounded from the FP64 position; FP64: (x, y, vx, vy), the FP64
//         position itself
//   pred  (v^x, v^y, s rho^, p / rho^2): predicted velocity and density,
//         s = +1 for fluid, -1 for boundary, 0 for a particle that no
//         longer exists
// An entry holds the neighbour's slot in its low 26 bits and the offset of
// the neighbour's home cell from the particle's, (dcx + 3) | (dcy + 3) << 3,
// in its high 6, so that in FP32 r_i - r_j = xi_i - xi_j + (dcx, dcy) cell
// to a few 1e-9 m.  FP32 decides an entry from that difference unless its
// squared distance lies within 1e-5 of the cut-off (or a position lies far
// from its home cell), where it takes the FP64 positions and the reference's
// test; the rounding of xi stays far below that band (2e-6 of the cut-off).
//
// Step kernels: [density_sum_list] -> pair_list -> integrate_list (in place;
// it also writes the next step's records, so no reorder runs between builds;
// with a constant dt and no wave maker the pair pass integrates: fused_step_begin),
// the first of them with the step's prologue (list_step_begin).  A build step runs list_prologue -> counting
// sort (cell_sort.hpp) -> reorder_list_kernel -> list_build_kernel -> the same step kernels
// on the reordered copy, integrating into A.
#pragma once

#include "cell_sort.hpp"
#include "device_common.hpp"
#include "step_kernels.hpp"

namespace rrsph {

constexpr uint32_t kStatusRebuild = 101;       // internal: re-run this step as a list build
constexpr uint32_t kStatusUnfused = 103;       // internal: a fused step might have too many neighbours; run steps unfused
constexpr uint32_t kStatusListOverflow = 102;  // internal: a list ran out of room; run without lists

// The state a list step reads (the reordered copy B on a build step, A after).
constexpr uint32_t kSlotBits = 26;
constexpr uint32_t kSlotMask = (1u << kSlotBits) - 1;  // list steps take at most 2^26 particles

template <class R> struct ListState {
    const double2* pos;
    const real4<R>* va;
    const uint32_t* oid;
};

// The record of a slot: near and pred halves.
template <class R> struct alignas(2 * sizeof(real4<R>)) ListRec {
    real4<R> nr;
    real4<R> pr;
};

// The sign-encoded predicted density of the pred record.
template <class R> __device__ __forceinline__ R typed_rho(R rho, int itype) {
    return itype > 0 ? rho : (itype < 0 ? -rho : R(0));
}

// The density back from its record where the type is at hand: a flow that breaks
// up may predict a negative one, whose sign a fabs would lose.
template <class R> __device__ __forceinline__ R untyped_rho(R z, int itype) { return itype > 0 ? z : -z; }

// The near record of a particle at pos with velocity (vx, vy) and home cell
// `home` (a cell key cx ncy + cy).
template <class R> __device__ __forceinline__ real4<R> near_record(const StepParams& P, double2 pos, R vx, R vy,
                                                                   uint32_t home);
template <> __device__ __forceinline__ float4 near_record<float>(const StepParams& P, double2 pos, float vx, float vy,
                                                                 uint32_t home) {
    const uint32_t cx = home / (uint32_t)P.ncy, cy = home - cx * (uint32_t)P.ncy;
    const double ox = P.xmin + (double)cx * P.cell, oy = P.ymin + (double)cy * P.cell;
    return make_float4((float)(pos.x - ox), (float)(pos.y - oy), vx, vy);
}
template <> __device__ __forceinline__ double4 near_record<double>(const StepParams&, double2 pos, double vx,
                                                                   double vy, uint32_t) {
    return make_double4(pos.x, pos.y, vx, vy);
}

// The prediction of PredictHalfStep.cpp:16-22 (v^ = v + a dt/2, rho^ = rho +
// drho dt/2 with continuity) and the pressure of the current density
// (Density.h:112) as reorder_kernel computes them; p / rho^2 in w.
template <class R> __device__ __forceinline__ real4<R> predict_record(const StepParams& P, const real4<R>& va,
                                                                      R ax, R ay, R drho, R dt, R& p) {
    const bool cont = P.density_treatment != 0;
    real4<R> pr;
    pr.x = va.x + ax * dt * R(0.5);
    pr.y = va.y + ay * dt * R(0.5);
    pr.z = cont ? va.z + drho * dt * R(0.5) : va.z;
    p = eos_p<R>(va.z, (R)P.rho0, (R)P.eos_B);
    pr.w = p / (pr.z * pr.z);
    pr.z = typed_rho<R>(pr.z, (int)va.w);
    return pr;
}

// The reorder of a build step: reorder_kernel's gather, prediction,
// pressure and cell-start table, plus the records of the list pass and each
// slot's home cell (its cell key).  COUNTED: behind the counting sort, with
// perm as its scatter left it; the cell-start table is there, and the
// permutation goes to perm_out.
template <class R, bool COUNTED>
__global__ void __launch_bounds__(kBlock) reorder_list_kernel(StepParams P, const Ctrl* __restrict__ ctrl,
                                                              const uint32_t* __restrict__ skey,
                                                              const uint32_t* __restrict__ perm, StateA<R> A,
                                                              StateB<R> B, ListRec<R>* __restrict__ rec,
                                                              uint32_t* __restrict__ home, uint32_t* __restrict__ LB,
                                                              uint32_t* __restrict__ perm_out) {
    if (ctrl->halted) return;
    const uint32_t s0 = blockIdx.x * kBlock + threadIdx.x;
    const bool live = s0 < P.n;
    uint32_t s = live ? s0 : P.n - 1;
    const uint32_t k = skey[s];
    const uint32_t src = min(perm[s], P.n - 1);  // a permutation of [0, n); the clamp only guards memory
    if constexpr (COUNTED) s = cell_place(P, LB, perm, s, k);
    const double2 pos = A.pos[src];
    const real4<R> va = A.va[src];
    const real4<R> ad = A.ad[src];
    const uint32_t oid = A.oid[src];
    R p;
    const real4<R> pr = predict_record<R>(P, va, ad.x, ad.y, ad.z, (R)ctrl->cur_dt, p);
    if (live) {
        B.pos[s] = pos;
        B.va[s] = va;
        B.oid[s] = oid;
        B.pres[s] = p;
        ListRec<R> r;
        r.nr = near_record<R>(P, pos, va.x, va.y, k);
        r.pr = pr;
        rec[s] = r;
        home[s] = k;
        if constexpr (COUNTED) perm_out[s] = src;
    }
    if constexpr (!COUNTED) fill_cell_starts(P, s, live, k, skey, LB);
}

// ------------------------------------------------------------------ control of list steps
// A list step has no prologue launch: between steps the control block
// `next` holds the last step's outcome; the step's first kernel (pair or
// summation pass) reads only `next` and the displacement slots, every block
// deciding by itself whether the step runs (list_step_halts), and its block 0
// writes the commit and this step's snapshot to a second block `cur`; the
// later kernels of the step read `cur`, and the integrator's block 0 publishes
// `cur` with the step's outcome in `next`.  So no kernel writes what its
// other blocks read.  A prologue launch of one block took 4.8 us and 1.2 us
// of launch gap at the head of every step (97 us at 1M particles FP32, 42 at
// 188k, 22 at 7k); build steps keep one (list_prologue), since their sort
// needs the decision.
//
// What several blocks of a step raise lies outside the published words: the
// flags at the end of Ctrl, and maxima in slots, a set per parity of the step
// index - displacement slots dslots (the integrator of step k fills set k,
// the first kernel of step k + 1 reads it and clears the other; where steps
// fuse, four sets by the index modulo 4) and dt reduction slots, the kernels'
// maxslots (the pair pass of step k fills set k, its integrator reads it and
// clears the other).  A set is few slots, each in a 256-byte line of its own:
// every block of the next kernel reads them all, at addresses known before any
// other load returns, without a reduction across lanes or a barrier (256
// adjacent slots, reduced by shuffles through LDS, held every block up for
// about 1.5 us).
constexpr uint32_t kSlots = 16, kSlotStride = 32;      // 64-bit words between slots
constexpr uint32_t kSlotSet = kSlots * kSlotStride;    // words of a set
constexpr uint32_t kDtSet = 2 * kSlotSet;              // a dt set: largest a^2, then largest mu
__device__ __forceinline__ double slots_max(const unsigned long long* slots) {
    unsigned long long w[kSlots];
#pragma unroll
    for (uint32_t k = 0; k < kSlots; ++k) w[k] = slots[k * kSlotStride];
    double m = 0.0;
#pragma unroll
    for (uint32_t k = 0; k < kSlots; ++k) m = fmax(m, dbits(w[k]));
    return m;
}
__device__ __forceinline__ void clear_slots(unsigned long long* slots) {
    if (threadIdx.x < kSlots) slots[threadIdx.x * kSlotStride] = 0;
}

// The wave's maximum of a non-negative value in every lane's return value of
// lane 63: data-parallel moves within and across the rows of 16 lanes, no LDS.
template <int CTRL> __device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL> __device__ __forceinline__ double dpp_move(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
template <class R> __device__ __forceinline__ R wave_max_lane63(R v) {
    v = fmax(v, dpp_move<0x111>(v));  // row_shr:1 (lanes without a source get 0)
    v = fmax(v, dpp_move<0x112>(v));  // row_shr:2
    v = fmax(v, dpp_move<0x114>(v));  // row_shr:4
    v = fmax(v, dpp_move<0x118>(v));  // row_shr:8
    v = fmax(v, dpp_move<0x142>(v));  // row_bcast:15
    v = fmax(v, dpp_move<0x143>(v));  // row_bcast:31
    return v;
}
// The block's maxima of two non-negative values into a slot of each set.
template <class A, class B>
__device__ __forceinline__ void block_max_to_slots(A a, B b, unsigned long long* __restrict__ slots_a,
                                                   unsigned long long* __restrict__ slots_b, uint32_t blk) {
    __shared__ double s_a[kBlock / kWave], s_b[kBlock / kWave];
    a = wave_max_lane63(a);
    if (slots_b) b = wave_max_lane63(b);
    if (__lane_id() == kWave - 1) {
        s_a[threadIdx.x / kWave] = (double)a;
        s_b[threadIdx.x / kWave] = (double)b;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const double* w = threadIdx.x ? s_b : s_a;
        double m = w[0];
        for (int k = 1; k < kBlock / kWave; ++k) m = fmax(m, w[k]);
        unsigned long long* slots = threadIdx.x ? slots_b : slots_a;
        if (slots && m > 0.0)
            atomicMax(&slots[(blk % kSlots) * kSlotStride], (unsigned long long)__double_as_longlong(m));
    }
}

constexpr uint32_t kCtrlFlagWord = offsetof(Ctrl, nbr_overflow) / 8;
static_assert(offsetof(Ctrl, nbr_overflow) % 8 == 0 && offsetof(Ctrl, dt_new) % 8 == 0 &&
                  offsetof(Ctrl, pending) % 8 == 0 && offsetof(Ctrl, halted) == offsetof(Ctrl, pending) + 4 &&
                  offsetof(Ctrl, status) % 8 == 0,
              "publish_ctrl's words");

// The largest displacement of the step that `next` holds, the slots holding
// squares (of two sets both are loaded, so that the loads do not wait for the
// step index).
__device__ __forceinline__ double list_dmax(const StepParams& P, const Ctrl* next, const unsigned long long* dslots) {
    if (P.dset_mask == 3) return sqrt(slots_max(dslots + (uint32_t)(next->step & 3) * kSlotSet));
    const double even = slots_max(dslots), odd = slots_max(dslots + kSlotSet);
    return sqrt((next->step & 1) ? odd : even);
}

// The prologue of a list step (build: of a build step) in one block: the
// commit of the step that `next` holds, the staleness test of the lists (a
// list step also halts when no build has run since the last sort, e.g. a
// build launched while the run was stopped), the snapshot into `cur`.
// fused: of a step of one kernel (pair_list_kernel, FUSED with CONT), which
// publishes its outcome here: dt is known, and `next` gets all but the flags,
// which stay in `flags`.
__device__ __forceinline__ void list_block_prologue(const StepParams& P, const Ctrl* next, Ctrl* cur,
                                                    const Ctrl* flags, double dmax, bool build, bool fused) {
    const unsigned long long word = ctrl_word(next);
    uint32_t valid = 0;
    bool was_halted = false;
    block_prologue(
        P, cur, word,
        [&](Ctrl& c) {
            was_halted = c.halted != 0;
            if (fused) {
#pragma unroll
                for (int k = 0; k < 4; ++k) c.outside_l[k] = flags->outside_l[k];
            }
            if (!c.halted && c.pending) {  // the step being committed moved no particle further than dmax
                c.disp_acc += dmax;
                c.disp_last = dmax;
            }
            valid = c.list_valid;
            // a list step whose predecessor overflowed does not get here (its
            // integrator halted); other blocks of this kernel may be raising
            // the flag for this step already
            if (!build) c.nbr_overflow = 0;
        },
        [&](Ctrl& c) {
            c.halt_now = c.halted && !was_halted;
            if (c.halted) return;
            c.list_valid = build ? 1u : valid;
            if (build) {
                c.disp_acc = 0.0;
            } else if (!valid || !(c.disp_acc < P.skin_half)) {
                c.halted = 1;
                c.status = kStatusRebuild;
                c.halt_now = 1;
                if (c.wall_disappear) c.nwm_done = 0;  // the re-run prologue fires it again
            } else if (fused && P.consistency_check && flags->list_long) {
                c.halted = 1;
                c.status = kStatusUnfused;
                c.halt_now = 1;
            } else if (fused) {
                c.dt_new = c.cur_dt_const;
                c.pending = 1;
            }
        },
        fused ? kCtrlFlagWord : kCtrlWords);
}

// Whether list_block_prologue (not a build) halts, from the same fields
// (none of which the blocks of this kernel write).
__device__ __forceinline__ bool list_step_halts(const StepParams& P, const Ctrl& N, uint32_t outside, double dmax) {
    if (N.halted) return true;
    double t = N.time, disp = N.disp_acc;
    if (N.pending) {
        if (P.consistency_check && outside > 0 && P.consistency_treatment == 1) return true;
        t += N.dt_new;
        disp += dmax;
    }
    return t > N.t_end || !N.list_valid || !(disp < P.skin_half);
}

// The index of the step that a kernel starting from `next` runs, in scalar registers.
__device__ __forceinline__ unsigned long long list_step_index(const Ctrl* next) {
    const unsigned long long k = next->step + (next->pending ? 1 : 0);
    return (unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)k) |
           ((unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(k >> 32)) << 32);
}

// At the head of a list step's first kernel (every thread of the block):
// false when the step halts, else its step index in `step`.
__device__ __forceinline__ bool list_step_begin(const StepParams& P, Ctrl* next, Ctrl* cur,
                                                unsigned long long* dslots, unsigned long long& step) {
    const double dmax = list_dmax(P, next, dslots);
    step = list_step_index(next);
    const bool halts = list_step_halts(P, *next, ctrl_outside(*next), dmax);
    if (blockIdx.x == 0) {
        list_block_prologue(P, next, cur, next, dmax, false, false);
        if (!halts) {  // this step's sets, and of four the next one's; the blocks of this kernel read neither
            clear_slots(dslots + (uint32_t)(step & P.dset_mask) * kSlotSet);
            if (P.dset_mask == 3) clear_slots(dslots + (uint32_t)((step + 1) & 3) * kSlotSet);
            if (threadIdx.x < 2) next->outside_l[(step + threadIdx.x) & 3] = 0;
        }
    }
    return !halts;
}

// Fused steps (dt constant, no wave maker): the pair pass integrates too.
// It writes the next step's records to a second array, so that its other
// blocks still read this step's, and (FP32, whose near cut-off tests read
// the neighbours' FP64 positions) the positions to the other of two arrays.
// Steps go in pairs, back and forth, so that a pair leaves everything where
// the other kernels expect it; when the second of a pair halts, it puts the
// positions back instead.  Where the pair pass is the step's only kernel
// (continuity), the step also reads the control block in one place and
// publishes in another, for the same reason, and clears the next step's
// displacement set (of four) while its blocks fill their own; more entries
// than max_neighbours - 1 in some list halt it (kStatusUnfused): the step
// could not be undone if a particle had more neighbours.
//
// At the head of a fused continuity step (every thread): false when it halts.
__device__ __forceinline__ bool fused_step_begin(const StepParams& P, const Ctrl* in, Ctrl* out, Ctrl* flags,
                                                 unsigned long long* dslots, unsigned long long& step) {
    const double dmax = list_dmax(P, in, dslots);
    step = list_step_index(in);
    uint32_t outside = flags->outside_l[0];
#pragma unroll
    for (uint32_t k = 1; k < 4; ++k) outside = (in->step & 3) == k ? flags->outside_l[k] : outside;
    const bool halts = list_step_halts(P, *in, outside, dmax) || (P.consistency_check && flags->list_long);
    if (blockIdx.x == 0) {
        list_block_prologue(P, in, out, flags, dmax, false, true);
        if (!halts) {
            clear_slots(dslots + (uint32_t)((step + 1) & 3) * kSlotSet);
            if (threadIdx.x == 0) flags->outside_l[(step + 1) & 3] = 0;
        }
    }
    return !halts;
}

// The prologue of a build step (one block of kBlock threads): it also
// clears every reduction slot and the flags of the build.
__global__ void __launch_bounds__(kBlock) list_prologue(StepParams P, Ctrl* __restrict__ next, Ctrl* __restrict__ cur,
                                                        unsigned long long* __restrict__ dslots,
                                                        unsigned long long* __restrict__ maxslots) {
    const double dmax = list_dmax(P, next, dslots);
    list_block_prologue(P, next, cur, next, dmax, true, false);
    // (also when the step halts: the step after a halt is a build and reads none of them)
    for (uint32_t k = 0; k <= P.dset_mask; ++k) clear_slots(dslots + k * kSlotSet);
    for (uint32_t k = 0; k < 2; ++k) {
        clear_slots(maxslots + k * kDtSet);
        clear_slots(maxslots + k * kDtSet + kSlotSet);
    }
    if (threadIdx.x == 0) {
        for (int k = 0; k < 4; ++k) next->outside_l[k] = 0;
        next->list_overflow = 0;
        next->list_long = 0;
    }
}

// At the head of a later kernel of a list or build step: false when the
// step halted.
__device__ __forceinline__ bool list_step_goes(const Ctrl* cur) { return !cur->halted; }

// A build that found more entries for some particle than its list holds:
// the step halts before its pair pass and runs without lists.
__device__ __forceinline__ bool list_build_overflowed(const Ctrl* next, Ctrl* cur) {
    if (!next->list_overflow) return false;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        cur->halted = 1;
        cur->status = kStatusListOverflow;
    }
    return true;
}

// The summation density of step `step` is renormalised (as prologue_commit
// decides it).
__device__ __forceinline__ bool step_renorm(const StepParams& P, unsigned long long step) {
    return P.renorm && (step + 1) % P.renorm_every == 0;
}

// The integrator's block 0: `next` becomes `cur` with the step's outcome
// (dt: committed by the next step's prologue), or with the halt `status`.
__device__ __forceinline__ void publish_ctrl(const Ctrl* cur, Ctrl* next, double dt, uint32_t halt_status) {
    if (threadIdx.x >= kCtrlFlagWord) return;
    unsigned long long w = reinterpret_cast<const unsigned long long*>(cur)[threadIdx.x];
    if (!cur->halted) {
        if (threadIdx.x == offsetof(Ctrl, dt_new) / 8 && halt_status == 0)
            w = (unsigned long long)__double_as_longlong(dt);
        if (threadIdx.x == offsetof(Ctrl, pending) / 8) w = halt_status ? (1ull << 32) : 1ull;  // pending | halted << 32
        if (threadIdx.x == offsetof(Ctrl, status) / 8 && halt_status) w = (w & ~0xffffffffull) | halt_status;
    }
    reinterpret_cast<unsigned long long*>(next)[threadIdx.x] = w;
}

// Cell index (clamped to the grid) of coordinate r.
__device__ __forceinline__ int clamped_cell(double r, double rmin, double cell, int ncell) {
    const double t = floor((r - rmin) / cell);
    return t < 0.0 ? 0 : (t >= (double)ncell ? ncell - 1 : (int)t);
}

// ------------------------------------------------------------------ list builds
// A wave of the build walks the union of its lanes' columns of cells; a
// lane has one range of slots per column (none if the column is out of its
// reach).  The candidates of the union of the ranges are staged in LDS, from
// coalesced loads: each lane loading its own took an access per lane group
// and kept the vector L1 as busy as the arithmetic did the vector units (681
// thousand accesses per CU in 699 thousand busy cycles, 3D, 555,686
// particles).  Tests run in FP32 on positions relative to the column, 32
// candidates into a bit mask (the sign of |r|^2 - reach^2 shifted in); then each lane takes the hits off its mask.  Their entries go to
// the lane's column of an LDS buffer first; when a lane's column might
// overflow, the wave writes the buffered rows out together, so that the
// stores of a row are contiguous (written straight from the walk, they left
// lines partly written in L2).  3D 455 -> 339 us at 555,686 particles, 2020 ->
// 1593 at 2,899,370; 2D 113 -> 90 at 1,020,263, 22 -> 17 at 22,662.  Vector
// instructions, about 7 per candidate and 10 per entry, take 43 of 93 us in 2D at
// 1,020,263 particles and 1.86 of 3.15 ms in 3D at 6,595,366.
//
// The FP32 reach exceeds list_reach by build_margin (relative, of the square),
// above the rounding of positions `cells` cells from the wave's reference (half
// an ulp of each of two, cells 2^-24 of a cell together, twice that in the
// square): the lists hold every pair within list_reach and a few just beyond,
// which every list step tests again.
constexpr uint32_t kBuildStage = 96, kBuildTest = 32, kBuildRows = 32;
__device__ __forceinline__ double build_margin(int cells) { return 1e-4 + 2.5e-7 * cells; }
struct BuildLds {                             // of a wave; four blocks fill a CU's LDS
    float4 cand[kBuildStage + kBuildTest];    // position, entry word
    uint32_t rows[kBuildRows * kWave];
};
__device__ __forceinline__ uint32_t wave_of_block() {  // in a scalar register
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
}
// The wave's maximum, every lane active.
template <int CTRL> __device__ __forceinline__ uint32_t dpp_move_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t full_wave_max(uint32_t v) {
    v = max(v, dpp_move_u32<0x111>(v));  // row_shr:1 (lanes without a source get 0)
    v = max(v, dpp_move_u32<0x112>(v));  // row_shr:2
    v = max(v, dpp_move_u32<0x114>(v));  // row_shr:4
    v = max(v, dpp_move_u32<0x118>(v));  // row_shr:8
    v = max(v, dpp_move_u32<0x142>(v));  // row_bcast:15
    v = max(v, dpp_move_u32<0x143>(v));  // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane((int)v, kWave - 1);
}
__device__ __forceinline__ int full_wave_min_i32(int v) { return (int)~(full_wave_max(~((uint32_t)v ^ 0x80000000u)) ^ 0x80000000u); }
__device__ __forceinline__ int full_wave_max_i32(int v) { return (int)(full_wave_max((uint32_t)v ^ 0x80000000u) ^ 0x80000000u); }

// The first and last of n cells per axis within reach of a particle at
// `o` from the origin of its home cell h (reach a little widened for the
// rounding here).
__device__ __forceinline__ int reach_first(float o, float reach, float inv_cell, int h) {
    return max(0, h + (int)floorf((o - reach) * inv_cell));
}
__device__ __forceinline__ int reach_last(float o, float reach, float inv_cell, int h, int n) {
    return min(n - 1, h + (int)floorf((o + reach) * inv_cell));
}

struct ListBuilder {
    BuildLds& lds;
    uint32_t* nbl;
    uint32_t* my;  // this lane's column of the buffered rows
    uint32_t n, cap, s, cnt = 0, nh = 0;
    __device__ ListBuilder(const StepParams& P, BuildLds& l, uint32_t* lists, uint32_t slot)
        : lds(l), nbl(lists), my(l.rows + __lane_id()), n(P.n), cap(P.list_cap), s(slot) {}
    __device__ __forceinline__ void flush() {
        const uint32_t rows = cnt < cap ? min(nh, cap - cnt) : 0u;
        uint32_t* out = nbl + (size_t)cnt * n + s;
#pragma unroll 1
        for (uint32_t r = 0; r < rows; ++r, out += n) *out = my[r * kWave];
        cnt += nh;
        nh = 0;
    }
    // One column (every lane of the wave calls it): the candidates b .. e - 1 of
    // the lanes that need it against the lane's position (px, py, pz) in the
    // column's frame; an entry is the candidate's word + add.  load(i): the
    // candidate in that frame and its word.
    template <bool Z, class Load>
    __device__ __forceinline__ void column(bool need, uint32_t b, uint32_t e, float px, float py, float pz, float r2,
                                           uint32_t add, Load&& load) {
        const uint32_t lane = __lane_id();
        const uint32_t end = full_wave_max(need ? e : 0u), first = ~full_wave_max(need ? ~b : 0u);
#pragma unroll 1
        for (uint32_t t0 = first; t0 < end; t0 += kBuildStage) {
            __builtin_amdgcn_wave_barrier();  // the last stage's reads are issued
#pragma unroll
            for (uint32_t j = 0; j < kBuildStage; j += kWave)
                if (j + lane < kBuildStage && t0 + j + lane < end) lds.cand[j + lane] = load(t0 + j + lane);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const uint32_t i0 = max(b, t0), i1 = min(e, t0 + kBuildStage);
            const uint32_t len = need && i1 > i0 ? i1 - i0 : 0u, lmax = full_wave_max(len);
#pragma unroll 1
            for (uint32_t i = 0; i < lmax; i += kBuildTest) {
                const uint32_t at = i < len ? i0 - t0 + i : 0u;  // (past its range a lane tests the stage's first)
                const float4* c = lds.cand + at;
                uint32_t m = 0;  // candidate at + u in bit 31 - u
#pragma unroll
                for (uint32_t h = 0; h < kBuildTest; h += 8) {
                    if (i + h >= lmax) {
                        m <<= 8;
                        continue;
                    }
#pragma unroll
                    for (uint32_t u = 0; u < 8; ++u) {
                        const float dx = c[h + u].x - px, dy = c[h + u].y - py;
                        float d = fmaf(dy, dy, -r2);  // |r_i - r_j|^2 - r2, negative for a hit
                        if constexpr (Z) {
                            const float dz = c[h + u].z - pz;
                            d = fmaf(dz, dz, d);
                        }
                        d = fmaf(dx, dx, d);
                        m = __builtin_amdgcn_alignbit(m, __float_as_uint(d), 31);  // m << 1 | sign
                    }
                }
                const uint32_t valid = i < len ? len - i : 0u, self = s - (i0 + i);
                if (valid < kBuildTest) m &= ~(0xffffffffu >> valid);
                if (self < kBuildTest) m &= ~(0x80000000u >> self);
                const uint32_t hits = (uint32_t)__popc(m);
                if (__any(nh + hits > kBuildRows)) flush();  // wave-uniform
                uint32_t* out = my + nh * kWave;
#pragma unroll 1
                while (m) {
                    const uint32_t u = (uint32_t)__clz((int)m);
                    m ^= 0x80000000u >> u;
                    *out = __float_as_uint(c[u].w) + add;
                    out += kWave;
                }
                nh += hits;
            }
        }
    }
};

// The lists of a build step, on the reordered copy (pos, va) with its
// cell-start table LB: for each live particle, every live particle i != s
// within list_reach, in the order of the cell walk (columns, then rows
// within a column).  The cells visited are those within list_reach of the
// particle (3 or 4 per axis, the reach being under two cells).
template <class R>
__global__ void __launch_bounds__(kBlock) list_build_kernel(StepParams P, Ctrl* __restrict__ next,
                                                            const Ctrl* __restrict__ cur,
                                                            const double2* __restrict__ pos,
                                                            const real4<R>* __restrict__ va,
                                                            const uint32_t* __restrict__ skey,
                                                            const uint32_t* __restrict__ LB, uint32_t* __restrict__ nbl,
                                                            uint32_t* __restrict__ nbc) {
    __shared__ BuildLds s_build[kBlock / kWave];
    if (cur->halted) return;
    const uint32_t lb = xcd_block(P.blocks_per_xcd);
    if (lb >= P.nblocks) return;
    const uint32_t s0 = lb * kBlock + threadIdx.x;
    const bool inb = s0 < P.n;
    const uint32_t s = inb ? s0 : P.n - 1;
    const bool alive = inb && (int)va[s].w != 0;
    const double2 pj = pos[s];
    const uint32_t kj = skey[s];
    const int hx = (int)(kj / (uint32_t)P.ncy), hy = (int)kj - hx * P.ncy;
    // the list pass takes the FP32 positions relative to the home cell
    // for within 2.1 cells of its origin: a particle outside the cell
    // grid (keyed to the nearest edge cell) runs the step without lists
    const double ox = pj.x - (P.xmin + hx * P.cell), oy = pj.y - (P.ymin + hy * P.cell);
    bool bad = alive && !(ox > -P.cell && ox < 2.0 * P.cell && oy > -P.cell && oy < 2.0 * P.cell);
    const float reach = (float)(P.list_reach * (1.0 + 1e-5)), inv_cell = (float)(1.0 / P.cell);
    int x0 = 0, x1 = -1, y0 = 0, y1 = 0;  // (no column for lanes with nothing to list)
    if (alive && !bad) {
        x0 = reach_first((float)ox, reach, inv_cell, hx);
        x1 = reach_last((float)ox, reach, inv_cell, hx, P.ncx);
        y0 = reach_first((float)oy, reach, inv_cell, hy);
        y1 = reach_last((float)oy, reach, inv_cell, hy, P.ncy);
        bad |= x0 < hx - 2 || x1 > hx + 2 || y0 < hy - 2 || y1 > hy + 2;
    }
    ListBuilder out(P, s_build[wave_of_block()], nbl, s);
    const int wx0 = full_wave_min_i32(x0 <= x1 ? x0 : INT_MAX), wx1 = full_wave_max_i32(x1);
    const double yref = P.ymin + (double)__builtin_amdgcn_readfirstlane(hy) * P.cell;
    const float py = (float)(pj.y - yref), r2 = (float)(P.list_r2 * (1.0 + build_margin(P.ncy)));
#pragma unroll 1
    for (int col = wx0; col <= wx1; ++col) {
        const bool need = col >= x0 && col <= x1;
        if (!__any(need)) continue;
        const uint32_t col0 = (uint32_t)(col * P.ncy);
        const uint32_t b = need ? LB[col0 + y0] : 0u, e = need ? LB[col0 + y1 + 1] : 0u;
        const double xref = P.xmin + col * P.cell;
        // the slot, the row of the candidate's home cell (its key's) in the
        // word; the offsets from the lane's home cell complete the code
        const uint32_t add = ((uint32_t)(col - hx + 3) << kSlotBits) + ((uint32_t)(3 - hy) << (kSlotBits + 3));
        out.column<false>(need, b, e, (float)(pj.x - xref), py, 0.f, r2, add, [&](uint32_t i) {
            const double2 q = pos[i];
            return make_float4((float)(q.x - xref), (float)(q.y - yref), 0.f,
                               __uint_as_float(i + ((skey[i] - col0) << (kSlotBits + 3))));
        });
    }
    out.flush();
    if (out.cnt > P.list_cap || bad) atomicOr(&next->list_overflow, 1u);
    if (out.cnt > P.max_nbr - 1) atomicOr(&next->list_long, 1u);
    if (inb) nbc[s] = min(out.cnt, P.list_cap);
}

// One list entry as the pair pass sees it.
template <class R> struct ListEntry {
    bool take;        // a neighbour: within the cut-off, alive, among the first `cap`
    R dx, dy;         // r_i - r_j
    real4<R> nr;      // near record of i: (xi or x, xi or y, vx, vy)
    real4<R> pr;      // pred record of i: (v^x, v^y, s rho^, p / rho^2)
};

// r_i - r_j of an entry and whether it is within the cut-off.  FP32: from
// the near records and the offset of the two home cells (a table in LDS
// indexed by the entry's code), the reference's FP64 test on the FP64
// positions only inside the band around the cut-off.  The build guarantees
// that every listed position lies within a cell of its home cell, and the
// lists go stale before any particle moves half the skin, so xi stays below
// 2.1 cells and its rounding far inside the band.  FP64: the reference's test
// on the FP64 positions of the near records.
struct CutFP32 {
    float lo, hi;
};
__device__ __forceinline__ CutFP32 cut_band(const StepParams& P) {
    CutFP32 C;
    C.lo = (float)(P.cut2 * (1.0 - 1e-5));
    C.hi = (float)(P.cut2 * (1.0 + 1e-5));
    return C;
}
__device__ __forceinline__ bool list_cut(const StepParams& P, const CutFP32& C, const float2* s_off, uint32_t e,
                                         const float4& ni, const float4& nj, uint32_t s,
                                         const double2* __restrict__ pos, float& dx, float& dy) {
    const float2 o = s_off[e >> kSlotBits];
    dx = (ni.x - nj.x) + o.x;
    dy = (ni.y - nj.y) + o.y;
    const float d2 = dx * dx + dy * dy;
    if (!(d2 > C.lo && d2 < C.hi)) return d2 <= C.lo;  // on the band's edge: within a rounding of lo < cut2
    const double2 q = pos[e & kSlotMask], pj = pos[s];  // rare: the band around the cut-off
    const double ddx = __dsub_rn(q.x, pj.x), ddy = __dsub_rn(q.y, pj.y);
    dx = (float)ddx;
    dy = (float)ddy;
    return dist2_exact(ddx, ddy) < P.cut2;
}
__device__ __forceinline__ bool list_cut(const StepParams& P, const CutFP32&, const float2*, uint32_t,
                                         const double4& ni, const double4& nj, uint32_t, const double2* __restrict__,
                                         double& dx, double& dy) {
    dx = __dsub_rn(ni.x, nj.x);
    dy = __dsub_rn(ni.y, nj.y);
    return dist2_exact(dx, dy) < P.cut2;
}

// The table of home-cell offsets of the entry codes, code = (dcx + 3) |
// (dcy + 3) << 3 -> (dcx cell, dcy cell) rounded to FP32, filled by the
// first 64 threads of the block (a barrier must follow).
__device__ __forceinline__ void fill_cell_offsets(const StepParams& P, float2* s_off) {
    if (threadIdx.x < 64) {
        const int c = (int)threadIdx.x;
        s_off[c] = make_float2((float)(((c & 7) - 3) * P.cell), (float)(((c >> 3) - 3) * P.cell));
    }
}

// Entry k of slot s's list: the lists hold list_cap + kListPad rows, zero
// where no build wrote (so the loads of the entries after a list's last one
// stay in bounds and name valid slots), and the byte offsets fit 32 bits.
constexpr uint32_t kListPad = 8;
__device__ __forceinline__ uint32_t list_entry(const uint32_t* __restrict__ nbl, uint32_t byte_off) {
    return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(nbl) + byte_off);
}

// LPP lanes of a wave share a particle's list in the 2D passes: lane l takes
// the entries l, l + LPP, ..., and the partial sums are added across the
// lanes (lane_sum).  The lanes of one l are consecutive, so that a row of the
// lists is still read in runs of 64 / LPP entries.  A pass is bound by the
// latency of its dependent loads (entry, then record), so with few particles
// it is the number of rounds per lane that counts, and the lanes that fill
// the chip are free; with many, the extra lanes only repeat the work per
// particle.
template <int LPP> struct LaneGroup {
    static constexpr uint32_t kParticles = kWave / LPP;  // of a wave
    uint32_t l, s;                                       // this lane's share of the list, and its particle
    __device__ explicit LaneGroup(uint32_t lb)
        : l(__lane_id() / kParticles),
          s((lb * (kBlock / kWave) + threadIdx.x / kWave) * kParticles + __lane_id() % kParticles) {}
};
template <int LPP> __host__ __device__ inline uint32_t group_blocks(uint32_t n) {
    return (n + kBlock / LPP - 1) / (kBlock / LPP);
}
template <int LPP> __host__ __device__ inline uint32_t group_blocks_per_xcd(uint32_t n) {
    return (group_blocks<LPP>(n) + kNumXcd - 1) / kNumXcd;
}
template <int LPP, class R> __device__ __forceinline__ R lane_sum(R v) {
#pragma unroll
    for (int off = kWave / LPP; off < kWave; off <<= 1) v += __shfl_xor(v, off);
    return v;
}
template <int LPP, class R> __device__ __forceinline__ R lane_max(R v) {
#pragma unroll
    for (int off = kWave / LPP; off < kWave; off <<= 1) v = fmax(v, __shfl_xor(v, off));
    return v;
}

// Of the hits of one row of LPP entries of a particle (this lane's: hit),
// whether this lane's is among the first `cap` of the list, hits counting
// those of the rows before; every lane of the particle calls it.
template <int LPP>
__device__ __forceinline__ bool take_capped(bool hit, uint32_t l, uint32_t cap, uint32_t& hits, bool& over) {
    uint32_t before = hits;
    if (LPP == 1) {
        hits += hit ? 1u : 0u;
    } else {
#pragma unroll
        for (int q = 0; q < LPP; ++q) {
            const uint32_t h = (uint32_t)__shfl((int)hit, q * (kWave / LPP) + (int)(__lane_id() % (kWave / LPP)));
            before += q < (int)l ? h : 0u;
            hits += h;
        }
    }
    const bool take = hit & (before < cap);
    over |= hit & !take;
    return take;
}

// The entries of slot s's list, a row of LPP entries at a time: entry k + l
// for k a multiple of LPP, the row's offset in a scalar register (so that an
// entry costs no vector instruction but its load).  Rows past a list's end
// name valid slots (padding rows, or entries of an earlier build); the loads
// past the last allocated row read the last one instead.
template <int LPP> struct ListRows {
    __amdgpu_buffer_rsrc_t lists;
    uint32_t row, last, col;  // bytes of a row; the last row to start from; this lane's byte offset in one
    __device__ ListRows(const StepParams& P, const uint32_t* nbl, uint32_t s, uint32_t l)
        : lists(__builtin_amdgcn_make_buffer_rsrc((void*)nbl, 0, (int)((P.list_cap + kListPad) * P.n * 4u), 0x00027000)),
          row(P.n * 4u),
          last(P.list_cap + kListPad - LPP),
          col((l * P.n + min(s, P.n - 1)) * 4u) {}
    __device__ __forceinline__ uint32_t operator()(uint32_t k) const {
        return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(lists, (int)col, (int)(min(k, last) * row), 0);
    }
};

// Entries of slot s's list in rounds of G per lane: per round
// body(k, e, load) - k the list index of the lane's first entry, its entries
// k, k + LPP, ... in e; load fetches the next round's.
template <int LPP, uint32_t G, class Rows, class B>
__device__ __forceinline__ void list_rounds(const Rows& rows, uint32_t l, uint32_t cnt, B&& body) {
    uint32_t k = 0, e[G];
    auto load = [&](uint32_t (&e)[G]) {
#pragma unroll
        for (uint32_t u = 0; u < G; ++u) e[u] = rows(k + (G + u) * LPP);
    };
#pragma unroll
    for (uint32_t u = 0; u < G; ++u) e[u] = rows(u * LPP);
#pragma unroll 1
    for (; k < cnt; k += G * LPP) body(k + l, e, load);
}

// ------------------------------------------------------------------ wave gathers
// FP64 records fetched by the lanes of a wave together.  A lane that loads
// its own record of W 16-byte words takes W instructions, each with a
// cache-line access per lane or nearly (45 for 64 lanes, neighbouring lanes'
// neighbours lying close), and those accesses bound the plain passes, not
// bytes or arithmetic.  Here W consecutive lanes load the words of one
// record, the first instruction those of their first lane's, and so on, so
// that an instruction touches 64 / W records, each once.  The loads go
// straight to LDS (16 bytes per lane in lane order) and each lane reads its
// own record there.  Record t is lane t % W's of its W lanes: instruction
// t % W put its words at lanes t - t % W on, word p in place p ^ (t % W), so
// that lanes read from different banks.
template <uint32_t W, uint32_t STRIDE, uint32_t MASK> struct WaveGather {
    static_assert(W == 2 || W == 4, "words of a gathered record");
    static constexpr uint32_t kW = W;
    const char* records;
    uint4* buf;        // of the wave: W * 64 words per record in flight
    uint32_t part[W];  // byte offset of the word that this lane loads in the q-th instruction
    __device__ WaveGather(const void* rec, uint4* wave_buf) : records((const char*)rec), buf(wave_buf) {
#pragma unroll
        for (uint32_t q = 0; q < W; ++q) part[q] = ((__lane_id() % W) ^ q) * 16u;
    }
    // the value of the q-th of this lane's W lanes
    template <uint32_t q> __device__ __forceinline__ static uint32_t of_lane(uint32_t v) {
        constexpr int perm = W == 4 ? q * 0x55 : (q == 0 ? 0xa0 : 0xf5);  // quad_perm [q,q,q,q] or [q,q,q+2,q+2]
        return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, perm, 0xf, 0xf, true);
    }
    template <uint32_t q> __device__ __forceinline__ void fetch_one(uint32_t u, uint32_t off) const {
        using Global = const __attribute__((address_space(1))) void*;
        using Lds = __attribute__((address_space(3))) void*;
        __builtin_amdgcn_global_load_lds((Global)(records + (of_lane<q>(off) | part[q])),
                                         (Lds)(buf + (u * W + q) * kWave), 16, 0, 0);
        if constexpr (q + 1 < W) fetch_one<q + 1>(u, off);
    }
    // starts the loads of the records that the lanes' entries e name, the u-th in flight
    __device__ __forceinline__ void fetch(uint32_t u, uint32_t e) const { fetch_one<0>(u, (e & MASK) * STRIDE); }
    __device__ __forceinline__ void read(uint32_t u, uint4* w) const {
        const uint32_t t = __lane_id(), q = t % W;
#pragma unroll
        for (uint32_t p = 0; p < W; ++p) w[p] = buf[(u * W + q) * kWave + t - q + (p ^ q)];
    }
};
// Records of two arrays under one entry.
template <class A, class B> struct WaveGatherBoth {
    static constexpr uint32_t kW = A::kW + B::kW;
    A a;
    B b;
    __device__ __forceinline__ void fetch(uint32_t u, uint32_t e) const {
        a.fetch(u, e);
        b.fetch(u, e);
    }
    __device__ __forceinline__ void read(uint32_t u, uint4* w) const {
        a.read(u, w);
        b.read(u, w + A::kW);
    }
};
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0f70); }  // vmcnt(0)
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }    // lgkmcnt(0)

// list_rounds with the records gathered by the wave (every lane calls it;
// cnt 0: no entries): body(k, e, w) - k the list index of the lane's first
// entry of the round, e the entries, w the words of their records.  The next
// round's records are on their way while body works on this one's, which are
// in registers by then.
template <int LPP, uint32_t G, class S_, class B>
__device__ __forceinline__ void gather_rounds(const StepParams& P, const uint32_t* __restrict__ nbl, const S_& src,
                                              uint32_t s, uint32_t l, uint32_t cnt, B&& body) {
    const uint32_t cmax = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_max_u32(cnt));
    if (cmax == 0) return;
    const ListRows<LPP> rows(P, nbl, s, l);
    uint32_t e[G], en[G];
    auto load = [&](uint32_t k) {
#pragma unroll
        for (uint32_t u = 0; u < G; ++u) en[u] = rows(k + u * LPP);
    };
    auto fetch = [&]() {
#pragma unroll
        for (uint32_t u = 0; u < G; ++u) {
            e[u] = en[u];
            src.fetch(u, e[u]);
        }
    };
    load(0);
    fetch();
    load(G * LPP);
#pragma unroll 1
    for (uint32_t k = 0; k < cmax; k += G * LPP) {
        uint4 w[G][S_::kW];
        uint32_t ec[G];
        wait_loads();
#pragma unroll
        for (uint32_t u = 0; u < G; ++u) {
            src.read(u, w[u]);
            ec[u] = e[u];
        }
        wait_lds();  // the records are in registers: the next ones may land
        __builtin_amdgcn_sched_barrier(0);
        if (k + G * LPP < cmax) {
            fetch();
            load(k + 2 * G * LPP);
        }
        body(k + l, ec, w);
    }
}
__device__ __forceinline__ float4 record_real4(const uint4* w, float) {
    return make_float4(__uint_as_float(w[0].x), __uint_as_float(w[0].y), __uint_as_float(w[0].z),
                       __uint_as_float(w[0].w));
}
__device__ __forceinline__ double4 record_real4(const uint4* w, double) {
    auto d = [](uint32_t lo, uint32_t hi) { return __hiloint2double((int)hi, (int)lo); };
    return make_double4(d(w[0].x, w[0].y), d(w[0].z, w[0].w), d(w[1].x, w[1].y), d(w[1].z, w[1].w));
}
// Records in flight per lane of the 2D FP64 pass: 1,020,263 particles, 105 us
// per pass with 2 (119 with 3; 127 when each lane gathered its own).
constexpr uint32_t kGather2 = 2;

// Visits the entries of slot s's list: f(ListEntry) for every entry (f must
// add nothing when take is false: every entry runs the same instructions,
// most entries being neighbours).  kCap: count the neighbours, and entries
// beyond the first `cap` set `overflow` (GridFind.cpp:158-188); a wave
// whose lists are all no longer than cap cannot overflow and skips the
// count.  Entries go in groups of G: the group's records are gathered
// together and the next group's entries loaded behind them, so that no
// gathered value lives across iterations (the loop waits only on its own
// loads).  Larger groups keep more gathers in flight per wave but take
// registers: the pass is bound by load latency, and 2 entries per group
// (74 VGPRs, 6 waves per SIMD) gave the least time.
template <class R, bool kCap, int LPP, class F>
__device__ __forceinline__ void for_each_listed(const StepParams& P, const float2* s_off, uint32_t cap, uint32_t s,
                                                uint32_t l, const real4<R>& nj, const double2* __restrict__ pos,
                                                const ListRec<R>* __restrict__ rec, const uint32_t* __restrict__ nbl,
                                                uint32_t cnt, uint4* buf, bool& overflow, F&& f) {
    const CutFP32 C = cut_band(P);
    uint32_t hits = 0;
    bool over = false;
    auto entry = [&](uint32_t k, uint32_t e, const real4<R>& nr, const real4<R>& pr) {
        ListEntry<R> E;
        const bool in = list_cut(P, C, s_off, e, nr, nj, s, pos, E.dx, E.dy);
        const bool hit = in & (pr.z != R(0)) & (k < cnt);
        E.take = kCap ? take_capped<LPP>(hit, l, cap, hits, over) : hit;
        E.nr = nr;
        E.pr = pr;
        f(E);
    };
    if constexpr (sizeof(R) == 8) {
        constexpr uint32_t G = kGather2;
        gather_rounds<LPP, G>(P, nbl, WaveGather<4, 64, kSlotMask>(rec, buf), s, l, cnt,
                              [&](uint32_t k, const uint32_t (&e)[G], const auto& w) {
#pragma unroll
                                  for (uint32_t u = 0; u < G; ++u)
                                      entry(k + u * LPP, e[u], record_real4(w[u], R(0)), record_real4(w[u] + 2, R(0)));
                              });
    } else {
        constexpr uint32_t G = 2;  // measured at C1-1M FP32: 57.7 us per pass against 58.8 (3), 61.4 (4), 65.1 (1)
        list_rounds<LPP, G>(ListRows<LPP>(P, nbl, s, l), l, cnt, [&](uint32_t k, uint32_t (&e)[G], auto& load) {
            ListRec<R> r[G];
            uint32_t en[G];
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) r[u] = rec[e[u] & kSlotMask];
            load(en);
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) {
                entry(k + u * LPP, e[u], r[u].nr, r[u].pr);
                e[u] = en[u];
            }
        });
    }
    overflow |= over;
}

// The cubic configuration's pair terms (fast_pair_term) for list entries,
// 2D and 3D, arranged for instruction count, the largest share of the FP32
// passes' time (a wave of the 2D pass issues 1,557 VALU instructions, 40 of its
// 59 us at 1M particles):
//   * with t = h - |r| / 2 the outer piece is W = f / h^3 (4/3 t^3) and grad W
//     = diff (-2f / h^3) t^2 / |r|, the inner one with the same scales 2/3 h^3 -
//     |r|^2 t and t - |r| / 4; one comparison selects both, and the scales are
//     applied once per particle (lp_mF, lp_mW).  At most one operand of each
//     instruction is uniform: a second would take vector registers, which
//     spills in FP64.  (With u = h - |r| above 0 the inner piece is the
//     outer less multiples of u^2 and u^3, without the comparison; but the
//     difference loses the bits of close pairs: FP32 gradients off by up to
//     6.9e-6 of their value at q = 0.02 to 0.05 and 8.7e-7 at 0.2 to 0.4, 2e-7
//     here);
//   * an entry that is no neighbour gets |r| = 2 h, where both vanish;
//   * artificial viscosity from x = min(vr, 0) / (d^2 + eta^2), mu = h x:
//     the term is zero by itself where particles separate.
// CONT: continuity density; ALL: artificial viscosity, XSPH and the wall
// force are all on (else each by its switch).
template <class R, bool CONT, bool ALL> struct ListPair {
    static constexpr bool cont = CONT;
    R h, h2, h23, a2, b2, eta2, lj_r0, lj_D;
    bool lj_on, av_on, xsph_on;
    __device__ explicit ListPair(const StepParams& P)
        : h((R)P.h), h2((R)(2.0 * P.h)), h23((R)(2.0 / 3.0 * P.h * P.h * P.h)), a2((R)P.lp_a2),
          b2((R)P.lp_b2), eta2((R)P.av_eta2), lj_r0((R)P.lj_r0), lj_D((R)P.lj_D), lj_on(ALL || P.lj_on),
          av_on(ALL || P.av_on), xsph_on(ALL || P.xsph_on) {}
};
// What a pair gives, but for the direction: the gradient factor F (grad W =
// diff F lp_mF / m), the XSPH weight w of fluid neighbours (W / (rho_i +
// rho_j), to be scaled by lp_mW), the coefficient of the pressure and
// viscosity terms, and whether the wall force acts.
template <class R> struct ListTerm {
    R F, w, coef, rinv;
    bool wall;
};
// min(a, b) for b not NaN; the median takes no canonicalising instruction
__device__ __forceinline__ float running_min(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, -INFINITY); }
__device__ __forceinline__ double running_min(double a, double b) { return b < a ? b : a; }
// d2 = |diff|^2, vr = (v^_i - v^_j) . diff, zi and zj the typed densities, pw the sum
// of the p / rho^2; xmin collects the least x (mu = h x).
template <class R, class K_>
__device__ __forceinline__ ListTerm<R> list_pair(const K_& K, bool take, R d2, R vr, R zi, R zj, R pw, R& xmin) {
    ListTerm<R> T;
    T.rinv = fast_rsqrt<R>(d2 + (sizeof(R) == 4 ? R(1e-30f) : R(1e-200)));
    const R dist = take ? d2 * T.rinv : K.h2;
    const R t = fma(dist, R(-0.5), K.h), t2 = t * t;
    const bool inner = dist <= K.h;  // (then taken, and d2 = |r|^2)
    T.F = inner ? fma(dist, R(-0.25), t) : T.rinv * t2;
    const R inv_rs = fast_rcp<R>(fabs(zi) + fabs(zj));
    T.coef = pw;
    if (K.av_on) {
        const R x = take ? fmin(vr, R(0)) * fast_rcp<R>(d2 + K.eta2) : R(0);
        xmin = running_min(xmin, x);
        T.coef += (K.b2 * x - K.a2) * x * inv_rs;
    }
    const R w = inner ? fma(-d2, t, K.h23) : t2 * t * R(4.0 / 3.0);
    T.w = K.xsph_on && zi > R(0) ? w * inv_rs : R(0);
    T.wall = K.lj_on && take && zj > R(0) && zi < R(0) && dist < K.lj_r0;
    return T;
}
// The wall force's factor on diff (0 for coincident particles).
template <class R, class K_> __device__ __forceinline__ R list_wall(const K_& K, R d2, R rinv) {
    const R ri = d2 > R(0) ? rinv : R(0);
    const R rn = K.lj_r0 * ri;
    const R rn2 = rn * rn, rn4 = rn2 * rn2;
    return K.lj_D * (rn4 * rn4 * rn4 - rn4) * (ri * ri);
}

// One entry in 2D; nj, prj: the particle's own record.
template <class R> struct ListSums {
    R sx = 0, sy = 0, sd = 0, xx = 0, xy = 0, xmin = 0, ljx = 0, ljy = 0;
};
template <class R, class K_>
__device__ __forceinline__ void list_pair_term(const K_& K, ListSums<R>& S, const ListEntry<R>& E,
                                               const real4<R>& nj, const real4<R>& prj) {
    const R dx = E.dx, dy = E.dy, d2 = dx * dx + dy * dy;
    const R dvx = E.pr.x - prj.x, dvy = E.pr.y - prj.y;
    const ListTerm<R> T = list_pair<R>(K, E.take, d2, dvx * dx + dvy * dy, E.pr.z, prj.z, E.pr.w + prj.w, S.xmin);
    if (K.cont) S.sd += T.F * ((E.nr.z - nj.z) * dx + (E.nr.w - nj.w) * dy);
    const R fc = T.F * T.coef;
    S.sx += fc * dx;
    S.sy += fc * dy;
    S.xx += dvx * T.w;
    S.xy += dvy * T.w;
    if (T.wall) {
        const R f = list_wall<R>(K, d2, T.rinv);
        S.ljx -= dx * f;
        S.ljy -= dy * f;
    }
}

// The dt reductions of a pair pass: the block's largest a^2 and mu into the
// step's slots (the integrator takes the square root of the largest: the
// same value as the largest root).
template <class R>
__device__ __forceinline__ void list_dt_maxima(const StepParams& P, double a2, R mu,
                                               unsigned long long* __restrict__ slots, uint32_t lb) {
    if (P.dt_method == 2 && P.dt_dynamic_mode == 1) block_max_to_slots(a2, mu, slots, slots + kSlotSet, lb);
}

// The summed density of a particle that no longer exists, which has no
// neighbours: its own term, renormalised by itself (w0 = W(0)).  Its record holds
// 0 instead, the sign of its type, so that the integrator works it out again.
template <class R> __device__ __forceinline__ R dead_density(const StepParams& P, R w0, R rho_old, bool renorm) {
    const R m = (R)P.mass, rho = m * w0;
    return renorm ? rho / (m / rho_old * w0) : rho;
}
template <class R> __device__ __forceinline__ R density_w0(const StepParams& P) {
    return kernel_w<R>(kernel_consts<R>(P), P.skf_density, R(0));
}

// Summation density from the lists (Density.h:25-61): rho = m W(0) +
// sum m W_ij, p = EOS(rho), into the pred records (the forces use this rho)
// and the pressure array; renormalised on the steps that ask for it
// (ModelParams.tex:124-133, rho_i the density before the step).  Cubic
// spline.  Aliveness and the old densities come from va (pred is being
// rewritten by this pass).
template <class R, bool FIRST, int LPP>
__global__ void __launch_bounds__(kBlock) density_sum_list(StepParams P, Ctrl* next, Ctrl* cur, ListState<R> X,
                                                           ListRec<R>* __restrict__ rec, R* __restrict__ pres,
                                                           const uint32_t* __restrict__ nbl,
                                                           const uint32_t* __restrict__ nbc,
                                                           unsigned long long* __restrict__ dslots) {
    const uint32_t lb = xcd_block(group_blocks_per_xcd<LPP>(P.n));
    if (lb >= group_blocks<LPP>(P.n)) return;
    __shared__ float2 s_off[64];
    fill_cell_offsets(P, s_off);
    const LaneGroup<LPP> g(lb);
    const uint32_t s = g.s;
    const bool live = s < P.n;
    real4<R> vaj{}, nj{};
    uint32_t cnt = 0;
    if (live) {
        vaj = X.va[s];
        nj = rec[s].nr;
        cnt = nbc[s];
    }
    unsigned long long step;
    if constexpr (FIRST) {
        if (!list_step_begin(P, next, cur, dslots, step)) return;
    } else {
        if (!list_step_goes(cur)) return;
        step = cur->step;
    }
    __syncthreads();  // the offset table
    const KernelConsts<R> K = kernel_consts<R>(P);
    const R m = (R)P.mass;
    const R w0 = kernel_w<R>(K, P.skf_density, R(0));
    const bool renorm = step_renorm(P, step);
    R rho = R(0), wsum = R(0);
    bool overflow = false;
    if ((int)vaj.w == 0) cnt = 0;
    if (cnt) {
        const CutFP32 C = cut_band(P);
        const uint32_t cap = P.max_nbr - 1;
        constexpr uint32_t G = 2;
        const bool capped = __ballot(cnt > cap) != 0;  // some list of the wave may hold more than cap neighbours
        uint32_t hits = 0;
        list_rounds<LPP, G>(ListRows<LPP>(P, nbl, s, g.l), g.l, cnt, [&](uint32_t k, uint32_t (&e)[G], auto& load) {
            real4<R> ni[G], va[G];
            uint32_t en[G];
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) {
                ni[u] = rec[e[u] & kSlotMask].nr;
                va[u] = X.va[e[u] & kSlotMask];
            }
            load(en);
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) {
                R dx, dy;
                bool take = list_cut(P, C, s_off, e[u], ni[u], nj, s, X.pos, dx, dy) & ((int)va[u].w != 0) &
                            (k + u * LPP < cnt);
                if (capped) take = take_capped<LPP>(take, g.l, cap, hits, overflow);
                const R w = take ? kernel_w<R>(K, P.skf_density, pair_dist<R>(dx, dy, 0.0)) : R(0);
                rho += m * w;
                if (renorm && take) wsum += m / va[u].z * w;
            }
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) e[u] = en[u];
        });
    }
    if (overflow) atomicOr(&next->nbr_overflow, 1u);
    rho = m * w0 + lane_sum<LPP>(rho);
    if (renorm) rho = rho / (m / vaj.z * w0 + lane_sum<LPP>(wsum));
    if (!live || g.l != 0) return;
    real4<R> pr = rec[s].pr;
    const R p = eos_p<R>(rho, (R)P.rho0, (R)P.eos_B);
    pr.z = typed_rho<R>(rho, (int)vaj.w);
    pr.w = p / (rho * rho);
    rec[s].pr = pr;
    pres[s] = p;
}

// Where a 2D step leaves the state, the next step's records and keys, and
// the control block with the flags it raises.
template <class R> struct ListOut {
    double2* pos;
    real4<R>* va;
    ListRec<R>* rec;
    const uint32_t* home;
    uint32_t* key_next;
    Ctrl* flags;
    bool second;  // fused steps: the second of a pair
};
// whole_step of slot s, its cell key for the next build and the records of
// the next step's pair pass: near (the new position relative to the home
// cell, the new velocity) and pred (PredictHalfStep.cpp:16-22 with this
// step's dt, which is the next step's).  The square of its displacement.
template <class R>
__device__ __forceinline__ double step_listed(const StepParams& P, const Ctrl& c, uint32_t s, double2 p0,
                                              const real4<R>& va, const real4<R>& pr, uint32_t oid, uint32_t h,
                                              const real4<R>& d, const real2<R>& x, double dt, const ListOut<R>& O,
                                              uint32_t& outside, uint32_t& bad) {
    const Stepped2<R> o = whole_step_one<R>(P, c, p0, va, pr, oid, d.x, d.y, d.z, x.x, x.y, dt, outside);
    O.pos[s] = o.pos;
    O.va[s] = o.va;
    O.key_next[s] = (int)o.va.w == 0 ? P.ncells : cell_key(P, o.pos.x, o.pos.y, bad);
    R p;
    ListRec<R> r;
    r.pr = predict_record<R>(P, o.va, d.x, d.y, d.z, (R)dt, p);
    r.nr = near_record<R>(P, o.pos, o.va.x, o.va.y, h);
    O.rec[s] = r;
    const double mx = o.pos.x - p0.x, my = o.pos.y - p0.y;
    return mx * mx + my * my;
}
// The flags of step `step` and its largest displacement (every thread).
__device__ __forceinline__ void finish_listed(const StepParams& P, Ctrl* flags, unsigned long long step,
                                              uint32_t outside, uint32_t bad, double moved2,
                                              unsigned long long* dslots, uint32_t blk) {
    wave_count_add(&flags->outside_l[step & 3], outside);
    if (bad) atomicOr(&flags->grid_overflow, 1u);
    block_max_to_slots(moved2, 0.0, dslots + (uint32_t)(step & P.dset_mask) * kSlotSet, nullptr, blk);
}

// At the head of a fused pair pass behind the summation pass (every thread):
// as list_dt, dt being constant; too many neighbours were found by the
// summation pass.
__device__ __forceinline__ bool fused_pair_begin(const StepParams& P, Ctrl* next, const Ctrl* cur) {
    const bool halted = cur->halted != 0;
    const uint32_t halt_status = !halted && P.consistency_check && next->nbr_overflow ? 3u : 0u;
    if (blockIdx.x == 0) publish_ctrl(cur, next, cur->cur_dt_const, halt_status);
    return !halted && halt_status == 0;
}

// Pair pass from the lists: continuity density rate, pressure, artificial
// viscosity, Lennard-Jones walls and XSPH (the cubic configuration of
// pair_fast_kernel), the dt maxima, and the fields for the integrator.  With
// continuity it also writes the pressure of the current density (the
// reference's p array).
// In FP64 with 8 lanes a bound of 3 waves per SIMD, about as many as 25,000
// particles give: 4 spill (17.7 us a step of 11,842 particles, 16.5 with 3).
// FUSED: see fused_step_begin.  200 steps of 6,923 particles (FP64) take 2.35 ms
// so, 2.88 with an integrator of their own (4 us of a step's 14, and a launch
// gap); 30 of 134,603 (summation, FP32) 1.50 against 1.58.
template <class R, bool FIRST, int LPP, bool CONT, bool ALL, bool FUSED>
__global__ void __launch_bounds__(kBlock, sizeof(R) == 8 ? (FUSED || LPP == 8 ? 3 : 4) : LPP == 1 ? (FUSED ? 5 : 6) : 1)
    pair_list_kernel(StepParams P, Ctrl* next, Ctrl* cur, ListState<R> X, const ListRec<R>* __restrict__ rec,
                     R* __restrict__ pres, const uint32_t* __restrict__ nbl, const uint32_t* __restrict__ nbc,
                     real4<R>* __restrict__ der, real2<R>* __restrict__ xs,
                     unsigned long long* __restrict__ maxslots, unsigned long long* __restrict__ dslots,
                     ListOut<R> O) {
    const uint32_t lb = xcd_block(group_blocks_per_xcd<LPP>(P.n));
    if (lb >= group_blocks<LPP>(P.n)) return;
    __shared__ float2 s_off[64];
    fill_cell_offsets(P, s_off);
    const LaneGroup<LPP> g(lb);
    const uint32_t s = g.s;
    const bool live = s < P.n;
    // in flight while the block decides whether the step runs
    real4<R> prj{}, nj{};
    uint32_t cnt = 0;
    if (live) {
        prj = rec[s].pr;
        nj = rec[s].nr;
        cnt = nbc[s];
    }
    unsigned long long step;
    double dt = 0;
    if constexpr (FUSED) {
        bool goes, back;  // back: the pair's first step left the positions in the other array
        if constexpr (CONT) {
            back = !next->halted;
            goes = fused_step_begin(P, next, cur, O.flags, dslots, step);
            dt = next->pending ? next->dt_new : next->dt;
        } else {
            back = cur->halt_now || !cur->halted;
            goes = fused_pair_begin(P, next, cur);
            step = cur->step;
            dt = cur->cur_dt_const;
        }
        if (!goes) {
            if (O.second && back && X.pos != O.pos && live && g.l == 0) O.pos[s] = X.pos[s];
            return;
        }
    } else if constexpr (FIRST) {
        if (!list_step_begin(P, next, cur, dslots, step)) return;
    } else {
        if (!list_step_goes(cur)) return;
        if (list_build_overflowed(next, cur)) return;
        step = cur->step;
    }
    __syncthreads();  // the offset table
    maxslots += (uint32_t)(step & 1) * kDtSet;
    const ListPair<R, CONT, ALL> K(P);
    ListSums<R> S;
    bool overflow = false;
    if (prj.z == R(0)) cnt = 0;  // died since the build
    const uint32_t cap = P.max_nbr - 1;
    {
        __shared__ uint4 s_rec[kBlock / kWave][sizeof(R) == 8 ? kGather2 * 4 * kWave : 1];
        uint4* buf = s_rec[wave_of_block()];
        auto term = [&](const ListEntry<R>& E) { list_pair_term<R>(K, S, E, nj, prj); };
        if (__ballot(cnt > cap))  // some list of the wave may hold more than cap neighbours
            for_each_listed<R, true, LPP>(P, s_off, cap, s, g.l, nj, X.pos, rec, nbl, cnt, buf, overflow, term);
        else
            for_each_listed<R, false, LPP>(P, s_off, cap, s, g.l, nj, X.pos, rec, nbl, cnt, buf, overflow, term);
        // a dead particle's lanes went along with their wave's: its density is
        // 0, so that a pair of dead particles gives no number
        if (cnt == 0) S = ListSums<R>();
    }
    if (!FUSED && overflow) atomicOr(&next->nbr_overflow, 1u);
    const R mF = (R)P.lp_mF, mW = K.xsph_on ? (R)P.lp_mW : R(0);
    const R ax = lane_sum<LPP>(S.ljx + mF * S.sx);
    const R ay = -(R)P.g + lane_sum<LPP>(S.ljy + mF * S.sy);
    const R drho = mF * lane_sum<LPP>(S.sd);
    const R xx = mW * lane_sum<LPP>(S.xx), xy = mW * lane_sum<LPP>(S.xy);
    const R amu = (R)P.h * lane_max<LPP>(-S.xmin);
    list_dt_maxima<R>(P, live ? (double)ax * ax + (double)ay * ay : 0.0, live ? amu : R(0), maxslots, lb);
    if (live && g.l == 0) {
        real4<R> d;
        d.x = ax;
        d.y = ay;
        d.z = drho;
        d.w = amu;
        der[s] = d;
        real2<R> x;
        x.x = xx;
        x.y = xy;
        xs[s] = x;
        if (P.density_treatment != 0) pres[s] = eos_p<R>(X.va[s].z, (R)P.rho0, (R)P.eos_B);
    }
    if constexpr (FUSED) {
        uint32_t outside = 0, bad = 0;
        double moved2 = 0.0;
        if (live && g.l == 0) {
            Ctrl c{};  // what whole_step reads of it without a wave maker
            c.cur_first = step == 0;
            const real4<R> d{ax, ay, drho, amu};
            const real2<R> x{xx, xy};
            real4<R> pr{};
            const real4<R> va = X.va[s];
            if constexpr (!CONT)  // the summed density
                pr.z = (int)va.w != 0 ? fabs(prj.z) : dead_density<R>(P, density_w0<R>(P), va.z, cur->cur_renorm != 0);
            moved2 = step_listed<R>(P, c, s, X.pos[s], va, pr, 0u, O.home[s], d, x, dt, O, outside, bad);
        }
        finish_listed(P, O.flags, step, outside, bad, moved2, dslots, lb);
    }
}

// W and the gradient factor F (grad W = (r_i - r_j) F) of kernel type skf at
// q = |r| / h, iq = h / |r| (infinite for coincident particles): the pieces
// of kernel_w and kernel_gradf (physics.hpp) without their divisions, with
// 1 / h^2 in the gradients' factors.  Wendland's s^4 - (2 q + 1) s^3 is
// q times -5/2 s^3, without the difference (q iq is 1 but for q's rounding,
// which offsets part of what that does to s^3).
template <class R>
__device__ __forceinline__ void kernel_wf(const StepParams& P, int skf, R q, R iq, R& W, R& F) {
    const R t = R(2) - q;
    switch (skf) {
    case 2:
        W = (R)P.f_gauss * exp(-q * q);
        F = (R)P.g_gauss * W;
        break;
    case 3: {
        const R s = R(0.5) * t, s3 = s * s * s;
        W = q > R(2) ? R(0) : (R)P.f_wend * (s3 * s) * (R(2) * q + R(1));
        F = q < R(1.e-6f) || q >= R(2) ? R(0) : (R)P.g_wend * (s3 * (q * iq));
        break;
    }
    case 4:
        W = q <= R(2) ? (R)P.f_desb * (t * t * t) : R(0);
        F = q < R(2) ? (R)P.g_desb * (t * t) * iq : R(0);
        break;
    default:
        if (q <= R(1)) {
            W = (R)P.f_cubic * (R(2) / R(3) - q * q + q * q * q * R(0.5));
            F = (R)P.c_q1 * (R(-2) + R(1.5) * q);
        } else {
            W = q <= R(2) ? (R)P.f_cubic * (R(1) / R(6) * (t * t * t)) : R(0);
            F = q <= R(2) ? (R)P.c_q1 * (t * t * R(-0.5)) * iq : R(0);
        }
        break;
    }
}

// Pair pass from the lists with every switch of pair_kernel: any smoothing
// kernel per term, both pressure approximations, artificial pressure,
// summation, continuity and delta-SPH density.  Same terms and neighbours as
// pair_kernel on the same FP64 positions.  An entry gathers the neighbour's
// position, state and pred record; entries in groups of G as in
// for_each_listed.  Terms whose kernel type is the pressure's share one
// evaluation, and no term divides: the cell walk over ~55 candidates with a
// division or more per term took 167 us at 187,530 particles (FP64, Wendland
// kernels, delta-SPH, artificial pressure), the ~20 entries of a list 45.  The reciprocal root and 1 / h alone would leave |r| / h
// with half as much error again (43 us).
template <class R, bool FIRST, int LPP>
__global__ void __launch_bounds__(kBlock, sizeof(R) == 8 ? 3 : 1) pair_list_general_kernel(
    StepParams P, Ctrl* next, Ctrl* cur, ListState<R> X, const ListRec<R>* __restrict__ rec, R* __restrict__ pres,
    const uint32_t* __restrict__ nbl, const uint32_t* __restrict__ nbc, real4<R>* __restrict__ der,
    real2<R>* __restrict__ xs, unsigned long long* __restrict__ maxslots, unsigned long long* __restrict__ dslots) {
    const uint32_t lb = xcd_block(group_blocks_per_xcd<LPP>(P.n));
    if (lb >= group_blocks<LPP>(P.n)) return;
    const LaneGroup<LPP> g(lb);
    const uint32_t s = g.s;
    const bool live = s < P.n;
    double2 pj = make_double2(0, 0);
    real4<R> vaj{}, prj{};
    uint32_t cnt = 0;
    if (live) {
        pj = X.pos[s];
        vaj = X.va[s];
        prj = rec[s].pr;
        cnt = nbc[s];
    }
    unsigned long long step;
    if constexpr (FIRST) {
        if (!list_step_begin(P, next, cur, dslots, step)) return;
    } else {
        if (!list_step_goes(cur)) return;
        if (list_build_overflowed(next, cur)) return;
        step = cur->step;
    }
    maxslots += (uint32_t)(step & 1) * kDtSet;
    const KernelConsts<R> K = kernel_consts<R>(P);
    const R m = (R)P.mass;
    R ax = R(0), ay = R(0), drho = R(0), avx = R(0), avy = R(0), amu = R(0);
    bool overflow = false;
    const int tj = (int)vaj.w;
    if (tj == 0) cnt = 0;
    if (cnt) {
        const bool cont = P.density_treatment != 0, delta = P.density_treatment == 2;
        const R rhohj = untyped_rho<R>(prj.z, tj), pjres = prj.w * (rhohj * rhohj);
        const R alpha_c = (R)P.av_alpha * (R)P.av_c, beta = (R)P.av_beta, eta2 = (R)P.av_eta2;
        const R two_eps_m = R(2) * (R)P.xsph_eps * m, lj_r0 = (R)P.lj_r0, lj_D = (R)P.lj_D;
        const R dhc2m = R(2) * (R)P.dhc * m, ap_iw = P.art_pressure ? (R)(1.0 / P.ap_wdelta) : R(0);
        const uint32_t cap = P.max_nbr - 1;
        // FP64 (187,530 particles, Wendland kernels): 42 us per pass with one
        // entry a round and 3 waves per SIMD, 47 with two and 2 waves
        constexpr uint32_t G = sizeof(R) == 8 ? 1 : 2;
        const bool capped = __ballot(cnt > cap) != 0;  // some list of the wave may hold more than cap neighbours
        uint32_t hits = 0;
        list_rounds<LPP, G>(ListRows<LPP>(P, nbl, s, g.l), g.l, cnt, [&](uint32_t k, uint32_t (&e)[G], auto& load) {
            double2 pos[G];
            real4<R> va[G], pr[G];
            uint32_t en[G];
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) {
                const uint32_t i = e[u] & kSlotMask;
                pos[u] = X.pos[i];
                va[u] = X.va[i];
                pr[u] = rec[i].pr;
            }
            load(en);
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) {
                const double dxd = __dsub_rn(pos[u].x, pj.x), dyd = __dsub_rn(pos[u].y, pj.y);
                const int ti = (int)va[u].w;
                bool take = (k + u * LPP < cnt) & (ti != 0) & (dist2_exact(dxd, dyd) < P.cut2);
                if (capped) take = take_capped<LPP>(take, g.l, cap, hits, overflow);
                if (!take) continue;
                const R dx = (R)dxd, dy = (R)dyd;  // r_i - r_j
                const R d2 = (R)(dxd * dxd + dyd * dyd);
                const bool apart = d2 > R(0);
                const R rinv = apart ? fast_rsqrt<R>(d2) : R(INFINITY);
                // |r| and |r| / h within half a unit of the last place, as sqrt and a
                // division give them: near the cut-off the kernels amplify their errors
                const R r1 = d2 * rinv;
                const R dist = apart ? fma(fma(-r1, r1, d2), R(0.5) * rinv, r1) : R(0);
                const R q1 = dist * K.inv_h, q = fma(fma(-q1, K.h, dist), K.inv_h, q1), iq = K.h * rinv;
                R W, F;
                kernel_wf<R>(P, P.skf_intf, q, iq, W, F);
                // continuity density with v and rho of the current step
                if (cont) {
                    R Wd = W, Fd = F;
                    if (P.skf_density != P.skf_intf) kernel_wf<R>(P, P.skf_density, q, iq, Wd, Fd);
                    const R gx = dx * Fd, gy = dy * Fd;
                    drho += m * ((va[u].x - vaj.x) * gx + (va[u].y - vaj.y) * gy);
                    if (delta) {
                        const R rf = -(dx * gx + dy * gy) * (rinv * rinv);
                        drho += dhc2m * ((va[u].z - vaj.z) * fast_rcp<R>(va[u].z) * rf);
                    }
                }
                // Lennard-Jones wall force on fluid from boundary particles
                if (P.lj_on && tj > 0 && ti < 0 && dist < lj_r0) {
                    const R r2 = lj_r0 * rinv, rn = fma(fma(-r2, dist, lj_r0), rinv, r2);  // (its 12th power)
                    const R rn2 = rn * rn, rn4 = rn2 * rn2;
                    const R f = lj_D * (rn4 * rn4 * rn4 - rn4) * (rinv * rinv);
                    ax -= dx * f;
                    ay -= dy * f;
                }
                // pressure: p / rho^2 of both from the pred records
                const R rhohi = untyped_rho<R>(pr[u].z, ti);
                R pf = P.intf_approx == 1 ? (pjres + pr[u].w * (rhohi * rhohi)) * fast_rcp<R>(rhohj * rhohi)
                                          : pr[u].w + prj.w;
                if (P.art_pressure && (pr[u].w < R(0) || prj.w < R(0))) {
                    R Wa = W, Fa = F;
                    if (P.skf_ap != P.skf_intf) kernel_wf<R>(P, P.skf_ap, q, iq, Wa, Fa);
                    const R api = pr[u].w < R(0) ? -(R)P.ap_coef * pr[u].w : R(0);
                    const R apj = prj.w < R(0) ? -(R)P.ap_coef * prj.w : R(0);
                    pf += (api + apj) * pow(Wa * ap_iw, (R)P.ap_index);
                }
                R cx = F * pf * m;
                // artificial viscosity and XSPH with the predicted velocity and density
                const R dvx = pr[u].x - prj.x, dvy = pr[u].y - prj.y;
                const R inv_rs = fast_rcp<R>(rhohi + rhohj);
                if (P.av_on) {
                    const R vr = dvx * dx + dvy * dy;  // (v_j - v_i) . (r_j - r_i)
                    if (vr < R(0)) {
                        const R mu = K.h * vr * fast_rcp<R>(d2 + eta2);
                        amu = fmax(amu, fabs(mu));
                        R Wv = W, Fv = F;
                        if (P.skf_av != P.skf_intf) kernel_wf<R>(P, P.skf_av, q, iq, Wv, Fv);
                        cx += Fv * ((beta * mu - alpha_c) * mu * R(2) * inv_rs) * m;
                    }
                }
                ax += dx * cx;
                ay += dy * cx;
                if (P.xsph_on && ti > 0) {
                    R Wx = W, Fx = F;
                    if (P.skf_xsph != P.skf_intf) kernel_wf<R>(P, P.skf_xsph, q, iq, Wx, Fx);
                    const R c = two_eps_m * inv_rs * Wx;
                    avx += dvx * c;
                    avy += dvy * c;
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) e[u] = en[u];
        });
    }
    if (overflow) atomicOr(&next->nbr_overflow, 1u);
    ax = lane_sum<LPP>(ax);
    ay = -(R)P.g + lane_sum<LPP>(ay);
    drho = lane_sum<LPP>(drho);
    avx = lane_sum<LPP>(avx);
    avy = lane_sum<LPP>(avy);
    amu = lane_max<LPP>(amu);
    list_dt_maxima<R>(P, live ? (double)ax * ax + (double)ay * ay : 0.0, live ? amu : R(0), maxslots, lb);
    if (live && g.l == 0) {
        real4<R> d;
        d.x = ax;
        d.y = ay;
        d.z = drho;
        d.w = amu;
        der[s] = d;
        real2<R> x;
        x.x = avx;
        x.y = avy;
        xs[s] = x;
        if (P.density_treatment != 0) pres[s] = eos_p<R>(vaj.z, (R)P.rho0, (R)P.eos_B);
    }
}

// At the head of a list step's integrator (every thread): the step's dt;
// block 0 publishes the control block and clears the next step's dt slots.
// False when the step halted or halts here (dt below the reference's
// never-ending bound, more neighbours than max_neighbours - 1).  keep: a
// tape's copy of the published words, or null.
__device__ __forceinline__ bool list_dt(const StepParams& P, Ctrl* next, const Ctrl* cur,
                                        unsigned long long* maxslots, double& dt, Ctrl* keep = nullptr) {
    uint32_t halt_status = 0;
    const bool halted = cur->halted != 0;
    if (!halted) {
        const uint32_t par = (uint32_t)(cur->step & 1);
        if (P.dt_method == 2 && P.dt_dynamic_mode == 1) {
            const double a2max = slots_max(maxslots + par * kDtSet), mumax = slots_max(maxslots + par * kDtSet + kSlotSet);
            dt = P.cfl * fmin(sqrt(P.h / sqrt(a2max)), P.h / (P.c0 + mumax));
        } else {
            dt = cur->cur_dt_const;
        }
        const bool never = P.dt_method == 2 && dt <= P.never_ending;
        const bool nbr_err = P.consistency_check && next->nbr_overflow;
        halt_status = nbr_err ? 3u : (never ? 4u : 0u);
        if (blockIdx.x == 0) {
            clear_slots(maxslots + (par ^ 1) * kDtSet);
            clear_slots(maxslots + (par ^ 1) * kDtSet + kSlotSet);
        }
    }
    if (blockIdx.x == 0) {
        publish_ctrl(cur, next, dt, halt_status);
        if (keep) publish_ctrl(cur, keep, dt, halt_status);
    }
    return !halted && halt_status == 0;
}

// Whether whole_step of a particle looks at its original index: the wall that
// disappears, wave-maker particles (4 bytes a particle that the others need
// not read).
__device__ __forceinline__ bool step_needs_oid(const StepParams& P, const Ctrl& c, int itype) {
    return c.wall_disappear || (P.boundary_motion && c.piston_active && itype < 0);
}

// whole_step of every slot from X into A (in place on list steps, but for a
// tape's, which go from one kept state to the next), the cell
// key for the next build, the step's largest displacement, and the records
// of the next step's pair pass: near (the new position relative to the home
// cell, the new velocity) and pred (PredictHalfStep.cpp:16-22 with this
// step's dt, which is the next step's).  The step's accelerations are in
// A.ad already: the pair pass writes them there (its der), since what the
// step reads of the last ones is in the records.  Bound by HBM traffic: 124
// bytes a particle in FP32, 208 in FP64 (148 and 249 with A.ad written here
// and every original index read).  The loads go before the wait for dt.
template <class R>
__global__ void __launch_bounds__(kBlock) integrate_list_kernel(StepParams P, Ctrl* next, const Ctrl* cur,
                                                                ListState<R> X, const real2<R>* __restrict__ xs,
                                                                ListRec<R>* __restrict__ rec,
                                                                const uint32_t* __restrict__ home, StateA<R> A,
                                                                uint32_t* __restrict__ key_next,
                                                                unsigned long long* maxslots,
                                                                unsigned long long* dslots, Ctrl* keep) {
    const uint32_t s0 = blockIdx.x * kBlock + threadIdx.x;
    const bool live = s0 < P.n;
    const uint32_t s = live ? s0 : P.n - 1;
    const real4<R> d = A.ad[s];
    const real2<R> x = xs[s];
    const double2 p0 = X.pos[s];
    const real4<R> va = X.va[s];
    const uint32_t h = home[s];
    real4<R> pr{};
    if (P.density_treatment == 0) pr.z = fabs(rec[s].pr.z);  // the summed density (sign-encoded)
    const Ctrl& c = *cur;
    double dt;
    if (!list_dt(P, next, cur, maxslots, dt, keep)) return;
    uint32_t outside = 0, bad = 0;
    double moved2 = 0.0;
    if (live) {
        const bool reordered = A.oid != X.oid;
        const uint32_t oid = reordered || step_needs_oid(P, c, (int)va.w) ? X.oid[s] : 0u;
        if (P.density_treatment == 0 && (int)va.w == 0)
            pr.z = dead_density<R>(P, density_w0<R>(P), va.z, c.cur_renorm != 0);
        moved2 = step_listed<R>(P, c, s, p0, va, pr, oid, h, d, x, dt, ListOut<R>{A.pos, A.va, rec, home, key_next, next, false},
                                outside, bad);
        if (reordered) A.oid[s] = oid;
    }
    finish_listed(P, next, c.step, outside, bad, moved2, dslots, blockIdx.x);
}

}  // namespace rrsph
