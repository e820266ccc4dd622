// Neighbour-list steps in 3D: the design of list_step.hpp (builds that sort
// the cells and list every particle within k h + skin, list steps that
// decide each entry with the reference's cut-off test, a device-side
// staleness halt) with three-dimensional records.
//
// Per slot, in slot order:
//   rec.nr  FP32: (xi_x, xi_y, xi_z, p / rho^2), xi the position relative to
//           the origin of the home cell; FP64: (x, y, z, p / rho^2)
//   rec.pr  (v^x, v^y, v^z, s rho^), s = +1 fluid, -1 boundary, 0 dead
//   dens    (xi or x, s rho), rho the density before the step: what the
//           summation density pass gathers (its own record, so that the
//           pass can write the predicted density and p / rho^2 of its slot
//           into rec while others read dens)
// An entry holds the neighbour's slot in its low 25 bits and the offset of
// the two home cells, (dcx + 2) + 5 (dcy + 2) + 25 (dcz + 2), in its high 7.
// The FP32 cut-off test takes r_i - r_j = xi_i - xi_j + dc cell, the
// offsets from a table in LDS, and the FP64 positions and the reference's
// test (GridFind.cpp:144-176, dist2_exact3) within 1e-5 of the cut-off.
//
// Step kernels: [density_sum_list3] -> pair_list3_kernel ->
// integrate_list3_kernel (in place), the first of them with the step's
// prologue (list_step_begin).  A build step runs list_prologue -> counting sort
// -> reorder_list3_kernel -> list_build3_kernel -> the same step kernels on
// the reordered copy, integrating into A.
#pragma once

#include "list_step.hpp"
#include "step3d.hpp"

namespace rrsph {

constexpr uint32_t kSlotBits3 = 25;
constexpr uint32_t kSlotMask3 = (1u << kSlotBits3) - 1;  // 3D list steps take fewer than 2^25 particles
constexpr uint32_t kCodes3 = 125;

template <class R> struct ListState3 {
    const double4* pos;
    const real4<R>* va;
    const uint32_t* oid;
};

// Origin of home cell `home` (a key (cx ncy + cy) ncz + cz).
__device__ __forceinline__ double3 cell_origin3(const StepParams& P, uint32_t home) {
    const uint32_t cz = home % (uint32_t)P.ncz;
    const uint32_t cxy = home / (uint32_t)P.ncz;
    const uint32_t cx = cxy / (uint32_t)P.ncy, cy = cxy - cx * (uint32_t)P.ncy;
    return make_double3(P.xmin + (double)cx * P.cell, P.ymin + (double)cy * P.cell, P.zmin + (double)cz * P.cell);
}

// A record's position half with w in the fourth component.
template <class R> __device__ __forceinline__ real4<R> near3(const StepParams& P, double4 pos, R w, uint32_t home);
template <> __device__ __forceinline__ float4 near3<float>(const StepParams& P, double4 pos, float w, uint32_t home) {
    const double3 o = cell_origin3(P, home);
    return make_float4((float)(pos.x - o.x), (float)(pos.y - o.y), (float)(pos.z - o.z), w);
}
template <> __device__ __forceinline__ double4 near3<double>(const StepParams&, double4 pos, double w, uint32_t) {
    return make_double4(pos.x, pos.y, pos.z, w);
}

// The prediction of PredictHalfStep.cpp:16-22 as reorder3_kernel makes it:
// (v^, s rho^) and p / rho^2 with p the pressure of the current density.
template <class R>
__device__ __forceinline__ real4<R> predict3(const StepParams& P, const real4<R>& va, int itype, const real4<R>& ad,
                                              R dt, R& pw, R& p) {
    real4<R> pr;
    pr.x = va.x + ad.x * dt * R(0.5);
    pr.y = va.y + ad.y * dt * R(0.5);
    pr.z = va.z + ad.z * dt * R(0.5);
    const R rho_hat = P.density_treatment != 0 ? va.w + ad.w * dt * R(0.5) : va.w;
    p = eos_p<R>(va.w, (R)P.rho0, (R)P.eos_B);
    pw = p / (rho_hat * rho_hat);
    pr.w = typed_rho<R>(rho_hat, itype);
    return pr;
}

// The reorder of a 3D build step: reorder3_kernel's gather, pressure and
// cell-start table, plus the records, each slot's home cell and its
// candidate record for the build's walk, cand = (position relative to the
// home cell's origin in FP32, the home cell's z index).  COUNTED as in 2D.
template <class R, bool COUNTED>
__global__ void __launch_bounds__(kBlock) reorder_list3_kernel(StepParams P, const Ctrl* __restrict__ ctrl,
                                                               const uint32_t* __restrict__ skey,
                                                               const uint32_t* __restrict__ perm, StateA3<R> A,
                                                               StateB3<R> B, ListRec<R>* __restrict__ rec,
                                                               real4<R>* __restrict__ dens, uint32_t* __restrict__ home,
                                                               float4* __restrict__ cand, uint32_t* __restrict__ LB,
                                                               uint32_t* __restrict__ perm_out) {
    if (ctrl->halted) return;
    const uint32_t s0 = blockIdx.x * kBlock + threadIdx.x;
    const bool live = s0 < P.n;
    uint32_t s = live ? s0 : P.n - 1;
    const uint32_t k = skey[s];
    const uint32_t src = min(perm[s], P.n - 1);  // a permutation of [0, n); the clamp only guards memory
    if constexpr (COUNTED) s = cell_place(P, LB, perm, s, k);
    const double4 pos = A.pos[src];
    const real4<R> va = A.va[src];
    const real4<R> ad = A.ad[src];
    const uint32_t oid = A.oid[src];
    const int itype = (int)pos.w;
    R pw, p;
    const real4<R> pr = predict3<R>(P, va, itype, ad, (R)ctrl->cur_dt, pw, p);
    if (live) {
        B.pos[s] = pos;
        B.va[s] = va;
        B.oid[s] = oid;
        B.pres[s] = p;
        ListRec<R> r;
        r.nr = near3<R>(P, pos, pw, k);
        r.pr = pr;
        rec[s] = r;
        dens[s] = near3<R>(P, pos, typed_rho<R>(va.w, itype), k);
        home[s] = k;
        const double3 o = cell_origin3(P, k);
        cand[s] = make_float4((float)(pos.x - o.x), (float)(pos.y - o.y), (float)(pos.z - o.z),
                              __int_as_float((int)(k % (uint32_t)P.ncz)));
        if constexpr (COUNTED) perm_out[s] = src;
    }
    if constexpr (!COUNTED) fill_cell_starts(P, s, live, k, skey, LB);
}

// The lists of a 3D build step on the reordered copy: for each live
// particle, every live particle i != s within list_reach, in the order of
// the reference's cell walk (x-major columns, then y, each column's z range
// contiguous).  The cells visited are those within list_reach (3 or 4 per
// axis; a column off the particle's own needs a shorter z range, corner
// columns most).
constexpr uint32_t kCollectL3 = 4;
__global__ void __launch_bounds__(kBlock) list_build3_kernel(StepParams P, Ctrl* __restrict__ next,
                                                             const Ctrl* __restrict__ cur,
                                                             const double4* __restrict__ pos,
                                                             const float4* __restrict__ cand,
                                                             const uint32_t* __restrict__ skey,
                                                             const uint32_t* __restrict__ LB,
                                                             uint32_t* __restrict__ nbl, uint32_t* __restrict__ nbc) {
    __shared__ BuildLds s_build[kBlock / kWave];
    if (cur->halted) return;
    const uint32_t lb = xcd_block(P.blocks_per_xcd);
    if (lb >= P.nblocks) return;
    const uint32_t s0 = lb * kBlock + threadIdx.x;
    const bool inb = s0 < P.n;
    const uint32_t s = inb ? s0 : P.n - 1;
    bool bad = false;
    const double4 pj = pos[s];
    const bool alive = inb && (int)pj.w != 0;
    const uint32_t kj = skey[s];
    const int hz = (int)(kj % (uint32_t)P.ncz);
    const uint32_t hxy = kj / (uint32_t)P.ncz;
    const int hx = (int)(hxy / (uint32_t)P.ncy), hy = (int)hxy - hx * P.ncy;
    const float4 cj = cand[s];
    const float cell = (float)P.cell, inv_cell = (float)(1.0 / P.cell);
    const float reach = (float)(P.list_reach * (1.0 + 1e-5));
    // empty ranges (x0 > x1) for lanes with nothing to list
    int x0 = 0, x1 = -1, y0 = 0, y1 = -1, z0 = 0, z1 = 0;
    if (alive) {
        // the list pass takes the FP32 positions relative to the home cell
        // for within 2.1 cells of its origin: a particle outside the cell
        // grid (keyed to the nearest edge cell) runs the step without lists
        const double3 o = cell_origin3(P, kj);
        const double ox = pj.x - o.x, oy = pj.y - o.y, oz = pj.z - o.z;
        bad = !(ox > -P.cell && ox < 2.0 * P.cell && oy > -P.cell && oy < 2.0 * P.cell && oz > -P.cell &&
                oz < 2.0 * P.cell);
        if (!bad) {
            x0 = reach_first(cj.x, reach, inv_cell, hx);
            x1 = reach_last(cj.x, reach, inv_cell, hx, P.ncx);
            y0 = reach_first(cj.y, reach, inv_cell, hy);
            y1 = reach_last(cj.y, reach, inv_cell, hy, P.ncy);
            z0 = reach_first(cj.z, reach, inv_cell, hz);
            z1 = reach_last(cj.z, reach, inv_cell, hz, P.ncz);
        }
        bad |= x0 < hx - 2 || x1 > hx + 2 || y0 < hy - 2 || y1 > hy + 2 || z0 < hz - 2 || z1 > hz + 2;
    }
    ListBuilder out(P, s_build[wave_of_block()], nbl, s);
    const int wx0 = full_wave_min_i32(x0 <= x1 ? x0 : INT_MAX), wx1 = full_wave_max_i32(x1);
    const int wy0 = full_wave_min_i32(y0 <= y1 ? y0 : INT_MAX), wy1 = full_wave_max_i32(y1);
    // positions relative to the column in x and y and to one cell of the
    // wave in z, from the candidate records (relative to their home cells)
    const float r2 = (float)(P.list_r2 * (1.0 + build_margin(P.ncz)));
    const int zref = __builtin_amdgcn_readfirstlane(hz);
    const float pz = cj.z + (float)(hz - zref) * cell;
#pragma unroll 1
    for (int x = wx0; x <= wx1; ++x) {
        const bool need_x = x >= x0 && x <= x1;
        if (!__any(need_x)) continue;
        const float px = cj.x + (float)(hx - x) * cell;
        const float dxm = fmaxf(0.f, fmaxf(-px, px - cell));  // distance to the column's x slab
        const float rem_x = r2 - dxm * dxm;
#pragma unroll 1
        for (int y = wy0; y <= wy1; ++y) {
            const float py = cj.y + (float)(hy - y) * cell;
            const float dym = fmaxf(0.f, fmaxf(-py, py - cell));
            const float rem = rem_x - dym * dym;
            const bool need = need_x && y >= y0 && y <= y1 && rem >= 0.f;
            if (!__any(need)) continue;
            const uint32_t col = ((uint32_t)x * (uint32_t)P.ncy + (uint32_t)y) * (uint32_t)P.ncz;
            uint32_t b = 0, e = 0;
            if (need) {
                // the z cells of this column within reach, a little widened
                // for the rounding here
                const float zr = __builtin_amdgcn_sqrtf(rem) * (1.f + 1e-5f) + 1e-5f * cell;
                const int za = max(z0, hz + (int)floorf((cj.z - zr) * inv_cell));
                const int zb = min(z1, hz + (int)floorf((cj.z + zr) * inv_cell));
                b = LB[col + za];
                e = LB[col + zb + 1];
            }
            // the word holds the slot and the z cell; the offsets from the
            // lane's home cell complete the code (modulo 2^32)
            const uint32_t add = (uint32_t)((x - hx + 2) + 5 * (y - hy + 2) + 25 * (2 - hz)) << kSlotBits3;
            out.column<true>(need, b, e, px, py, pz, r2, add, [&](uint32_t i) {
                const float4 q = cand[i];
                const int cz = __float_as_int(q.w);
                return make_float4(q.x, q.y, q.z + (float)(cz - zref) * cell,
                                   __uint_as_float(i + ((uint32_t)(25 * cz) << kSlotBits3)));
            });
        }
    }
    out.flush();
    if (!inb) return;
    if (out.cnt > P.list_cap || bad) atomicOr(&next->list_overflow, 1u);
    if (out.cnt > P.max_nbr - 1) atomicOr(&next->list_long, 1u);
    nbc[s] = min(out.cnt, P.list_cap);
}

// collect_neighbours3 over a particle's list instead of the cell walk: the
// entries within the cut-off (the reference's FP64 test on pos), alive, in
// list order, first `cap` kept, into the lane's column of the LDS hit list,
// flushed wave-uniformly.  Every lane of the wave calls it; lanes with
// active = false have no entries.
template <uint32_t kChunk, class F>
__device__ __forceinline__ void collect_listed3(const StepParams& P, bool active, uint32_t cap, uint32_t s,
                                                double4 pj, const double4* __restrict__ pos,
                                                const uint32_t* __restrict__ nbl, const uint32_t* __restrict__ nbc,
                                                uint32_t* __restrict__ hits, bool& overflow, F&& flush) {
    static_assert(kChunk >= 2 * kCollectL3, "hit list too short");
    const uint32_t cnt = active ? nbc[s] : 0u;
    const uint32_t cmax = wave_max_u32(cnt);
    const uint32_t row = P.n * 4u;
    uint32_t nh = 0, done = 0;
#pragma unroll 1
    for (uint32_t k = 0; k < cmax; k += kCollectL3) {
        uint32_t i[kCollectL3];
        double4 q[kCollectL3];
#pragma unroll
        for (uint32_t u = 0; u < kCollectL3; ++u) i[u] = list_entry(nbl, (k + u) * row + s * 4u) & kSlotMask3;
#pragma unroll
        for (uint32_t u = 0; u < kCollectL3; ++u) q[u] = pos[i[u]];
#pragma unroll
        for (uint32_t u = 0; u < kCollectL3; ++u) {
            const double dx = __dsub_rn(q[u].x, pj.x), dy = __dsub_rn(q[u].y, pj.y), dz = __dsub_rn(q[u].z, pj.z);
            const bool hit = (k + u < cnt) & ((int)q[u].w != 0) & (dist2_exact3(dx, dy, dz) < P.cut2);
            if (hit) {
                if (done + nh < cap) {
                    hits[nh * kBlock] = i[u];
                    ++nh;
                } else {
                    overflow = true;
                }
            }
        }
        if (__any(nh + kCollectL3 > kChunk)) {  // wave-uniform
            flush(nh);
            done += nh;
            nh = 0;
        }
    }
    flush(nh);
}

// The table of home-cell offsets of the 3D entry codes (first kCodes3
// threads; a barrier must follow).
__device__ __forceinline__ void fill_cell_offsets3(const StepParams& P, float4* s_off) {
    if (threadIdx.x < kCodes3) {
        const int c = (int)threadIdx.x;
        const int dx = c % 5 - 2, dy = (c / 5) % 5 - 2, dz = c / 25 - 2;
        s_off[c] = make_float4((float)(dx * P.cell), (float)(dy * P.cell), (float)(dz * P.cell), 0.f);
    }
}

// r_i - r_j of an entry and whether it is within the cut-off (see the
// header): FP32 from the records, FP64 on the band; FP64 from the FP64
// record positions.
__device__ __forceinline__ bool list_cut3(const StepParams& P, const CutFP32& C, const float4* s_off, uint32_t e,
                                          const float4& ni, const float4& nj, uint32_t s,
                                          const double4* __restrict__ pos, float& dx, float& dy, float& dz) {
    const float4 o = s_off[e >> kSlotBits3];
    dx = (ni.x - nj.x) + o.x;
    dy = (ni.y - nj.y) + o.y;
    dz = (ni.z - nj.z) + o.z;
    const float d2 = dx * dx + dy * dy + dz * dz;
    if (!(d2 > C.lo && d2 < C.hi)) return d2 <= C.lo;  // on the band's edge: within a rounding of lo < cut2
    const double4 q = pos[e & kSlotMask3], pj = pos[s];  // rare: the band around the cut-off
    const double ddx = __dsub_rn(q.x, pj.x), ddy = __dsub_rn(q.y, pj.y), ddz = __dsub_rn(q.z, pj.z);
    dx = (float)ddx;
    dy = (float)ddy;
    dz = (float)ddz;
    return dist2_exact3(ddx, ddy, ddz) < P.cut2;
}
__device__ __forceinline__ bool list_cut3(const StepParams& P, const CutFP32&, const float4*, uint32_t,
                                          const double4& ni, const double4& nj, uint32_t,
                                          const double4* __restrict__, double& dx, double& dy, double& dz) {
    dx = __dsub_rn(ni.x, nj.x);
    dy = __dsub_rn(ni.y, nj.y);
    dz = __dsub_rn(ni.z, nj.z);
    return dist2_exact3(dx, dy, dz) < P.cut2;
}

// collect_listed3 from the near records of the list steps (position
// relative to the home cell of the build, and type, in nearf): each entry
// decided as the FP32 list pass decides it (list_cut3: FP32, the FP64 test
// on pos inside the band), the same hits; the hit list keeps the whole
// entry (slot and home-cell offset code).
template <uint32_t kChunk, class F>
__device__ __forceinline__ void collect_near3(const StepParams& P, bool active, uint32_t cap, uint32_t s,
                                              const float4* s_off, const float4& nk, const float4* __restrict__ nearf,
                                              const double4* __restrict__ pos,
                                              const uint32_t* __restrict__ nbl, const uint32_t* __restrict__ nbc,
                                              uint32_t* __restrict__ hits, bool& overflow, F&& flush) {
    static_assert(kChunk >= 2 * kCollectL3, "hit list too short");
    const CutFP32 C = cut_band(P);
    const uint32_t cnt = active ? nbc[s] : 0u;
    const uint32_t cmax = wave_max_u32(cnt);
    const uint32_t row = P.n * 4u;
    uint32_t nh = 0, done = 0;
#pragma unroll 1
    for (uint32_t k = 0; k < cmax; k += kCollectL3) {
        uint32_t e[kCollectL3];
        float4 q[kCollectL3];
#pragma unroll
        for (uint32_t u = 0; u < kCollectL3; ++u) e[u] = list_entry(nbl, (k + u) * row + s * 4u);
#pragma unroll
        for (uint32_t u = 0; u < kCollectL3; ++u) q[u] = nearf[e[u] & kSlotMask3];
#pragma unroll
        for (uint32_t u = 0; u < kCollectL3; ++u) {
            float dx, dy, dz;
            const bool in = list_cut3(P, C, s_off, e[u], q[u], nk, s, pos, dx, dy, dz);
            const bool hit = (k + u < cnt) & (q[u].w != 0.f) & in;
            if (hit) {
                if (done + nh < cap) {
                    hits[nh * kBlock] = e[u];
                    ++nh;
                } else {
                    overflow = true;
                }
            }
        }
        if (__any(nh + kCollectL3 > kChunk)) {  // wave-uniform
            flush(nh);
            done += nh;
            nh = 0;
        }
    }
    flush(nh);
}

// ListRows with the row's offset added in a vector register: the FP32 passes,
// which keep 6 or 12 entries in flight, take 703 us at 2,899,370 particles
// (pair pass) this way and 728 with scalar row offsets.
struct ListRowsVector {
    const uint32_t* nbl;
    uint32_t row, last, col;
    __device__ ListRowsVector(const StepParams& P, const uint32_t* lists, uint32_t s)
        : nbl(lists), row(P.n * 4u), last(P.list_cap + kListPad - 1), col(s * 4u) {}
    __device__ __forceinline__ uint32_t operator()(uint32_t k) const {
        return list_entry(nbl, min(k, last) * row + col);
    }
};

template <class R> __device__ __forceinline__ R density_w0_3(const StepParams& P) {
    return (R)P.f_cubic * (R(2) / R(3));
}

// Summation density from the lists (Density.h:25-61) with the
// renormalisation of the steps that ask for it (ModelParams.tex:124-133):
// rho into rec.pr.w (sign-typed), p / rho^2 into rec.nr.w, p into pres.
template <class R, bool FIRST>
__global__ void __launch_bounds__(kBlock) density_sum_list3(StepParams P, Ctrl* next, Ctrl* cur, ListState3<R> X,
                                                            const real4<R>* __restrict__ dens,
                                                            ListRec<R>* __restrict__ rec, R* __restrict__ pres,
                                                            const uint32_t* __restrict__ nbl,
                                                            const uint32_t* __restrict__ nbc,
                                                            unsigned long long* __restrict__ dslots) {
    const uint32_t lb = xcd_block(P.blocks_per_xcd);
    if (lb >= P.nblocks) return;
    __shared__ float4 s_off[kCodes3];
    fill_cell_offsets3(P, s_off);
    unsigned long long step;
    if constexpr (FIRST) {
        if (!list_step_begin(P, next, cur, dslots, step)) return;
    } else {
        if (!list_step_goes(cur)) return;
        step = cur->step;
    }
    __syncthreads();  // the offset table
    const uint32_t s0 = lb * kBlock + threadIdx.x;
    const bool live = s0 < P.n;
    const uint32_t s = live ? s0 : P.n - 1;
    const R m = (R)P.mass, inv_h = (R)(1.0 / P.h), w_q1 = (R)P.f_cubic, w_q2 = (R)(P.f_cubic / 6.0);
    const real4<R> dj = dens[s];
    const R w0 = density_w0_3<R>(P);
    R rho = m * w0;
    const bool renorm = step_renorm(P, step);
    R wsum = renorm && dj.w != R(0) ? m / fabs(dj.w) * w0 : R(0);
    bool overflow = false;
    const uint32_t cnt = live && dj.w != R(0) ? nbc[s] : 0u;
    const CutFP32 C = cut_band(P);
    const uint32_t cap = P.max_nbr - 1;
    uint32_t hits = 0;
    auto entry_term = [&](uint32_t k, uint32_t e, const real4<R>& di) {
        R dx, dy, dz;
        const bool hit = list_cut3(P, C, s_off, e, di, dj, s, X.pos, dx, dy, dz) & (di.w != R(0)) & (k < cnt);
        const bool take = hit & (hits < cap);
        overflow |= hit & !take;
        hits += take ? 1u : 0u;
        const R q = pair_dist<R>(dx, dy, dz) * inv_h;
        const R t = R(2) - q;
        const R w = q <= R(1) ? w_q1 * (R(2) / R(3) - q * q + R(0.5) * q * q * q) : w_q2 * t * t * t;
        const R wt = take ? w : R(0);
        rho += m * wt;
        // (a neighbour that died since the build has density 0 in its
        // record: only taken entries enter the sum)
        if (renorm && take) wsum += m / fabs(di.w) * wt;
    };
    if constexpr (sizeof(R) == 4) {
        // 2,899,370 particles: 466 us per pass with 12 in flight (492 with 8, 538 with 4)
        constexpr uint32_t G = 12;
        list_rounds<1, G>(ListRowsVector(P, nbl, s), 0, cnt, [&](uint32_t k, uint32_t (&e)[G], auto& load) {
            real4<R> di[G];
            uint32_t en[G];
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) di[u] = dens[e[u] & kSlotMask3];
            load(en);
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) {
                entry_term(k + u, e[u], di[u]);
                e[u] = en[u];
            }
        });
    } else {
        // 555,686 particles: 158 us per pass with 8 in flight (184 with 4, 225
        // with 12), 181 when each lane gathered its own
        constexpr uint32_t G = 8;
        __shared__ uint4 s_rec[kBlock / kWave][G * 2 * kWave];
        const WaveGather<2, 32, kSlotMask3> src(dens, s_rec[wave_of_block()]);
        gather_rounds<1, G>(P, nbl, src, s0, 0, cnt, [&](uint32_t k, const uint32_t (&e)[G], const auto& w) {
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) entry_term(k + u, e[u], record_real4(w[u], R(0)));
        });
    }
    if (!live) return;
    const int itype = (int)X.pos[s].w;
    if (itype == 0) rho = dead_density<R>(P, w0, X.va[s].w, renorm);  // (its record's density is 0)
    else if (renorm) rho = rho / wsum;
    if (overflow) atomicOr(&next->nbr_overflow, 1u);
    const R p = eos_p<R>(rho, (R)P.rho0, (R)P.eos_B);
    ListRec<R> r = rec[s];
    r.pr.w = typed_rho<R>(rho, itype);
    r.nr.w = p / (rho * rho);
    rec[s] = r;
    pres[s] = p;
}

// One entry in 3D (list_pair).  i's records: nr (position half, p / rho^2),
// pr (v^, s rho^), vai (its current velocity; continuity only).
template <class R> struct ListSums3 {
    R sx = 0, sy = 0, sz = 0, sd = 0, xx = 0, xy = 0, xz = 0, xmin = 0, ljx = 0, ljy = 0, ljz = 0;
};
template <class R, class K_>
__device__ __forceinline__ void list_pair_term3(const K_& K, ListSums3<R>& S, bool take, R dx, R dy, R dz,
                                                const real4<R>& nri, const real4<R>& pri, const real4<R>& vai,
                                                const real4<R>& vaj, const real4<R>& prj, R pwj) {
    const R d2 = dx * dx + dy * dy + dz * dz;
    const R dvx = pri.x - prj.x, dvy = pri.y - prj.y, dvz = pri.z - prj.z;
    const ListTerm<R> T =
        list_pair<R>(K, take, d2, dvx * dx + dvy * dy + dvz * dz, pri.w, prj.w, nri.w + pwj, S.xmin);
    if (K.cont) S.sd += T.F * ((vai.x - vaj.x) * dx + (vai.y - vaj.y) * dy + (vai.z - vaj.z) * dz);
    const R fc = T.F * T.coef;
    S.sx += fc * dx;
    S.sy += fc * dy;
    S.sz += fc * dz;
    S.xx += dvx * T.w;
    S.xy += dvy * T.w;
    S.xz += dvz * T.w;
    if (T.wall) {
        const R f = list_wall<R>(K, d2, T.rinv);
        S.ljx -= dx * f;
        S.ljy -= dy * f;
        S.ljz -= dz * f;
    }
}

// As ListOut and step_listed in 3D (dens only where the summation pass reads it).
template <class R> struct ListOut3 {
    double4* pos;
    real4<R>* va;
    ListRec<R>* rec;
    real4<R>* dens;
    const uint32_t* home;
    uint32_t* key_next;
    Ctrl* flags;
    bool second;
};
template <class R>
__device__ __forceinline__ double step_listed3(const StepParams& P, const Ctrl& c, uint32_t s, double4 p0,
                                               const real4<R>& va, const real4<R>& pr, uint32_t oid, uint32_t h,
                                               const real4<R>& d, const real4<R>& x, double dt, const ListOut3<R>& O,
                                               uint32_t& outside, uint32_t& bad) {
    const Stepped3<R> o = whole_step_one3<R>(P, c, p0, va, pr, oid, d.x, d.y, d.z, d.w, x.x, x.y, x.z, dt, outside);
    O.pos[s] = o.pos;
    O.va[s] = o.va;
    const int itype = (int)o.pos.w;
    O.key_next[s] = itype == 0 ? P.ncells : cell_key3(P, o.pos.x, o.pos.y, o.pos.z, bad);
    R pw, p;
    ListRec<R> r;
    r.pr = predict3<R>(P, o.va, itype, d, (R)dt, pw, p);
    r.nr = near3<R>(P, o.pos, pw, h);
    O.rec[s] = r;
    if (P.density_treatment == 0) O.dens[s] = near3<R>(P, o.pos, typed_rho<R>(o.va.w, itype), h);
    const double mx = o.pos.x - p0.x, my = o.pos.y - p0.y, mz = o.pos.z - p0.z;
    return mx * mx + my * my + mz * mz;
}

// Pair pass from the 3D lists: the cubic configuration of pair3_kernel
// (continuity, pressure, artificial viscosity, Lennard-Jones walls, XSPH),
// the dt maxima and the fields for the integrator.  Entries in rounds of G,
// the records gathered by each lane in FP32 (6 in flight: 706 us per pass at
// 2,899,370 particles, summation; 724 at 8, 793 at 4; by the wave, two lanes a
// record, 807: vector instructions take two thirds of the pass's time, 1.04 of
// 1.53 ms at 6,595,366 particles) and by the wave in
// FP64 (555,686 particles, summation: 224 us per pass with 4 in flight, 235
// with 3, 253 with 2; 310 when each lane gathered its own; 943,906 particles,
// continuity, which gathers the velocity too: 515 with 3, 576 with 2, 633 by
// lane).  Two blocks per CU hold enough loads in flight then.
// FUSED (behind the summation pass): see fused_step_begin; 16 steps of 6.6M
// particles (FP32) 62.0 -> 60.5 ms, of which 8 are copies.
template <class R, bool FIRST, bool CONT, bool ALL, bool FUSED>
__global__ void __launch_bounds__(kBlock, 3) pair_list3_kernel(
    StepParams P, Ctrl* next, Ctrl* cur, ListState3<R> X, const ListRec<R>* __restrict__ rec, R* __restrict__ pres,
    const uint32_t* __restrict__ nbl, const uint32_t* __restrict__ nbc, real4<R>* __restrict__ der,
    real4<R>* __restrict__ xs, unsigned long long* __restrict__ maxslots, unsigned long long* __restrict__ dslots,
    ListOut3<R> O) {
    static_assert(!(FUSED && CONT), "a fused 3D step has a summation pass");
    const uint32_t lb = xcd_block(P.blocks_per_xcd);
    if (lb >= P.nblocks) return;
    __shared__ float4 s_off[kCodes3];
    fill_cell_offsets3(P, s_off);
    unsigned long long step;
    if constexpr (FUSED) {
        const bool back = cur->halt_now || !cur->halted;  // as in pair_list_kernel
        if (!fused_pair_begin(P, next, cur)) {
            const uint32_t s = lb * kBlock + threadIdx.x;
            if (O.second && back && X.pos != O.pos && s < P.n) O.pos[s] = X.pos[s];
            return;
        }
        step = cur->step;
    } else if constexpr (FIRST) {
        if (!list_step_begin(P, next, cur, dslots, step)) return;
    } else {
        if (!list_step_goes(cur)) return;
        if (list_build_overflowed(next, cur)) return;
        step = cur->step;
    }
    __syncthreads();  // the offset table
    maxslots += (uint32_t)(step & 1) * kDtSet;
    const uint32_t s = lb * kBlock + threadIdx.x;
    const bool live = s < P.n;
    const ListPair<R, CONT, ALL> K(P);
    ListSums3<R> S;
    bool overflow = false;
    real4<R> vaj{};
    ListRec<R> rj{};
    if (live) {
        vaj = X.va[s];
        rj = rec[s];
    }
    const uint32_t cnt = rj.pr.w != R(0) ? nbc[s] : 0u;  // 0: died since the build
    const uint32_t cap = P.max_nbr - 1;
    {
        const bool capped = __ballot(cnt > cap) != 0;  // some list of the wave may hold more than cap neighbours
        const CutFP32 C = cut_band(P);
        uint32_t hits = 0;
        auto entry = [&](uint32_t k, uint32_t e, const real4<R>& nr, const real4<R>& pr, const real4<R>& va) {
            R dx, dy, dz;
            const bool in = list_cut3(P, C, s_off, e, nr, rj.nr, s, X.pos, dx, dy, dz);
            const bool hit = in & (pr.w != R(0)) & (k < cnt);
            bool take = hit;
            if (capped) {
                take = hit & (hits < cap);
                overflow |= hit & !take;
                hits += take ? 1u : 0u;
            }
            list_pair_term3<R>(K, S, take, dx, dy, dz, nr, pr, va, vaj, rj.pr, rj.nr.w);
        };
        if constexpr (sizeof(R) == 8) {
            constexpr uint32_t G = CONT ? 3 : 4;
            __shared__ uint4 s_rec[kBlock / kWave][G * (CONT ? 6 : 4) * kWave];
            uint4* buf = s_rec[wave_of_block()];
            const WaveGather<4, 64, kSlotMask3> of_rec(rec, buf);
            auto body = [&](uint32_t k, const uint32_t (&e)[G], const auto& w) {
#pragma unroll
                for (uint32_t u = 0; u < G; ++u) {
                    real4<R> va{};
                    if constexpr (CONT) va = record_real4(w[u] + 4, R(0));
                    entry(k + u, e[u], record_real4(w[u], R(0)), record_real4(w[u] + 2, R(0)), va);
                }
            };
            if constexpr (CONT) {
                using Va = WaveGather<2, 32, kSlotMask3>;
                const WaveGatherBoth<WaveGather<4, 64, kSlotMask3>, Va> both{of_rec, Va(X.va, buf + G * 4 * kWave)};
                gather_rounds<1, G>(P, nbl, both, s, 0, cnt, body);
            } else {
                gather_rounds<1, G>(P, nbl, of_rec, s, 0, cnt, body);
            }
            // a dead particle's lane went along with its wave's: its density is
            // 0, so that a pair of dead particles gives no number
            if (cnt == 0) S = ListSums3<R>();
        } else if (cnt) {
            constexpr uint32_t G = 6;
            list_rounds<1, G>(ListRowsVector(P, nbl, s), 0, cnt, [&](uint32_t k, uint32_t (&e)[G], auto& load) {
                ListRec<R> r[G];
                real4<R> va[G]{};
                uint32_t en[G];
#pragma unroll
                for (uint32_t u = 0; u < G; ++u) {
                    r[u] = rec[e[u] & kSlotMask3];
                    if (K.cont) va[u] = X.va[e[u] & kSlotMask3];
                }
                load(en);
#pragma unroll
                for (uint32_t u = 0; u < G; ++u) {
                    entry(k + u, e[u], r[u].nr, r[u].pr, va[u]);
                    e[u] = en[u];
                }
            });
        }
    }
    if (!FUSED && overflow) atomicOr(&next->nbr_overflow, 1u);
    const R mF = (R)P.lp_mF, mW = K.xsph_on ? (R)P.lp_mW : R(0);
    const R ax = S.ljx + mF * S.sx;
    const R ay = -(R)P.g + S.ljy + mF * S.sy;
    const R az = S.ljz + mF * S.sz;
    const R drho = mF * S.sd;
    const R amu = (R)P.h * -S.xmin;
    list_dt_maxima<R>(P, live ? (double)ax * ax + (double)ay * ay + (double)az * az : 0.0, live ? amu : R(0), maxslots,
                      lb);
    if (live) {
        real4<R> d;
        d.x = ax;
        d.y = ay;
        d.z = az;
        d.w = drho;
        der[s] = d;
        real4<R> x;
        x.x = mW * S.xx;
        x.y = mW * S.xy;
        x.z = mW * S.xz;
        x.w = amu;
        xs[s] = x;
        if (P.density_treatment != 0) pres[s] = eos_p<R>(vaj.w, (R)P.rho0, (R)P.eos_B);
    }
    if constexpr (FUSED) {
        uint32_t outside = 0, bad = 0;
        double moved2 = 0.0;
        if (live) {
            Ctrl c{};  // what whole_step reads of it without a wave maker
            c.cur_first = step == 0;
            const real4<R> d{ax, ay, az, drho}, x{mW * S.xx, mW * S.xy, mW * S.xz, amu};
            real4<R> pr{};
            const double4 p0 = X.pos[s];
            pr.w = (int)p0.w != 0 ? fabs(rj.pr.w)  // the summed density
                                  : dead_density<R>(P, density_w0_3<R>(P), vaj.w, cur->cur_renorm != 0);
            moved2 = step_listed3<R>(P, c, s, p0, vaj, pr, 0u, O.home[s], d, x, cur->cur_dt_const, O, outside,
                                     bad);
        }
        finish_listed(P, O.flags, step, outside, bad, moved2, dslots, lb);
    }
}

// whole_step of every slot from X into A (in place on list steps), the
// cell key for the next build, the step's largest displacement, and the
// next step's records (dens only where the summation pass reads it); the
// accelerations are in A.ad already, as in integrate_list_kernel.
template <class R>
__global__ void __launch_bounds__(kBlock) integrate_list3_kernel(StepParams P, Ctrl* next, const Ctrl* cur,
                                                                 ListState3<R> X, const real4<R>* __restrict__ xs,
                                                                 ListRec<R>* __restrict__ rec,
                                                                 real4<R>* __restrict__ dens,
                                                                 const uint32_t* __restrict__ home, StateA3<R> A,
                                                                 uint32_t* __restrict__ key_next,
                                                                 unsigned long long* maxslots,
                                                                 unsigned long long* dslots, Ctrl* keep) {
    const uint32_t s0 = blockIdx.x * kBlock + threadIdx.x;
    const bool live = s0 < P.n;
    const uint32_t s = live ? s0 : P.n - 1;
    const real4<R> d = A.ad[s];
    const real4<R> x = xs[s];
    const double4 p0 = X.pos[s];
    const real4<R> va = X.va[s];
    const uint32_t h = home[s];
    real4<R> pr{};
    if (P.density_treatment == 0) pr.w = fabs(rec[s].pr.w);  // the summed density
    const Ctrl& c = *cur;
    double dt;
    if (!list_dt(P, next, cur, maxslots, dt, keep)) return;
    uint32_t outside = 0, bad = 0;
    double moved2 = 0.0;
    if (live) {
        const bool reordered = A.oid != X.oid;
        const uint32_t oid = reordered || step_needs_oid(P, c, (int)p0.w) ? X.oid[s] : 0u;
        if (P.density_treatment == 0 && (int)p0.w == 0)
            pr.w = dead_density<R>(P, density_w0_3<R>(P), va.w, c.cur_renorm != 0);
        moved2 = step_listed3<R>(P, c, s, p0, va, pr, oid, h, d, x, dt,
                                 ListOut3<R>{A.pos, A.va, rec, dens, home, key_next, next, false}, outside, bad);
        if (reordered) A.oid[s] = oid;
    }
    finish_listed(P, next, c.step, outside, bad, moved2, dslots, blockIdx.x);
}

}  // namespace rrsph
