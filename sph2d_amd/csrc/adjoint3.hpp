// Discrete adjoint of the FP64 3D step: the 2D adjoint (adjoint.hpp) with a
// z component, the state of step3d.hpp (positions carry the type), the
// wave-uniform neighbour walk, and a segmented piston whose paddles each
// collect their own velocity adjoint.
//
// Adjoint state per particle (original order, 12 doubles):
//   lam = (r x y z, v x y z, rho, a_prev x y z, drho_prev, 0)
// Output adjoints of the step (sorted order), packed by adj_prep3 with the
// state a neighbour's pair adjoint reads into one record per slot (AdjRec3):
//   oa = (a x y z, drho),  ox = (av x y z)
// Gauges: gauge g sits at (x_g, z_g) and weighs fluid particles by
// w = (1 - ((x - x_g)^2 + (z - z_g)^2) / R^2)^3 inside the disc of radius R;
// eta_g = y_ref + tau log(sum w e / sum w), e = exp((y - y_ref) / tau).
#pragma once

#include "adjoint.hpp"
#include "list_step3.hpp"
#include "step3d.hpp"

namespace rrsph {

constexpr uint32_t kLam3 = 12;
constexpr uint32_t kDirect3 = 8;

// What the pair adjoint of a neighbour reads of slot s, in one record:
// the output adjoints oa = (a x y z, drho) and ox = (av x y z), p / R^2,
// the velocity v and the predicted (u, R): 128 bytes in FP64.  The FP32
// step's record is 64 bytes, two slots per cache line (a hit's gather costs
// by the lines it touches, and the neighbours of a particle lie in runs of
// slots): the state in its FP32 and the adjoints rounded to FP32 (the
// arithmetic stays FP64).  The position comes from the packed position
// array, whose lines the neighbour walk has just read.
template <class R> struct AdjRec3;
template <> struct alignas(128) AdjRec3<double> {
    double4 oa;
    double ox, oy, oz, pw;
    double4 v;  // (v x y z, unused)
    double4 u;  // (u x y z, R)
};
template <> struct alignas(64) AdjRec3<float> {
    float4 vp;  // (v x y z, p / R^2)
    float4 u;   // (u x y z, R)
    float4 oa;
    float4 ox;  // (av x y z, unused)
};
static_assert(sizeof(AdjRec3<float>) == 64 && sizeof(AdjRec3<double>) == 128, "words of a wave gather");

// The fields of a record, widened to FP64, with its position.
struct AdjHit3 {
    double4 pos, v, u, oa, ox;
    double pw;
};
__device__ __forceinline__ AdjHit3 adj_hit3(const AdjRec3<double>& r, const double4& pos) {
    return AdjHit3{pos, r.v, r.u, r.oa, make_double4(r.ox, r.oy, r.oz, 0.0), r.pw};
}
__device__ __forceinline__ AdjHit3 adj_hit3(const AdjRec3<float>& r, const double4& pos) {
    return AdjHit3{pos,
                   make_double4(r.vp.x, r.vp.y, r.vp.z, 0.0),
                   make_double4(r.u.x, r.u.y, r.u.z, r.u.w),
                   make_double4(r.oa.x, r.oa.y, r.oa.z, r.oa.w),
                   make_double4(r.ox.x, r.ox.y, r.ox.z, 0.0),
                   (double)r.vp.w};
}

__device__ __forceinline__ AdjParticle<3> adj_particle(const AdjHit3& h, int t) {
    return AdjParticle<3>{{h.pos.x, h.pos.y, h.pos.z}, {h.u.x, h.u.y, h.u.z},    {h.v.x, h.v.y, h.v.z},
                          {h.oa.x, h.oa.y, h.oa.z},    {h.ox.x, h.ox.y, h.ox.z}, h.u.w,
                          h.pw,                        h.oa.w,                   t};
}

struct GaugeSpec3 {
    GaugeSpec g;
    double z[kMaxGauges];
};

__device__ __forceinline__ double gauge_weight3(const GaugeSpec3& G, uint32_t g, double x, double z, double inv_r2,
                                                double& dx, double& dz) {
    dx = x - G.g.x[g];
    dz = z - G.z[g];
    const double u = 1.0 - (dx * dx + dz * dz) * inv_r2;
    return u > 0.0 ? u : 0.0;
}

// Block partial sums (sum w e, sum w) of every gauge (layout of
// gauge_block_sums).
__global__ void __launch_bounds__(kBlock) smooth_gauge_partials3(uint32_t n, const double4* __restrict__ pos,
                                                                 GaugeSpec3 G, double* __restrict__ partials,
                                                                 size_t stride) {
    __shared__ GaugeLds L;
    // row y of the grid: the state y strides further on, its partials in a row of their own
    pos = (const double4*)((const char*)pos + blockIdx.y * stride);
    partials += (size_t)blockIdx.y * 2 * G.g.n * gridDim.x;
    gauge_lds_clear(G.g, L);
    const double inv_r2 = 1.0 / (G.g.radius * G.g.radius);
    for (uint32_t base = blockIdx.x * kBlock; base < n; base += gridDim.x * kBlock) {
        const uint32_t s = base + threadIdx.x;
        bool in = false;
        double4 p = make_double4(0, 0, 0, 0);
        if (s < n) {
            p = pos[s];
            in = (int)p.w == G.g.ptype;
        }
        auto d2 = [&](uint32_t g) {
            const double dx = p.x - G.g.x[g], dz = p.z - G.z[g];
            return dx * dx + dz * dz;
        };
        gauge_chunk_sums(G.g, in, p.y, d2, inv_r2, L);
    }
    gauge_block_store(G.g, L, partials);
}

// (gx, gy, gz) = sum_g eta_bar[g] d eta_g / d r at p; false outside every window.
__device__ __forceinline__ bool gauge_gradient3(const GaugeSpec3& G, const double4& p,
                                                const double* __restrict__ eta_bar, const double* __restrict__ zsum,
                                                const double* __restrict__ wsum, double& gx, double& gy, double& gz) {
    const double inv_r2 = 1.0 / (G.g.radius * G.g.radius);
    gx = gy = gz = 0;
    bool seen = false;  // inside a window: only those particles update lam
    for (uint32_t g = 0; g < G.g.n; ++g) {
        double dx, dz;
        const double u = gauge_weight3(G, g, p.x, p.z, inv_r2, dx, dz);
        if (!(u > 0.0) || !(wsum[g] > 0.0) || eta_bar[g] == 0.0) continue;
        seen = true;
        const double w = u * u * u;
        const double wr = -6.0 * inv_r2 * u * u;  // dw/dx = wr dx, dw/dz = wr dz
        const double e = exp((p.y - G.g.y_ref) / G.g.tau);
        const double z = zsum[g], ws = wsum[g];
        const double c = eta_bar[g] * G.g.tau * wr * (e / z - 1.0 / ws);
        gy += eta_bar[g] * w * e / z;
        gx += c * dx;
        gz += c * dz;
    }
    return seen;
}

// lam[oid].r += sum_g eta_bar[g] d eta_g / d r (state in sorted order).
__global__ void __launch_bounds__(kBlock) smooth_gauge_grad3(uint32_t n, const double4* __restrict__ pos,
                                                             const uint32_t* __restrict__ oid, GaugeSpec3 G,
                                                             const double* __restrict__ eta_bar,
                                                             const double* __restrict__ zsum,
                                                             const double* __restrict__ wsum,
                                                             double* __restrict__ lam) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= n) return;
    const double4 p = pos[s];
    if ((int)p.w != G.g.ptype) return;
    double gx, gy, gz;
    if (!gauge_gradient3(G, p, eta_bar, zsum, wsum, gx, gy, gz)) return;
    double* l = lam + kLam3 * (size_t)oid[s];
    l[0] += gx;
    l[1] += gy;
    l[2] += gz;
}

// Cell keys of a restored FP64 3D state (dead particles get the dead key).
__global__ void __launch_bounds__(kBlock) state_keys3_kernel(StepParams P, const double4* __restrict__ pos,
                                                             uint32_t* __restrict__ key_next) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= P.n) return;
    uint32_t bad = 0;
    const double4 p = pos[s];
    key_next[s] = (int)p.w == 0 ? P.ncells : cell_key3(P, p.x, p.y, p.z, bad);
}

// whole_step reverse (WholeStep.cpp:19-61 with the boundary motion of
// cl/TimeIntegration.cl:190-245).  piston_sum[g] += adjoint of paddle g's
// velocity (one entry per paddle of this step).
// PREDICT: B's positions, velocities and indices are a kept state in the
// step's slot order and ad its last accelerations; the prediction, pressure
// and p / rho^2 that reorder3_kernel gives are made here (943,906 particles
// FP32: a reorder of 27 us and 64 before, 67 now).
template <class R, bool PREDICT>
__global__ void __launch_bounds__(kBlock) adj_prep3(StepParams P, AdjStep T, StateB3<R> B,
                                                    const real4<R>* __restrict__ ad,
                                                    const double* __restrict__ lam_in, AdjRec3<R>* __restrict__ rec,
                                                    double* __restrict__ direct, double* __restrict__ piston_sum,
                                                    const uint32_t* __restrict__ home, float4* __restrict__ nearf) {
    __shared__ double s_p[kMaxSegments][kBlock / kWave];
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    double pist = 0.0;
    int seg = 0;
    if (s < P.n) {
        const uint32_t o = B.oid[s];
        const double4 ps = B.pos[s];
        const double* l = lam_in + kLam3 * (size_t)o;
        const double rx = l[0], ry = l[1], rz = l[2], vx = l[3], vy = l[4], vz = l[5], rb = l[6];
        const double ax = l[7], ay = l[8], az = l[9], db = l[10];
        const int t = (int)ps.w;
        const double vdt = T.first ? T.dt * 0.5 : T.dt;
        double4 oa, ox;
        double dvx = 0, dvy = 0, dvz = 0;
        if (t > 0) {
            const double tx = vx + rx * T.dt, ty = vy + ry * T.dt, tz = vz + rz * T.dt;  // updated-v adjoint
            oa = make_double4(tx * vdt + ax, ty * vdt + ay, tz * vdt + az, 0.0);
            ox = P.xsph_on ? make_double4(tx, ty, tz, 0.0) : make_double4(0, 0, 0, 0);
            dvx = tx;
            dvy = ty;
            dvz = tz;
        } else {
            oa = make_double4(ax, ay, az, 0.0);
            ox = make_double4(0, 0, 0, 0);
            const bool moving = P.boundary_motion && t < 0;
            const bool piston = moving && T.piston && o >= P.nwm_start && o < P.nwm_end && o >= P.nfluid;
            if (piston) {
                const double tv[3] = {vx + rx * T.dt, vy + ry * T.dt, vz + rz * T.dt};
                pist = tv[P.nwm_axis];
                seg = P.piston_segments > 1 ? piston_segment(P, ps.z) : 0;
            } else if (moving) {
                dvx = vx + rx * T.dt;
                dvy = vy + ry * T.dt;
                dvz = vz + rz * T.dt;
            } else {
                dvx = vx;
                dvy = vy;
                dvz = vz;
            }
        }
        if (t == 0) oa.x = oa.y = oa.z = 0.0;  // no neighbours, no acceleration dependence
        oa.w = P.density_treatment != 0 ? rb * vdt + db : 0.0;
        AdjRec3<R> r;
        const real4<R> va = B.va[s];
        real4<R> pr;
        R pw;
        if constexpr (PREDICT) {
            R p;
            pr = predict3<R>(P, va, 1, ad[s], (R)T.dt_pred, pw, p);
            B.pred[s] = pr;
            B.pres[s] = p;
        } else {
            pr = B.pred[s];
            pw = B.pw[s];
        }
        if constexpr (sizeof(R) == 4) {
            r.vp = make_float4(va.x, va.y, va.z, pw);
            r.u = pr;
            r.oa = make_float4((float)oa.x, (float)oa.y, (float)oa.z, (float)oa.w);
            r.ox = make_float4((float)ox.x, (float)ox.y, (float)ox.z, 0.f);
        } else {
            r.oa = oa;
            r.ox = ox.x;
            r.oy = ox.y;
            r.oz = ox.z;
            r.pw = pw;
            r.v = va;
            r.u = pr;
        }
        rec[s] = r;
        if (nearf) nearf[s] = near3<float>(P, ps, (float)t, home[s]);  // type in w
        double* d = direct + kDirect3 * (size_t)s;
        d[0] = rx;
        d[1] = ry;
        d[2] = rz;
        d[3] = dvx;
        d[4] = dvy;
        d[5] = dvz;
        d[6] = rb;
        d[7] = 0.0;
    }
    for (int g = 0; g < P.piston_segments; ++g) {
        double v = seg == g ? pist : 0.0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if (__lane_id() == 0) s_p[g][threadIdx.x / kWave] = v;
    }
    __syncthreads();
    if (threadIdx.x < (uint32_t)P.piston_segments) {
        double b = 0;
        for (int w = 0; w < kBlock / kWave; ++w) b += s_p[threadIdx.x][w];
        if (b != 0.0) atomicAdd(piston_sum + threadIdx.x, b);
    }
}

// Gather over neighbours, both orientations of every pair, then the
// predict and EOS reverse; writes lam_out.  Every lane of a block runs the
// wave-uniform walk (lanes past n walk empty ranges).  LISTS: the
// neighbours come from the lists of the build the step read (nbl, nbc, in
// B's slot order) instead of the cell walk, and the gradient of the gauges of
// the state it reverses into is added (eta_bar null: none).
template <class R, bool LISTS>
__global__ void __launch_bounds__(kBlock) adj_pair3(StepParams P, AdjStep T, StateB3<R> B,
                                                    const uint32_t* __restrict__ skey,
                                                    const uint32_t* __restrict__ LB,
                                                    const uint32_t* __restrict__ nbl,
                                                    const uint32_t* __restrict__ nbc,
                                                    const AdjRec3<R>* __restrict__ rec,
                                                    const double* __restrict__ direct, double* __restrict__ lam_out,
                                                    uint32_t* __restrict__ overflow_flag,
                                                    const float4* __restrict__ nearf, GaugeSpec3 G,
                                                    const double* __restrict__ eta_bar,
                                                    const double* __restrict__ zsum,
                                                    const double* __restrict__ wsum) {
    // FP32 step over lists: entries decided and hits' r_i - r_k taken from
    // the near records (16 bytes, as the list pass does) instead of the FP64
    // positions (32 bytes)
    constexpr bool kNear = LISTS && sizeof(R) == 4;
    __shared__ uint32_t hits[kAdjChunk * kBlock];
    __shared__ float4 s_off[kNear ? kCodes3 : 1];
    constexpr bool kGathered = LISTS && sizeof(R) == 8;
    __shared__ uint4 s_rec[kBlock / kWave][kGathered ? 8 * kWave : 1];
    // XCD-aware: each XCD walks one contiguous slice of the slots
    const uint32_t lb = xcd_block(P.blocks_per_xcd);
    if (lb >= P.nblocks) return;
    if constexpr (kNear) {
        fill_cell_offsets3(P, s_off);
        __syncthreads();
    }
    const uint32_t s = lb * kBlock + threadIdx.x;
    const bool live = s < P.n;
    const uint32_t sc = live ? s : P.n - 1;
    const AdjConsts K = adj_consts(P);
    const double4 pk = B.pos[sc];
    const double4 vak = to_d4<R>(B.va[sc]);    // (v, rho)
    const double4 prk = to_d4<R>(B.pred[sc]);  // (u, R)
    const double pres_k = B.pres[sc];
    const AdjHit3 hk = adj_hit3(rec[sc], pk);
    float4 nk{};
    if constexpr (kNear) nk = nearf[sc];
    const int tk = (int)pk.w;
    // (the own velocities and p / R^2 are those of its record)
    const AdjParticle<3> own = adj_particle(hk, tk);
    AdjSums<3> S;
    bool overflow = false;
    uint32_t* my = hits + threadIdx.x;
    // Over lists in FP64 the wave fetches the records of its lanes' next hits
    // together (WaveGather) while it works on their last ones: lanes loading their
    // own made 10 accesses of up to 64 lines a hit, which bound the loop
    // (509,126 particles 503 -> 427 us).  In FP32, 5 accesses a hit, it made no
    // difference (943,906 particles: 623 us, 638 and with two records in flight
    // 632 gathered), nor did 3 waves per SIMD, which spill (791).
    auto flush = [&](uint32_t nh) {
        if constexpr (kGathered) {
            const uint32_t nmax = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_max_u32(nh));
            if (nmax == 0) return;
            auto hit = [&](uint32_t u) { return u < nh ? my[u * kBlock] : sc; };  // past its hits: its own slot
            uint4* buf = s_rec[wave_of_block()];
            using Half = WaveGather<4, sizeof(AdjRec3<R>), kSlotMask3>;
            const WaveGatherBoth<Half, Half> src{Half(rec, buf), Half((const char*)rec + 64, buf + 4 * kWave)};
            uint32_t in = hit(0), next = hit(1);
            double4 pn{};
            auto fetch = [&]() {
                pn = B.pos[in];
                src.fetch(0, in);
            };
            fetch();
#pragma unroll 1
            for (uint32_t u = 0; u < nmax; ++u) {
                uint4 w[8];
                wait_loads();
                src.read(0, w);
                const double4 p = pn;
                in = next;
                next = hit(u + 2);
                wait_lds();  // the records are in registers: the next ones may land
                __builtin_amdgcn_sched_barrier(0);
                if (u + 1 < nmax) fetch();
                if (u >= nh) continue;
                AdjRec3<R> r;
                __builtin_memcpy(&r, w, sizeof r);
                const double e[3] = {p.x - pk.x, p.y - pk.y, p.z - pk.z};  // r_i - r_k
                adj_pair_term<3>(K, own, adj_particle(adj_hit3(r, p), (int)p.w), e, S);
            }
        } else {
            // the loads of hit u + 1 are issued before the arithmetic of hit u (the
            // kernel runs at 2 waves per SIMD either way, so the registers are free;
            // a second record in flight needs more registers than 2 waves leave)
            if (nh == 0) return;
            // kNear: the hit list holds whole entries (slot and home-cell code)
            uint32_t in = my[0];
            AdjRec3<R> rn = rec[kNear ? in & kSlotMask3 : in];
            double4 pn{};
            float4 qn{};
            if constexpr (kNear) qn = nearf[in & kSlotMask3];
            else pn = B.pos[in];
#pragma unroll 1
            for (uint32_t u = 0; u < nh; ++u) {
                const AdjHit3 h = adj_hit3(rn, pn);
                int ti;
                double e[3];  // r_i - r_k
                if constexpr (kNear) {
                    const float4 o = s_off[in >> kSlotBits3];
                    e[0] = (double)((qn.x - nk.x) + o.x);
                    e[1] = (double)((qn.y - nk.y) + o.y);
                    e[2] = (double)((qn.z - nk.z) + o.z);
                    ti = (int)qn.w;
                } else {
                    e[0] = h.pos.x - pk.x;
                    e[1] = h.pos.y - pk.y;
                    e[2] = h.pos.z - pk.z;
                    ti = (int)h.pos.w;
                }
                in = my[min(u + 1, nh - 1) * kBlock];
                rn = rec[kNear ? in & kSlotMask3 : in];
                if constexpr (kNear) qn = nearf[in & kSlotMask3];
                else pn = B.pos[in];
                adj_pair_term<3>(K, own, adj_particle(h, ti), e, S);
            }
        }
    };
    if constexpr (kNear)
        collect_near3<kAdjChunk>(P, live && tk != 0, P.max_nbr - 1, sc, s_off, nk, nearf, B.pos, nbl, nbc, my,
                                 overflow, flush);
    else if (LISTS)
        collect_listed3<kAdjChunk>(P, live && tk != 0, P.max_nbr - 1, sc, pk, B.pos, nbl, nbc, my, overflow, flush);
    else
        collect_neighbours3<kAdjChunk>(P, live && tk != 0, P.max_nbr - 1, sc, skey[sc], pk, B.pos, LB, my,
                                       overflow, flush);
    if (overflow) atomicOr(overflow_flag, 1u);
    if (!live) return;
    double l[kLam3];
    adj_predict<3>(P, T.dt_pred, S, prk.w, pres_k, vak.w, direct + kDirect3 * (size_t)s, l);
    l[kLam3 - 1] = 0.0;
    if (LISTS && eta_bar && tk == G.g.ptype) {
        double gx, gy, gz;
        if (gauge_gradient3(G, pk, eta_bar, zsum, wsum, gx, gy, gz)) {
            l[0] += gx;
            l[1] += gy;
            l[2] += gz;
        }
    }
    double2* out = (double2*)(lam_out + kLam3 * (size_t)B.oid[s]);
#pragma unroll
    for (uint32_t c = 0; c < kLam3 / 2; ++c) out[c] = make_double2(l[2 * c], l[2 * c + 1]);
}

}  // namespace rrsph
