// Discrete adjoint of the FP64 WCSPH step (continuity density, cubic
// spline, pressure p_i/rho_i^2 + p_j/rho_j^2, artificial viscosity, Lennard-
// Jones walls, XSPH, boundary motion with the Fourier piston), and the
// smooth gauge surrogate it is driven by.
//
// The step maps S_n = (r, v, rho, a_prev, drho_prev) to S_{n+1}:
//   u = v + a_prev dt/2, R = rho + drho_prev dt/2, p = EOS(rho), P = p / R^2
//   drho_j = m sum_i F_ij (v_i - v_j).e        (e = r_i - r_j, grad W = F e)
//   a_j    = -g y + LJ_j + m sum_i F_ij coef_ij e,  coef = P_i + P_j + AV_ij
//   av_j   = 2 eps m sum_{i fluid} (u_i - u_j) W_ij / (R_i + R_j)
//   whole_step (dt/2 for v and rho on the first step), piston velocity on
//   the wave-maker particles, a_prev' = a, drho_prev' = drho.
// Neighbour sets are those of the step (the kernel, its gradient, the LJ
// force and the AV switch are continuous at their thresholds, so the sets
// are constant on the pieces the derivative is taken on).
//
// Kernels (sorted order of the replayed step, adjoints stored in original
// particle order, lam = (r, v, rho, a_prev, drho_prev) adjoints, 8 doubles):
//   adj_prep  whole_step reverse: output adjoints (a, av, drho) per particle,
//             the direct input adjoints, and the piston sum
//             s_n = sum over wave-maker particles of (v' + dt r')-adjoints
//   adj_pair  gather over neighbours: every pair is differentiated in both
//             orientations (the particle as owner of the sum and as
//             neighbour), then predict and EOS reverse; writes lam_n
//   adj_prep_list, adj_pair_list  the same on the lists of the build that the
//             step read, in its slot order
//   smooth_gauge_* the surrogate eta_g = y_ref + tau log(sum w e / sum w)
//             with w = (1 - (x - x_g)^2 / R^2)^3 inside |x - x_g| < R and
//             e = exp((y - y_ref) / tau); tau -> 0 gives max y in the window,
//             the definition of HeightTesting::maxInLayer
//             (tools/WaterProfile/include/HeightTesting.h:25-54)
#pragma once

#include "device_common.hpp"
#include "list_step.hpp"
#include "step_kernels.hpp"

namespace rrsph {

constexpr uint32_t kMaxGauges = 64;
constexpr uint32_t kAdjChunk = 32;

// The adjoint runs in FP64 on the state of either precision (an FP32 state
// is the FP32 step's trajectory; its Jacobian is taken in FP64).
template <class R> __device__ __forceinline__ double4 to_d4(const real4<R>& v) {
    return make_double4((double)v.x, (double)v.y, (double)v.z, (double)v.w);
}

struct GaugeSpec {
    uint32_t n;          // gauges
    int32_t ptype;       // particle type the gauge looks at
    double radius, tau, y_ref;
    double x[kMaxGauges];
};

// ------------------------------------------------------------------ smooth gauges
// Block partial sums (sum w e, sum w) of every gauge, gauge-major:
// partials[(2 g) nb + b] = sum w e, partials[(2 g + 1) nb + b] = sum w of
// block b (nb = gridDim.x).  The grid is at most kGaugeBlocks blocks; block
// b sums the particle chunks b, b + nb, b + 2 nb, ... of kBlock particles.
// A chunk with no particle inside any window adds nothing and skips the
// per-gauge reductions (its sums are exactly zero).
constexpr uint32_t kGaugeBlocks = 1024;

struct GaugeLds {
    double z[kBlock / kWave][kMaxGauges], w[kBlock / kWave][kMaxGauges];
};

__device__ __forceinline__ void gauge_lds_clear(const GaugeSpec& G, GaugeLds& L) {
    for (uint32_t i = threadIdx.x; i < (kBlock / kWave) * G.n; i += kBlock) {
        L.z[i / G.n][i % G.n] = 0.0;
        L.w[i / G.n][i % G.n] = 0.0;
    }
    __syncthreads();
}

// One chunk: every thread of the block calls it (uniform control flow).
template <class D2>
__device__ __forceinline__ void gauge_chunk_sums(const GaugeSpec& G, bool in, double y, D2&& d2, double inv_r2,
                                                 GaugeLds& L) {
    const uint32_t wave = threadIdx.x / kWave;
    bool near = false;
    for (uint32_t g = 0; g < G.n; ++g) near |= in && d2(g) * inv_r2 < 1.0;
    if (!__syncthreads_or(near)) return;
    for (uint32_t g = 0; g < G.n; ++g) {
        const double u = 1.0 - d2(g) * inv_r2;
        const double w = in && u > 0.0 ? u * u * u : 0.0;
        double z = w > 0.0 ? w * exp((y - G.y_ref) / G.tau) : 0.0;
        double ww = w;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            z += __shfl_xor(z, off);
            ww += __shfl_xor(ww, off);
        }
        if (__lane_id() == 0) {  // each wave owns its row
            L.z[wave][g] += z;
            L.w[wave][g] += ww;
        }
    }
}

__device__ __forceinline__ void gauge_block_store(const GaugeSpec& G, GaugeLds& L, double* __restrict__ partials) {
    __syncthreads();
    const uint32_t nb = gridDim.x;
    for (uint32_t g = threadIdx.x; g < G.n; g += kBlock) {
        double z = 0, ww = 0;
        for (uint32_t w = 0; w < kBlock / kWave; ++w) {
            z += L.z[w][g];
            ww += L.w[w][g];
        }
        partials[(size_t)(2 * g) * nb + blockIdx.x] = z;
        partials[(size_t)(2 * g + 1) * nb + blockIdx.x] = ww;
    }
}

__host__ __device__ inline uint32_t gauge_blocks(uint32_t n) {
    const uint32_t chunks = (n + kBlock - 1) / kBlock;
    return chunks < kGaugeBlocks ? (chunks ? chunks : 1u) : kGaugeBlocks;
}

template <class R>
__global__ void __launch_bounds__(kBlock) smooth_gauge_partials(uint32_t n, const double2* __restrict__ pos,
                                                                const real4<R>* __restrict__ va, GaugeSpec G,
                                                                double* __restrict__ partials, size_t stride) {
    __shared__ GaugeLds L;
    // row y of the grid: the state y strides further on, its partials in a row of their own
    pos = (const double2*)((const char*)pos + blockIdx.y * stride);
    va = (const real4<R>*)((const char*)va + blockIdx.y * stride);
    partials += (size_t)blockIdx.y * 2 * G.n * gridDim.x;
    gauge_lds_clear(G, L);
    const double inv_r2 = 1.0 / (G.radius * G.radius);
    for (uint32_t base = blockIdx.x * kBlock; base < n; base += gridDim.x * kBlock) {
        const uint32_t s = base + threadIdx.x;
        bool in = false;
        double x = 0, y = 0;
        if (s < n) {
            const double2 p = pos[s];
            in = (int)va[s].w == G.ptype;
            x = p.x;
            y = p.y;
        }
        auto d2 = [&](uint32_t g) { return (x - G.x[g]) * (x - G.x[g]); };
        gauge_chunk_sums(G, in, y, d2, inv_r2, L);
    }
    gauge_block_store(G, L, partials);
}

// One block per gauge: each thread sums a fixed stride of the block
// partials, then a fixed shuffle tree and wave order (deterministic);
// writes eta[g], Z[g] = sum w e and Wsum[g] = sum w.  With ctrl, the three
// arrays are a tape of nsteps rows of kMaxGauges and the row is the step
// index of the step just launched - base, as adj_record takes it.
__global__ void __launch_bounds__(kBlock) smooth_gauge_final(uint32_t nblocks, GaugeSpec G,
                                                             const double* __restrict__ partials,
                                                             double* __restrict__ eta, double* __restrict__ zsum,
                                                             double* __restrict__ wsum, const Ctrl* __restrict__ ctrl,
                                                             uint64_t base, uint32_t nsteps) {
    __shared__ double s_z[kBlock / kWave], s_w[kBlock / kWave];
    const uint32_t g = blockIdx.x;
    if (g >= G.n) return;
    partials += (size_t)blockIdx.y * 2 * G.n * nblocks;  // row y of the grid: the next state's
    eta += (size_t)blockIdx.y * kMaxGauges;
    zsum += (size_t)blockIdx.y * kMaxGauges;
    wsum += (size_t)blockIdx.y * kMaxGauges;
    if (ctrl) {
        const size_t row = (size_t)min(ctrl->step - base, (uint64_t)nsteps - 1) * kMaxGauges;
        eta += row;
        zsum += row;
        wsum += row;
    }
    const double* pz = partials + (size_t)(2 * g) * nblocks;
    const double* pw = partials + (size_t)(2 * g + 1) * nblocks;
    double z = 0, ww = 0;
    for (uint32_t b = threadIdx.x; b < nblocks; b += kBlock) {
        z += pz[b];
        ww += pw[b];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        z += __shfl_xor(z, off);
        ww += __shfl_xor(ww, off);
    }
    if (__lane_id() == 0) {
        s_z[threadIdx.x / kWave] = z;
        s_w[threadIdx.x / kWave] = ww;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        z = 0;
        ww = 0;
        for (uint32_t w = 0; w < kBlock / kWave; ++w) {
            z += s_z[w];
            ww += s_w[w];
        }
        eta[g] = ww > 0.0 ? G.y_ref + G.tau * log(z / ww) : 0.0;
        zsum[g] = z;
        wsum[g] = ww;
    }
}

// (gx, gy) = sum_g eta_bar[g] d eta_g / d r at p; false outside every window.
__device__ __forceinline__ bool gauge_gradient(const GaugeSpec& G, double2 p, const double* __restrict__ eta_bar,
                                               const double* __restrict__ zsum, const double* __restrict__ wsum,
                                               double& gx, double& gy) {
    const double inv_r2 = 1.0 / (G.radius * G.radius);
    gx = gy = 0;
    bool seen = false;  // inside a window: only those particles update lam
    for (uint32_t g = 0; g < G.n; ++g) {
        const double dx = p.x - G.x[g];
        const double u = 1.0 - dx * dx * inv_r2;
        if (!(u > 0.0) || !(wsum[g] > 0.0) || eta_bar[g] == 0.0) continue;
        seen = true;
        const double w = u * u * u;
        const double wp = -6.0 * dx * inv_r2 * u * u;  // dw/dx
        const double e = exp((p.y - G.y_ref) / G.tau);
        const double z = zsum[g], ws = wsum[g];
        gy += eta_bar[g] * w * e / z;
        gx += eta_bar[g] * G.tau * wp * (e / z - 1.0 / ws);
    }
    return seen;
}

// lam[oid].r += sum_g eta_bar[g] d eta_g / d r (state in sorted order).
template <class R>
__global__ void __launch_bounds__(kBlock) smooth_gauge_grad(uint32_t n, const double2* __restrict__ pos,
                                                            const real4<R>* __restrict__ va,
                                                            const uint32_t* __restrict__ oid, GaugeSpec G,
                                                            const double* __restrict__ eta_bar,
                                                            const double* __restrict__ zsum,
                                                            const double* __restrict__ wsum,
                                                            double* __restrict__ lam) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= n) return;
    if ((int)va[s].w != G.ptype) return;
    double gx, gy;
    if (!gauge_gradient(G, pos[s], eta_bar, zsum, wsum, gx, gy)) return;
    double* l = lam + 8 * (size_t)oid[s];
    l[0] += gx;
    l[1] += gy;
}

// Cell keys of a restored FP64 state (dead particles get the dead key).
template <class R>
__global__ void __launch_bounds__(kBlock) state_keys_kernel(StepParams P, const double2* __restrict__ pos,
                                                            const real4<R>* __restrict__ va,
                                                            uint32_t* __restrict__ key_next) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= P.n) return;
    uint32_t bad = 0;
    const double2 p = pos[s];
    key_next[s] = (int)va[s].w == 0 ? P.ncells : cell_key(P, p.x, p.y, bad);
}

// The gradients with respect to the initial state as a caller takes them:
// r and v as D-tuples, rho, from the adjoint state lam (lw doubles per
// particle, original order, beginning with r, v, rho).  At 943,906 particles
// in 3D, downloading all of lam and picking it apart on the host took 28 of
// the 41 ms of a 12-step reverse pass.
__global__ void __launch_bounds__(kBlock) unpack_gradients_kernel(uint32_t n, const double* __restrict__ lam,
                                                                  uint32_t lw, uint32_t D, double* __restrict__ gr,
                                                                  double* __restrict__ gv,
                                                                  double* __restrict__ grho) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double* l = lam + (size_t)lw * i;
    for (uint32_t c = 0; c < D; ++c) {
        gr[(size_t)D * i + c] = l[c];
        gv[(size_t)D * i + c] = l[D + c];
    }
    grho[i] = l[2 * D];
}

// ------------------------------------------------------------------ step adjoint
struct AdjStep {
    double t;         // time at the start of the step
    double dt;        // dt of whole_step and of the time advance
    double dt_pred;   // dt of predict_half_step
    uint32_t first;   // first step: v and rho advance with dt / 2
    uint32_t piston;  // the wave maker moves its particles this step
    uint32_t halted;  // the step did not run
    uint32_t pad;
};

// After a step: what its adjoint needs from the control block.
__device__ __forceinline__ AdjStep step_record(const Ctrl& c) {
    AdjStep r;
    r.t = c.cur_time;
    r.dt = c.dt_new;
    r.dt_pred = c.cur_dt;
    r.first = c.cur_first;
    r.piston = c.piston_active;
    r.halted = c.halted;
    r.pad = 0;
    return r;
}
// Record of the step just launched, at rec[k], k = its step index (the
// control block's step count, committed at the next prologue) - base,
// clamped to the tape's nsteps records: a step after a halt does not run,
// and its record lands on the halted step's, which the resumed range
// writes again.
__global__ void adj_record(const Ctrl* __restrict__ ctrl, AdjStep* __restrict__ rec, uint64_t base, uint32_t nsteps) {
    const uint64_t k = min(ctrl->step - base, (uint64_t)nsteps - 1);
    rec[k] = step_record(*ctrl);
}
// Records of every step, from the control blocks kept with the state after
// each: `first` and on, stride bytes apart, and `last`.
__global__ void __launch_bounds__(kBlock) tape_records_kernel(const char* __restrict__ first, size_t stride,
                                                              const char* __restrict__ last,
                                                              AdjStep* __restrict__ rec, uint32_t nsteps) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k < nsteps) rec[k] = step_record(*(const Ctrl*)(k + 1 < nsteps ? first + k * stride : last));
}

// whole_step reverse of one particle of type t and original index o with
// output adjoints l: out = adjoints of (a_x, a_y, av_x, av_y), drho that of
// drho; d = adjoints of (r_x, r_y, v_x, v_y, rho) that do not pass through
// the pair sums.  Returns the wave maker's velocity adjoint.
__device__ __forceinline__ double adj_whole_step(const StepParams& P, const AdjStep& T, int t, uint32_t o,
                                                 const double* __restrict__ l, double4& out, double& drho, double* d) {
    const double rx = l[0], ry = l[1], vx = l[2], vy = l[3], rb = l[4], ax = l[5], ay = l[6], db = l[7];
    const double vdt = T.first ? T.dt * 0.5 : T.dt;
    double pist = 0.0, dvx = 0, dvy = 0;
    if (t > 0) {
        const double tx = vx + rx * T.dt, ty = vy + ry * T.dt;  // adjoint of the updated v
        out.x = tx * vdt + ax;
        out.y = ty * vdt + ay;
        out.z = P.xsph_on ? tx : 0.0;
        out.w = P.xsph_on ? ty : 0.0;
        dvx = tx;
        dvy = ty;
    } else {
        out.x = ax;
        out.y = ay;
        out.z = 0.0;
        out.w = 0.0;
        const bool moving = P.boundary_motion && t < 0;
        const bool piston = moving && T.piston && o >= P.nwm_start && o < P.nwm_end && o >= P.nfluid;
        if (piston) {
            pist = P.nwm_axis == 0 ? vx + rx * T.dt : vy + ry * T.dt;
        } else if (moving) {
            dvx = vx + rx * T.dt;
            dvy = vy + ry * T.dt;
        } else {
            dvx = vx;
            dvy = vy;
        }
    }
    if (t == 0) out.x = out.y = 0.0;  // no neighbours, no acceleration dependence
    drho = P.density_treatment != 0 ? rb * vdt + db : 0.0;
    d[0] = rx;
    d[1] = ry;
    d[2] = dvx;
    d[3] = dvy;
    d[4] = rb;
    return pist;
}
// piston_sum += the block's wave-maker velocity adjoints (every thread).
__device__ __forceinline__ void adj_piston_sum(double pist, double* __restrict__ piston_sum) {
    __shared__ double s_p[kBlock / kWave];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) pist += __shfl_xor(pist, off);
    if (__lane_id() == 0) s_p[threadIdx.x / kWave] = pist;
    __syncthreads();
    if (threadIdx.x == 0) {
        double b = 0;
        for (int w = 0; w < kBlock / kWave; ++w) b += s_p[w];
        if (b != 0.0) atomicAdd(piston_sum, b);
    }
}

// whole_step reverse on the re-sorted state: out_adj, drho_adj and direct[5 s]
// as adj_whole_step gives them.
template <class R>
__global__ void __launch_bounds__(kBlock) adj_prep(StepParams P, AdjStep T, StateB<R> B,
                                                   const double* __restrict__ lam_in,
                                                   double4* __restrict__ out_adj, double* __restrict__ drho_adj,
                                                   double* __restrict__ direct, double* __restrict__ piston_sum) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    double pist = 0.0;
    if (s < P.n) {
        const uint32_t o = B.oid[s];
        double4 oa;
        double drho;
        pist = adj_whole_step(P, T, (int)B.va[s].w, o, lam_in + 8 * (size_t)o, oa, drho, direct + 5 * (size_t)s);
        out_adj[s] = oa;
        drho_adj[s] = drho;
    }
    adj_piston_sum(pist, piston_sum);
}

struct AdjConsts {
    double h, inv_h, two_inv_h, c1a, c1b, c1ah, c2, w1, w2, alpha_c, beta, two_beta, eta2, r0, lj_Dm, m, eps2;
    bool av_on, lj_on;
};
__device__ __forceinline__ AdjConsts adj_consts(const StepParams& P) {
    const double c1 = P.f_cubic / (P.h * P.h);
    AdjConsts K;
    K.h = P.h;
    K.inv_h = 1.0 / P.h;
    K.two_inv_h = 2.0 / P.h;
    K.c1a = 1.5 * c1;
    K.c1b = -2.0 * c1;
    K.c1ah = 1.5 * c1 / P.h;
    K.c2 = 0.5 * P.f_cubic / P.h;
    K.w1 = P.f_cubic;
    K.w2 = P.f_cubic / 6.0;
    K.alpha_c = P.av_alpha * P.av_c;
    K.beta = P.av_beta;
    K.two_beta = 2.0 * P.av_beta;
    K.eta2 = P.av_eta2;
    K.r0 = P.lj_r0;
    K.lj_Dm = P.lj_D / P.mass;
    K.m = P.mass;
    K.eps2 = 2.0 * P.xsph_eps;
    K.av_on = P.av_on;
    K.lj_on = P.lj_on;
    return K;
}

// What a pair's adjoint reads of a particle in D dimensions: position p,
// predicted velocity u and density R = rho^, velocity v, p / rho^2, type, and
// the output adjoints a, x (of av; 0 for all but fluid) and da (of drho).
template <int D> struct AdjParticle {
    double p[D], u[D], v[D], a[D], x[D];
    double R, pw, da;
    int t;
};
// The pair sums of a particle, over the particle mass: adjoints of r, v, u, R and p / R^2.
template <int D> struct AdjSums {
    double r[D] = {}, v[D] = {}, u[D] = {};
    double R = 0, P = 0;
    template <class F> __device__ __forceinline__ void each(F&& f) {
#pragma unroll
        for (int c = 0; c < D; ++c) {
            r[c] = f(r[c]);
            v[c] = f(v[c]);
            u[c] = f(u[c]);
        }
        R = f(R);
        P = f(P);
    }
};
template <int D> __device__ __forceinline__ double adj_dot(const double (&a)[D], const double (&b)[D]) {
    double s = a[0] * b[0];
#pragma unroll
    for (int c = 1; c < D; ++c) s = fma(a[c], b[c], s);
    return s;
}
// The pair of k and its neighbour i at e = r_i - r_k.
//
// k's own sum has the terms T1 = F (dv . e), T2 = F coef e, T4 = du W IR (i
// and k fluid: elsewhere the av-adjoints or the term vanish) and the wall
// force T3 = -e f(d) of a fluid particle near a wall one; dv = v_i - v_k, du =
// u_i - u_k, IR = 1 / (R_i + R_k), coef = P_i + P_k + A with A = 2 IR (beta mu
// - alpha c) mu, mu = h (du . e) / (d^2 + eta^2) where particles approach.
// i's sum has them at (-e, -dv, -du), entering rb, vb, ub with the opposite
// sign and Rb, Pb with the same.  Every output is linear in the owner's
// adjoints, and even (the a- and av-adjoint terms, the wall force) or odd
// (the drho-adjoint terms) in (e, dv, du), so the two make one evaluation at
// (e, dv, du) with the adjoints a_k - a_i, da_k + da_i, x_k - x_i, and for
// the wall force a_k, or -a_i where i is the fluid particle.
//
// Bound by FP64 instructions: everything along e goes through one factor
// (ce), and the mass multiplies the sums once.  Pair passes before (one
// orientation's terms written out) and now: 3D FP32, 943,906 particles, 687
// and 622 us; 2D over lists, 134,042 particles, 33.1 and 31.2 us.
template <int D>
__device__ __forceinline__ void adj_pair_term(const AdjConsts& K, const AdjParticle<D>& k, const AdjParticle<D>& i,
                                              const double (&e)[D], AdjSums<D>& S) {
#pragma clang fp contract(off)  // the same roundings in every kernel that calls it
    const double d2 = adj_dot<D>(e, e);
    const double rinv = d2 > 0.0 ? fast_rsqrt<double>(d2) : 0.0;
    const double d = d2 * rinv, q = d * K.inv_h, t = 2.0 - q, tr = t * rinv;
    const bool in = q <= 1.0;
    const double F = in ? fma(K.c1a, q, K.c1b) : -K.c2 * (t * tr);
    const double Fpe = rinv * (in ? K.c1ah : K.c2 * (tr * (tr + K.two_inv_h)));  // grad_e F = Fpe e
    const double W = in ? K.w1 * fma(q * q, fma(0.5, q, -1.0), 2.0 / 3.0) : K.w2 * (t * t * t);
    const double IR = fast_rcp<double>(i.R + k.R);
    double du[D], dv[D], a[D], x[D];
#pragma unroll
    for (int c = 0; c < D; ++c) {
        du[c] = i.u[c] - k.u[c];
        dv[c] = i.v[c] - k.v[c];
        a[c] = k.a[c] - i.a[c];
        x[c] = k.x[c] - i.x[c];
    }
    const double vr = adj_dot<D>(du, e);
    const double den = K.av_on && vr < 0.0 ? fast_rcp<double>(d2 + K.eta2) : 0.0;  // 0: no artificial viscosity
    const double hden = K.h * den, mu = hden * vr, IR2 = 2.0 * IR;
    const double A = IR2 * (fma(K.beta, mu, -K.alpha_c) * mu);
    const double coef = i.pw + k.pw + A;
    const double s1 = k.da + i.da;
    const double ae = adj_dot<D>(a, e);
    const double coefb = F * ae;
    const double mub = (IR2 * coefb) * fma(K.two_beta, mu, -K.alpha_c);
    const double vrb = mub * hden;              // adjoint of vr
    const double em = -2.0 * (mub * mu) * den;  // of d^2 in mu, along e
    const double IRx = k.t > 0 && i.t > 0 ? K.eps2 * IR : 0.0;
    const double xdu = IRx * adj_dot<D>(x, du);
    const double WI = IRx * W, s1F = s1 * F, coefF = coef * F;
    const double ce = fma(Fpe, fma(s1, adj_dot<D>(dv, e), coef * ae), fma(F, xdu, em));
#pragma unroll
    for (int c = 0; c < D; ++c) {
        S.r[c] -= fma(ce, e[c], fma(vrb, du[c], fma(s1F, dv[c], coefF * a[c])));
        S.v[c] = fma(-s1F, e[c], S.v[c]);
        S.u[c] -= fma(vrb, e[c], WI * x[c]);
    }
    S.R = fma(-IR, fma(coefb, A, W * xdu), S.R);
    S.P += coefb;
    if (K.lj_on && d < K.r0 && ((k.t > 0 && i.t < 0) || (i.t > 0 && k.t < 0))) {
        double L[D];
#pragma unroll
        for (int c = 0; c < D; ++c) L[c] = k.t > 0 ? k.a[c] : -i.a[c];
        const double rn = K.r0 * rinv, rn2 = rn * rn, rn4 = rn2 * rn2, rn12 = rn4 * rn4 * rn4, ri2 = rinv * rinv;
        const double f = K.lj_Dm * (rn12 - rn4) * ri2;
        const double g = K.lj_Dm * fma(-14.0, rn12, 6.0 * rn4) * ri2 * ri2 * adj_dot<D>(L, e);  // df/dd / d (L . e)
#pragma unroll
        for (int c = 0; c < D; ++c) S.r[c] += fma(f, L[c], g * e[c]);
    }
}
// The predict and EOS reverse of a particle, into l (r, v, rho, a_prev,
// drho_prev adjoints): P = p / R^2, p = EOS(rho) = B ((rho / rho0)^7 - 1), u =
// v + a_prev dt/2, R = rho + drho_prev dt/2.
template <int D>
__device__ __forceinline__ void adj_predict(const StepParams& P, double dt_pred, AdjSums<D> S, double Rk, double pres,
                                            double rho, const double* __restrict__ d, double* __restrict__ l) {
#pragma clang fp contract(off)
    S.each([&](double v) { return v * P.mass; });
    const double pb = S.P / (Rk * Rk);
    const double Rb = S.R - 2.0 * S.P * pres / (Rk * Rk * Rk);
    const double x = rho / P.rho0;
    const double x2 = x * x, x3 = x2 * x;
    const double dpdrho = 7.0 * P.eos_B * x3 * x3 / P.rho0;
    const double h2 = dt_pred * 0.5;
#pragma unroll
    for (int c = 0; c < D; ++c) {
        l[c] = d[c] + S.r[c];
        l[D + c] = d[D + c] + S.v[c] + S.u[c];
        l[2 * D + 1 + c] = S.u[c] * h2;
    }
    l[2 * D] = d[2 * D] + (P.density_treatment != 0 ? Rb : 0.0) + pb * dpdrho;
    l[3 * D + 1] = P.density_treatment != 0 ? Rb * h2 : 0.0;
}

template <class R>
__global__ void __launch_bounds__(kBlock) adj_pair(StepParams P, AdjStep T, StateB<R> B,
                                                   const uint32_t* __restrict__ skey,
                                                   const uint32_t* __restrict__ LB,
                                                   const double4* __restrict__ out_adj,
                                                   const double* __restrict__ drho_adj,
                                                   const double* __restrict__ direct, double* __restrict__ lam_out,
                                                   uint32_t* __restrict__ overflow_flag) {
    __shared__ uint32_t hits[kAdjChunk * kBlock];
    // XCD-aware: each XCD walks one contiguous slice of the slots
    const uint32_t lb = xcd_block(P.blocks_per_xcd);
    const uint32_t s = lb * kBlock + threadIdx.x;
    if (lb >= P.nblocks || s >= P.n) return;
    const AdjConsts K = adj_consts(P);
    auto particle = [&](uint32_t i) {
        const double4 va = to_d4<R>(B.va[i]), pr = to_d4<R>(B.pred[i]);
        const double2 pos = B.pos[i];
        const double4 oa = out_adj[i];
        return AdjParticle<2>{{pos.x, pos.y}, {pr.x, pr.y}, {va.x, va.y},    {oa.x, oa.y}, {oa.z, oa.w},
                              pr.z,           pr.w,         drho_adj[i], (int)va.w};
    };
    const AdjParticle<2> k = particle(s);
    AdjSums<2> S;
    bool overflow = false;
    if (k.t != 0) {
        uint32_t* my = hits + threadIdx.x;
        auto flush = [&](uint32_t nh) {
#pragma unroll 1
            for (uint32_t u = 0; u < nh; ++u) {
                const AdjParticle<2> i = particle(my[u * kBlock]);
                const double e[2] = {i.p[0] - k.p[0], i.p[1] - k.p[1]};
                adj_pair_term<2>(K, k, i, e, S);
            }
        };
        collect_neighbours<kAdjChunk>(P, P.max_nbr - 1, s, skey[s], make_double2(k.p[0], k.p[1]), B.pos, LB, my, overflow, flush);
    }
    if (overflow) atomicOr(overflow_flag, 1u);
    adj_predict<2>(P, T.dt_pred, S, k.R, (double)B.pres[s], (double)B.va[s].z, direct + 5 * (size_t)s,
                lam_out + 8 * (size_t)B.oid[s]);
}

// ------------------------------------------------------------------ step adjoint over lists
// The reverse of a step that read neighbour lists, in the slot order of
// their build.  adj_prep_list takes the kept state as it is (or, for a build
// step, through the build's permutation) and writes one record per slot with
// all that the pair adjoint reads of a particle: 128 bytes, which the wave
// fetches as WaveGather does, in two halves of four words.
// Per step of 134,042 particles (FP64): reorder 8.9 us, prep 6.9, cell walk
// 41.2 and gauge gradients 5.0 us before; prep 9.9 and pair with gauges 30.9 now.
struct alignas(128) AdjRec2 {
    double2 pos, u, v;
    double R, pw;      // R = typed_rho: the sign of the type, 0 for a dead particle
    double4 oa;
    double da, rho, pres;
    uint32_t oid;
    int32_t itype;
};
static_assert(sizeof(AdjRec2) == 128, "eight words of a wave gather");
constexpr uint32_t kAdjListMax = 1u << 25;  // particles whose records' byte offsets fit 32 bits
__device__ __forceinline__ AdjParticle<2> adj_particle(const AdjRec2& r) {
    return AdjParticle<2>{{r.pos.x, r.pos.y}, {r.u.x, r.u.y}, {r.v.x, r.v.y}, {r.oa.x, r.oa.y}, {r.oa.z, r.oa.w},
                          fabs(r.R),          r.pw,           r.da,           r.R > 0.0 ? 1 : (r.R < 0.0 ? -1 : 0)};
}

// perm: the build step's permutation, or null where the state is in slot
// order.  A wave's records go through LDS, so that its stores are contiguous:
// every lane storing its own wrote 16 bytes of each of 64 lines at a time
// (134,042 particles 16.0 -> 9.9 us, 40 bytes of direct adjoints left out too).
// (word p of record t in place p ^ t % 8, for the banks)
template <class R>
__global__ void __launch_bounds__(kBlock) adj_prep_list(StepParams P, AdjStep T, StateA<R> A,
                                                        const uint32_t* __restrict__ perm,
                                                        const double* __restrict__ lam_in, AdjRec2* __restrict__ rec,
                                                        double* __restrict__ piston_sum) {
    __shared__ uint4 s_rec[kBlock / kWave][8 * kWave];
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x, lane = __lane_id();
    uint4* buf = s_rec[wave_of_block()];
    double pist = 0.0;
    if (s < P.n) {
        const uint32_t src = perm ? min(perm[s], P.n - 1) : s;
        const real4<R> va = A.va[src], ad = A.ad[src];
        R p;
        const real4<R> pr = predict_record<R>(P, va, ad.x, ad.y, ad.z, (R)T.dt_pred, p);
        AdjRec2 r;
        r.oid = A.oid[src];
        r.itype = (int)va.w;
        r.pos = A.pos[src];
        r.u = make_double2((double)pr.x, (double)pr.y);
        r.v = make_double2((double)va.x, (double)va.y);
        r.R = (double)pr.z;
        r.pw = (double)pr.w;
        r.rho = (double)va.z;
        r.pres = (double)p;
        double direct[5];  // (the pair adjoint works these out again)
        pist = adj_whole_step(P, T, r.itype, r.oid, lam_in + 8 * (size_t)r.oid, r.oa, r.da, direct);
        uint4 w[8];
        __builtin_memcpy(w, &r, sizeof r);
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) buf[8 * lane + (q ^ (lane & 7))] = w[q];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const uint32_t first = s - lane;  // the wave's first slot
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) {
        const uint32_t t = 8 * q + lane / 8, w = lane & 7;
        if (first + t < P.n) ((uint4*)rec)[8 * (size_t)(first + t) + w] = buf[8 * t + (w ^ (t & 7))];
    }
    adj_piston_sum(pist, piston_sum);
}

// The pair adjoint over lists, LPP lanes per particle, and the gradient of
// the gauges of the state it reverses into (gauges: eta_bar null for none).
// Every entry is decided as the step decided it (FP32 steps too: their test
// ends in the same FP64 comparison).
template <int LPP>
__global__ void __launch_bounds__(kBlock) adj_pair_list(StepParams P, AdjStep T, const AdjRec2* __restrict__ rec,
                                                        const uint32_t* __restrict__ nbl,
                                                        const uint32_t* __restrict__ nbc,
                                                        const double* __restrict__ lam_in,
                                                        double* __restrict__ lam_out,
                                                        uint32_t* __restrict__ overflow_flag, GaugeSpec G,
                                                        const double* __restrict__ eta_bar,
                                                        const double* __restrict__ zsum,
                                                        const double* __restrict__ wsum) {
    using Half = WaveGather<4, sizeof(AdjRec2), kSlotMask>;
    __shared__ uint4 s_rec[kBlock / kWave][8 * kWave];
    const uint32_t lb = xcd_block(group_blocks_per_xcd<LPP>(P.n));
    if (lb >= group_blocks<LPP>(P.n)) return;
    const LaneGroup<LPP> g(lb);
    const bool live = g.s < P.n;
    const uint32_t s = live ? g.s : P.n - 1;
    const AdjConsts K = adj_consts(P);
    const AdjParticle<2> k = adj_particle(rec[s]);
    const uint32_t cnt = live && k.t != 0 ? nbc[s] : 0u;
    AdjSums<2> S;
    uint32_t hits = 0;
    uint4* buf = s_rec[wave_of_block()];
    const WaveGatherBoth<Half, Half> src{Half(rec, buf), Half((const char*)rec + 64, buf + 4 * kWave)};
    gather_rounds<LPP, 1>(P, nbl, src, s, g.l, cnt, [&](uint32_t e0, const uint32_t (&)[1], const auto& w) {
        const double4 a = record_real4(w[0], 0.0), b = record_real4(w[0] + 2, 0.0);  // (pos, u), (v, R, pw)
        const double e[2] = {__dsub_rn(a.x, k.p[0]), __dsub_rn(a.y, k.p[1])};
        if (e0 < cnt && b.z != 0.0 && dist2_exact(e[0], e[1]) < P.cut2) {
            const double4 oa = record_real4(w[0] + 4, 0.0);
            const AdjParticle<2> i{{a.x, a.y}, {a.z, a.w}, {b.x, b.y}, {oa.x, oa.y}, {oa.z, oa.w}, fabs(b.z), b.w,
                                   record_real4(w[0] + 6, 0.0).x, b.z > 0.0 ? 1 : -1};
            adj_pair_term<2>(K, k, i, e, S);
            ++hits;
        }
    });
    S.each([](double v) { return lane_sum<LPP>(v); });
    if (lane_sum<LPP>((int)hits) > (int)(P.max_nbr - 1)) atomicOr(overflow_flag, 1u);
    if (!live || g.l != 0) return;
    double l[8], direct[5], da;
    double4 oa;
    const AdjRec2& own = rec[s];
    adj_whole_step(P, T, own.itype, own.oid, lam_in + 8 * (size_t)own.oid, oa, da, direct);
    // (a dead particle has no sums, and no density in its record)
    adj_predict<2>(P, T.dt_pred, S, k.t != 0 ? k.R : 1.0, own.pres, own.rho, direct, l);
    if (eta_bar && own.itype == G.ptype) {
        double gx, gy;
        if (gauge_gradient(G, own.pos, eta_bar, zsum, wsum, gx, gy)) {
            l[0] += gx;
            l[1] += gy;
        }
    }
    double2* out = (double2*)(lam_out + 8 * (size_t)own.oid);
#pragma unroll
    for (int c = 0; c < 4; ++c) out[c] = make_double2(l[2 * c], l[2 * c + 1]);
}

}  // namespace rrsph
