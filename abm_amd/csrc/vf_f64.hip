// vf_f64.hip -- float64 VSWRM step.  Two kernels with the same decisions and
// fields, whose sums differ in rounding: the guarded one (below), and the plain
// one, the reference arithmetic on the GPU, for what the guarded one does not
// take (steps that count near ties, R beyond 4096).
//
// The plain kernel: one workgroup per replica.  The replica's poses live in LDS for the whole
// step and are updated in place, agent by agent in id order, which is the
// reference's Group.update semantics (vf_sims.py:302; agent k sees agents <k
// at their new poses).  Per agent:
//   1. lanes over objects: exact float64 pair decision (vf_exact.hpp), and
//      each drawn interval written as bytes into a per-ray LDS field;
//   2. lanes over rays: numpy's trapz terms and dPhi spike terms
//      (vf_supcalc.py:199-254, 257-277) summed with a block reduction;
//   3. one lane: VSWRM motion, Euler step and boundary (vf_agent.py:188-204,
//      263-326; agent.py:347-395, 605-610).
// Built with -ffp-contract=off.
#include <algorithm>

#include "vf_batch.hpp"
#include "vf_exact.hpp"
#include "vf_f32_common.hpp"

namespace abm {

namespace {

__device__ inline double wave_sum(double x) {
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}

// Block-wide float64 sums over the raw raster field V (0/1 bytes in LDS):
// trapz(cos(PHI)*(-V), PHI), trapz(sin(PHI)*(-V), PHI), sum(cos(PHI)*dPhi_V^2),
// sum(sin(PHI)*dPhi_V^2) (vf_supcalc.py:199-238, 257-277).  Each trapz term is
// numpy's d_k*(y_{k+1}+y_k)/2 with y = cos(PHI)*G, G = -V + ALP2*0.  Leaves the
// per-wave partial sums in red[4*wave + 0..3]; the caller synchronises.
__device__ void integrals_f64(const uint8_t* V, int R, const double* cs, const double* sn,
                              const double* dp, int tid, int nthr, double* red) {
#pragma clang fp contract(off)
    const bool case1 = V[0] == 1 && V[R - 1] == 0;
    double tc = 0.0, ts = 0.0, ec = 0.0, es = 0.0;
    for (int r = tid; r < R; r += nthr) {
        const double vr = V[r] ? 1.0 : 0.0;
        const double gr = -vr + 0.0;
        if (r < R - 1) {
            const double vn = V[r + 1] ? 1.0 : 0.0;
            const double gn = -vn + 0.0;
            const double yc = cs[r] * gr, ycn = cs[r + 1] * gn;
            const double ys = sn[r] * gr, ysn = sn[r + 1] * gn;
            tc += (dp[r] * (ycn + yc)) / 2.0;
            ts += (dp[r] * (ysn + ys)) / 2.0;
        }
        double o;
        if (case1) o = vr - (V[r == 0 ? R - 1 : r - 1] ? 1.0 : 0.0);
        else o = (V[r == R - 1 ? 0 : r + 1] ? 1.0 : 0.0) - vr;
        const double sq = o * o;
        ec += cs[r] * sq;
        es += sn[r] * sq;
    }
    tc = wave_sum(tc); ts = wave_sum(ts); ec = wave_sum(ec); es = wave_sum(es);
    if ((tid & 63) == 0) {
        red[4 * (tid >> 6) + 0] = tc; red[4 * (tid >> 6) + 1] = ts;
        red[4 * (tid >> 6) + 2] = ec; red[4 * (tid >> 6) + 3] = es;
    }
}

__global__ void __launch_bounds__(256)
vf_step_f64_kernel(const VFRep* __restrict__ reps, const double* __restrict__ tcos,
                   const double* __restrict__ tsin, const double* __restrict__ tdphi,
                   abm_vf_state_f64 st, uint32_t* __restrict__ bits_out,
                   double* __restrict__ diag, uint32_t flags, unsigned long long* __restrict__ counters) {
#pragma clang fp contract(off)
    extern __shared__ double smem[];
    const VFRep P = reps[blockIdx.x];
    // near-tie margin count: pairs whose bin or half-width decision lies
    // within 1e-12 of its tie, where the device's and the host's libm (acos,
    // atan) may round the deciding value to opposite sides
    const bool count = (flags & ABM_COUNT_RECHECKS) != 0 && counters != nullptr;
    unsigned long long n_near = 0;
    const int N = P.n_agents, R = P.n_rays;
    const int tid = threadIdx.x, nthr = blockDim.x, nw = nthr >> 6;
    const bool sync_order = (flags & ABM_ORDER_SYNCHRONOUS) != 0;

    double* sx = smem;
    double* sy = sx + N;
    double* sth = sy + N;
    double* sv = sth + N;
    double* srad = sv + N;
    double* ox = sync_order ? srad + N : sx;   // object positions
    double* oy = sync_order ? srad + 2 * N : sy;
    double* red = (sync_order ? srad + 3 * N : srad + N);
    double* shared_out = red + 4 * nw;          // 2 doubles: dv, dpsi broadcast
    uint8_t* V = reinterpret_cast<uint8_t*>(shared_out + 8);

    const int a0 = P.agent_offset;
    for (int i = tid; i < N; i += nthr) {
        sx[i] = st.x[a0 + i];
        sy[i] = st.y[a0 + i];
        sth[i] = st.theta[a0 + i];
        sv[i] = st.v[a0 + i];
        srad[i] = (double)st.radius[a0 + i];
        if (sync_order) { ox[i] = sx[i]; oy[i] = sy[i]; }
    }
    const double* cs = tcos + P.table_offset;
    const double* sn = tsin + P.table_offset;
    const double* dp = tdphi + P.table_offset;
    const bool torus = P.boundary == ABM_BOUNDARY_INFINITE;
    __syncthreads();

    for (int k = 0; k < N; ++k) {
        for (int r = tid; r < R; r += nthr) V[r] = 0;
        __syncthreads();
        const Focal f = make_focal(sx[k], sy[k], sth[k], srad[k]);
        for (int j = tid; j < N; j += nthr) {
            if (j == k) continue;
            PairVF p = pair_vf_exact(f, ox[j], oy[j], srad[j], torus, P.width, P.height,
                                     R, P.step, P.fov_px0, P.fov_px1);
            if (count && !p.skipped) {
                const double ca = p.closed_angle;
                const double dt = fabs(linspace_at(p.t, R, P.step) - ca);
                double dn = 1e300;
                if (p.t > 0) dn = fmin(dn, fabs(linspace_at(p.t - 1, R, P.step) - ca));
                if (p.t < R - 1) dn = fmin(dn, fabs(linspace_at(p.t + 1, R, P.step) - ca));
                const double hf = p.half_f, fr = hf - floor(hf);
                const bool near_bin = dn - dt < 1e-12;
                const bool near_half = hf >= 0.5 && (fr < 1e-12 * hf || 1.0 - fr < 1e-12 * hf);
                if (near_bin || near_half) ++n_near;
            }
            if (p.skipped || !p.drawn) continue;
            int a0p, b0p, a1p, b1p;
            vf_pieces(p.start, p.end, R, &a0p, &b0p, &a1p, &b1p);
            for (int r = a0p; r < b0p; ++r) V[r] = 1;
            for (int r = a1p; r < b1p; ++r) V[r] = 1;
        }
        __syncthreads();

        integrals_f64(V, R, cs, sn, dp, tid, nthr, red);
        // pack the field for output while the sums settle
        if (bits_out) {
            const int W = P.words;
            uint32_t* dst = bits_out + P.field_offset + (int64_t)k * W;
            for (int w = tid; w < W; w += nthr) {
                uint32_t m = 0;
                for (int b = 0; b < 32; ++b) {
                    int r = w * 32 + b;
                    if (r < R && V[r]) m |= 1u << b;
                }
                dst[w] = m;
            }
        }
        __syncthreads();
        if (tid == 0) {
            double Tc = 0.0, Ts = 0.0, Ec = 0.0, Es = 0.0;
            for (int w = 0; w < nw; ++w) {
                Tc += red[4 * w]; Ts += red[4 * w + 1]; Ec += red[4 * w + 2]; Es += red[4 * w + 3];
            }
            const int ag = a0 + k;
            const double alp0 = st.alp0 ? st.alp0[ag] : P.alp0;
            const double bet0 = st.bet0 ? st.bet0[ag] : P.bet0;
            const double v0 = st.v0 ? st.v0[ag] : P.v0;
            double dv = 0.0, dpsi = 0.0, ab = 0.0, ae = 0.0, bb = 0.0, be = 0.0;
            const double vel = sv[k];
            if (P.phi_ok) {
                ab = alp0 * Tc;
                ae = (alp0 * P.alp1) * Ec;
                bb = bet0 * Ts;
                be = (bet0 * P.bet1) * Es;
                dv = P.gam * (v0 - vel) + ab + ae;
                dpsi = bb + be;
            }
            Pose p{sx[k], sy[k], sth[k], vel};
            p = vf_move(p, dpsi, dv, P.limit_movement, P.max_th, P.max_vel);
            if (torus) p = teleport(p, srad[k], P.pad, P.width, P.height);
            else p = reflect_walls(p, srad[k], P.pad, P.width, P.height);
            sx[k] = p.x; sy[k] = p.y; sth[k] = p.theta; sv[k] = p.v;
            if (diag && (flags & ABM_WANT_DIAG)) {
                double* d = diag + 6 * (int64_t)ag;
                d[0] = dv; d[1] = dpsi; d[2] = ab; d[3] = ae; d[4] = bb; d[5] = be;
            }
        }
        __syncthreads();
    }
    for (int i = tid; i < N; i += nthr) {
        st.x[a0 + i] = sx[i];
        st.y[a0 + i] = sy[i];
        st.theta[a0 + i] = sth[i];
        st.v[a0 + i] = sv[i];
    }
    if (count && n_near) atomicAdd(&counters[3], n_near);
}

// ---------------------------------------------------------------------------
// The same step with the pairs' integer decisions made in float32 where
// float32 is certain of them and by the exact float64 replica elsewhere;
// state, sums and motion stay float64.  A pair's decision is its bin and its
// half-width; the centre difference (periodic image included) is the float64
// one, rounded once, the heading the float64 sine and cosine, rounded once, so
// the float32 angle is within 1e-6 rad of the exact one and the guard bands of
// the fused kernels (4e-6 rad around a bin tie and the +-pi wrap, 4e-6 relative
// + 1e-6 around an integer half-width) cover it and the reference's own error
// (vf_f32_common.hpp).  About 1 pair in 1000 takes the replica, and every pair of
// a focal agent whose heading the reference loses (heading_kept).
//
// One workgroup of NW waves per replica, largest first.  Lanes over objects
// decide and OR each interval into a bit-packed field in LDS; every lane owns
// RPL rays whose table entries it keeps in registers for the whole step; the
// sums meet by lane swaps and DPP.  Bound by VALU
// issue (batches) or the id-order chain's latency (few replicas).  Against the
// plain kernel (exact decisions, a byte per ray, tables from memory): 4096
// replicas of 50 agents at R = 512 0.773 -> 0.167 ms a step (1332 -> 439 VALU
// instructions per agent-step, an eighth of them the motion's sincos; 0.88 of
// the VALU issue slots filled), 512 of 37 at R = 300 in a walled arena 0.265 ->
// 0.088 ms.
// On the CPU, with the reciprocals one ulp off either way, no decision of 96
// million pairs differs from the exact one at any of nine scales (positions of 20
// to 1e10 radii; an eighth of the pairs near bin ties, as many ahead and behind):
// the angle is within 5.6e-7 rad up to 3e9 radii, the half-width within 5.3e-7.
constexpr int kGuardMaxWaves = 8;

struct GuardSmem {
    double *x, *y, *th, *v, *a0, *b0, *v0, *ox, *oy, *red;
    float2* u;       // heading vectors (agents move only in their own turn)
    int* rad;
    uint2* D;        // the focal agent's field and its edges, a word of each
    uint32_t* F;     // the field as the pairs set it
};

constexpr int kGuardRays = 8;   // at most, per lane

__host__ __device__ inline size_t guard_lds_bytes(int N, int R, int nw, bool sync_order) {
    return (size_t)N * (sizeof(double) * (sync_order ? 9 : 7) + sizeof(float2) + sizeof(int)) +
           sizeof(double) * 4 * nw + sizeof(uint2) * 2 * kGuardRays * nw + sizeof(uint32_t) * ((size_t)(R + 31) / 32) + 16;
}

__device__ inline GuardSmem guard_carve(void* base, int N, int nw, bool sync_order) {
    GuardSmem s;
    char* p = reinterpret_cast<char*>(base);
    for (double** d : {&s.x, &s.y, &s.th, &s.v, &s.a0, &s.b0, &s.v0}) {
        *d = reinterpret_cast<double*>(p);
        p += sizeof(double) * N;
    }
    s.ox = s.x; s.oy = s.y;
    if (sync_order) {
        s.ox = reinterpret_cast<double*>(p); p += sizeof(double) * N;
        s.oy = reinterpret_cast<double*>(p); p += sizeof(double) * N;
    }
    s.red = reinterpret_cast<double*>(p); p += sizeof(double) * 4 * nw;
    s.u = reinterpret_cast<float2*>(p); p += sizeof(float2) * N;
    s.D = reinterpret_cast<uint2*>(p); p += sizeof(uint2) * 2 * kGuardRays * nw;
    s.rad = reinterpret_cast<int*>(p); p += sizeof(int) * N;
    s.F = reinterpret_cast<uint32_t*>(p);
    return s;
}

// The float64 decision of a pair inside a guard band, out of line.
struct Interval {
    int start, end, drawn;
};
__device__ __noinline__ Interval exact_interval(double px, double py, double theta, double radius, double ox,
                                                double oy, double osize, const VFRep* rp) {
    const Focal f = make_focal(px, py, theta, radius);
    const PairVF p = pair_vf_exact(f, ox, oy, osize, rp->boundary == ABM_BOUNDARY_INFINITE ? 1 : 0, rp->width,
                                   rp->height, rp->n_rays, rp->step, rp->fov_px0, rp->fov_px1);
    return Interval{p.start, p.end, p.skipped ? 0 : p.drawn};
}

// sincos out of line: inlined, its constants are held over the agent loop and
// spilled to scratch, nine loads per agent.
__device__ __noinline__ double2 sincos_f64(double x) {
    double s, c;
    sincos(x, &s, &c);
    return make_double2(s, c);
}

template <int CTRL>
__device__ inline double dpp_f64(double v) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true));
}
__device__ inline double lane_f64(double x, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                            __builtin_amdgcn_readlane(__double2loint(x), l));
}
// The wave sums of four values, to every lane, in one pass over lanes 32, 16, 8,
// 4, 2 and 1 apart (the plain kernel's order).  A swap of halves leaves the first
// value's pairs in the lower lanes and the second's in the upper ones, a swap of
// rows one value a row: 29 instructions, where two sums by themselves are 40.
__device__ inline void wave_totals_f64(double (&c)[4]) {
    double h[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {   // c[2q] | c[2q + 1]
        const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)__double2loint(c[2 * q]), (uint32_t)__double2loint(c[2 * q + 1]), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)__double2hiint(c[2 * q]), (uint32_t)__double2hiint(c[2 * q + 1]), false, false);
        h[q] = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
    }
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)__double2loint(h[0]), (uint32_t)__double2loint(h[1]), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)__double2hiint(h[0]), (uint32_t)__double2hiint(h[1]), false, false);
    double x = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);   // by row: c[0], c[2], c[1], c[3]
    x += dpp_f64<0x128>(x);
    x += dpp_f64<0x124>(x);
    x += dpp_f64<0x4E>(x);
    x += dpp_f64<0xB1>(x);
    c[0] = lane_f64(x, 0); c[2] = lane_f64(x, 16); c[1] = lane_f64(x, 32); c[3] = lane_f64(x, 48);
}

// The sums over the workgroup's NW waves, by way of red (4 NW doubles).
template <int NW>
__device__ inline void block_totals_f64(double (&c)[4], double* red) {
    wave_totals_f64(c);
    if (NW == 1) return;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[4 * (threadIdx.x >> 6) + q] = c[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        c[q] = 0.0;
#pragma unroll
        for (int w = 0; w < NW; ++w) c[q] += red[4 * w + q];
    }
}

// OR the rays [a, b) into the field: one or two words nearly always.
__device__ inline void or_rays(uint32_t* F, int a, int b) {
    if (a >= b) return;
    const int w0 = a >> 5, w1 = (b - 1) >> 5;
    const uint32_t m0 = 0xffffffffu << (a & 31), m1 = 0xffffffffu >> (31 - ((b - 1) & 31));
    atomicOr(&F[w0], w0 == w1 ? m0 & m1 : m0);
    if (w0 < w1) {
        atomicOr(&F[w1], m1);
        for (int w = w0 + 1; w < w1; ++w) atomicOr(&F[w], 0xffffffffu);
    }
}

template <int NW, int RPL>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4)))
vf_step_f64_guard_kernel(const VFRep* __restrict__ reps, const int32_t* __restrict__ order,
                         const double* __restrict__ tcos, const double* __restrict__ tsin,
                         const double* __restrict__ tdphi, abm_vf_state_f64 st,
                         uint32_t* __restrict__ bits_out, double* __restrict__ diag, uint32_t flags, int maxN) {
#pragma clang fp contract(off)
    extern __shared__ double smem[];
    constexpr int NT = 64 * NW;
    const VFRep* rp = reps + order[blockIdx.x];
    const int N = rp->n_agents, R = rp->n_rays, W = rp->words, a0 = rp->agent_offset;
    const int tid = threadIdx.x, lane = tid & 63;
    const bool sync_order = (flags & ABM_ORDER_SYNCHRONOUS) != 0;
    const bool want_diag = diag != nullptr && (flags & ABM_WANT_DIAG) != 0;
    const GuardSmem S = guard_carve(smem, maxN, NW, sync_order);
    // this lane's rays, tid + NT i, and their table entries (zero at or beyond
    // R): cos, sin and the trapz weight d_{r-1} / 2 + d_r / 2 (numpy's trapz
    // terms d_k (y_{k+1} + y_k) / 2 gathered by ray).  Rays spread over the circle
    // cancel within a lane, so the lanes' sums stay small and the tree rounds as
    // little as the plain kernel's (spans of consecutive rays: 1.5 times its error).
    double tw[RPL], tc[RPL], ts[RPL];
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
        const int r = tid + NT * i, e = rp->table_offset + (r < R ? r : 0);
        const double left = r > 0 && r < R ? tdphi[e - 1] : 0.0, right = r < R - 1 ? tdphi[e] : 0.0;
        tw[i] = left / 2.0 + right / 2.0;
        tc[i] = r < R ? tcos[e] : 0.0;
        ts[i] = r < R ? tsin[e] : 0.0;
    }
    for (int w = tid; w < 2 * kGuardRays * NW; w += NT) S.D[w] = make_uint2(0u, 0u);   // beyond the field: no ray
    for (int i = tid; i < N; i += NT) {
        const int g = a0 + i;
        const double th = st.theta[g];
        S.x[i] = st.x[g]; S.y[i] = st.y[g]; S.th[i] = th; S.v[i] = st.v[g];
        S.rad[i] = st.radius[g];
        S.a0[i] = st.alp0 ? st.alp0[g] : rp->alp0;
        S.b0[i] = st.bet0 ? st.bet0[g] : rp->bet0;
        S.v0[i] = st.v0 ? st.v0[g] : rp->v0;
        const double2 sc = sincos_f64(th);
        // unit(v1) = (cos th, -sin th), or NaN, which no guard lets through
        S.u[i] = make_float2(heading_kept(S.x[i], S.y[i], (double)S.rad[i]) ? (float)sc.y : NAN, -(float)sc.x);
        if (sync_order) { S.ox[i] = S.x[i]; S.oy[i] = S.y[i]; }
    }
    const bool torus = rp->boundary == ABM_BOUNDARY_INFINITE;
    const double Wd = rp->width, Hd = rp->height, hw = Wd / 2.0, hh = Hd / 2.0;
    const float inv_step = (float)(1.0 / rp->step), hs = (float)((double)R / kTwoPi);
    const float g_bins = (float)(f32::kAngleGuardF / rp->step + 1.5e-7 * R);
    const int px0 = rp->fov_px0, px1 = rp->fov_px1;
    __syncthreads();

    for (int k = 0; k < N; ++k) {
        // a SIMD's arbiter favours its oldest wave: each lowers its own
        // priority as it advances, so that a batch's waves finish together
        if (NW == 1) {
            if (k == 0) __builtin_amdgcn_s_setprio(3);
            else if (k == N / 2) __builtin_amdgcn_s_setprio(2);
            else if (k == 3 * N / 4) __builtin_amdgcn_s_setprio(1);
            else if (k == 15 * N / 16) __builtin_amdgcn_s_setprio(0);
        }
        for (int w = tid; w < W; w += NT) S.F[w] = 0u;
        const double fx = S.x[k], fy = S.y[k], fr = (double)S.rad[k], cx = fx + fr, cy = fy + fr;
        const float2 u = S.u[k];
        __syncthreads();
        // ---- pairs
        for (int j = tid; j < N; j += NT) {
            const double ojx = S.ox[j], ojy = S.oy[j], os = (double)S.rad[j];
            if (j == k || (ojx == fx && ojy == fy)) continue;   // coincident (vf_supcalc.py:57)
            // the centre difference exactly as pair_vf_exact forms it (a
            // difference beyond half the arena is not zero, so its sign is
            // that of the comparison there)
            const double ocx = ojx + os, ocy = ojy + os;
            double vx = ocx - cx, vy = ocy - cy;
            if (torus) {
                vx = (ocx - (fabs(vx) > hw ? copysign(Wd, vx) : 0.0)) - cx;
                vy = (ocy - (fabs(vy) > hh ? copysign(Hd, vy) : 0.0)) - cy;
            }
            const float dx = (float)vx, dy = (float)vy;
            const float d2 = fmaf(dy, dy, dx * dx);
            const float a = f32::atan2_f32(fmaf(u.x, dy, -u.y * dx), fmaf(u.x, dx, u.y * dy));
            const float z = (float)os * __builtin_amdgcn_rsqf(d2);
            const float xb = (f32::kPiF - a) * inv_step;   // bin coordinate of the closed angle -a
            const float tr = rintf(xb), dfr = xb - tr;
            const float half = f32::atan_unit_f32(z) * hs;   // proj_size / 2
            const float hfl = floorf(half), hfrac = half - hfl, hg = 4e-6f * fabsf(half) + 1e-6f;
            const bool ok = (d2 > 1e-30f) & (fabsf(z) < 1.0f) & (fabsf(a) < f32::kPiF - f32::kAngleGuardF) &
                            (hfrac >= hg) & (hfrac <= 1.0f - hg) & (fabsf(dfr) <= 0.5f - g_bins);
            const int t = (int)tr, h = (int)hfl;
            Interval p{t - h, t + h, 0};
            p.drawn = ((px0 < p.start) & (p.start < px1)) | ((px0 < p.end) & (p.end < px1));
            if (!ok) p = exact_interval(fx, fy, S.th[k], fr, ojx, ojy, os, rp);
            if (p.drawn) {
                // vf_pieces: the part inside, and the part that wraps (at
                // most one end does; an end at or beyond R wraps one ray less)
                or_rays(S.F, clamp_ray(p.start, R), p.end >= R ? R : clamp_ray(p.end, R));
                if (p.start < 0 || p.end >= R)
                    or_rays(S.F, p.end >= R ? 0 : clamp_ray(R + p.start, R), p.end >= R ? clamp_ray(p.end - (R - 1), R) : R);
            }
        }
        __syncthreads();
        // ---- sums: the field's edges by the dPhi alignment rule
        // (vf_supcalc.py:266-274), then the table entries added where a bit is
        // set (as fma(bit ? w : 0, t, acc), one rounding)
        const bool case1 = (S.F[0] & 1u) == 1u && f32::field_bit(S.F, R - 1) == 0u;
        for (int w = tid; w < W; w += NT) {
            const uint32_t cur = S.F[w];
            const int nb = w == W - 1 ? R - 32 * w : 32;   // the word's rays
            const uint32_t other = case1 ? (cur << 1) | (w ? S.F[w - 1] >> 31 : 0u)
                                         : (cur >> 1) | ((w == W - 1 ? S.F[0] & 1u : S.F[w + 1] & 1u) << (nb - 1));
            S.D[w] = make_uint2(cur, (cur ^ other) & f32::low_mask(nb));
        }
        __syncthreads();
        const uint2* const D = S.D + (tid >> 5);
        const int sh = tid & 31;
        double bc = 0.0, bs = 0.0, ec = 0.0, es = 0.0;
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
            const uint2 d = D[(NT / 32) * i];
            const int vm = __builtin_amdgcn_sbfe((int)d.x, sh, 1), sm = __builtin_amdgcn_sbfe((int)d.y, sh, 1);
            const double vb = __hiloint2double(vm & __double2hiint(tw[i]), vm & __double2loint(tw[i]));
            const double sb = __hiloint2double(sm & 0x3ff00000, 0);
            bc = __builtin_fma(vb, tc[i], bc);
            bs = __builtin_fma(vb, ts[i], bs);
            ec = __builtin_fma(sb, tc[i], ec);
            es = __builtin_fma(sb, ts[i], es);
        }
        const double alp0 = S.a0[k], bet0 = S.b0[k], vel = S.v[k];
        const double ae0 = alp0 * rp->alp1, be0 = bet0 * rp->bet1;
        // blob terms: trapz(cos(PHI) * (-V)) = -sum(w cos V).  The speed's two sums
        // are weighted and added by lane, which rounds least; the heading's stay
        // apart, as the plain kernel has them: in a field that mirrors itself each
        // cancels, and a residue could take a heading of 0 to 2 pi.
        double c[4] = {__builtin_fma(ae0, ec, -(alp0 * bc)), bs, es, 0.0};
        block_totals_f64<NW>(c, S.red);
        const double Sv = c[0];
        double bb = bet0 * -c[1], be = be0 * c[2], ab = 0.0, ae = 0.0;
        const double Sp = __builtin_fma(be0, c[2], bb);
        if (want_diag) {
            double d[4] = {bc, ec, 0.0, 0.0};
            if (NW > 1) __syncthreads();   // red is read
            block_totals_f64<NW>(d, S.red);
            ab = alp0 * -d[0]; ae = ae0 * d[1];
        }
        if (bits_out) {
            uint32_t* dst = bits_out + rp->field_offset + (int64_t)k * W;
            for (int w = tid; w < W; w += NT) dst[w] = S.F[w];
        }
        // ---- motion, on every lane (one writes it)
        double dv = 0.0, dpsi = 0.0;
        if (rp->phi_ok) {
            dv = __builtin_fma(rp->gam, S.v0[k] - vel, Sv);
            dpsi = Sp;
        } else {
            ab = ae = bb = be = 0.0;
        }
        // vf_move with one sincos for both values
        double turn = dpsi;
        if (rp->limit_movement && fabs(turn) > rp->max_th) turn = turn < 0.0 ? -rp->max_th : rp->max_th;
        Pose p{fx, fy, prove_orientation(S.th[k] + turn), vel + dv};
        if (rp->limit_movement && fabs(p.v) > rp->max_vel) p.v = p.v < 0.0 ? -rp->max_vel : rp->max_vel;
        const double2 sc = sincos_f64(p.theta);
        p.x = fx + p.v * sc.y;
        p.y = fy - p.v * sc.x;
        p = torus ? teleport(p, fr, rp->pad, Wd, Hd) : reflect_walls(p, fr, rp->pad, Wd, Hd);
        // every wave has read agent k's pose and the field
        if (NW > 1) __syncthreads();
        if (tid == 0) {
            S.x[k] = p.x; S.y[k] = p.y; S.th[k] = p.theta; S.v[k] = p.v;
            if (want_diag) {
                double* d = diag + 6 * (int64_t)(a0 + k);
                d[0] = dv; d[1] = dpsi; d[2] = ab; d[3] = ae; d[4] = bb; d[5] = be;
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < N; i += NT) {
        const int g = a0 + i;
        st.x[g] = S.x[i];
        st.y[g] = S.y[i];
        st.theta[g] = S.th[i];
        st.v[g] = S.v[i];
    }
}

}  // namespace

size_t vf_f64_lds_bytes(int max_agents, int max_rays, int nthr, bool sync_order) {
    size_t d = (size_t)max_agents * (sync_order ? 7 : 5) + 4 * (nthr / 64) + 8;
    return d * sizeof(double) + (size_t)max_rays + 16;
}

namespace {

// Waves per replica of the guarded kernel, 0 where it does not apply: the
// near-tie count (it needs every pair's float64 angle), R beyond 4096 (eight
// waves of eight rays a lane) or replicas beyond its LDS.  As few waves as hold
// the rays at eight a lane, or, while the batch leaves SIMDs with fewer than two
// waves, up to four that bring the rays to four a lane or the objects to one
// (us a step with 1, 2, 4, 8 waves: one replica of 100 agents at R = 1024 -, 251,
// 235, 288; of 300 at 512 1279, 961, 842, 903; 256 replicas of 100 at 512 281,
// 224, 236, 289; 512 of 150 at 300 496, 432, 381, 522; 1000 of 64 at 1000 -, 190,
// 220, 450; 2048 of 50 at 512 139, 168, 304, 654).
int guard_waves(const abm_vf_batch* b, uint32_t flags) {
    if ((flags & ABM_COUNT_RECHECKS) != 0 || b->max_rays > 64 * 8 * kGuardMaxWaves) return 0;
    int nw = 1;
    while (64 * 8 * nw < b->max_rays) nw *= 2;
    const int want = std::max((b->max_rays + 255) / 256, (b->max_agents + 63) / 64);
    while (nw < want && nw < 4 && (int64_t)b->n_replicas * nw * 2 <= 8ll * b->n_cu) nw *= 2;
    const size_t lds = guard_lds_bytes(b->max_agents, b->max_rays, nw, (flags & ABM_ORDER_SYNCHRONOUS) != 0);
    return lds <= (size_t)b->dev_max_lds ? nw : 0;
}

int launch_guard(abm_vf_batch* b, const abm_vf_state_f64* st, uint32_t* bits, double* diag, uint32_t flags,
                 hipStream_t s, int nw, int rpl) {
    const size_t lds = guard_lds_bytes(b->max_agents, b->max_rays, nw, (flags & ABM_ORDER_SYNCHRONOUS) != 0);
    auto kern = rpl == 4 ? (nw == 1 ? vf_step_f64_guard_kernel<1, 4>
                            : nw == 2 ? vf_step_f64_guard_kernel<2, 4>
                            : nw == 4 ? vf_step_f64_guard_kernel<4, 4> : vf_step_f64_guard_kernel<8, 4>)
                         : (nw == 1 ? vf_step_f64_guard_kernel<1, 8>
                            : nw == 2 ? vf_step_f64_guard_kernel<2, 8>
                            : nw == 4 ? vf_step_f64_guard_kernel<4, 8> : vf_step_f64_guard_kernel<8, 8>);
    if (lds > 65536)
        if (int rc = check_hip(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   (int)lds), "hipFuncSetAttribute"))
            return rc;
    hipLaunchKernelGGL(kern, dim3(b->n_replicas), dim3(64 * nw), lds, s, b->reps_dev, b->order_dev, b->tab_cos,
                       b->tab_sin, b->tab_dphi, *st, bits, diag, flags, b->max_agents);
    b->last_kernels = ABM_KERNEL_F64;
    return check_hip(hipGetLastError(), "vf_step_f64_guard_kernel launch");
}

}  // namespace

int launch_vf_step_f64(abm_vf_batch* b, const abm_vf_state_f64* st, uint32_t* bits,
                       double* diag, uint32_t flags, hipStream_t s) {
    const bool sync_order = (flags & ABM_ORDER_SYNCHRONOUS) != 0;
    if (const int nw = guard_waves(b, flags)) {
        const int per = (b->max_rays + 64 * nw - 1) / (64 * nw);
        return launch_guard(b, st, bits, diag, flags, s, nw, per <= 4 ? 4 : 8);
    }
    int nthr = 64;
    if (b->max_rays >= 1024 || b->max_agents > 128) nthr = 128;
    if (b->max_agents > 512) nthr = 256;
    size_t lds = vf_f64_lds_bytes(b->max_agents, b->max_rays, nthr, sync_order);
    if (lds > (size_t)b->dev_max_lds)
        return set_error(ABM_ERR_UNSUPPORTED,
                         "abm_vf_step_f64: %d agents need %zu B of LDS per replica (device max %d)",
                         b->max_agents, lds, b->dev_max_lds);
    if (lds > 65536) {
        if (int rc = check_hip(hipFuncSetAttribute((const void*)vf_step_f64_kernel,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   (int)lds), "hipFuncSetAttribute"))
            return rc;
    }
    hipLaunchKernelGGL(vf_step_f64_kernel, dim3(b->n_replicas), dim3(nthr), lds, s,
                       b->reps_dev, b->tab_cos, b->tab_sin, b->tab_dphi, *st, bits, diag, flags,
                       (unsigned long long*)b->counters);
    b->last_kernels = ABM_KERNEL_F64;
    return check_hip(hipGetLastError(), "vf_step_f64_kernel launch");
}

// ---------------------------------------------------------------- probes
namespace {

__global__ void vf_projection_rows_kernel(int R, double step, int fov_px0, int fov_px1,
                                          int torus, double W, double H, double fx, double fy,
                                          double ftheta, double fradius,
                                          const double* __restrict__ ox,
                                          const double* __restrict__ oy,
                                          const double* __restrict__ osize, int n_obj,
                                          uint32_t* __restrict__ rows, int32_t* __restrict__ rec) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_obj) return;
    const Focal f = make_focal(fx, fy, ftheta, fradius);
    const PairVF p = pair_vf_exact(f, ox[i], oy[i], osize[i], torus, W, H, R, step,
                                   fov_px0, fov_px1);
    const int words = (R + 31) / 32;
    uint32_t* row = rows + (int64_t)i * words;
    int a0 = 0, b0 = 0, a1 = 0, b1 = 0;
    if (!p.skipped && p.drawn) vf_pieces(p.start, p.end, R, &a0, &b0, &a1, &b1);
    for (int w = 0; w < words; ++w) {
        uint32_t m = 0;
        for (int b = 0; b < 32; ++b) {
            const int r = w * 32 + b;
            if ((r >= a0 && r < b0) || (r >= a1 && r < b1)) m |= 1u << b;
        }
        row[w] = m;
    }
    if (rec) {
        int32_t* q = rec + 5 * (int64_t)i;
        q[0] = p.t; q[1] = p.half; q[2] = p.start; q[3] = p.end;
        q[4] = p.skipped ? -1 : p.drawn;
    }
}

__global__ void __launch_bounds__(256)
vf_state_variables_kernel(int R, const uint32_t* __restrict__ bits, const double* __restrict__ vel,
                          const double* __restrict__ alp0, const double* __restrict__ bet0,
                          const double* __restrict__ v0, double gam, double alp1, double bet1,
                          const double* __restrict__ tcos, const double* __restrict__ tsin,
                          const double* __restrict__ tdphi, int phi_ok,
                          double* __restrict__ out, int8_t* __restrict__ dphi) {
#pragma clang fp contract(off)
    extern __shared__ double smem[];
    const int row = blockIdx.x, tid = threadIdx.x, nthr = blockDim.x, nw = nthr >> 6;
    double* red = smem;
    uint8_t* V = reinterpret_cast<uint8_t*>(smem + 4 * nw);
    const int words = (R + 31) / 32;
    const uint32_t* src = bits + (int64_t)row * words;
    for (int r = tid; r < R; r += nthr) V[r] = (src[r >> 5] >> (r & 31)) & 1u;
    __syncthreads();
    integrals_f64(V, R, tcos, tsin, tdphi, tid, nthr, red);
    if (dphi) {
        const bool case1 = V[0] == 1 && V[R - 1] == 0;
        for (int r = tid; r < R; r += nthr) {
            int o;
            if (case1) o = (int)V[r] - (int)V[r == 0 ? R - 1 : r - 1];
            else o = (int)V[r == R - 1 ? 0 : r + 1] - (int)V[r];
            dphi[(int64_t)row * R + r] = (int8_t)o;
        }
    }
    __syncthreads();
    if (tid == 0) {
        double Tc = 0.0, Ts = 0.0, Ec = 0.0, Es = 0.0;
        for (int w = 0; w < nw; ++w) {
            Tc += red[4 * w]; Ts += red[4 * w + 1]; Ec += red[4 * w + 2]; Es += red[4 * w + 3];
        }
        const double a0 = alp0[row], b0 = bet0[row], vv0 = v0[row], vn = vel[row];
        double* o = out + 6 * (int64_t)row;
        if (phi_ok) {
            const double ab = a0 * Tc, ae = (a0 * alp1) * Ec;
            const double bb = b0 * Ts, be = (b0 * bet1) * Es;
            o[0] = gam * (vv0 - vn) + ab + ae;
            o[1] = bb + be;
            o[2] = ab; o[3] = ae; o[4] = bb; o[5] = be;
        } else {
            for (int q = 0; q < 6; ++q) o[q] = 0.0;
        }
    }
}

}  // namespace

int launch_vf_projection_rows(int R, double fov0, double fov1, int boundary, double W, double H,
                              double fx, double fy, double ftheta, double fradius,
                              const double* ox, const double* oy, const double* osize, int n_obj,
                              uint32_t* rows, int32_t* rec, hipStream_t s) {
    const double step = linspace_step(R);
    const int px0 = linspace_argmin(fov0, R, step), px1 = linspace_argmin(fov1, R, step);
    if (n_obj == 0) return ABM_OK;
    hipLaunchKernelGGL(vf_projection_rows_kernel, dim3((n_obj + 63) / 64), dim3(64), 0, s, R, step,
                       px0, px1, boundary == ABM_BOUNDARY_INFINITE ? 1 : 0, W, H, fx, fy, ftheta,
                       fradius, ox, oy, osize, n_obj, rows, rec);
    return check_hip(hipGetLastError(), "vf_projection_rows_kernel launch");
}

int launch_vf_state_variables(int R, int n, const uint32_t* bits, const double* vel,
                              const double* alp0, const double* bet0, const double* v0,
                              double gam, double alp1, double bet1, const double* tcos,
                              const double* tsin, const double* tdphi, int phi_ok, double* out,
                              int8_t* dphi, hipStream_t s) {
    if (n == 0) return ABM_OK;
    const int nthr = R >= 1024 ? 256 : 64;
    const size_t lds = (size_t)4 * (nthr / 64) * sizeof(double) + (size_t)R + 16;
    hipLaunchKernelGGL(vf_state_variables_kernel, dim3(n), dim3(nthr), lds, s, R, bits, vel, alp0,
                       bet0, v0, gam, alp1, bet1, tcos, tsin, tdphi, phi_ok, out, dphi);
    return check_hip(hipGetLastError(), "vf_state_variables_kernel launch");
}

}  // namespace abm
