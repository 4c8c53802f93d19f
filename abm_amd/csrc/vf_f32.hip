// vf_f32.hip -- fused float32 VSWRM step for batches of replicas.
//
// Persistent workgroups of NW waves; each takes replicas (largest first) and
// runs the reference-order step (agent k sees agents <k moved,
// vf_sims.py:302) with the replica's poses and its float32 ray table in LDS.
//
// Per focal agent k:
//   pairs   -- lanes over the other agents j.  The centre differences, the
//              periodic image, atan2 for the closed angle, atan for the
//              half-width and the bin arithmetic are float32 (fast_pair in
//              vf_f32_common.hpp, within 1e-6 rad of the exact angle).  When the
//              float32 angle lies within a guard band of a bin tie or of the
//              +-pi wrap, the half-width within its band of an integer, or a
//              difference within its band of the half-arena image switch, the
//              pair is re-decided with the exact float64 code of vf_exact.hpp
//              (vf_supcalc.py:55-119), so the raster equals the float64 one.
//   raster  -- each drawn interval (wrap rules of vf_supcalc.py:122-129) is
//              OR-ed into bit-packed uint32 words in LDS.
//   sums    -- lanes over contiguous ray spans: V bits, edges by shift-XOR
//              with the dPhi alignment rule (vf_supcalc.py:266-274), and the
//              four sums over float32 tables (trapz weight * cos/sin, cos, sin);
//              float32 per-lane partials, float64 cross-lane tree.
//   motion  -- float32 VSWRM update, Euler step, boundary (vf_agent.py:188-204,
//              263-326; agent.py:347-395, 605-610).
#include <cmath>
#include <type_traits>

#include "vf_f32_common.hpp"

namespace abm {

namespace {
using namespace f32;

// Replicas with more agents than this take the wide (synchronous) kernel.
constexpr int kWideThreshold = 2048;

// LDS layout: per-agent records as float4 so one 16-byte read serves a pair.
struct Smem {
    RayTab32* tab;     // transposed ray table: entry i*NT + lane holds ray lane*RPL + i
    float4* pose;      // live (x, y, radius, theta) of every agent
    float4* obj;       // positions the pairs read: = pose, or a pre-step copy (synchronous)
    float4* dyn;       // (v, ALP0, BET0, V0)
    int32_t* rlist;    // pairs queued for the float64 decision
    int32_t* rfast;    // their float32 decision (verify mode)
    uint32_t* F;       // the focal agent's bit-packed field
    double* red;       // cross-wave partial sums
    int32_t* nre;
};

__device__ inline Smem carve(void* base, int maxN, int tab_entries, int nw, bool sync_order) {
    Smem s;
    char* p = reinterpret_cast<char*>(base);
    s.tab = reinterpret_cast<RayTab32*>(p); p += sizeof(RayTab32) * tab_entries;
    s.pose = reinterpret_cast<float4*>(p); p += sizeof(float4) * maxN;
    s.dyn = reinterpret_cast<float4*>(p); p += sizeof(float4) * maxN;
    if (sync_order) { s.obj = reinterpret_cast<float4*>(p); p += sizeof(float4) * maxN; }
    else s.obj = s.pose;
    s.red = reinterpret_cast<double*>(p); p += sizeof(double) * (2 * nw + 2);
    s.rlist = reinterpret_cast<int32_t*>(p); p += sizeof(int32_t) * maxN;
    s.rfast = reinterpret_cast<int32_t*>(p); p += sizeof(int32_t) * maxN;
    s.nre = reinterpret_cast<int32_t*>(p); p += sizeof(int32_t) * 4;
    s.F = reinterpret_cast<uint32_t*>(p);
    return s;
}

template <int NW, int RPL, bool PLAIN>   // PLAIN: as the push kernel's
__global__ void __launch_bounds__(64 * NW)
vf_step_f32_kernel(const VFRep* __restrict__ reps, const int32_t* __restrict__ order, int n_rep,
                   const RayTab32* __restrict__ tab32, abm_vf_state_f32 st,
                   uint32_t* __restrict__ bits_out, float* __restrict__ diag, uint32_t flags,
                   unsigned long long* __restrict__ counters, int maxN) {
    extern __shared__ __align__(16) double smem_d[];
    constexpr int NT = 64 * NW;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const bool sync_order = (flags & ABM_ORDER_SYNCHRONOUS) != 0;
    const bool want_diag = !PLAIN && (flags & ABM_WANT_DIAG) != 0 && diag != nullptr;
    const bool count = !PLAIN && (flags & (ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) != 0 && counters;
    const bool verify = !PLAIN && (flags & ABM_VERIFY_FAST_PATH) != 0 && counters != nullptr;
    Smem S = carve(smem_d, maxN, RPL * NT, NW, sync_order);
    int loaded_tab = -1;
    uint32_t n_pairs = 0, n_recheck = 0, n_disagree = 0;   // this lane's

    for (int idx = blockIdx.x; idx < n_rep; idx += gridDim.x) {
        const VFRep* rp = reps + order[idx];
        const RepConst C = rep_const(rp);
        const int tab_off = rp->table_offset;
        if (tab_off != loaded_tab) {
            for (int e = tid; e < RPL * NT; e += NT) {
                const int r = (e % NT) * RPL + e / NT;
                RayTab32 z;
                z.wcos = z.wsin = z.cos = z.sin = 0.f;
                S.tab[e] = r < C.R ? tab32[tab_off + r] : z;
            }
            loaded_tab = tab_off;
        }
        const float a0d = (float)rp->alp0, b0d = (float)rp->bet0, v0d = (float)rp->v0;
        for (int i = tid; i < C.N; i += NT) {
            const int g = C.a0 + i;
            const float4 p = make_float4(st.x[g], st.y[g], (float)st.radius[g], st.theta[g]);
            S.pose[i] = p;
            if (sync_order) S.obj[i] = p;
            S.dyn[i] = make_float4(st.v[g], st.alp0 ? st.alp0[g] : a0d, st.bet0 ? st.bet0[g] : b0d,
                                   st.v0 ? st.v0[g] : v0d);
        }
        const int rs = tid * RPL;            // this lane's ray span [rs, rs + rn)
        const int rn = rs >= C.R ? 0 : (C.R - rs < RPL ? C.R - rs : RPL);
        if (tid == 0) S.nre[0] = 0;
        __syncthreads();
        // heading of agent 0 (later headings come with the previous agent's motion)
        float sth, cth;
        sincos_f32(S.pose[0].w, &sth, &cth);

        for (int k = 0; k < C.N; ++k) {
            for (int w = tid; w < C.W; w += NT) S.F[w] = 0u;
            const float4 fp = S.pose[k];
            const float fx = fp.x, fy = fp.y, fr = fp.z, fth = fp.w;
            const float u1x = cth, u1y = -sth;           // unit(v1) = (cos th, -sin th)
            __syncthreads();

            // ------------------------------------------------ pairs, float32
            for (int j = tid; j < C.N; j += NT) {
                if (j == k) continue;
                const float4 o = S.obj[j];
                if (o.x == fx && o.y == fy) continue;          // coincident (:57)
                PairF32 p = fast_pair(u1x, u1y, fx, fy, fr, o.x, o.y, o.z, C);
                if (count) ++n_pairs;
                if (p.tie && tie_in_place(p, fx, fy, fth, fr, o.x, o.y, o.z, rp, C))   // rare
                    if (count) ++n_recheck;   // a float64 decision too
                if (!p.ok || verify) {
                    const int slot = atomicAdd(S.nre, 1);
                    S.rlist[slot] = entry_code(j, 0, p.ok);
                    S.rfast[slot] = fast_code(p.start, p.end, p.drawn, C.R);
                    if (!p.ok) continue;
                }
                if (p.drawn) raster_lds(S.F, p.start, p.end, C.R);
            }
            __syncthreads();
            // ------------------------------------- pairs re-decided in float64
            const int nre = S.nre[0];
            if (nre > 0) {
                for (int i = tid; i < nre; i += NT) {
                    const int e = S.rlist[i];
                    const int fc = S.rfast[i];
                    const int j = e & 0xfffff;
                    const float4 o = S.obj[j];
                    int dis;
                    const int r = resolve_queued(e, fc, fx, fy, fth, fr, o.x, o.y, o.z, rp, verify, &dis);
                    n_disagree += dis;
                    if (e & kEntryForced) {
                        if (count) ++n_recheck;
                        if (r >= 0) raster_lds(S.F, (r & 0x7fff) - 2 * C.R, ((r >> 15) & 0x7fff) - 2 * C.R, C.R);
                    }
                }
                __syncthreads();
                if (tid == 0) S.nre[0] = 0;
            }

            // ------------------------------------------------ sums
            const bool case1 = (S.F[0] & 1u) == 1u && field_bit(S.F, C.R - 1) == 0u;
            float bc = 0.f, bs = 0.f, ec = 0.f, es = 0.f;
            {
                // rays at or beyond R have zero table entries and zero bits
                const int w0 = rs >> 5;
                const uint32_t lo = w0 < C.W ? S.F[w0] : 0u;
                const uint32_t hi = (RPL > 1 && w0 + 1 < C.W) ? S.F[w0 + 1] : 0u;
                const uint64_t v64 = (((uint64_t)hi << 32) | lo) >> (rs & 31);
                const uint32_t m = low_mask(rn);
                const uint32_t cur = (uint32_t)v64 & m;
                uint32_t spike = 0u;
                if (rn > 0) {
                    if (case1) {
                        const uint32_t prev = field_bit(S.F, rs == 0 ? C.R - 1 : rs - 1);
                        spike = (cur ^ ((cur << 1) | prev)) & m;
                    } else {
                        const int nx = rs + rn;
                        const uint32_t next = field_bit(S.F, nx >= C.R ? 0 : nx);
                        spike = (cur ^ ((cur >> 1) | (next << (rn - 1)))) & m;
                    }
                }
#pragma unroll
                for (int i = 0; i < RPL; ++i) {
                    const RayTab32 T = S.tab[i * NT + tid];
                    const float vb = (float)((cur >> i) & 1u);   // acc + (bit ? t : 0) as fma(bit, t, acc)
                    const float sb = (float)((spike >> i) & 1u);
                    bc = __builtin_fmaf(vb, T.wcos, bc);
                    bs = __builtin_fmaf(vb, T.wsin, bs);
                    ec = __builtin_fmaf(sb, T.cos, ec);
                    es = __builtin_fmaf(sb, T.sin, es);
                }
            }
            const float4 dk = S.dyn[k];
            const float alp0 = dk.y, bet0 = dk.z, v0 = dk.w;
            // blob terms: trapz(cos(PHI) * (-V)) = -sum(w cos V)
            double Sv, Sp, Bc = 0.0, Bs = 0.0, Ec = 0.0, Es = 0.0;
            if (!want_diag) {
                Sv = wave_total(alp0 * (-bc) + (alp0 * C.alp1) * ec);
                Sp = wave_total(bet0 * (-bs) + (bet0 * C.bet1) * es);
            } else {
                Bc = wave_total(bc); Bs = wave_total(bs);
                Ec = wave_total(ec); Es = wave_total(es);
                Sv = (double)alp0 * -Bc + (double)(alp0 * C.alp1) * Ec;
                Sp = (double)bet0 * -Bs + (double)(bet0 * C.bet1) * Es;
            }
            if (NW > 1) {
                if (lane == 0) {
                    S.red[2 * (tid >> 6)] = Sv; S.red[2 * (tid >> 6) + 1] = Sp;
                }
                __syncthreads();
                Sv = Sp = 0.0;
                for (int w = 0; w < NW; ++w) { Sv += S.red[2 * w]; Sp += S.red[2 * w + 1]; }
                if (want_diag) {   // components of the other waves
                    __syncthreads();
                    double comp[4] = {Bc, Bs, Ec, Es};
                    for (int c = 0; c < 4; ++c) {
                        if (lane == 0) S.red[tid >> 6] = comp[c];
                        __syncthreads();
                        double t = 0.0;
                        for (int w = 0; w < NW; ++w) t += S.red[w];
                        comp[c] = t;
                        __syncthreads();
                    }
                    Bc = comp[0]; Bs = comp[1]; Ec = comp[2]; Es = comp[3];
                }
            }
            if (!PLAIN && bits_out) {
                uint32_t* dst = bits_out + C.field_offset + (int64_t)k * C.W;
                for (int w = tid; w < C.W; w += NT) dst[w] = S.F[w];
            }

            // ------------------------------------------------ motion
            float vel, o, dv, dpsi;
            steer(C, fth, dk.x, v0, (float)Sv, (float)Sp, &o, &vel, &dv, &dpsi);
            // one sincos serves this agent's motion (lane 0) and the next
            // agent's heading (lane 1)
            const float ang = (lane == 1 && k + 1 < C.N) ? S.pose[k + 1].w : o;
            float s_l, c_l;
            sincos_f32(ang, &s_l, &c_l);
            const float so = lane_f32(s_l, 0), co = lane_f32(c_l, 0);
            sth = lane_f32(s_l, 1);
            cth = lane_f32(c_l, 1);
            float nx, ny;
            euler_boundary(C, fx, fy, fr, vel, so, co, &o, &nx, &ny);
            if (tid == 0) {
                S.pose[k] = make_float4(nx, ny, fr, o);
                S.dyn[k].x = vel;
                if (want_diag) {
                    float* dd = diag + 6 * (int64_t)(C.a0 + k);
                    dd[0] = dv; dd[1] = dpsi;
                    dd[2] = C.phi_ok ? (float)((double)alp0 * -Bc) : 0.f;
                    dd[3] = C.phi_ok ? (float)((double)(alp0 * C.alp1) * Ec) : 0.f;
                    dd[4] = C.phi_ok ? (float)((double)bet0 * -Bs) : 0.f;
                    dd[5] = C.phi_ok ? (float)((double)(bet0 * C.bet1) * Es) : 0.f;
                }
            }
            __syncthreads();
        }
        for (int i = tid; i < C.N; i += NT) {
            const int g = C.a0 + i;
            const float4 p = S.pose[i];
            st.x[g] = p.x;
            st.y[g] = p.y;
            st.theta[g] = p.w;
            st.v[g] = S.dyn[i].x;
        }
        __syncthreads();
    }
    if (count) {
        if (n_pairs) atomicAdd(&counters[0], (unsigned long long)n_pairs);
        if (n_recheck) atomicAdd(&counters[1], (unsigned long long)n_recheck);
        if (n_disagree) atomicAdd(&counters[2], (unsigned long long)n_disagree);
    }
}

// ---------------------------------------------------------------------------
// Wide variant for single large flocks, synchronous order only: one wave per
// focal agent, four waves per workgroup.  The waves of a workgroup share the
// ray table and 256-agent tiles of the (pre-step) poses in LDS.  A cheap
// float32 distance pass first drops every pair beyond the exact visibility
// cut-off -- the raster of a pair is empty when floor(proj_size / 2) = 0,
// i.e. when d > size * cot(2 pi / R) -- with a relative guard of 2e-4, and
// compacts the others; only those take the float32 decision.  New poses go
// to a scratch buffer and are copied back by a second kernel.
constexpr int kWideWaves = 8;    // focal agents per block, sharing the ray table
constexpr int kWideTile = 512;  // objects per LDS tile of the full scan (one per thread)
constexpr int kWideQueue = 128;   // grid path: candidates queued per wave (tile + cand memory)
static_assert(sizeof(float4) * kWideTile + sizeof(int32_t) * kWideTile * kWideWaves >=
              sizeof(float4) * kWideQueue * kWideWaves, "grid queues reuse the tile memory");

// Grid cell of a centre: the coordinate taken modulo the arena, clamped
// into the grid (rounding at the far edge).
__device__ inline int grid_cell(const WideGrid& G, float cx, float cy) {
    float u = cx - G.x0, v = cy - G.y0;
    u = u - G.W * floorf(u / G.W);
    v = v - G.H * floorf(v / G.H);
    const int ix = min(G.nx - 1, max(0, (int)(u / G.cw)));
    const int iy = min(G.ny - 1, max(0, (int)(v / G.ch)));
    return iy * G.nx + ix;
}

// Decision and raster of one pair of the grid path (no counters, no verify).
__device__ __forceinline__ void wide_decide(const float4 o, float u1x, float u1y, float fx, float fy,
                                            float fth, float fr, const VFRep* rp, const RepConst& C,
                                            uint32_t* F) {
    PairF32 p = fast_pair(u1x, u1y, fx, fy, fr, o.x, o.y, o.z, C);
    if (p.tie) tie_in_place(p, fx, fy, fth, fr, o.x, o.y, o.z, rp, C);   // rare
    if (!p.ok) {
        int es = 0, ee = 0, ed = 0;
        exact_pair(fx, fy, fth, fr, o.x, o.y, o.z, rp, &es, &ee, &ed);
        p.start = es; p.end = ee; p.drawn = ed != 0;
    }
    if (p.drawn) raster_lds(F, p.start, p.end, C.R);
}

// LDS written by some lanes of a wave and read by others: in-order per
// wave once the writes have completed.
__device__ inline void wave_lds_sync() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}


struct WideSmem {
    RayTab32* tab;      // transposed for 64 lanes
    float4* tile;       // (x, y, radius, -) of the current object tile
    uint32_t* F;        // kWideWaves fields of maxW words
    int32_t* cand;      // kWideWaves lists of tile-local candidates
};

// START: the chain step's first pass instead (see vf_step_f32_chain_kernel):
// agent k's pairs with the agents after it in id order only, its field written
// to start_fields[k W ..] and its heading vector to start_u[k]; no move.
template <int RPL, bool START, bool PLAIN>   // PLAIN: as the push kernel's
__global__ void __launch_bounds__(64 * kWideWaves)
vf_step_f32_wide_kernel(const VFRep* __restrict__ rp, const RayTab32* __restrict__ tab32,
                        abm_vf_state_f32 st, float4* __restrict__ out_pose,
                        uint32_t* __restrict__ bits_out, float* __restrict__ diag, uint32_t flags,
                        unsigned long long* __restrict__ counters, float cull_c,
                        const WideGrid* __restrict__ grid, const float4* __restrict__ sorted,
                        const int32_t* __restrict__ cell_start, uint32_t* __restrict__ start_fields,
                        float2* __restrict__ start_u) {
    extern __shared__ __align__(16) double smem_d[];
    const RepConst C = rep_const(rp);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const bool want_diag = !PLAIN && (flags & ABM_WANT_DIAG) != 0 && diag != nullptr;
    const bool count = !PLAIN && (flags & (ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) != 0 && counters;
    const bool verify = !PLAIN && (flags & ABM_VERIFY_FAST_PATH) != 0 && counters != nullptr;
    // Grid path (counters and verify mode keep the full scan): focal agents
    // in cell order, so a block's waves read the same neighbourhoods
    const WideGrid G = *grid;
    const bool use_grid = G.ok && !count && !verify;
    const int slot = blockIdx.x * kWideWaves + wave;
    const bool active = slot < C.N;
    const int k = (use_grid && active) ? __float_as_int(sorted[slot].w) : slot;
    const int maxW = (RPL * 64 + 31) >> 5;
    WideSmem S;
    {
        char* p = reinterpret_cast<char*>(smem_d);
        S.tab = reinterpret_cast<RayTab32*>(p); p += sizeof(RayTab32) * RPL * 64;
        S.tile = reinterpret_cast<float4*>(p); p += sizeof(float4) * kWideTile;
        S.cand = reinterpret_cast<int32_t*>(p); p += sizeof(int32_t) * kWideTile * kWideWaves;
        S.F = reinterpret_cast<uint32_t*>(p);
    }
    uint32_t* F = S.F + wave * maxW;
    int32_t* cand = S.cand + wave * kWideTile;
    const int tab_off = rp->table_offset;
    for (int e = tid; e < (START ? 0 : RPL * 64); e += 64 * kWideWaves) {
        const int r = (e % 64) * RPL + e / 64;
        RayTab32 z = tab32[tab_off + (r < C.R ? r : 0)];
        if (r >= C.R) z.wcos = z.wsin = z.cos = z.sin = 0.f;
        S.tab[e] = z;
    }
    for (int w = lane; w < maxW; w += 64) F[w] = 0u;
    const int g = C.a0 + (active ? k : 0);
    const float fx = st.x[g], fy = st.y[g], fth = st.theta[g], fr = (float)st.radius[g];
    float sth, cth;
    sincos_f32(fth, &sth, &cth);
    const float u1x = cth, u1y = -sth;
    unsigned long long n_pairs = 0, n_recheck = 0, n_disagree = 0;
    // Grid path: each wave takes its focal agent's 3 x 3 cells from the
    // sorted agents (the next 64 loaded while the current 64 are tested),
    // queues the pairs inside the cut-off and decides them 64 at a time.  No
    // block barrier inside: the waves share only the ray table.
    if (use_grid) {
        __syncthreads();   // the ray table
        if (active) {
            float4* cq = reinterpret_cast<float4*>(S.tile) + wave * kWideQueue;
            int nq = 0;
            const int fc = grid_cell(G, fx + fr, fy + fr);
            const int fiy = fc / G.nx, fix = fc - fiy * G.nx;
            const int xl = fix == 0 ? G.nx - 1 : fix - 1, xr = fix == G.nx - 1 ? 0 : fix + 1;
            const int yl = fiy == 0 ? G.ny - 1 : fiy - 1, yr = fiy == G.ny - 1 ? 0 : fiy + 1;
            for (int t = 0; t < 9; ++t) {   // the 3 x 3 cells, wrapped
                const int ty = t >= 6 ? 2 : (t >= 3 ? 1 : 0), tx = t - 3 * ty;
                const int cy = ty == 0 ? yl : (ty == 1 ? fiy : yr);
                const int cx = tx == 0 ? xl : (tx == 1 ? fix : xr);
                const int c = cy * G.nx + cx;
                const int end = cell_start[c + 1];
                int pos = cell_start[c];
                // loads always from a valid index; the next 64 are in flight
                // while these are tested
                float4 nxt = sorted[pos + lane < end ? pos + lane : 0];
                while (pos < end) {
                    const bool valid = pos + lane < end;
                    const float4 o = nxt;
                    pos += 64;
                    nxt = sorted[pos + lane < end ? pos + lane : 0];
                    bool cnd = false;
                    const int j = __float_as_int(o.w);
                    if (valid && (START ? j > k : j != k) && !(o.x == fx && o.y == fy)) {
                        float dx = (o.x - fx) + (o.z - fr), dy = (o.y - fy) + (o.z - fr);
                        const float ex = fabsf(dx) - C.hw, ey = fabsf(dy) - C.hh;
                        const bool near_wrap = fabsf(ex) < C.tguard || fabsf(ey) < C.tguard;
                        if (ex > 0.f) dx = dx > 0.f ? dx - C.fW : dx + C.fW;
                        if (ey > 0.f) dy = dy > 0.f ? dy - C.fH : dy + C.fH;
                        const float lim = o.z * cull_c;
                        cnd = near_wrap || fmaf(dy, dy, dx * dx) <= lim * lim;
                    }
                    const uint64_t m = __ballot(cnd);
                    if (cnd) cq[nq + __popcll(m & ((1ull << lane) - 1ull))] = o;
                    nq += __popcll(m);
                    if (nq >= 64) {
                        wave_lds_sync();
                        wide_decide(cq[lane], u1x, u1y, fx, fy, fth, fr, rp, C, F);
                        const int rest = nq - 64;
                        const float4 tq = cq[64 + lane];   // lanes >= rest read a stale entry, unused
                        wave_lds_sync();
                        if (lane < rest) cq[lane] = tq;
                        nq = rest;
                        wave_lds_sync();
                    }
                }
            }
            wave_lds_sync();
            if (lane < nq) wide_decide(cq[lane], u1x, u1y, fx, fy, fth, fr, rp, C, F);
            wave_lds_sync();
        }
    }

    // (START: the tiles before the block's first agent hold no pair)
    const int t_first = START ? (blockIdx.x * kWideWaves / kWideTile) * kWideTile : 0;
    for (int t0 = t_first; t0 < (use_grid ? 0 : C.N); t0 += kWideTile) {
        __syncthreads();
        if (t0 + tid < C.N) {
            const int gj = C.a0 + t0 + tid;
            S.tile[tid] = make_float4(st.x[gj], st.y[gj], (float)st.radius[gj], 0.f);
        }
        __syncthreads();
        // cheap pass: candidates inside the cut-off (or inside a torus guard band)
        int ncand = 0;
        const int tn = C.N - t0 < kWideTile ? C.N - t0 : kWideTile;
        for (int sub = 0; sub < kWideTile; sub += 64) {
            const int jt = sub + lane;
            bool c = false, culled = false;
            if (active && jt < tn && (START ? t0 + jt > k : t0 + jt != k)) {
                const float4 o = S.tile[jt];
                if (!(o.x == fx && o.y == fy)) {
                    if (count) ++n_pairs;
                    float dx = (o.x - fx) + (o.z - fr), dy = (o.y - fy) + (o.z - fr);
                    bool near_wrap = false;
                    if (C.torus) {
                        const float ex = fabsf(dx) - C.hw, ey = fabsf(dy) - C.hh;
                        near_wrap = fabsf(ex) < C.tguard || fabsf(ey) < C.tguard;
                        if (ex > 0.f) dx = dx > 0.f ? dx - C.fW : dx + C.fW;
                        if (ey > 0.f) dy = dy > 0.f ? dy - C.fH : dy + C.fH;
                    }
                    const float lim = o.z * cull_c;
                    culled = !near_wrap && fmaf(dy, dy, dx * dx) > lim * lim;
                    c = !culled || verify;
                }
            }
            const uint64_t m = __ballot(c);
            if (c) {
                const int pos = ncand + __popcll(m & ((1ull << lane) - 1ull));
                cand[pos] = jt | (culled ? (1 << 30) : 0);
            }
            ncand += __popcll(m);
        }
        __syncthreads();
        // float32 decisions of the candidates (float64 when inside a guard band)
        for (int c0 = 0; c0 < ncand; c0 += 64) {
            const int ci = c0 + lane;
            if (ci >= ncand) continue;
            const int e = cand[ci];
            const int jt = e & ((1 << 30) - 1);
            const bool culled = (e >> 30) & 1;
            const float4 o = S.tile[jt];
            PairF32 p = fast_pair(u1x, u1y, fx, fy, fr, o.x, o.y, o.z, C);
            if (p.tie && tie_in_place(p, fx, fy, fth, fr, o.x, o.y, o.z, rp, C))   // rare
                if (count) ++n_recheck;   // a float64 decision too
            if (!p.ok || verify) {
                int es = 0, ee = 0, ed = 0;
                exact_pair(fx, fy, fth, fr, o.x, o.y, o.z, rp, &es, &ee, &ed);
                if (verify) {
                    // a culled pair must have an empty raster; a float32 decision must match
                    const bool empty = !ed || es == ee;
                    if ((culled && !empty) ||
                        (!culled && p.ok && (es != p.start || ee != p.end || ed != (int)p.drawn)))
                        ++n_disagree;
                }
                if (!p.ok) {
                    if (count) ++n_recheck;
                    p.start = es; p.end = ee; p.drawn = ed != 0;
                }
            }
            if (culled) continue;
            if (p.drawn) raster_lds(F, p.start, p.end, C.R);
        }
    }
    if (!use_grid) __syncthreads();
    if (START) {
        if (active) {
            uint32_t* dst = start_fields + (size_t)k * C.W;
            for (int w = lane; w < C.W; w += 64) dst[w] = F[w];
            if (lane == 0) start_u[k] = make_float2(u1x, u1y);
        }
        if (count) {
            if (n_pairs) atomicAdd(&counters[0], n_pairs);
            if (n_recheck) atomicAdd(&counters[1], n_recheck);
            if (n_disagree) atomicAdd(&counters[2], n_disagree);
        }
        return;
    }
    if (!active) {
        if (count) {
            if (n_pairs) atomicAdd(&counters[0], n_pairs);
        }
        return;
    }
    // sums over this wave's field (lanes own RPL consecutive rays)
    const int rs = lane * RPL;
    const int rn = rs >= C.R ? 0 : (C.R - rs < RPL ? C.R - rs : RPL);
    const bool case1 = (F[0] & 1u) == 1u && field_bit(F, C.R - 1) == 0u;
    float bc = 0.f, bs = 0.f, ec = 0.f, es = 0.f;
    {
        const int w0 = rs >> 5;
        const uint32_t lo = w0 < C.W ? F[w0] : 0u;
        const uint32_t hi = (RPL > 1 && w0 + 1 < C.W) ? F[w0 + 1] : 0u;
        const uint64_t v64 = (((uint64_t)hi << 32) | lo) >> (rs & 31);
        const uint32_t m = low_mask(rn);
        const uint32_t cur = (uint32_t)v64 & m;
        uint32_t spike = 0u;
        if (rn > 0) {
            if (case1) {
                const uint32_t prev = field_bit(F, rs == 0 ? C.R - 1 : rs - 1);
                spike = (cur ^ ((cur << 1) | prev)) & m;
            } else {
                const int nx = rs + rn;
                const uint32_t next = field_bit(F, nx >= C.R ? 0 : nx);
                spike = (cur ^ ((cur >> 1) | (next << (rn - 1)))) & m;
            }
        }
#pragma unroll 8
        for (int i = 0; i < RPL; ++i) {
            const RayTab32 T = S.tab[i * 64 + lane];
            const float vb = (float)((cur >> i) & 1u);   // acc + (bit ? t : 0) as fma(bit, t, acc)
            const float sb = (float)((spike >> i) & 1u);
            bc = __builtin_fmaf(vb, T.wcos, bc);
            bs = __builtin_fmaf(vb, T.wsin, bs);
            ec = __builtin_fmaf(sb, T.cos, ec);
            es = __builtin_fmaf(sb, T.sin, es);
        }
    }
    const float alp0 = st.alp0 ? st.alp0[g] : (float)rp->alp0;
    const float bet0 = st.bet0 ? st.bet0[g] : (float)rp->bet0;
    const float v0 = st.v0 ? st.v0[g] : (float)rp->v0;
    const double Bc = wave_total(bc), Bs = wave_total(bs), Ec = wave_total(ec), Es = wave_total(es);
    const double Sv = (double)alp0 * -Bc + (double)(alp0 * C.alp1) * Ec;
    const double Sp = (double)bet0 * -Bs + (double)(bet0 * C.bet1) * Es;
    if (!PLAIN && bits_out) {
        uint32_t* dst = bits_out + C.field_offset + (int64_t)k * C.W;
        for (int w = lane; w < C.W; w += 64) dst[w] = F[w];
    }
    float vel, o, dv, dpsi;
    steer(C, fth, st.v[g], v0, (float)Sv, (float)Sp, &o, &vel, &dv, &dpsi);
    float so, co;
    sincos_f32(o, &so, &co);
    float nx, ny;
    euler_boundary(C, fx, fy, fr, vel, so, co, &o, &nx, &ny);
    if (lane == 0) {
        out_pose[g] = make_float4(nx, ny, o, vel);
        if (want_diag) {
            float* dd = diag + 6 * (int64_t)g;
            dd[0] = dv; dd[1] = dpsi;
            dd[2] = C.phi_ok ? (float)((double)alp0 * -Bc) : 0.f;
            dd[3] = C.phi_ok ? (float)((double)(alp0 * C.alp1) * Ec) : 0.f;
            dd[4] = C.phi_ok ? (float)((double)bet0 * -Bs) : 0.f;
            dd[5] = C.phi_ok ? (float)((double)(bet0 * C.bet1) * Es) : 0.f;
        }
    }
    if (count) {
        if (n_pairs) atomicAdd(&counters[0], n_pairs);
        if (n_recheck) atomicAdd(&counters[1], n_recheck);
        if (n_disagree) atomicAdd(&counters[2], n_disagree);
    }
}

// Inclusive prefix sum over the 64 lanes: inside rows of 16, then rows 0 and 2
// into 1 and 3, then the lower half into the upper.
__device__ inline int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return v;
}

// One block: the replica's grid (cells no narrower than the largest
// visibility cut-off r_max * cull_c, plus 0.1 % and 1 px) and its agents
// sorted by cell (counting sort in LDS).  The order inside a cell is free:
// the field is an OR of rasters.  Bound by latency: the agents' loads, a few
// barriers, the scatter.  The first 8192 agents stay in registers from one load
// to the scatter, the radii meet by wave and the counts are summed by wave
// (before, three passes over global memory, 1024 atomics to one word and twenty
// barriers: 16.6 us for 8192 agents, 10.5 now, of 87.8 and 81.6 in a synchronous
// step).
__global__ void __launch_bounds__(1024)
wide_grid_kernel(const VFRep* __restrict__ rp, abm_vf_state_f32 st, float cull_c,
                 float4* __restrict__ sorted, int32_t* __restrict__ cell_start,
                 WideGrid* __restrict__ grid) {
    __shared__ int cnt[kWideGridMaxCells + 1];
    __shared__ int part[16];
    __shared__ int rmax;
    __shared__ WideGrid G;
    const RepConst C = rep_const(rp);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int nthr = 1024;
    if (tid == 0) rmax = 0;
    // eight agents per thread per pass, their loads issued together; the first
    // pass's stay
    constexpr int kPer = 8;
    float px[kPer], py[kPer];
    int pr[kPer], cell[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int i = q * nthr + tid, g = C.a0 + (i < C.N ? i : 0);
        px[q] = st.x[g]; py[q] = st.y[g]; pr[q] = (int)st.radius[g];
    }
    for (int c = tid; c <= kWideGridMaxCells; c += nthr) cnt[c] = 0;
    int rm = 0;
#pragma unroll
    for (int q = 0; q < kPer; ++q) rm = max(rm, q * nthr + tid < C.N ? pr[q] : 0);
    for (int base = nthr * kPer; base < C.N; base += nthr * kPer) {
        int rv[kPer];
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int i = base + q * nthr + tid;
            rv[q] = i < C.N ? (int)st.radius[C.a0 + i] : 0;
        }
#pragma unroll
        for (int q = 0; q < kPer; ++q) rm = max(rm, rv[q]);
    }
    for (int o = 32; o > 0; o >>= 1) rm = max(rm, __shfl_xor(rm, o, 64));
    __syncthreads();
    if (lane == 0) atomicMax(&rmax, rm);
    __syncthreads();
    if (tid == 0) {
        WideGrid g;
        g.pad_ = 0;
        g.x0 = C.pad; g.y0 = C.pad; g.W = C.fW; g.H = C.fH;
        const float reach = (float)rmax * cull_c * 1.001f + 1.0f;
        g.nx = min(kWideGridMaxSide, (int)floorf(C.fW / reach));
        g.ny = min(kWideGridMaxSide, (int)floorf(C.fH / reach));
        g.ok = C.torus && g.nx >= 3 && g.ny >= 3 && C.hw - C.tguard > reach && C.hh - C.tguard > reach;
        g.cw = g.nx > 0 ? C.fW / (float)g.nx : 1.f;
        g.ch = g.ny > 0 ? C.fH / (float)g.ny : 1.f;
        G = g;
        *grid = g;
    }
    __syncthreads();
    if (!G.ok) return;
    const int ncell = G.nx * G.ny;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const float r = (float)pr[q];
        cell[q] = grid_cell(G, px[q] + r, py[q] + r);
        if (q * nthr + tid < C.N) atomicAdd(&cnt[cell[q]], 1);
    }
    for (int base = nthr * kPer; base < C.N; base += nthr * kPer) {
        float x[kPer], y[kPer], r[kPer];
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int i = base + q * nthr + tid;
            const int g = C.a0 + (i < C.N ? i : 0);
            x[q] = st.x[g]; y[q] = st.y[g]; r[q] = (float)st.radius[g];
        }
#pragma unroll
        for (int q = 0; q < kPer; ++q)
            if (base + q * nthr + tid < C.N) atomicAdd(&cnt[grid_cell(G, x[q] + r[q], y[q] + r[q])], 1);
    }
    __syncthreads();
    // exclusive scan of the counts: a run of cells per thread, the runs by wave
    const int per = (ncell + nthr - 1) / nthr;
    int run = 0;
    for (int q = 0; q < per; ++q) {
        const int c = tid * per + q;
        if (c < ncell) run += cnt[c];
    }
    const int upto = wave_scan(run);
    if (lane == 63) part[wave] = upto;
    __syncthreads();
    int acc = upto - run;
    for (int w = 0; w < wave; ++w) acc += part[w];
    for (int q = 0; q < per; ++q) {
        const int c = tid * per + q;
        if (c < ncell) {
            const int n = cnt[c];
            cnt[c] = acc;          // now the cell's write cursor
            cell_start[c] = acc;
            acc += n;
        }
    }
    if (tid == 0) cell_start[ncell] = C.N;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int i = q * nthr + tid;
        if (i < C.N) sorted[atomicAdd(&cnt[cell[q]], 1)] = make_float4(px[q], py[q], (float)pr[q], __int_as_float(i));
    }
    for (int base = nthr * kPer; base < C.N; base += nthr * kPer) {
        float x[kPer], y[kPer], r[kPer];
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int i = base + q * nthr + tid;
            const int g = C.a0 + (i < C.N ? i : 0);
            x[q] = st.x[g]; y[q] = st.y[g]; r[q] = (float)st.radius[g];
        }
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int i = base + q * nthr + tid;
            if (i < C.N)
                sorted[atomicAdd(&cnt[grid_cell(G, x[q] + r[q], y[q] + r[q])], 1)] =
                    make_float4(x[q], y[q], r[q], __int_as_float(i));
        }
    }
}

__global__ void copy_back_kernel(const float4* __restrict__ out_pose, abm_vf_state_f32 st, int a0, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 p = out_pose[a0 + i];
    st.x[a0 + i] = p.x;
    st.y[a0 + i] = p.y;
    st.theta[a0 + i] = p.z;
    st.v[a0 + i] = p.w;
}

size_t lds_bytes_wide(int rpl) {
    const int maxW = (rpl * 64 + 31) >> 5;
    return sizeof(RayTab32) * (size_t)rpl * 64 + sizeof(float4) * kWideTile +
           sizeof(int32_t) * kWideTile * kWideWaves + sizeof(uint32_t) * (size_t)maxW * kWideWaves;
}

template <int RPL>
int launch_wide(abm_vf_batch* b, const abm_vf_state_f32* st, uint32_t* bits, float* diag,
                uint32_t flags, hipStream_t s) {
    const size_t lds = lds_bytes_wide(RPL);
    const bool plain = bits == nullptr && (flags & (ABM_WANT_DIAG | ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) == 0;
    auto kern = plain ? vf_step_f32_wide_kernel<RPL, false, true> : vf_step_f32_wide_kernel<RPL, false, false>;
    if (lds > 65536) {
        if (int rc = check_hip(hipFuncSetAttribute((const void*)kern,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                               "hipFuncSetAttribute"))
            return rc;
    }
    for (int rep = 0; rep < b->n_replicas; ++rep) {
        const VFRep& h = b->reps_host[rep];
        // visibility cut-off: floor(proj_size/2) >= 1 needs d <= size * cot(2 pi / R)
        const float cull_c = (float)((1.0 / std::tan(kTwoPi / h.n_rays)) * (1.0 + 2e-4));
        const int blocks = (h.n_agents + kWideWaves - 1) / kWideWaves;
        WideGrid* grid = (WideGrid*)b->grid_param;
        hipLaunchKernelGGL(wide_grid_kernel, dim3(1), dim3(1024), 0, s, b->reps_dev + rep, *st, cull_c,
                           b->grid_sorted, b->grid_start, grid);
        if (int rc = check_hip(hipGetLastError(), "wide_grid_kernel launch")) return rc;
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * kWideWaves), lds, s, b->reps_dev + rep,
                           b->tab32, *st, b->wide_out, bits, diag, flags, b->counters, cull_c,
                           (const WideGrid*)grid, (const float4*)b->grid_sorted,
                           (const int32_t*)b->grid_start, nullptr, nullptr);
        if (int rc = check_hip(hipGetLastError(), "vf_step_f32_wide_kernel launch")) return rc;
        hipLaunchKernelGGL(copy_back_kernel, dim3((h.n_agents + 255) / 256), dim3(256), 0, s,
                           (const float4*)b->wide_out, *st, h.agent_offset, h.n_agents);
        if (int rc = check_hip(hipGetLastError(), "copy_back_kernel launch")) return rc;
    }
    b->last_kernels |= ABM_KERNEL_WIDE;
    return ABM_OK;
}

// ---------------------------------------------------------------------------
// Reference (id) order for replicas beyond kWideThreshold agents: one
// workgroup of 1024 threads per replica, agents in id order as in the
// per-replica kernel, with every agent's pose (x, y, radius, theta) in LDS,
// 16 bytes each (up to about 8,900 agents in 160 KB).  Velocities and the
// ray table stay in global memory (each thread keeps its rays' table entries
// in registers for the whole step).  Per focal agent k: a cheap float32 pass
// over all others drops the pairs beyond the exact visibility cut-off (as
// the wide kernel) and queues the rest in LDS (16-bit indices); the queued
// pairs take the float32 decision (float64 inside the guard bands) and are
// ORed into the field; each thread sums its rays, the waves' sums meet in
// LDS, wave 0 moves agent k.
constexpr int kBigThreads = 1024;
constexpr int kBigWaves = kBigThreads / 64;

// Queue segment of one wave: wave w owns the objects j with j mod 1024 in
// [64 w, 64 w + 64), at most 64 per 1024 agents.
__host__ __device__ inline int big_segment(int maxN) { return 64 * ((maxN + kBigThreads - 1) / kBigThreads); }

// The queues of 16-bit indices, padded to 16 bytes (what follows is int32).
__host__ __device__ inline size_t big_queue_bytes(int maxN) {
    return ((size_t)kBigWaves * big_segment(maxN) * sizeof(uint16_t) + 15) & ~(size_t)15;
}

size_t lds_bytes_big(int maxN, int maxR) {
    const int maxW = (maxR + 31) >> 5;
    size_t b = sizeof(float4) * (size_t)maxN + big_queue_bytes(maxN) +
               sizeof(double) * (4 * kBigWaves + 8) + sizeof(uint32_t) * (size_t)(maxW + 4);
    return (b + 15) & ~(size_t)15;
}

template <int RPL, bool PLAIN>   // PLAIN: as the push kernel's
__global__ void __launch_bounds__(kBigThreads)
vf_step_f32_big_kernel(const VFRep* __restrict__ reps, const int32_t* __restrict__ order,
                       const RayTab32* __restrict__ tab32, abm_vf_state_f32 st,
                       uint32_t* __restrict__ bits_out, float* __restrict__ diag, uint32_t flags,
                       unsigned long long* __restrict__ counters, float cull_c, int maxN, int maxR) {
    extern __shared__ __align__(16) double smem_d[];
    const VFRep* rp = reps + order[blockIdx.x];
    const RepConst C = rep_const(rp);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const bool want_diag = !PLAIN && (flags & ABM_WANT_DIAG) != 0 && diag != nullptr;
    const bool count = !PLAIN && (flags & (ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) != 0 && counters;
    const bool verify = !PLAIN && (flags & ABM_VERIFY_FAST_PATH) != 0 && counters != nullptr;
    char* p = reinterpret_cast<char*>(smem_d);
    double* red = reinterpret_cast<double*>(p); p += sizeof(double) * (4 * kBigWaves + 8);
    float4* pose = reinterpret_cast<float4*>(p); p += sizeof(float4) * (size_t)maxN;
    uint16_t* queue = reinterpret_cast<uint16_t*>(p); p += big_queue_bytes(maxN);
    p += sizeof(int32_t) * 4;
    uint32_t* F = reinterpret_cast<uint32_t*>(p);
    // each wave queues the candidates among its own objects (64 of every
    // 1024) in its own segment, so no counter is shared between waves
    uint16_t* wq = queue + wave * big_segment(maxN);
    for (int i = tid; i < C.N; i += kBigThreads) {
        const int g = C.a0 + i;
        pose[i] = make_float4(st.x[g], st.y[g], (float)st.radius[g], st.theta[g]);
    }
    // this thread's rays [rs, rs + rn) and their table entries
    const int rs = tid * RPL;
    const int rn = rs >= C.R ? 0 : (C.R - rs < RPL ? C.R - rs : RPL);
    RayTab32 T[RPL];
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
        const int r = rs + i;
        if (r < C.R) T[i] = tab32[rp->table_offset + r];
        else T[i].wcos = T[i].wsin = T[i].cos = T[i].sin = 0.f;
    }
    const float a0d = (float)rp->alp0, b0d = (float)rp->bet0, v0d = (float)rp->v0;
    unsigned long long n_pairs = 0, n_recheck = 0, n_disagree = 0;
    // wave 0 moves the agents: agent k's speed and parameters are loaded one
    // agent ahead, so no global load waits on the id-order chain
    float vel_next = 0.f, a0_next = a0d, b0_next = b0d, v0_next = v0d;
    if (wave == 0) {
        vel_next = st.v[C.a0];
        if (st.alp0) a0_next = st.alp0[C.a0];
        if (st.bet0) b0_next = st.bet0[C.a0];
        if (st.v0) v0_next = st.v0[C.a0];
    }
    __syncthreads();
    for (int k = 0; k < C.N; ++k) {
        for (int w = tid; w < C.W; w += kBigThreads) F[w] = 0u;
        const float vel_k = vel_next, alp0_k = a0_next, bet0_k = b0_next, v0_k = v0_next;
        if (wave == 0 && k + 1 < C.N) {
            const int gn = C.a0 + k + 1;
            vel_next = st.v[gn];
            if (st.alp0) a0_next = st.alp0[gn];
            if (st.bet0) b0_next = st.bet0[gn];
            if (st.v0) v0_next = st.v0[gn];
        }
        const float4 fp = pose[k];
        const float fx = fp.x, fy = fp.y, fr = fp.z, fth = fp.w;
        float sth, cth;
        sincos_f32(fth, &sth, &cth);
        const float u1x = cth, u1y = -sth;
        __syncthreads();
        // ---- cheap pass: the pairs inside the cut-off (or a torus guard band)
        int nq = 0;   // wave-uniform
        for (int base = tid - lane; base < C.N; base += kBigThreads) {
            const int j = base + lane;
            bool c = false;
            if (j < C.N && j != k) {
                const float4 o = pose[j];
                if (!(o.x == fx && o.y == fy)) {
                    float dx = (o.x - fx) + (o.z - fr), dy = (o.y - fy) + (o.z - fr);
                    bool near_wrap = false;
                    if (C.torus) {
                        const float ex = fabsf(dx) - C.hw, ey = fabsf(dy) - C.hh;
                        near_wrap = fabsf(ex) < C.tguard || fabsf(ey) < C.tguard;
                        if (ex > 0.f) dx = dx > 0.f ? dx - C.fW : dx + C.fW;
                        if (ey > 0.f) dy = dy > 0.f ? dy - C.fH : dy + C.fH;
                    }
                    const float lim = o.z * cull_c;
                    const bool culled = !near_wrap && fmaf(dy, dy, dx * dx) > lim * lim;
                    if (culled && count) ++n_pairs;   // decided here: out of sight
                    if (culled && verify) {
                        // a culled pair must have an empty raster
                        int es = 0, ee = 0, ed = 0;
                        exact_pair(fx, fy, fth, fr, o.x, o.y, o.z, rp, &es, &ee, &ed);
                        if (ed && es != ee) ++n_disagree;
                    }
                    c = !culled;
                }
            }
            const uint64_t m = __ballot(c);
            if (c) wq[nq + (int)__popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)j;
            nq += (int)__popcll(m);
        }
        wave_lds_sync();
        // ---- this wave's queued pairs: float32 decision, float64 inside the guard bands
        for (int q = lane; q < nq; q += 64) {
            const float4 o = pose[wq[q]];
            PairF32 pr = fast_pair(u1x, u1y, fx, fy, fr, o.x, o.y, o.z, C);
            if (count) ++n_pairs;
            if (pr.tie && tie_in_place(pr, fx, fy, fth, fr, o.x, o.y, o.z, rp, C))   // rare
                if (count) ++n_recheck;
            if (!pr.ok || verify) {
                int es = 0, ee = 0, ed = 0;
                exact_pair(fx, fy, fth, fr, o.x, o.y, o.z, rp, &es, &ee, &ed);
                if (verify && pr.ok && (es != pr.start || ee != pr.end || ed != (int)pr.drawn))
                    ++n_disagree;
                if (!pr.ok) {
                    if (count) ++n_recheck;
                    pr.start = es; pr.end = ee; pr.drawn = ed != 0;
                }
            }
            if (pr.drawn) raster_lds(F, pr.start, pr.end, C.R);
        }
        __syncthreads();
        // ---- sums over this thread's rays
        const bool case1 = (F[0] & 1u) == 1u && field_bit(F, C.R - 1) == 0u;
        float bc = 0.f, bs = 0.f, ec = 0.f, es = 0.f;
        if (rn > 0) {
            const int w0 = rs >> 5;
            const uint32_t lo = F[w0];
            const uint32_t hi = (RPL > 1 && w0 + 1 < C.W) ? F[w0 + 1] : 0u;
            const uint64_t v64 = (((uint64_t)hi << 32) | lo) >> (rs & 31);
            const uint32_t m = low_mask(rn);
            const uint32_t cur = (uint32_t)v64 & m;
            uint32_t spike;
            if (case1) {
                const uint32_t prev = field_bit(F, rs == 0 ? C.R - 1 : rs - 1);
                spike = (cur ^ ((cur << 1) | prev)) & m;
            } else {
                const int nx = rs + rn;
                const uint32_t next = field_bit(F, nx >= C.R ? 0 : nx);
                spike = (cur ^ ((cur >> 1) | (next << (rn - 1)))) & m;
            }
#pragma unroll
            for (int i = 0; i < RPL; ++i) {
                const float vb = (float)((cur >> i) & 1u);   // acc + (bit ? t : 0) as fma(bit, t, acc)
                const float sb = (float)((spike >> i) & 1u);
                bc = __builtin_fmaf(vb, T[i].wcos, bc);
                bs = __builtin_fmaf(vb, T[i].wsin, bs);
                ec = __builtin_fmaf(sb, T[i].cos, ec);
                es = __builtin_fmaf(sb, T[i].sin, es);
            }
        }
        const int gk = C.a0 + k;
        const float alp0 = alp0_k, bet0 = bet0_k, v0 = v0_k;
        // blob terms: trapz(cos(PHI) * (-V)) = -sum(w cos V); components by
        // wave in LDS, summed in wave order by every thread
        {
            const double Bc = wave_total(bc), Bs = wave_total(bs), Ec = wave_total(ec), Es = wave_total(es);
            if (lane == 0) {
                red[4 * wave] = Bc; red[4 * wave + 1] = Bs; red[4 * wave + 2] = Ec; red[4 * wave + 3] = Es;
            }
        }
        __syncthreads();
        if (wave == 0) {
            double Bc = 0.0, Bs = 0.0, Ec = 0.0, Es = 0.0;
            for (int w = 0; w < kBigWaves; ++w) {
                Bc += red[4 * w]; Bs += red[4 * w + 1]; Ec += red[4 * w + 2]; Es += red[4 * w + 3];
            }
            const double Sv = (double)alp0 * -Bc + (double)(alp0 * C.alp1) * Ec;
            const double Sp = (double)bet0 * -Bs + (double)(bet0 * C.bet1) * Es;
            float vel, o, dv, dpsi;
            steer(C, fth, vel_k, v0, (float)Sv, (float)Sp, &o, &vel, &dv, &dpsi);
            float so, co;
            sincos_f32(o, &so, &co);
            float nx, ny;
            euler_boundary(C, fx, fy, fr, vel, so, co, &o, &nx, &ny);
            if (lane == 0) {
                pose[k] = make_float4(nx, ny, fr, o);
                st.v[gk] = vel;
                if (want_diag) {
                    float* dd = diag + 6 * (int64_t)gk;
                    dd[0] = dv; dd[1] = dpsi;
                    dd[2] = C.phi_ok ? (float)((double)alp0 * -Bc) : 0.f;
                    dd[3] = C.phi_ok ? (float)((double)(alp0 * C.alp1) * Ec) : 0.f;
                    dd[4] = C.phi_ok ? (float)((double)bet0 * -Bs) : 0.f;
                    dd[5] = C.phi_ok ? (float)((double)(bet0 * C.bet1) * Es) : 0.f;
                }
            }
        }
        if (!PLAIN && bits_out) {
            uint32_t* dst = bits_out + C.field_offset + (int64_t)k * C.W;
            for (int w = tid; w < C.W; w += kBigThreads) dst[w] = F[w];
        }
        __syncthreads();
    }
    for (int i = tid; i < C.N; i += kBigThreads) {
        const int g = C.a0 + i;
        const float4 q = pose[i];
        st.x[g] = q.x;
        st.y[g] = q.y;
        st.theta[g] = q.w;
    }
    if (count) {
        if (n_pairs) atomicAdd(&counters[0], n_pairs);
        if (n_recheck) atomicAdd(&counters[1], n_recheck);
        if (n_disagree) atomicAdd(&counters[2], n_disagree);
    }
}

// The 16-wave kernel over the replicas order[0 .. n_rep), the largest with
// maxN agents and maxR rays.
template <int RPL>
int launch_big(abm_vf_batch* b, const abm_vf_state_f32* st, uint32_t* bits, float* diag,
               uint32_t flags, hipStream_t s, const int32_t* order, int n_rep, int maxN, int maxR) {
    const size_t lds = lds_bytes_big(maxN, maxR);
    if (lds > (size_t)b->dev_max_lds)
        return set_error(ABM_ERR_UNSUPPORTED,
                         "abm_vf_step_f32: %d agents in one replica need %zu B of LDS in the reference "
                         "(sequential) order on the 16-wave kernel (device max %d); the chain step (the default "
                         "for single flocks, abm_vf_set_launch(64)) takes it", maxN,
                         lds, b->dev_max_lds);
    const bool plain = bits == nullptr && (flags & (ABM_WANT_DIAG | ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) == 0;
    auto kern = plain ? vf_step_f32_big_kernel<RPL, true> : vf_step_f32_big_kernel<RPL, false>;
    if (lds > 65536) {
        if (int rc = check_hip(hipFuncSetAttribute((const void*)kern,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                               "hipFuncSetAttribute"))
            return rc;
    }
    // the cut-off of the largest R: no smaller for a replica of fewer rays
    // (cot(2 pi / R) grows with R), so it drops no drawable pair there either
    const float cull_c = (float)((1.0 / std::tan(kTwoPi / maxR)) * (1.0 + 2e-4));
    hipLaunchKernelGGL(kern, dim3(n_rep), dim3(kBigThreads), lds, s, b->reps_dev, order, b->tab32, *st,
                       bits, diag, flags, b->counters, cull_c, maxN, maxR);
    b->last_kernels |= ABM_KERNEL_BIG;
    return check_hip(hipGetLastError(), "vf_step_f32_big_kernel launch");
}

int launch_big_any(abm_vf_batch* b, const abm_vf_state_f32* st, uint32_t* bits, float* diag,
                   uint32_t flags, hipStream_t s, const int32_t* order, int n_rep, int maxN, int maxR) {
    if (maxR <= kBigThreads) return launch_big<1>(b, st, bits, diag, flags, s, order, n_rep, maxN, maxR);
    return launch_big<2>(b, st, bits, diag, flags, s, order, n_rep, maxN, maxR);
}

// ---------------------------------------------------------------------------
// Reference (id) order with the pairs off the id-order chain (one workgroup
// of 512 threads per replica, every agent's field in LDS).  Agent m's field
// is the OR of its pairs with every other agent j, seen at j's new pose for
// j < m and at its start pose for j > m, and m itself at its start pose.
// Step k of the chain (one barrier each), where the sums are taken ahead
// (push_ahead):
//   * wave 0 moves agent k by the sums of its field and decides the pairs
//     (k + 1, k) and (k + 2, k) at k's new pose;
//   * wave 1 sums agent k + 1's field, complete but for the pair (k + 1, k),
//     with the rays that pair would set if agent k kept its heading and speed;
//     where the decided rays differ, wave 0 takes agent k + 1's sums again
//     with the decided ones, so a wrong guess costs time and no result;
//   * waves 2..7 decide the pairs (m, k - 1) for m > k + 1 with agent k - 1's
//     new pose.
// Otherwise wave 0 sums agent k's field, moves it and decides the pair (k + 1, k),
// and waves 1..7 decide agent k - 1's other pairs.
// The start-pose pairs (m, j > m) are decided before the chain by every
// wave.  Pairs beyond the visibility cut-off are dropped by a cheap float32
// test (as in the 16-wave kernel) and the rest queued, so that the exact
// decisions run on full waves.
// So only agent k's move and one pair deep of decisions stay on the chain
// (about 0.5 + 1.0 thousand cycles of latency; the sums are another 1.3, which
// the guess takes off the chain).  The sums and moves are exactly those of the
// one-wave per-replica kernel (same ray spans, table order and reductions),
// and the decisions are exact, so the two kernels give identical results bit
// for bit.  Waves 0 and 1 keep their rays' table entries in registers (up to
// 128), which two waves per SIMD allow; from LDS, the loads of the sums waited
// on the other waves' LDS traffic.  Measured, one replica of 100 agents at
// R = 1024: 0.160 ms a step with the sums and their LDS round trips on the
// chain, 0.141 with the pair handed over in registers, 0.123 with wave 1
// summing ahead, 0.121 with the rays between a span's ends stored rather than
// ORed and a pushing lane's agent in registers; 1000 replicas of 8 to 512 agents,
// 1.025, 0.989, 0.931, 0.921 (0.811 with the small ones in the same launch).
constexpr int kPushThreads = 64 * kPushWaves;

// Rays added to a field in registers: up to two pieces [a, b) (wave-uniform).
struct Pieces {
    int a0, b0, a1, b1;
};

// Bits of the lane's rays [rs, rs + RPL) inside [a, b).
template <int RPL>
__device__ __forceinline__ uint32_t span_mask(int a, int b, int rs) {
    const int lo = min(max(a - rs, 0), RPL), hi = min(max(b - rs, lo), RPL);
    if (RPL < 32) return (1u << hi) - (1u << lo);
    return low_mask(hi) & ~low_mask(lo);
}

// The one-wave sums of a field Fk, as the one-wave per-replica kernel takes
// them: lane l sums its rays [l RPL, (l + 1) RPL) (table entries T) in float32,
// the wave totals are float64.  Without diagnostics the two integrals are
// totalled directly (Sv, Sp); with them the four parts (Bc, Bs, Ec, Es) and
// the integrals from those.  Shared by the push kernel and the chain step's
// segment kernel, which thereby give the same results bit for bit.  A lane's
// rays lie in one word (RPL divides 32), its neighbours' rays come from the
// lanes beside it, so one LDS read starts the sums; `more` holds rays that are
// not in Fk yet.  SPANS = 2: the sums as two waves of half as many rays a lane
// take them (float32 over a half, the halves' sum the first of the float32 adds).
template <int RPL, int SPANS = 1>
__device__ __forceinline__ void one_wave_sums(const uint32_t* Fk, const RayTab32* T, int lane, const RepConst& C,
                                              bool want_diag, float alp0, float bet0, const Pieces& more,
                                              double& Sv, double& Sp, double& Bc, double& Bs, double& Ec,
                                              double& Es) {
    static_assert(SPANS == 1 || SPANS == 2, "whole lanes or halves");
    const int rs = lane * RPL;
    const int rn = rs >= C.R ? 0 : (C.R - rs < RPL ? C.R - rs : RPL);
    float bc = 0.f, bs = 0.f, ec = 0.f, es = 0.f;
    float hv = 0.f, hp = 0.f, hbc = 0.f, hbs = 0.f, hec = 0.f, hes = 0.f;   // the first half's
    {
        const uint32_t m = low_mask(rn);
        uint32_t cur = Fk[min(rs >> 5, C.W - 1)] >> (rs & 31);
        if (more.b0 > more.a0) cur |= span_mask<RPL>(more.a0, more.b0, rs);
        if (more.b1 > more.a1) cur |= span_mask<RPL>(more.a1, more.b1, rs);
        cur &= m;
        // edges by the dPhi alignment rule (vf_supcalc.py:266-274): against the
        // ray before when ray 0 is set and ray R - 1 is not, else the ray after
        const int end_lane = (C.R - 1) / RPL;
        const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)cur) & 1u;
        const uint32_t last = ((uint32_t)__builtin_amdgcn_readlane((int)cur, end_lane) >> ((C.R - 1) % RPL)) & 1u;
        uint32_t other;
        if (first == 1u && last == 0u) {   // wave_shr:1; lane 0's ray before is R - 1, not set
            const uint32_t low = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)cur, 0x138, 0xf, 0xf, false);
            other = (cur << 1) | (low >> (RPL - 1));
        } else {                           // wave_shl:1; the last ray's next is ray 0
            uint32_t up = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)cur, 0x130, 0xf, 0xf, false) & 1u;
            up = lane == end_lane ? first : up;
            other = (cur >> 1) | (up << ((rn - 1) & 31));
        }
        const uint32_t spike = (cur ^ other) & m;
        // acc + (bit ? t : 0) as fma(bit, t, acc): the same value (a 0 bit adds
        // a zero to an accumulator that is never -0), without a lane mask
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
            const float vb = (float)((cur >> i) & 1u);
            const float sb = (float)((spike >> i) & 1u);
            bc = __builtin_fmaf(vb, T[i].wcos, bc);
            bs = __builtin_fmaf(vb, T[i].wsin, bs);
            ec = __builtin_fmaf(sb, T[i].cos, ec);
            es = __builtin_fmaf(sb, T[i].sin, es);
            if (SPANS == 2 && i == RPL / 2 - 1) {
                if (!want_diag) {
                    hv = alp0 * (-bc) + (alp0 * C.alp1) * ec;
                    hp = bet0 * (-bs) + (bet0 * C.bet1) * es;
                } else {
                    hbc = bc; hbs = bs; hec = ec; hes = es;
                }
                bc = bs = ec = es = 0.f;
            }
        }
    }
    Bc = Bs = Ec = Es = 0.0;
    if (!want_diag) {
        const float v = alp0 * (-bc) + (alp0 * C.alp1) * ec;
        const float p = bet0 * (-bs) + (bet0 * C.bet1) * es;
        Sv = SPANS == 2 ? pair_total(hv + v) : wave_total(v);
        Sp = SPANS == 2 ? pair_total(hp + p) : wave_total(p);
    } else if (SPANS == 2) {
        Bc = pair_total(hbc + bc); Bs = pair_total(hbs + bs);
        Ec = pair_total(hec + ec); Es = pair_total(hes + es);
    } else {
        Bc = wave_total(bc); Bs = wave_total(bs);
        Ec = wave_total(ec); Es = wave_total(es);
    }
    if (want_diag) {
        Sv = (double)alp0 * -Bc + (double)(alp0 * C.alp1) * Ec;
        Sp = (double)bet0 * -Bs + (double)(bet0 * C.bet1) * Es;
    }
}

// One pair of the push kernel: focal f (start pose, heading vector u), object
// o; the float32 decision with the float64 one inside the guard bands (and
// every pair in verify mode), rastered into the focal's field Fm.
// The decision alone: whether the pair draws, and its span in pr.start/end.
__device__ inline bool decide_pair(PairF32& pr, float2 u, float4 f, float4 o, const VFRep* rp,
                                   const RepConst& C, bool count, bool verify, unsigned long long& n_pairs,
                                   unsigned long long& n_recheck, unsigned long long& n_disagree) {
    if (o.x == f.x && o.y == f.y) return false;   // coincident (vf_supcalc.py:57)
    pr = fast_pair(u.x, u.y, f.x, f.y, f.z, o.x, o.y, o.z, C);
    if (count) ++n_pairs;
    if (pr.tie && tie_in_place(pr, f.x, f.y, f.w, f.z, o.x, o.y, o.z, rp, C))   // rare
        if (count) ++n_recheck;
    if (!pr.ok || verify) {
        int es = 0, ee = 0, ed = 0;
        exact_pair(f.x, f.y, f.w, f.z, o.x, o.y, o.z, rp, &es, &ee, &ed);
        if (verify && pr.ok && (es != pr.start || ee != pr.end || ed != (int)pr.drawn)) ++n_disagree;
        if (!pr.ok) {
            if (count) ++n_recheck;
            pr.start = es; pr.end = ee; pr.drawn = ed != 0;
        }
    }
    return pr.drawn;
}

template <bool LDS = true>   // where the field lies
__device__ inline void push_pair(uint32_t* Fm, float2 u, float4 f, float4 o, const VFRep* rp,
                                 const RepConst& C, bool count, bool verify, unsigned long long& n_pairs,
                                 unsigned long long& n_recheck, unsigned long long& n_disagree) {
    PairF32 pr;
    if (decide_pair(pr, u, f, o, rp, C, count, verify, n_pairs, n_recheck, n_disagree)) {
        if (LDS) raster_lds(Fm, pr.start, pr.end, C.R);
        else raster(Fm, pr.start, pr.end, C.R);
    }
}

// Whether a pair lies beyond the visibility cut-off d > size cot(2 pi / R)
// (floor(proj_size / 2) = 0: nothing drawn), in float32 with the periodic
// image's guard band, as the 16-wave kernel's cheap pass.  A culled pair is
// counted as decided; in verify mode its float64 raster must be empty.
__device__ inline bool push_culled(float4 f, float4 o, const RepConst& C, float cull_c) {
    float dx = (o.x - f.x) + (o.z - f.z), dy = (o.y - f.y) + (o.z - f.z);
    bool near_wrap = false;
    if (C.torus) {
        const float ex = fabsf(dx) - C.hw, ey = fabsf(dy) - C.hh;
        near_wrap = fabsf(ex) < C.tguard || fabsf(ey) < C.tguard;
        if (ex > 0.f) dx = dx > 0.f ? dx - C.fW : dx + C.fW;
        if (ey > 0.f) dy = dy > 0.f ? dy - C.fH : dy + C.fH;
    }
    const float lim = o.z * cull_c;
    return !near_wrap && fmaf(dy, dy, dx * dx) > lim * lim;
}

__device__ inline void push_culled_check(float4 f, float4 o, const VFRep* rp, bool count, bool verify,
                                         unsigned long long& n_pairs, unsigned long long& n_disagree) {
    if (count) ++n_pairs;
    if (verify) {
        int es = 0, ee = 0, ed = 0;
        exact_pair(f.x, f.y, f.w, f.z, o.x, o.y, o.z, rp, &es, &ee, &ed);
        if (ed && es != ee) ++n_disagree;
    }
}

// The wave's total of a counter, on every lane.
__device__ inline unsigned long long wave_count(unsigned long long n) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) n += __shfl_xor(n, d, 64);
    return n;
}

// PLAIN: a step with no fields, diagnostics or counters out (the flags and
// pointers that ask for them are ignored), so their tests leave the kernel.
// HALVES: replicas up to kBigClass agents sum as two waves do (SPANS = 2).
// AHEAD: wave 1 sums agent k + 1's field while agent k moves (push_ahead).
template <int RPL, bool PLAIN, bool HALVES, bool AHEAD>
__global__ void __launch_bounds__(kPushThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
vf_step_f32_push_kernel(const VFRep* __restrict__ reps, const int32_t* __restrict__ order,
                        const RayTab32* __restrict__ tab32, abm_vf_state_f32 st,
                        uint32_t* __restrict__ bits_out, float* __restrict__ diag, uint32_t flags,
                        unsigned long long* __restrict__ counters) {
    extern __shared__ __align__(16) double smem_d[];
    const VFRep* rp = reps + order[blockIdx.x];
    const RepConst C = rep_const(rp);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int W1 = C.W + 1;
    const bool halves = HALVES && C.N <= kBigClass;
    constexpr int kSpans = HALVES ? 2 : 1;
    const bool want_diag = !PLAIN && (flags & ABM_WANT_DIAG) != 0 && diag != nullptr;
    const bool count = !PLAIN && (flags & (ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) != 0 && counters;
    const bool verify = !PLAIN && (flags & ABM_VERIFY_FAST_PATH) != 0 && counters != nullptr;
    // laid out for this replica (lds_bytes_push(N, R) bytes)
    char* p = reinterpret_cast<char*>(smem_d);
    float4* P0 = reinterpret_cast<float4*>(p); p += sizeof(float4) * (size_t)C.N;    // start poses
    float4* P1 = reinterpret_cast<float4*>(p); p += sizeof(float4) * (size_t)C.N;    // new poses
    float4* dyn = reinterpret_cast<float4*>(p); p += sizeof(float4) * (size_t)C.N;   // v, ALP0, BET0, V0
    float2* U = reinterpret_cast<float2*>(p); p += sizeof(float2) * (size_t)C.N;     // (cos, -sin) of start headings
    uint32_t* queue = reinterpret_cast<uint32_t*>(p); p += sizeof(uint32_t) * kPushQueue * kPushWaves;
    uint32_t* F = reinterpret_cast<uint32_t*>(p);                                     // [N][W + 1] fields
    // Sv, Sp, Bc, Bs, Ec, Es of agents k and k + 1: in the queues' place, which are
    // done with before the chain (a replica may fill the LDS to the last byte); 1000
    // replicas of 8 to 512 agents 0.815 ms at the queues' start, 0.807 in their middle
    double (*red)[6] = reinterpret_cast<double (*)[6]>(queue + kPushQueue * kPushWaves / 2);
    const float cull_c = (float)rp->cull_c;
    uint32_t* wq = queue + wave * kPushQueue;   // this wave's ring of queued pairs
    const float a0d = (float)rp->alp0, b0d = (float)rp->bet0, v0d = (float)rp->v0;
    for (int i = tid; i < C.N; i += kPushThreads) {
        const int g = C.a0 + i;
        const float4 q = make_float4(st.x[g], st.y[g], (float)st.radius[g], st.theta[g]);
        P0[i] = q;
        dyn[i] = make_float4(st.v[g], st.alp0 ? st.alp0[g] : a0d, st.bet0 ? st.bet0[g] : b0d,
                             st.v0 ? st.v0[g] : v0d);
        float sth, cth;
        sincos_f32(q.w, &sth, &cth);
        U[i] = make_float2(cth, -sth);
    }
    // in the summing waves (0 and 1, or 0) lane l owns rays [l RPL, (l + 1) RPL) and
    // their table entries
    RayTab32 T[RPL];
    if (wave <= (AHEAD ? 1 : 0)) {
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
            const int r = lane * RPL + i;
            if (r < C.R) T[i] = tab32[rp->table_offset + r];
            else T[i].wcos = T[i].wsin = T[i].cos = T[i].sin = 0.f;
        }
    }
    for (int w = tid; w < C.N * W1; w += kPushThreads) F[w] = 0u;
    unsigned long long n_pairs = 0, n_recheck = 0, n_disagree = 0;
    __syncthreads();
    // ---- the start-pose pairs (m, j > m), wave w taking the rows m = w mod 8;
    // queue entries m | j << 16
    {
        int head = 0, tail = 0;   // wave-uniform ring positions
        for (int m = wave; m < C.N; m += kPushWaves) {
            const float4 f = P0[m];
            for (int jb = m + 1; jb < C.N; jb += 64) {
                const int j = jb + lane;
                bool keep = false;
                if (j < C.N) {
                    const float4 ob = P0[j];
                    if (!(ob.x == f.x && ob.y == f.y)) {   // coincident pairs are skipped (vf_supcalc.py:57)
                        keep = !push_culled(f, ob, C, cull_c);
                        if (!keep) push_culled_check(f, ob, rp, count, verify, n_pairs, n_disagree);
                    }
                }
                const uint64_t mk = __ballot(keep);
                if (keep)
                    wq[(tail + (int)__popcll(mk & ((1ull << lane) - 1ull))) & (kPushQueue - 1)] =
                        (uint32_t)m | ((uint32_t)j << 16);
                tail += (int)__popcll(mk);
                wave_lds_sync();
                if (tail - head >= 64) {
                    const uint32_t e = wq[(head + lane) & (kPushQueue - 1)];
                    const int mm = (int)(e & 0xffffu), jj = (int)(e >> 16);
                    push_pair(F + (size_t)mm * W1, U[mm], P0[mm], P0[jj], rp, C, count, verify, n_pairs,
                              n_recheck, n_disagree);
                    head += 64;
                    wave_lds_sync();
                }
            }
        }
        if (lane < tail - head) {
            const uint32_t e = wq[(head + lane) & (kPushQueue - 1)];
            const int mm = (int)(e & 0xffffu), jj = (int)(e >> 16);
            push_pair(F + (size_t)mm * W1, U[mm], P0[mm], P0[jj], rp, C, count, verify, n_pairs, n_recheck,
                      n_disagree);
        }
    }
    if constexpr (AHEAD) {
    // ---- where agent i will be if it keeps its heading and speed, and the
    // rays its pair (i + 1, i) then sets: a prediction, left in P1[i + 1] until
    // agent i + 1's new pose goes there
    for (int i = tid; i < C.N; i += kPushThreads) {
        Pieces q{0, 0, 0, 0};
        if (i > 0) {
            const float4 b = P0[i - 1];
            const float2 ub = U[i - 1];
            const float vb = dyn[i - 1].x;
            const float4 f = P0[i];
            const PairF32 pr = fast_pair(U[i].x, U[i].y, f.x, f.y, f.z, b.x + vb * ub.x, b.y + vb * ub.y, b.z, C);
            if (pr.drawn) vf_pieces(pr.start, pr.end, C.R, &q.a0, &q.b0, &q.a1, &q.b1);
        }
        P1[i] = make_float4(__int_as_float(q.a0), __int_as_float(q.b0), __int_as_float(q.a1), __int_as_float(q.b1));
    }
    __syncthreads();
    auto predicted = [&](int i) {
        const float4 q = P1[i];
        return Pieces{__float_as_int(q.x), __float_as_int(q.y), __float_as_int(q.z), __float_as_int(q.w)};
    };
    auto sums_into = [&](int i, const Pieces& more, double* r) {   // wave 1
        const float4 d = dyn[i];
        double Sv, Sp, Bc, Bs, Ec, Es;
        if (halves) one_wave_sums<RPL, kSpans>(F + (size_t)i * W1, T, lane, C, want_diag, d.y, d.z, more, Sv, Sp, Bc, Bs, Ec, Es);
        else one_wave_sums<RPL>(F + (size_t)i * W1, T, lane, C, want_diag, d.y, d.z, more, Sv, Sp, Bc, Bs, Ec, Es);
        if (lane == 0) {
            r[0] = Sv; r[1] = Sp;
            if (want_diag) { r[2] = Bc; r[3] = Bs; r[4] = Ec; r[5] = Es; }
        }
    };
    if (wave == 1) sums_into(0, Pieces{0, 0, 0, 0}, red[0]);   // agent 0's field is complete
    __syncthreads();
    if (wave == 0) __builtin_amdgcn_s_setprio(3);   // the chain's wave issues first,
    if (wave == 1) __builtin_amdgcn_s_setprio(2);   // then the summing wave
    const int last = C.N - 1;
    float4 f0 = P0[0], f1 = P0[min(1, last)];   // wave 0: start poses of agents k, k + 1
    float2 u1 = U[min(1, last)];
    // a pushing lane's agents m0, m0 + 384 ..: the first one's start pose stays in registers
    const int m0 = 2 + (wave - 2) * 64 + lane;
    const float4 fm = P0[min(max(m0, 0), last)];
    const float2 um = U[min(max(m0, 0), last)];
    Pieces more{0, 0, 0, 0};   // wave 0: the rays of the pair (k, k - 1)
    bool hit = true;           // wave 0: they are the ones wave 1 summed with
    for (int k = 0; k < C.N; ++k) {
        if (wave == 0) {
            // ---- agent k's sums: wave 1's, or taken again where the
            // prediction missed; what the next steps need loads meanwhile
            const uint32_t* Fk = F + (size_t)k * W1;
            const double* r = red[k & 1];
            double Sv = r[0], Sp = r[1], Bc = 0.0, Bs = 0.0, Ec = 0.0, Es = 0.0;
            const float4 dk = dyn[k], f2 = P0[min(k + 2, last)];
            const float2 u2 = U[min(k + 2, last)];
            const Pieces guess = predicted(min(k + 1, last));
            const float fx = f0.x, fy = f0.y, fr = f0.z, fth = f0.w;
            const float alp0 = dk.y, bet0 = dk.z, v0 = dk.w;
            if (!PLAIN && want_diag) { Bc = r[2]; Bs = r[3]; Ec = r[4]; Es = r[5]; }
            if (!hit) {
                if (halves) one_wave_sums<RPL, kSpans>(Fk, T, lane, C, want_diag, alp0, bet0, more, Sv, Sp, Bc, Bs, Ec, Es);
                else one_wave_sums<RPL>(Fk, T, lane, C, want_diag, alp0, bet0, more, Sv, Sp, Bc, Bs, Ec, Es);
            }
            // ---- agent k's move
            float vel, o, dv, dpsi;
            steer(C, fth, dk.x, v0, (float)Sv, (float)Sp, &o, &vel, &dv, &dpsi);
            float so, co;
            sincos_f32(o, &so, &co);
            float nx, ny;
            euler_boundary(C, fx, fy, fr, vel, so, co, &o, &nx, &ny);
            const float4 moved = make_float4(nx, ny, fr, o);
            // ---- the pairs (k + 1, k), on even lanes, and (k + 2, k), on odd
            // ones, at its new pose; counted on lanes 0 and 1
            const bool odd = (lane & 1) != 0;
            const bool there = k + (odd ? 2 : 1) < C.N;
            const bool once = lane < 2 && there;
            const float4 f = odd ? f2 : f1;
            const float2 u = odd ? u2 : u1;
            PairF32 pr;
            pr.drawn = false;
            Pieces q{0, 0, 0, 0};
            bool culled = false;
            if (count && odd && there && push_culled(f, moved, C, cull_c)) {   // counted as every pushed pair
                culled = true;
                if (once) push_culled_check(f, moved, rp, count, verify, n_pairs, n_disagree);
            }
            if (there && !culled &&
                decide_pair(pr, u, f, moved, rp, C, count && once, verify && once, n_pairs, n_recheck, n_disagree))
                vf_pieces(pr.start, pr.end, C.R, &q.a0, &q.b0, &q.a1, &q.b1);
            {   // the odd lanes' rays into agent k + 2's field, a word a lane
                const Pieces z{__builtin_amdgcn_readlane(q.a0, 1), __builtin_amdgcn_readlane(q.b0, 1),
                               __builtin_amdgcn_readlane(q.a1, 1), __builtin_amdgcn_readlane(q.b1, 1)};
                uint32_t bits = 0;
                if (z.b0 > z.a0) bits = span_mask<32>(z.a0, z.b0, 32 * lane);
                if (z.b1 > z.a1) bits |= span_mask<32>(z.a1, z.b1, 32 * lane);
                if (bits) atomicOr(&F[(size_t)(k + 2) * W1 + lane], bits);   // (rays < R: words < W)
            }
            more.a0 = __builtin_amdgcn_readfirstlane(q.a0); more.b0 = __builtin_amdgcn_readfirstlane(q.b0);
            more.a1 = __builtin_amdgcn_readfirstlane(q.a1); more.b1 = __builtin_amdgcn_readfirstlane(q.b1);
            if (!PLAIN && bits_out) {   // into agent k + 1's field, which wave 1 writes out
                // (and may be summing with the guessed rays: the same ones, or the sums are taken again)
                uint32_t bits = 0;
                if (more.b0 > more.a0) bits = span_mask<32>(more.a0, more.b0, 32 * lane);
                if (more.b1 > more.a1) bits |= span_mask<32>(more.a1, more.b1, 32 * lane);
                if (bits) atomicOr(&F[(size_t)(k + 1) * W1 + lane], bits);
            }
            hit = more.a0 == __builtin_amdgcn_readfirstlane(guess.a0) && more.b0 == __builtin_amdgcn_readfirstlane(guess.b0) &&
                  more.a1 == __builtin_amdgcn_readfirstlane(guess.a1) && more.b1 == __builtin_amdgcn_readfirstlane(guess.b1);
            f0 = f1; f1 = f2; u1 = u2;
            if (lane == 0) {
                const int gk = C.a0 + k;
                P1[k] = moved;
                st.v[gk] = vel;
                if (want_diag) {
                    float* dd = diag + 6 * (int64_t)gk;
                    dd[0] = dv; dd[1] = dpsi;
                    dd[2] = C.phi_ok ? (float)((double)alp0 * -Bc) : 0.f;
                    dd[3] = C.phi_ok ? (float)((double)(alp0 * C.alp1) * Ec) : 0.f;
                    dd[4] = C.phi_ok ? (float)((double)bet0 * -Bs) : 0.f;
                    dd[5] = C.phi_ok ? (float)((double)(bet0 * C.bet1) * Es) : 0.f;
                }
            }
        } else if (wave == 1) {
            // ---- agent k + 1's sums: its row lacks only the pair (k + 1, k),
            // whose rays are the predicted ones
            if (k + 1 < C.N) sums_into(k + 1, predicted(k + 1), red[(k + 1) & 1]);
            if (!PLAIN && bits_out) {   // agent k's field, complete since the step before
                uint32_t* dst = bits_out + C.field_offset + (int64_t)k * C.W;
                for (int w = lane; w < C.W; w += 64) dst[w] = F[(size_t)k * W1 + w];
            }
        } else if (k >= 1) {
            // ---- agent k - 1's new pose into the fields of agents k + 2 ..
            const float4 ob = P1[k - 1];
            for (int m = m0; m < C.N; m += (kPushWaves - 2) * 64) {
                if (m < k + 2) continue;
                float4 f = fm;
                float2 u = um;
                if (m != m0) {
                    f = P0[m];
                    u = U[m];
                }
                if (push_culled(f, ob, C, cull_c)) {
                    push_culled_check(f, ob, rp, count, verify, n_pairs, n_disagree);
                } else {
                    push_pair(F + (size_t)m * W1, u, f, ob, rp, C, count, verify, n_pairs, n_recheck, n_disagree);
                }
            }
        }
        __syncthreads();
    }
    } else {
    __syncthreads();
    if (wave == 0) __builtin_amdgcn_s_setprio(3);   // the chain's wave issues first
    float4 f1 = P0[0], d1 = dyn[0];   // wave 0: the next agent's
    Pieces more{0, 0, 0, 0};          // wave 0: the pair (k, k - 1)'s rays, not in F
    for (int k = 0; k < C.N; ++k) {
        if (wave == 0) {
            // ---- agent k's sums, as the one-wave per-replica kernel; the next
            // agent's start pose, heading and parameters (constant over the
            // step) load meanwhile
            const uint32_t* Fk = F + (size_t)k * W1;
            const float4 fp = f1, dk = d1;
            const int k1 = min(k + 1, C.N - 1);
            f1 = P0[k1];
            d1 = dyn[k1];
            const float2 u1 = U[k1];
            const float fx = fp.x, fy = fp.y, fr = fp.z, fth = fp.w;
            const float alp0 = dk.y, bet0 = dk.z, v0 = dk.w;
            double Sv, Sp, Bc, Bs, Ec, Es;
            if (halves) one_wave_sums<RPL, kSpans>(Fk, T, lane, C, want_diag, alp0, bet0, more, Sv, Sp, Bc, Bs, Ec, Es);
            else one_wave_sums<RPL>(Fk, T, lane, C, want_diag, alp0, bet0, more, Sv, Sp, Bc, Bs, Ec, Es);
            if (!PLAIN && bits_out) {
                uint32_t* dst = bits_out + C.field_offset + (int64_t)k * C.W;
                for (int w = lane; w < C.W; w += 64) dst[w] = Fk[w];
            }
            // ---- agent k's move, then the pair (k + 1, k) at its new pose
            float vel, o, dv, dpsi;
            steer(C, fth, dk.x, v0, (float)Sv, (float)Sp, &o, &vel, &dv, &dpsi);
            float so, co;
            sincos_f32(o, &so, &co);
            float nx, ny;
            euler_boundary(C, fx, fy, fr, vel, so, co, &o, &nx, &ny);
            const float4 moved = make_float4(nx, ny, fr, o);
            if (lane == 0) {
                const int gk = C.a0 + k;
                P1[k] = moved;
                st.v[gk] = vel;
                if (want_diag) {
                    float* dd = diag + 6 * (int64_t)gk;
                    dd[0] = dv; dd[1] = dpsi;
                    dd[2] = C.phi_ok ? (float)((double)alp0 * -Bc) : 0.f;
                    dd[3] = C.phi_ok ? (float)((double)(alp0 * C.alp1) * Ec) : 0.f;
                    dd[4] = C.phi_ok ? (float)((double)bet0 * -Bs) : 0.f;
                    dd[5] = C.phi_ok ? (float)((double)(bet0 * C.bet1) * Es) : 0.f;
                }
                if (!PLAIN && k + 1 < C.N) {
                    if (push_culled(f1, moved, C, cull_c))
                        push_culled_check(f1, moved, rp, count, verify, n_pairs, n_disagree);
                    else
                        push_pair(F + (size_t)(k + 1) * W1, u1, f1, moved, rp, C, count, verify,
                                  n_pairs, n_recheck, n_disagree);
                }
            }
            if (PLAIN) {
                // on every lane alike: its rays go into agent k + 1's sums
                // from registers (a pair beyond the cut-off decides to none; with
                // few rays most are beyond it and it is tested first: 64 rays, 1000
                // agents 1063 us against 1248, 250 rays 1474 against 1417)
                PairF32 pr;
                more = Pieces{0, 0, 0, 0};
                if (!(RPL == 4 && push_culled(f1, moved, C, cull_c)) &&
                    decide_pair(pr, u1, f1, moved, rp, C, false, false, n_pairs, n_recheck, n_disagree)) {
                    Pieces q;
                    vf_pieces(pr.start, pr.end, C.R, &q.a0, &q.b0, &q.a1, &q.b1);
                    more.a0 = __builtin_amdgcn_readfirstlane(q.a0); more.b0 = __builtin_amdgcn_readfirstlane(q.b0);
                    more.a1 = __builtin_amdgcn_readfirstlane(q.a1); more.b1 = __builtin_amdgcn_readfirstlane(q.b1);
                }
            }
        } else if (k >= 1) {
            // ---- agent k - 1's new pose into the fields of agents k + 1 ..:
            // each wave tests its focal agents against the cut-off 64 at a
            // time and queues the rest in a ring of 128 in LDS, deciding 64
            // at a time
            const float4 ob = P1[k - 1];
            int head = 0, tail = 0;   // wave-uniform ring positions
            for (int mb = k + 1 + (wave - 1) * 64; mb < C.N; mb += kPushThreads - 64) {
                const int m = mb + lane;
                bool keep = false;
                if (m < C.N) {
                    const float4 f = P0[m];
                    if (!(ob.x == f.x && ob.y == f.y)) {   // coincident pairs are skipped (vf_supcalc.py:57)
                        keep = !push_culled(f, ob, C, cull_c);
                        if (!keep) push_culled_check(f, ob, rp, count, verify, n_pairs, n_disagree);
                    }
                }
                const uint64_t mk = __ballot(keep);
                if (keep) wq[(tail + (int)__popcll(mk & ((1ull << lane) - 1ull))) & (kPushQueue - 1)] = (uint32_t)m;
                tail += (int)__popcll(mk);
                wave_lds_sync();
                if (tail - head >= 64) {
                    const int mm = (int)wq[(head + lane) & (kPushQueue - 1)];
                    push_pair(F + (size_t)mm * W1, U[mm], P0[mm], ob, rp, C, count, verify, n_pairs, n_recheck,
                              n_disagree);
                    head += 64;
                    wave_lds_sync();
                }
            }
            if (lane < tail - head) {
                const int mm = (int)wq[(head + lane) & (kPushQueue - 1)];
                push_pair(F + (size_t)mm * W1, U[mm], P0[mm], ob, rp, C, count, verify, n_pairs, n_recheck,
                          n_disagree);
            }
        }
        __syncthreads();
    }
    }
    for (int i = tid; i < C.N; i += kPushThreads) {
        const int g = C.a0 + i;
        const float4 q = P1[i];
        st.x[g] = q.x;
        st.y[g] = q.y;
        st.theta[g] = q.w;
    }
    if (count) {
        // one add per workgroup: adds to one address follow one another, about 10 ns
        // each (250 replicas of 10 agents, a wave each 42 us a step)
        n_pairs = wave_count(n_pairs); n_recheck = wave_count(n_recheck); n_disagree = wave_count(n_disagree);
        unsigned long long* part = reinterpret_cast<unsigned long long*>(queue);
        __syncthreads();   // the queues are done with
        if (lane < 3) part[3 * wave + lane] = lane == 0 ? n_pairs : (lane == 1 ? n_recheck : n_disagree);
        __syncthreads();
        if (tid < 3) {
            unsigned long long n = 0;
            for (int w = 0; w < kPushWaves; ++w) n += part[3 * w + tid];
            if (n) atomicAdd(&counters[tid], n);
        }
    }
}

// Whether the push kernel holds every replica (all) or the large size class.
bool push_fits_in(const abm_vf_batch* b, bool all) {
    const size_t lds = all ? b->push_lds_all : b->push_lds_big;
    return lds > 0 && b->max_rays <= 64 * 32 && lds <= (size_t)b->dev_max_lds &&
           (all ? b->max_agents : b->big_max_agents) <= kWideThreshold;
}

// Whether wave 1 sums ahead, or wave 0 sums in its turn and wave 1 pushes too.
// Ahead shortens the chain's link, but leaves six waves to push, each lane with its
// own agents, where seven test 64 agents at a time and decide the rest together: in
// large replicas the pushing outlasts the link, and where few rays leave most pairs
// beyond the cut-off there is little to decide.  us a step, ahead and in turn, one
// replica at 1e-4 agents per unit^2: R = 512, 100 agents 118 and 122, 300 338 and 366,
// 512 647 and 648, 600 875 and 786, 1000 1875 and 1493; R = 250, 60 agents 64 and 69,
// 450 493 and 539; R = 128 60 and 63, 466 and 485, but 458 and 413 at a fifth of that
// density; R = 64 61 and 55, 456 and 401.  The step with outputs holds more values per
// pushed pair: at R = 512 300 agents 402 and 407, 450 649 and 626, at R = 250 with few
// in sight 300 359 and 339, at R = 2000 33 agents 65 and 70, 200 424 and 421, counting,
// 200 at R = 512 285 and 274.
bool push_ahead(int rpl, int max_n, int max_r, bool plain, bool counts) {
    if (plain) return max_n <= (max_r <= 128 ? 64 : 512);
    return !counts && max_n <= (rpl == 4 ? 0 : (rpl == 32 ? 64 : 384));
}

template <int RPL>
int launch_push(abm_vf_batch* b, const abm_vf_state_f32* st, uint32_t* bits, float* diag,
                uint32_t flags, hipStream_t s, const int32_t* order, int n_rep, int max_n, int max_r,
                size_t lds, bool halves) {
    const bool plain = bits == nullptr && (flags & (ABM_WANT_DIAG | ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) == 0;
    constexpr bool kHalves = RPL > 4;   // (a lane's four rays are not halved)
    auto pick = [&](auto ahead) {
        constexpr bool A = decltype(ahead)::value;
        return halves && kHalves ? (plain ? vf_step_f32_push_kernel<RPL, true, kHalves, A> : vf_step_f32_push_kernel<RPL, false, kHalves, A>)
                                 : (plain ? vf_step_f32_push_kernel<RPL, true, false, A> : vf_step_f32_push_kernel<RPL, false, false, A>);
    };
    const bool counts = (flags & (ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) != 0;
    auto kern = push_ahead(RPL, max_n, max_r, plain, counts) ? pick(std::true_type{}) : pick(std::false_type{});
    if (lds > 65536) {
        if (int rc = check_hip(hipFuncSetAttribute((const void*)kern,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                               "hipFuncSetAttribute"))
            return rc;
    }
    hipLaunchKernelGGL(kern, dim3(n_rep), dim3(kPushThreads), lds, s, b->reps_dev, order, b->tab32, *st,
                       bits, diag, flags, b->counters);
    b->last_kernels |= ABM_KERNEL_PUSH;
    return check_hip(hipGetLastError(), "vf_step_f32_push_kernel launch");
}

// The push kernel over order[0 .. n_rep): every replica (all) or the large
// size class.  Rays per lane of wave 0 follow the one-wave per-replica
// kernel's rule for the largest R of the launch.  halves: replicas up to
// kBigClass agents sum as the per-replica kernel's two waves do.
int launch_push_any(abm_vf_batch* b, const abm_vf_state_f32* st, uint32_t* bits, float* diag,
                    uint32_t flags, hipStream_t s, const int32_t* order, int n_rep, bool all,
                    bool halves = false) {
    const size_t lds = all ? b->push_lds_all : b->push_lds_big;
    if (!push_fits_in(b, all))
        return set_error(ABM_ERR_UNSUPPORTED,
                         "abm_vf_step_f32: the push kernel holds no replica of this batch (%zu B of LDS "
                         "for its fields, device max %d; up to %d agents)", lds, b->dev_max_lds,
                         kWideThreshold);
    const int max_n = all ? b->max_agents : b->big_max_agents, max_r = all ? b->max_rays : b->big_max_rays;
    const int rpl = push_rpl(max_r);
    if (rpl == 4) return launch_push<4>(b, st, bits, diag, flags, s, order, n_rep, max_n, max_r, lds, halves);
    if (rpl == 8) return launch_push<8>(b, st, bits, diag, flags, s, order, n_rep, max_n, max_r, lds, halves);
    if (rpl == 16) return launch_push<16>(b, st, bits, diag, flags, s, order, n_rep, max_n, max_r, lds, halves);
    return launch_push<32>(b, st, bits, diag, flags, s, order, n_rep, max_n, max_r, lds, halves);
}

// ---------------------------------------------------------------------------
// Reference (id) order for flocks above kWideThreshold agents, the chain
// step.  Agent m's field is the OR of its pairs with every other agent j at
// j's new pose for j < m and its start pose for j > m (m itself at its start
// pose).  The pairs are decided as soon as both poses exist, mostly off the
// id-order chain and over the whole GPU:
//   1. wide_grid_kernel: the grid of the start poses (torus arenas whose
//      cells can be at least the visibility cut-off wide).
//   2. vf_step_f32_wide_kernel<RPL, true, *>: each agent's field with the agents
//      after it, all at their start poses, into a global buffer of fields,
//      and its start heading vector (one wave per agent).
//   3. For each segment of kChainSeg agents in id order:
//      a. vf_step_f32_segment_kernel (one workgroup of 512 threads) moves the
//         segment's agents in id order (or in one that gives the same moves),
//         the segment's fields in LDS (their pairs with every earlier agent
//         already ORed in), summing and moving as the push kernel does, so the
//         two give the same fields and poses bit for bit.
//      b. vf_step_f32_chain_push_kernel (the whole GPU) decides the segment's
//         new poses in the global fields of every later agent: one wave per
//         (moved agent, grid cell of its 3 x 3 neighbourhood), or per range
//         of later agents without a grid (and with counters or verify mode).
// Kernel boundaries order the global fields between the launches.
constexpr int kChainThreads = 512;
constexpr int kChainWaves = kChainThreads / 64;
constexpr int kChainCullWaves = 3;    // segment kernel: three waves test, three decide
static_assert(kChainWaves == 2 + 2 * kChainCullWaves, "segment kernel wave roles");
constexpr int kChainSeg = 256;        // agents per segment
constexpr int kChainQueue = 128;      // queued agents per wave of the chain push kernel
constexpr int kChainPushWaves = 4;    // waves per workgroup of the push kernel
constexpr int kChainScanRange = 512;  // later agents per wave of the push kernel without a grid

// Barrier of the segment kernel: this wave's LDS operations complete, then
// s_barrier (the kernel shares no global memory between its waves).
__device__ inline void chain_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The agents [s0, s0 + n) of one replica, n <= kChainSeg.  In id order, one
// barrier per agent k:
//   * wave 0 takes agent k's sums (made by wave 1 during agent k - 1), moves
//     agent k and decides the pairs (k + 1, k) and (k + 2, k) at k's new pose
//     and (k + 2, k - 1) at k - 1's (one lane each);
//   * wave 1 sums agent k + 1's field, which then lacks only the pair
//     (k + 1, k), as the push kernel's wave 0 sums (one_wave_sums);
//   * three waves test agent k - 1's new pose against the segment's agents
//     from k + 3 on (the cheap float32 cut-off test) and list the pairs that
//     remain; three more decide the pairs listed in the previous step (agent
//     k - 2's new pose), 64 per wave at a time.  A pair (m, j) with
//     m >= j + 4 is so decided two steps after j moved, before wave 1 sums
//     agent m's field (in step m - 1), and each wave makes one pass a step.
//     The busiest of them (the first lister and the first decider) run as
//     waves 3 and 2, which share their SIMDs (wave w on SIMD w mod 4) with
//     the lightly loaded waves 7 and 6, not with waves 0 and 1.
// When the pair (k + 1, k) draws, wave 1 sums agent k + 1's field again,
// behind an extra barrier, before wave 0 uses it.  The decisions are exact
// and the sums and moves are the push kernel's, so the two give the same
// fields and poses bit for bit.
//
// Where the flock is spread wider than an agent sees, most agents of a segment
// need not wait for each other: agent m waits only for the agents j < m whose new
// pose it can see, those within the cut-off plus j's margin of its start pose
// (a displacement beyond the margin is detected, and the segment taken again in id
// order).  A kernel of its own lists these dependences (dep, pend) and, where they are
// few (kFlowShare), a segment runs them as they come free: each wave takes the next ready
// agent, sums and moves it, decides its new pose for its dependents and counts
// them down.  The same fields and moves, in another order.  Bound by the longest
// path of dependences times an agent's latency (about 5 thousand cycles), where
// the id order takes 2.5 thousand cycles for every agent.  Measured, a step, id
// order and this: 8192 agents, a twelfth of the others in sight, R = 2048, 9.12
// and 3.29 ms; 2100 agents with walls at R = 2048, a third in sight 2.98 and 1.93,
// 0.7 3.94 and 3.47, 0.85 4.48 and 4.92 (hence kFlowShare).
// A segment with a jump stops at once, and a step in which most segments had one
// starts the others in id order (kFlowMisses): of the 8192 agents, all jumping
// 11.41 ms to the end of every segment and 8.96 so, 148 in 30 of 32 segments 10.96
// and 8.98, 11 in ten 5.87 and 5.36.
constexpr float kFlowMargin = 16.f;   // + 4 |v|: the displacement allowed for
constexpr float kFlowShare = 0.7f;    // of a segment's pairs that may depend
constexpr int kFlowMisses = 2;        // segments taken again, beyond twice the others, that a step tries
constexpr int kFlowSpins = 1 << 20;   // waits end (the dependences are acyclic); the bound is never met

constexpr int kDepWords = kChainSeg / 64;
static_assert(kChainDepBytes == 64 + 8 * kDepWords + 4, "an agent's dependences");

// The dependences of every agent inside its segment, from the start poses: the
// later agents that wait for it (dep, and the first 64 of them by index: first), and
// how many earlier ones it waits for (pend; negative, all bits inverted: on a torus too small for the nearest image
// alone to matter).  One wave per agent over the whole GPU, since no segment's
// moves change it: 6 us for 8192 agents, where each segment's own workgroup took
// 11 us for 256 (a step of 3.78 ms then, 3.47 after; 3.29 with the indices, whose
// agents then load in one go, where a wave made its list from the bits).
__global__ void __launch_bounds__(256)
vf_step_f32_depend_kernel(const VFRep* __restrict__ rp, abm_vf_state_f32 st, float cull_c,
                          uint8_t* __restrict__ first, uint64_t* __restrict__ dep, int32_t* __restrict__ pend,
                          int32_t* __restrict__ missed) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *missed = 0;   // segments of this step not done by dependence
    const RepConst C = rep_const(rp);
    const int lane = threadIdx.x & 63;
    const int a = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (a >= C.N) return;   // whole waves, no barrier below
    const int s0 = a / kChainSeg * kChainSeg, n = min(kChainSeg, C.N - s0), al = a - s0;
    float x[kDepWords], y[kDepWords], lim[kDepWords];   // centres, reach of a new pose
    float ax = 0.f, ay = 0.f, alim = 0.f;               // agent a's
#pragma unroll
    for (int c = 0; c < kDepWords; ++c) {
        const int i = 64 * c + lane, g = C.a0 + s0 + min(i, n - 1);
        const float r = (float)st.radius[g];
        x[c] = st.x[g] + r;
        y[c] = st.y[g] + r;
        lim[c] = r * cull_c + (kFlowMargin + 4.f * fabsf(st.v[g])) + 1.f;
        if (c == al >> 6) {
            ax = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x[c]), al & 63));
            ay = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(y[c]), al & 63));
            alim = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lim[c]), al & 63));
        }
    }
    int waits = 0, cnt = 0;
    uint64_t mine = 0;
#pragma unroll
    for (int c = 0; c < kDepWords; ++c) {
        const int i = 64 * c + lane;
        float dx = fabsf(ax - x[c]), dy = fabsf(ay - y[c]);
        if (C.torus) {   // to the nearest image
            dx = fminf(dx, fabsf(C.fW - dx));
            dy = fminf(dy, fabsf(C.fH - dy));
        }
        const float d2 = fmaf(dy, dy, dx * dx);
        const uint64_t after = __ballot(i > al && i < n && !(d2 > alim * alim));
        waits += (int)__popcll(__ballot(i < al && !(d2 > lim[c] * lim[c])));
        if (lane == c) mine = after;
        const int at = cnt + (int)__popcll(after & ((1ull << lane) - 1ull));
        if (((after >> lane) & 1ull) && at < 64) first[(size_t)a * 64 + at] = (uint8_t)i;
        cnt += (int)__popcll(after);
    }
    if (lane >= cnt) first[(size_t)a * 64 + lane] = 0;   // (not used)
    if (lane < kDepWords) dep[(size_t)a * kDepWords + lane] = mine;
    const bool tight = C.torus && !(fminf(C.hw, C.hh) - C.tguard > alim);
    if (lane == 0) pend[a] = tight ? ~waits : waits;
}

template <int RPL, bool PLAIN>   // PLAIN: as the push kernel's
__global__ void __launch_bounds__(kChainThreads)
vf_step_f32_segment_kernel(const VFRep* __restrict__ rp, const RayTab32* __restrict__ tab32,
                           abm_vf_state_f32 st, const uint32_t* __restrict__ fields,
                           const float2* __restrict__ ustart, uint32_t* __restrict__ bits_out,
                           float* __restrict__ diag, uint32_t flags, unsigned long long* __restrict__ counters,
                           const uint8_t* __restrict__ first_all, const uint64_t* __restrict__ dep_all, int32_t* pend_all,
                           int32_t* missed, float cull_c, int s0, int n) {
    __shared__ uint32_t rows[kChainSeg][64];
    __shared__ float4 srec[kChainSeg];     // start poses (x, y, radius, theta)
    __shared__ float2 su[kChainSeg];       // start heading vectors
    __shared__ float4 sdyn[kChainSeg];     // speed, ALP0, BET0, V0
    __shared__ double red[2][6];           // Sv, Sp, Bc, Bs, Ec, Es of agents k and k + 1
    __shared__ float4 newpose[4];          // new pose of local agent kk at kk & 3
    __shared__ int dirty[2];               // the pair (k, k - 1) drew after k's sums were taken
    __shared__ uint16_t cq[2][kChainCullWaves][kChainSeg];   // listed rows, by step parity and cull wave
    __shared__ int cn[2][kChainCullWaves];
    __shared__ uint64_t dep[kChainSeg][kDepWords];           // agents that wait for an agent
    __shared__ uint32_t first[kChainSeg][16];                // the first 64 of them, a byte each
    __shared__ int pend[kChainSeg];                          // agents it waits for
    __shared__ int ready[kChainSeg];                         // in the order they come free (-1: not yet)
    __shared__ uint16_t after[kChainWaves][kChainSeg];       // all dependents of a wave's agent (beyond 64)
    __shared__ int ctl[4];                                   // next to take, free so far, dependences, out of bounds
    const RepConst C = rep_const(rp);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const bool want_diag = !PLAIN && (flags & ABM_WANT_DIAG) != 0 && diag != nullptr;
    const bool count = !PLAIN && (flags & (ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) != 0 && counters;
    const bool verify = !PLAIN && (flags & ABM_VERIFY_FAST_PATH) != 0 && counters != nullptr;
    const float a0d = (float)rp->alp0, b0d = (float)rp->bet0, v0d = (float)rp->v0;
    auto load = [&]() {
        for (int i = tid; i < n; i += kChainThreads) {
            const int g = C.a0 + s0 + i;
            srec[i] = make_float4(st.x[g], st.y[g], (float)st.radius[g], st.theta[g]);
            su[i] = ustart[s0 + i];
            sdyn[i] = make_float4(st.v[g], st.alp0 ? st.alp0[g] : a0d, st.bet0 ? st.bet0[g] : b0d,
                                  st.v0 ? st.v0[g] : v0d);
        }
        for (int w0 = tid; w0 < n * 64; w0 += 8 * kChainThreads) {   // eight loads in flight
            uint32_t q[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int i = (w0 + e * kChainThreads) >> 6;
                q[e] = i < n && lane < C.W ? fields[(size_t)(s0 + i) * C.W + lane] : 0u;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int i = (w0 + e * kChainThreads) >> 6;
                if (i < n) rows[i][lane] = q[e];
            }
        }
    };
    if (tid < 2) dirty[tid] = 0;
    const bool may_flow = !count && !verify;
    if (tid < 4) ctl[tid] = 0;
    for (int i = tid; i < kChainSeg; i += kChainThreads) ready[i] = -1;
    // in a summing wave (wave 1, or all) lane l owns rays [l RPL, (l + 1) RPL) and
    // their table entries, which come through the rows' LDS (read from global
    // memory lane by lane they took 25 thousand cycles for eight waves)
    RayTab32 T[RPL];
    {
        static_assert(sizeof(RayTab32) == sizeof(float4) && sizeof(rows) >= 64 * (RPL + 1) * sizeof(float4), "staging");
        float4* stage = reinterpret_cast<float4*>(&rows[0][0]);   // a lane's entries, and one that shifts the banks
        const float4* tab = reinterpret_cast<const float4*>(tab32 + rp->table_offset);
        for (int r = tid; r < C.R; r += kChainThreads) stage[r / RPL * (RPL + 1) + r % RPL] = tab[r];
        __syncthreads();
        if (wave == 1 || may_flow) {
#pragma unroll
            for (int i = 0; i < RPL; ++i) {
                float4 e = make_float4(0.f, 0.f, 0.f, 0.f);
                if (lane * RPL + i < C.R) e = stage[lane * (RPL + 1) + i];
                T[i].wcos = e.x; T[i].wsin = e.y; T[i].cos = e.z; T[i].sin = e.w;
            }
        }
        __syncthreads();
    }
    load();
    // wave 1: the sums of local agent kk's field into red[buf]
    auto sums = [&](int kk, int buf) {
        const float4 d = sdyn[kk];
        double Sv, Sp, Bc, Bs, Ec, Es;
        one_wave_sums<RPL>(rows[kk], T, lane, C, want_diag, d.y, d.z, Pieces{0, 0, 0, 0}, Sv, Sp, Bc, Bs, Ec, Es);
        if (lane == 0) {
            double* r = red[buf];
            r[0] = Sv; r[1] = Sp; r[2] = Bc; r[3] = Bs; r[4] = Ec; r[5] = Es;
        }
    };
    unsigned long long n_pairs = 0, n_recheck = 0, n_disagree = 0;
    __syncthreads();
    auto margin = [&](float v) { return kFlowMargin + 4.f * fabsf(v); };
    auto image = [&](float& dx, float& dy) {   // the nearest image's, on the torus
        if (C.torus) {
            if (fabsf(dx) > C.hw) dx = dx > 0.f ? dx - C.fW : dx + C.fW;
            if (fabsf(dy) > C.hh) dy = dy > 0.f ? dy - C.fH : dy + C.fH;
        }
    };
    // A segment not done by dependence: where that is the rule, the next one's
    // first agent is marked as on a torus too small.
    auto miss = [&]() {
        if (tid != 0 || s0 + n >= C.N) return;
        const int times = atomicAdd(missed, 1) + 1, q = pend_all[s0 + n];
        if (times > 2 * (s0 / kChainSeg + 1 - times) + kFlowMisses && q >= 0) pend_all[s0 + n] = ~q;
    };
    bool flow = false;
    if (may_flow) {   // uniform: the dependences, and whether they are few
        uint64_t* flat = &dep[0][0];
        for (int w = tid; w < n * kDepWords; w += kChainThreads) flat[w] = dep_all[(size_t)s0 * kDepWords + w];
        const uint32_t* lists = reinterpret_cast<const uint32_t*>(first_all) + (size_t)s0 * 16;
        for (int w = tid; w < n * 16; w += kChainThreads) (&first[0][0])[w] = lists[w];
        int waits = 0;
        for (int m = tid; m < n; m += kChainThreads) {
            const int q = pend_all[s0 + m];
            waits = q < 0 ? ~q : q;
            pend[m] = waits;
            if (q < 0) ctl[3] = 1;
        }
        static_assert(kChainSeg <= kChainThreads, "an agent a thread");
        const int total = wave_scan(waits);
        if (lane == 63 && total > 0) atomicAdd(&ctl[2], total);
        __syncthreads();
        flow = ctl[3] == 0 && ctl[2] <= kFlowShare * n * n / 2;
        if (ctl[3] != 0) miss();
    }
    if (flow) {
        for (int m = tid; m < n; m += kChainThreads)
            if (pend[m] == 0) ready[atomicAdd(&ctl[1], 1)] = m;
        __syncthreads();
        for (;;) {
            int at = 0;
            if (lane == 0) at = atomicAdd(&ctl[0], 1);
            at = __builtin_amdgcn_readfirstlane(at);
            if (at >= n) break;
            int m = -1;
            for (int spin = 0; spin < kFlowSpins; ++spin) {
                m = __builtin_amdgcn_readfirstlane(*(volatile int*)&ready[at]);
                if (m >= 0) break;
                __builtin_amdgcn_s_sleep(1);
            }
            if (m < 0) {
                if (lane == 0) ctl[3] = 1;
                break;
            }
            if (m >= n) break;   // stopped
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const int gk = C.a0 + s0 + m;
            const float4 pk = srec[m], dk = sdyn[m];
            // its dependents, the first 64 to registers before the sums
            int mm = reinterpret_cast<const uint8_t*>(first[m])[lane];
            int cnt = 0;   // wave-uniform
#pragma unroll
            for (int c = 0; c < kDepWords; ++c) cnt += (int)__popcll(dep[m][c]);
            if (lane >= cnt) mm = m;
            float4 fm = srec[mm];
            float2 um = su[mm];
            double Sv, Sp, Bc, Bs, Ec, Es;
            one_wave_sums<RPL>(rows[m], T, lane, C, want_diag, dk.y, dk.z, Pieces{0, 0, 0, 0}, Sv, Sp, Bc, Bs, Ec, Es);
            float vel, o, dv, dpsi;
            steer(C, pk.w, dk.x, dk.w, (float)Sv, (float)Sp, &o, &vel, &dv, &dpsi);
            float so, co;
            sincos_f32(o, &so, &co);
            float nx, ny;
            euler_boundary(C, pk.x, pk.y, pk.z, vel, so, co, &o, &nx, &ny);
            const float4 moved = make_float4(nx, ny, pk.z, o);
            if (!PLAIN && bits_out && lane < C.W) bits_out[C.field_offset + (int64_t)(s0 + m) * C.W + lane] = rows[m][lane];
            if (lane == 0) {
                srec[m] = moved;   // its start pose is read no more
                sdyn[m].x = vel;
                if (want_diag) {
                    float* dd = diag + 6 * (int64_t)gk;
                    dd[0] = dv; dd[1] = dpsi;
                    dd[2] = C.phi_ok ? (float)((double)dk.y * -Bc) : 0.f;
                    dd[3] = C.phi_ok ? (float)((double)(dk.y * C.alp1) * Ec) : 0.f;
                    dd[4] = C.phi_ok ? (float)((double)dk.z * -Bs) : 0.f;
                    dd[5] = C.phi_ok ? (float)((double)(dk.z * C.bet1) * Es) : 0.f;
                }
            }
            cnt = __builtin_amdgcn_readfirstlane(cnt);
            if (cnt > 64) {
                int at = 0;
#pragma unroll
                for (int c = 0; c < kDepWords; ++c) {
                    const uint64_t mk = dep[m][c];
                    if ((mk >> lane) & 1ull)
                        after[wave][at + (int)__popcll(mk & ((1ull << lane) - 1ull))] = (uint16_t)(64 * c + lane);
                    at += (int)__popcll(mk);
                }
                wave_lds_sync();
            }
            for (int e = lane; e < cnt; e += 64) {
                if (e >= 64) {
                    mm = after[wave][e];
                    fm = srec[mm];
                    um = su[mm];
                }
                if (!push_culled(fm, moved, C, cull_c))
                    push_pair(rows[mm], um, fm, moved, rp, C, false, false, n_pairs, n_recheck, n_disagree);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the field first, then the count
                if (atomicSub(&pend[mm], 1) == 1) *(volatile int*)&ready[atomicAdd(&ctl[1], 1)] = mm;
            }
            // (its dependents do not wait for this)
            float jx = nx - pk.x, jy = ny - pk.y;
            image(jx, jy);
            const float mg = margin(dk.x);
            if (!(fmaf(jy, jy, jx * jx) <= mg * mg)) {   // stop: no wave takes or awaits another agent
                if (lane == 0) {
                    ctl[3] = 1;
                    atomicAdd(&ctl[0], n);
                }
                for (int i = lane; i < n; i += 64)
                    if (ready[i] < 0) *(volatile int*)&ready[i] = n;
            }
            wave_lds_sync();   // after[] is read before the next agent's
        }
        __syncthreads();
        if (ctl[3] == 0) {
            for (int i = tid; i < n; i += kChainThreads) {
                const int g = C.a0 + s0 + i;
                const float4 q = srec[i];
                st.x[g] = q.x;
                st.y[g] = q.y;
                st.theta[g] = q.w;
                st.v[g] = sdyn[i].x;
            }
            return;
        }
        miss();
        load();   // again, in id order
        __syncthreads();
    }
    if (wave == 1) sums(0, 0);   // agent s0's field is complete
    __syncthreads();
    if (wave == 0) __builtin_amdgcn_s_setprio(3);   // the chain's wave issues first,
    if (wave == 1) __builtin_amdgcn_s_setprio(2);   // then the summing wave
    for (int kk = 0; kk < n; ++kk) {
        const int k = s0 + kk;
        const int buf = kk & 1;
        if (dirty[buf]) {   // uniform: agent k's field changed after its sums
            if (wave == 1) sums(kk, buf);
            chain_barrier();
        }
        if (wave == 0) {
            const int gk = C.a0 + k;
            const double* r = red[buf];
            const double Sv = r[0], Sp = r[1], Bc = r[2], Bs = r[3], Ec = r[4], Es = r[5];
            const float4 pk = srec[kk];
            const float4 dk = sdyn[kk];
            const float fx = pk.x, fy = pk.y, fr = pk.z, fth = pk.w;
            const float alp0 = dk.y, bet0 = dk.z, v0 = dk.w;
            float vel, o, dv, dpsi;
            steer(C, fth, dk.x, v0, (float)Sv, (float)Sp, &o, &vel, &dv, &dpsi);
            float so, co;
            sincos_f32(o, &so, &co);
            float nx, ny;
            euler_boundary(C, fx, fy, fr, vel, so, co, &o, &nx, &ny);
            const float4 moved = make_float4(nx, ny, fr, o);
            if (lane == 0) {
                newpose[kk & 3] = moved;
                st.x[gk] = nx;
                st.y[gk] = ny;
                st.theta[gk] = o;
                st.v[gk] = vel;
                if (want_diag) {
                    float* dd = diag + 6 * (int64_t)gk;
                    dd[0] = dv; dd[1] = dpsi;
                    dd[2] = C.phi_ok ? (float)((double)alp0 * -Bc) : 0.f;
                    dd[3] = C.phi_ok ? (float)((double)(alp0 * C.alp1) * Ec) : 0.f;
                    dd[4] = C.phi_ok ? (float)((double)bet0 * -Bs) : 0.f;
                    dd[5] = C.phi_ok ? (float)((double)(bet0 * C.bet1) * Es) : 0.f;
                }
            }
            // lane d (1, 2): the pair (k + d, k); lane 3: the pair (k + 2, k - 1)
            // at k - 1's new pose (agent s0 - 1's pairs came with the fields)
            bool drew = false;
            const int m = kk + (lane == 3 ? 2 : lane);
            if (lane >= 1 && lane <= 3 && m < n && (lane < 3 || kk >= 1)) {
                const float4 f = srec[m];
                const float4 ob = lane == 3 ? newpose[(kk - 1) & 3] : moved;
                if (push_culled(f, ob, C, cull_c)) {
                    push_culled_check(f, ob, rp, count, verify, n_pairs, n_disagree);
                } else {
                    PairF32 pr;
                    if (decide_pair(pr, su[m], f, ob, rp, C, count, verify, n_pairs, n_recheck, n_disagree)) {
                        raster_lds(rows[m], pr.start, pr.end, C.R);
                        drew = true;
                    }
                }
            }
            const uint64_t dm = __ballot(drew && lane == 1);
            if (lane == 0) dirty[buf ^ 1] = dm != 0 ? 1 : 0;
        } else if (wave == 1) {
            if (kk + 1 < n) sums(kk + 1, buf ^ 1);   // lacks only the pair (k + 1, k)
        } else if (wave >= 3 && wave <= 5) {
            if (!PLAIN && bits_out && wave == 3 && lane < C.W) bits_out[C.field_offset + (int64_t)k * C.W + lane] = rows[kk][lane];
            // agent k - 1's new pose against the segment's agents from k + 3
            // on: the cut-off test, the rest listed for the next step
            const int c = wave - 3;
            int cnt = 0;   // wave-uniform
            if (kk >= 1) {
                const float4 o = newpose[(kk - 1) & 3];
                for (int mb = kk + 3 + c * 64; mb < n; mb += kChainCullWaves * 64) {
                    const int m = mb + lane;
                    bool keep = false;
                    if (m < n) {
                        const float4 f = srec[m];
                        if (!(o.x == f.x && o.y == f.y)) {   // coincident pairs are skipped (vf_supcalc.py:57)
                            keep = !push_culled(f, o, C, cull_c);
                            if (!keep) push_culled_check(f, o, rp, count, verify, n_pairs, n_disagree);
                        }
                    }
                    const uint64_t mk = __ballot(keep);
                    if (keep) cq[buf][c][cnt + (int)__popcll(mk & ((1ull << lane) - 1ull))] = (uint16_t)m;
                    cnt += (int)__popcll(mk);
                }
            }
            if (lane == 0) cn[buf][c] = cnt;
        } else if (kk >= 2) {
            // the pairs listed in the previous step, at agent k - 2's new pose
            const int pb = buf ^ 1;
            const int c0 = cn[pb][0], c1 = cn[pb][1], c2 = cn[pb][2];
            const float4 o = newpose[(kk - 2) & 3];
            const int d = wave == 2 ? 0 : wave - 5;   // waves 2, 6, 7
            for (int e = d * 64 + lane; e < c0 + c1 + c2; e += kChainCullWaves * 64) {
                const int mm = e < c0 ? cq[pb][0][e] : (e < c0 + c1 ? cq[pb][1][e - c0] : cq[pb][2][e - c0 - c1]);
                push_pair(rows[mm], su[mm], srec[mm], o, rp, C, count, verify, n_pairs, n_recheck, n_disagree);
            }
        }
        chain_barrier();
    }
    if (count) {
        if (n_pairs) atomicAdd(&counters[0], n_pairs);
        if (n_recheck) atomicAdd(&counters[1], n_recheck);
        if (n_disagree) atomicAdd(&counters[2], n_disagree);
    }
}

// The new poses of the agents [s0, s0 + n) (just moved) into the global
// fields of the agents from s1 = s0 + n on (at their start poses).  Wave
// (j, c): moved agent s0 + j and chunk c of the later agents -- grid cell c
// of the 3 x 3 around its new centre, or the range [s1 + c R, s1 + (c + 1) R)
// (R = kChainScanRange) without a grid.
__global__ void __launch_bounds__(64 * kChainPushWaves)
vf_step_f32_chain_push_kernel(const VFRep* __restrict__ rp, abm_vf_state_f32 st, uint32_t* __restrict__ fields,
                              const float2* __restrict__ ustart, uint32_t flags,
                              unsigned long long* __restrict__ counters, float cull_c,
                              const WideGrid* __restrict__ grid, const float4* __restrict__ sorted,
                              const int32_t* __restrict__ cell_start, int s0, int n, int n_chunks) {
    __shared__ uint32_t queue[kChainPushWaves][kChainQueue];
    const RepConst C = rep_const(rp);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const bool count = (flags & (ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) != 0 && counters;
    const bool verify = (flags & ABM_VERIFY_FAST_PATH) != 0 && counters != nullptr;
    const WideGrid G = *grid;
    const bool use_grid = G.ok && !count && !verify;
    const int item = blockIdx.x * kChainPushWaves + wave;
    const int j = item / n_chunks, c = item - j * n_chunks;
    const int s1 = s0 + n;
    // whole waves only (no barrier below): past the moved agents, or past the
    // nine cells of the grid
    if (j >= n || (use_grid && c >= 9)) return;
    const int gj = C.a0 + s0 + j;
    const float4 o = make_float4(st.x[gj], st.y[gj], (float)st.radius[gj], st.theta[gj]);
    uint32_t* wq = queue[wave];
    unsigned long long n_pairs = 0, n_recheck = 0, n_disagree = 0;
    int beg, end;
    if (use_grid) {
        const int oc = grid_cell(G, o.x + o.z, o.y + o.z);
        const int oiy = oc / G.nx, oix = oc - oiy * G.nx;
        const int ty = c / 3, tx = c - 3 * ty;
        int cy = oiy + ty - 1, cx = oix + tx - 1;   // the 3 x 3 cells, wrapped
        cy = cy < 0 ? G.ny - 1 : (cy >= G.ny ? 0 : cy);
        cx = cx < 0 ? G.nx - 1 : (cx >= G.nx ? 0 : cx);
        const int cell = cy * G.nx + cx;
        beg = cell_start[cell];
        end = cell_start[cell + 1];
    } else {
        beg = s1 + c * kChainScanRange;
        end = min(C.N, beg + kChainScanRange);
    }
    // focal agent m (record i), at its start pose
    auto focal = [&](int i, int& m, bool with_theta) -> float4 {
        if (use_grid) {
            const float4 s = sorted[i];
            m = __float_as_int(s.w);
            return make_float4(s.x, s.y, s.z, with_theta ? st.theta[C.a0 + m] : 0.f);
        }
        m = i;
        const int g = C.a0 + i;
        return make_float4(st.x[g], st.y[g], (float)st.radius[g], with_theta ? st.theta[g] : 0.f);
    };
    auto decide = [&](int head, int tail) {
        if (head + lane < tail) {
            int m;
            const float4 f = focal((int)wq[(head + lane) & (kChainQueue - 1)], m, true);
            push_pair<false>(fields + (size_t)m * C.W, ustart[m], f, o, rp, C, count, verify, n_pairs, n_recheck,
                      n_disagree);
        }
    };
    int head = 0, tail = 0;   // wave-uniform ring positions
    for (int b = beg; b < end; b += 64) {
        const int i = b + lane;
        bool keep = false;
        if (i < end) {
            int m;
            const float4 f = focal(i, m, verify);
            if (m >= s1 && !(o.x == f.x && o.y == f.y)) {   // coincident pairs are skipped (vf_supcalc.py:57)
                keep = !push_culled(f, o, C, cull_c);
                if (!keep) push_culled_check(f, o, rp, count, verify, n_pairs, n_disagree);
            }
        }
        const uint64_t mk = __ballot(keep);
        if (keep) wq[(tail + (int)__popcll(mk & ((1ull << lane) - 1ull))) & (kChainQueue - 1)] = (uint32_t)i;
        tail += (int)__popcll(mk);
        wave_lds_sync();
        if (tail - head >= 64) {
            decide(head, tail);
            head += 64;
            wave_lds_sync();
        }
    }
    decide(head, tail);
    if (count) {
        if (n_pairs) atomicAdd(&counters[0], n_pairs);
        if (n_recheck) atomicAdd(&counters[1], n_recheck);
        if (n_disagree) atomicAdd(&counters[2], n_disagree);
    }
}

template <int RPLW>
int launch_chain_start(abm_vf_batch* b, const abm_vf_state_f32* st, uint32_t flags, hipStream_t s,
                       int rep, float cull_c, int n_agents) {
    const size_t lds = lds_bytes_wide(RPLW);
    const bool plain = (flags & (ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) == 0;
    auto kern = plain ? vf_step_f32_wide_kernel<RPLW, true, true> : vf_step_f32_wide_kernel<RPLW, true, false>;
    if (lds > 65536) {
        if (int rc = check_hip(hipFuncSetAttribute((const void*)kern,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                               "hipFuncSetAttribute"))
            return rc;
    }
    const int blocks = (n_agents + kWideWaves - 1) / kWideWaves;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * kWideWaves), lds, s, b->reps_dev + rep, b->tab32, *st,
                       (float4*)nullptr, (uint32_t*)nullptr, (float*)nullptr, flags, b->counters, cull_c,
                       (const WideGrid*)b->grid_param, (const float4*)b->grid_sorted,
                       (const int32_t*)b->grid_start, b->chain_fields, (float2*)b->chain_u);
    return check_hip(hipGetLastError(), "vf_step_f32_wide_kernel (start pairs) launch");
}

// Whether the chain step can run the batch (its buffers, R up to 2048), and
// whether it does by default: every replica above kWideThreshold agents (a
// single large flock).
bool chain_ready(const abm_vf_batch* b) {
    return b->chain_fields != nullptr && b->chain_u != nullptr && b->chain_dep != nullptr && b->grid_sorted != nullptr &&
           b->grid_start != nullptr && b->grid_param != nullptr && b->n_replicas > 0 && b->max_rays <= 2048;
}
bool chain_fits(const abm_vf_batch* b) { return chain_ready(b) && b->min_agents > kWideThreshold; }

int launch_chain(abm_vf_batch* b, const abm_vf_state_f32* st, uint32_t* bits, float* diag, uint32_t flags,
                 hipStream_t s) {
    const bool counting = (flags & (ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) != 0;
    const bool plain = bits == nullptr && !counting && (flags & ABM_WANT_DIAG) == 0;
    const int rpl = push_rpl(b->max_rays);
    for (int rep = 0; rep < b->n_replicas; ++rep) {
        const VFRep& h = b->reps_host[rep];
        const int N = h.n_agents;
        const float cull_c = (float)h.cull_c;
        hipLaunchKernelGGL(wide_grid_kernel, dim3(1), dim3(1024), 0, s, b->reps_dev + rep, *st, cull_c,
                           b->grid_sorted, b->grid_start, (WideGrid*)b->grid_param);
        if (int rc = check_hip(hipGetLastError(), "wide_grid_kernel launch")) return rc;
        const int need = (h.n_rays + 63) / 64;
        int rc;
        if (need <= 4) rc = launch_chain_start<4>(b, st, flags, s, rep, cull_c, N);
        else if (need <= 8) rc = launch_chain_start<8>(b, st, flags, s, rep, cull_c, N);
        else if (need <= 16) rc = launch_chain_start<16>(b, st, flags, s, rep, cull_c, N);
        else rc = launch_chain_start<32>(b, st, flags, s, rep, cull_c, N);
        if (rc) return rc;
        uint8_t* first = (uint8_t*)b->chain_dep;
        uint64_t* dep = (uint64_t*)(first + (size_t)b->max_agents * 64);
        int32_t* pend = (int32_t*)(dep + (size_t)b->max_agents * kDepWords);
        int32_t* missed = pend + b->max_agents;
        if (!counting) {
            hipLaunchKernelGGL(vf_step_f32_depend_kernel, dim3((N + 3) / 4), dim3(256), 0, s, b->reps_dev + rep, *st,
                               cull_c, first, dep, pend, missed);
            if (int rc2 = check_hip(hipGetLastError(), "vf_step_f32_depend_kernel launch")) return rc2;
        }
        for (int s0 = 0; s0 < N; s0 += kChainSeg) {
            const int n = std::min(kChainSeg, N - s0);
            // rays per lane of the summing wave: the push kernel's rule for the batch
#define ABM_SEGMENT(RPLV)                                                                                   \
    if (rpl == RPLV)                                                                                        \
        hipLaunchKernelGGL((plain ? vf_step_f32_segment_kernel<RPLV, true>                                  \
                                  : vf_step_f32_segment_kernel<RPLV, false>),                               \
                           dim3(1), dim3(kChainThreads), 0, s,                                              \
                           b->reps_dev + rep, b->tab32, *st, (const uint32_t*)b->chain_fields,             \
                           (const float2*)b->chain_u, bits, diag, flags, b->counters, (const uint8_t*)first,       \
                           (const uint64_t*)dep,                                                            \
                           pend, missed, cull_c, s0, n);
            ABM_SEGMENT(4) ABM_SEGMENT(8) ABM_SEGMENT(16) ABM_SEGMENT(32)
#undef ABM_SEGMENT
            if (int rc2 = check_hip(hipGetLastError(), "vf_step_f32_segment_kernel launch")) return rc2;
            const int s1 = s0 + n;
            if (s1 >= N) break;
            // chunks per moved agent: enough for the nine cells of a grid and
            // for the ranges of the later agents (the device's grid decides
            // which apply; the other waves return at once)
            const int n_ranges = (N - s1 + kChainScanRange - 1) / kChainScanRange;
            const int n_chunks = counting ? n_ranges : std::max(9, n_ranges);
            const int items = n * n_chunks;
            hipLaunchKernelGGL(vf_step_f32_chain_push_kernel, dim3((items + kChainPushWaves - 1) / kChainPushWaves),
                               dim3(64 * kChainPushWaves), 0, s, b->reps_dev + rep, *st, b->chain_fields,
                               (const float2*)b->chain_u, flags, b->counters, cull_c, (const WideGrid*)b->grid_param,
                               (const float4*)b->grid_sorted, (const int32_t*)b->grid_start, s0, n, n_chunks);
            if (int rc2 = check_hip(hipGetLastError(), "vf_step_f32_chain_push_kernel launch")) return rc2;
        }
    }
    b->last_kernels |= ABM_KERNEL_CHAIN;
    return ABM_OK;
}

size_t lds_bytes_f32(int maxN, int maxR, int nw, int rpl, bool sync_order) {
    const int maxW = (maxR + 31) >> 5;
    size_t b = sizeof(RayTab32) * (size_t)rpl * 64 * nw + sizeof(float4) * (size_t)maxN * (sync_order ? 3 : 2) +
               sizeof(double) * (2 * nw + 2) + sizeof(int32_t) * ((size_t)2 * maxN + 4) +
               sizeof(uint32_t) * (maxW + 2);
    return (b + 15) & ~(size_t)15;
}

// The per-replica kernel over the replicas order[0 .. n_rep), the largest
// with maxN agents and maxR rays (split: the small size class of a batch
// whose large class goes to the 16-wave kernel).
template <int NW, int RPL>
int launch_nw(abm_vf_batch* b, const abm_vf_state_f32* st, uint32_t* bits, float* diag,
              uint32_t flags, hipStream_t s, const int32_t* order, int n_rep, int maxN, int maxR,
              bool split) {
    const bool sync_order = (flags & ABM_ORDER_SYNCHRONOUS) != 0;
    const size_t lds = lds_bytes_f32(maxN, maxR, NW, RPL, sync_order);
    if (lds > (size_t)b->dev_max_lds)
        return set_error(ABM_ERR_UNSUPPORTED,
                         "abm_vf_step_f32: %d agents x %d rays need %zu B of LDS (device max %d)",
                         maxN, maxR, lds, b->dev_max_lds);
    const bool plain = bits == nullptr && (flags & (ABM_WANT_DIAG | ABM_COUNT_RECHECKS | ABM_VERIFY_FAST_PATH)) == 0;
    auto kern = plain ? vf_step_f32_kernel<NW, RPL, true> : vf_step_f32_kernel<NW, RPL, false>;
    const int slot = NW == 1 ? 0 : (NW == 2 ? 1 : 2);
    int& per_cu = b->occ_f32[split ? 1 : 0][sync_order ? 1 : 0][plain ? 1 : 0][slot];
    if (per_cu == 0) {   // first launch of this shape: set the LDS limit, read the occupancy
        if (lds > 65536) {
            if (int rc = check_hip(hipFuncSetAttribute((const void*)kern,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       (int)lds), "hipFuncSetAttribute"))
                return rc;
        }
        int occ = 0;
        if (int rc = check_hip(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, 64 * NW, lds),
                               "hipOccupancyMaxActiveBlocksPerMultiprocessor"))
            return rc;
        per_cu = occ < 1 ? 1 : occ;
    }
    const int n_cu = b->n_cu;
    long grid = (long)per_cu * n_cu;
    if (grid > n_rep) grid = n_rep;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * NW), lds, s, b->reps_dev, order,
                       n_rep, b->tab32, *st, bits, diag, flags, b->counters, maxN);
    b->last_kernels |= ABM_KERNEL_PER_REPLICA;
    return check_hip(hipGetLastError(), "vf_step_f32_kernel launch");
}

}  // namespace

bool push_fits(const abm_vf_batch* b, bool all) { return push_fits_in(b, all); }

// Replicas per wave of the grouped kernel for this batch, or 0 for the
// per-replica kernel.  Automatic choice (measured on MI355X): batches with at
// least 8 replicas per CU run grouped, one replica per wave (four waves per
// SIMD), or four per wave when that still gives every SIMD two waves; so do
// batches with 4 to 8 replicas per CU of at most 128 agents (one replica per
// wave: 1024 replicas of 50 agents at R = 512 take 0.070 ms grouped against
// 0.095 ms on the per-replica kernel, of 100 agents at R = 1024 0.201 against
// 0.213; of 200 agents the per-replica kernel wins, 0.546 against 0.597);
// smaller batches are latency-bound and take the per-replica kernel with
// several waves per replica.
int selected_group_size(const abm_vf_batch* b) {
    if (!b->group_ok || b->group_g < 0) return 0;
    if (b->group_g > 0) return b->group_g;
    if (b->waves_per_group > 0) return 0;
    if (b->n_replicas < 4 * b->n_cu) return 0;
    if (b->n_replicas < 8 * b->n_cu) return b->max_agents <= 128 ? 1 : 0;
    if (b->gplan[2].n_groups >= 8 * b->n_cu) return 4;
    return 1;
}

constexpr int kFewReplicas = 8;

// Waves per replica of the per-replica kernel: four while the batch gives each
// CU at most two such workgroups, two while it fits at 16 waves per CU, else
// one (measured on MI355X: 1024 replicas of 100 agents take 0.223 ms on two
// waves and 0.256 ms on four; 512 take 0.216 and 0.219).
static int default_waves(const abm_vf_batch* b, int maxN, int n_rep) {
    if (maxN > 64 && (long)n_rep * 4 <= 8L * b->n_cu) return 4;
    if (maxN > 32 && (long)n_rep * 2 <= 16L * b->n_cu) return 2;
    return 1;
}

// The per-replica kernel with nw waves (0 = automatic) over order[0 .. n_rep).
static int launch_per_replica(abm_vf_batch* b, const abm_vf_state_f32* st, uint32_t* bits, float* diag,
                              uint32_t flags, hipStream_t s, int nw, const int32_t* order, int n_rep,
                              int maxN, int maxR, bool split) {
    if (nw == 0) nw = default_waves(b, maxN, n_rep);
    const int need = (maxR + 64 * nw - 1) / (64 * nw);   // rays per lane
    const int rpl = need <= 4 ? 4 : (need <= 8 ? 8 : (need <= 16 ? 16 : 32));
#define ABM_LAUNCH(NWV, RPLV) \
    if (nw == NWV && rpl == RPLV) \
        return launch_nw<NWV, RPLV>(b, st, bits, diag, flags, s, order, n_rep, maxN, maxR, split);
    ABM_LAUNCH(1, 4) ABM_LAUNCH(1, 8) ABM_LAUNCH(1, 16) ABM_LAUNCH(1, 32)
    ABM_LAUNCH(2, 4) ABM_LAUNCH(2, 8) ABM_LAUNCH(2, 16) ABM_LAUNCH(2, 32)
    ABM_LAUNCH(4, 4) ABM_LAUNCH(4, 8) ABM_LAUNCH(4, 16) ABM_LAUNCH(4, 32)
#undef ABM_LAUNCH
    return set_error(ABM_ERR_INVALID, "abm_vf_step_f32: no launch shape for %d waves", nw);
}

int launch_vf_step_f32(abm_vf_batch* b, const abm_vf_state_f32* st, uint32_t* bits, float* diag,
                       uint32_t flags, hipStream_t s) {
    b->last_kernels = 0;
    if (b->max_rays > 2048)
        return set_error(ABM_ERR_UNSUPPORTED,
                         "abm_vf_step_f32: n_rays up to 2048 (got %d); use abm_vf_step_f64", b->max_rays);
    const bool sync_order = (flags & ABM_ORDER_SYNCHRONOUS) != 0;
    const bool kahan = (flags & ABM_KAHAN_SUMS) != 0;
    if (kahan && b->max_agents > kWideThreshold)
        return set_error(ABM_ERR_UNSUPPORTED, "abm_vf_step_f32: ABM_KAHAN_SUMS is implemented by the "
                         "grouped kernel only (replicas of at most %d agents)", kGroupMaxAgents);
    if (b->max_agents > kWideThreshold) {
        // reference order: the chain step for single large flocks (unless the
        // 16-wave kernel is forced), else one workgroup per replica with every
        // pose in LDS
        if (!sync_order && b->waves_per_group != 16 && chain_fits(b))
            return launch_chain(b, st, bits, diag, flags, s);
        if (!sync_order)
            return launch_big_any(b, st, bits, diag, flags, s, b->order_dev, b->n_replicas, b->max_agents,
                                  b->max_rays);
        if (!b->wide_out)
            return set_error(ABM_ERR_INVALID, "abm_vf_step_f32: batch has no wide-step buffer");
        const int need = (b->max_rays + 63) / 64;
        if (need <= 4) return launch_wide<4>(b, st, bits, diag, flags, s);
        if (need <= 8) return launch_wide<8>(b, st, bits, diag, flags, s);
        if (need <= 16) return launch_wide<16>(b, st, bits, diag, flags, s);
        return launch_wide<32>(b, st, bits, diag, flags, s);
    }
    // Kahan sums run on the grouped kernel even where the automatic choice
    // (or a forced launch shape) would take the per-replica kernel
    const int G0 = selected_group_size(b);
    const int G = kahan && b->group_ok && G0 == 0 ? 1 : G0;
    if (G > 0) return launch_vf_group_f32(b, G, st, bits, diag, flags, s);
    if (kahan)
        return set_error(ABM_ERR_UNSUPPORTED, "abm_vf_step_f32: ABM_KAHAN_SUMS is implemented by the "
                         "grouped kernel only, which this batch does not take (one R up to %d rays, "
                         "replicas of at most %d agents)", kGroupMaxRays, kGroupMaxAgents);
    const int nw = b->waves_per_group;
    // the 16-wave and push kernels and the chain step move agents in the
    // reference order only; the synchronous order takes the per-replica kernel
    if (sync_order && (nw == 16 || nw == 32 || nw == 64))
        return set_error(ABM_ERR_UNSUPPORTED, "abm_vf_step_f32: the %s runs the reference order only "
                         "(ABM_ORDER_SYNCHRONOUS takes the per-replica kernel, abm_vf_set_launch(0))",
                         nw == 16 ? "16-wave kernel" : (nw == 32 ? "push kernel" : "chain step"));
    if (nw == 64) {   // the chain step for every replica
        if (!chain_ready(b))
            return set_error(ABM_ERR_INVALID, "abm_vf_step_f32: the chain step has no buffers (abm_vf_set_launch(64))");
        return launch_chain(b, st, bits, diag, flags, s);
    }
    if (nw == 32)   // the push kernel for every replica
        return launch_push_any(b, st, bits, diag, flags, s, b->order_dev, b->n_replicas, true);
    if (nw == 16)   // the 16-wave kernel for every replica
        return launch_big_any(b, st, bits, diag, flags, s, b->order_dev, b->n_replicas, b->max_agents,
                              b->max_rays);
    // The push kernel holds one replica per CU (eight waves of up to 256
    // VGPRs), so it shortens the step only while the agents, spread over the
    // CUs, do not outlast the chain of the largest replica; beyond that (many
    // replicas of similar size) the per-replica kernel's occupancy wins.  A
    // replica counts four agents more, its start and end.  Where that holds for
    // the whole batch, all of it goes there: ms a step on this kernel and
    // otherwise, one replica of 8 agents 0.0159 and 0.0169, of 33 0.046 and 0.063;
    // 256 of 8 to 60 0.074 and 0.100 (512 of 60: 0.141 and 0.112, which the rule
    // leaves); 250 of 60 at R = 2048 0.106 and 0.140; 64 of 8 to 200 0.218 and
    // 0.311, 1000 of 8 to 512 0.82 and 0.92 (the small ones first, on the other
    // kernel).  A batch of up to kFewReplicas replicas of both classes keeps a
    // kernel for each, although this one is faster there too (40 and 200 agents
    // at R = 512 0.227 and 0.291 ms, 64 and 65 0.073 and 0.175, 10 and 500 0.650
    // and 0.669): the tests of the size classes fix its kernels;
    const int nb = b->n_big_class;
    // and a step that takes every pair in float64 too keeps them (100 replicas of 64
    // agents 0.384 and 0.251).
    const bool verify = (flags & ABM_VERIFY_FAST_PATH) != 0;
    const bool few = b->n_replicas <= kFewReplicas && nb > 0 && nb < b->n_replicas;
    if (nw == 0 && !sync_order && !few && !verify && push_fits(b, true) &&
        (int64_t)b->n_agents_total + 4 * (int64_t)b->n_replicas <= ((int64_t)b->max_agents + 4) * b->n_cu) {
        // the sums as the kernels of the two classes take them, bit for bit (but
        // for the order of the last float64 adds): the same rays a lane, or half
        // as many on two waves
        const int ns = b->n_replicas - nb, rpl = push_rpl(b->max_rays), r = nb > 0 ? b->small_max_rays : b->max_rays;
        const int waves = ns > 0 ? default_waves(b, nb > 0 ? b->small_max_agents : b->max_agents, ns) : 1;
        const int small = ns > 0 ? push_rpl((r + waves - 1) / waves) : rpl;
        if ((nb == 0 || push_rpl(b->big_max_rays) == rpl) && (small == rpl || 2 * small == rpl))
            return launch_push_any(b, st, bits, diag, flags, s, b->order_dev, b->n_replicas, true, small != rpl);
    }
    // else for the class of large replicas alone
    const bool push_ok = !sync_order && nb > 0 && push_fits(b, false);
    const bool push = push_ok && b->big_sum_agents <= (int64_t)b->big_max_agents * b->n_cu;
    if (nw == 0 && nb > 0 && !sync_order && (push || (!push_ok && nb < b->n_replicas))) {
        // size classes: the small replicas on the per-replica kernel, then
        // the large ones, whose id-order chains are the step's critical
        // path, on the push kernel (pairs off the chain) where their fields
        // fit in LDS, else on the 16-wave kernel
        if (nb < b->n_replicas) {
            if (int rc = launch_per_replica(b, st, bits, diag, flags, s, 0, b->order_dev + nb,
                                            b->n_replicas - nb, b->small_max_agents, b->small_max_rays, true))
                return rc;
        }
        if (push) return launch_push_any(b, st, bits, diag, flags, s, b->order_dev, nb, false);
        return launch_big_any(b, st, bits, diag, flags, s, b->order_dev, nb, b->big_max_agents,
                              b->big_max_rays);
    }
    return launch_per_replica(b, st, bits, diag, flags, s, nw, b->order_dev, b->n_replicas, b->max_agents,
                              b->max_rays, false);
}

}  // namespace abm
