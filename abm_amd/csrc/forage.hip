// forage.hip -- collective-foraging agent step (Agent.update for every agent
// in id order) in float64, plus the Agent.projection_field probe.
//
// One workgroup per replica; the replica's agents live in LDS.  Without
// visual exclusion all agents are updated at once (forage_update_kernel); with
// it one after another, in id order (Group.update, abm/simulation/sims.py:861).
// Per focal agent k:
//   1. lanes over the other agents: cue class (agent.py:396-419) and the
//      projection record of each obstacle (agent.py:501-556): closed angle with
//      the strict 0 < a' < pi rule, the focal radius for both centres, int()
//      truncation of t -+ proj_size/2, strict FOV test;
//   2. visual exclusion (agent.py:421-445): records ranked by (distance,
//      obstacle-list position); each record then walks the nearer ones in rank
//      order and applies the three interval rules sequentially;
//   3. raster of the social records with Python slice semantics
//      (agent.py:569-590) into a per-ray byte field; flip and FOV mask
//      (agent.py:593-595) when counting;
//   4. one lane: I_priv, w/u integrators, mode table, random walk from the
//      host-supplied uniforms of numpy's global stream, relocation force,
//      Euler step and walls (agent.py:168-283, supcalc.py:38-47, 81-92).
// Built with -ffp-contract=off.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <utility>
#include <vector>

#include "../../include/abm_amd.h"
#include "forage_batch.hpp"
#include "vf_exact.hpp"
#include "vf_f32_common.hpp"

namespace abm {
int set_error(int code, const char* fmt, ...);
int check_hip(hipError_t e, const char* what);

namespace {

// Obstacle classes, in the order the reference lists them to projection_field.
constexpr int kSocial = 0;      // exploiting agents of other patches (the cues)
constexpr int kNonExpl = 1;     // in-range agents that are not exploiting (self included)
constexpr int kSamePatch = 2;   // exploiting agents of the focal's own patch
constexpr int kNone = -1;

struct PairFG {
    int skipped, visible, t, start, end;
    double dist, vis;
};

// One obstacle of Agent.projection_field (agent.py:501-556).
ABM_HD PairFG pair_forage_exact(const Focal& f, double ox, double oy, int R, double step,
                                double fov0, double fov1) {
#pragma clang fp contract(off)
    PairFG p;
    p.skipped = 0; p.visible = 0; p.t = 0; p.start = 0; p.end = 0; p.dist = 0.0; p.vis = 0.0;
    if (ox == f.px && oy == f.py) { p.skipped = 1; return p; }
    const double v2ex = ox + f.radius;          // the focal radius for the obstacle too
    const double v2ey = oy + f.radius;
    const double v2x = v2ex - f.cx, v2y = v2ey - f.cy;
    const double n2 = norm2(v2x, v2y);
    const double u2x = v2x / n2, u2y = v2y / n2;
    double d = dot2(f.u1x, f.u1y, u2x, u2y);
    if (d < -1.0) d = -1.0;
    else if (d > 1.0) d = 1.0;
    double a = acos(d);
    const double cross = f.u1x * u2y - f.u1y * u2x;
    if (cross < 0.0) a = -a;
    a = remainder_2pi(a);
    const double ca = (0.0 < a && a < kPi) ? -a : kTwoPi - a;   // strict (agent.py:520)
    p.dist = n2;
    p.vis = 2.0 * atan(f.radius / (1.0 * n2));
    p.t = linspace_argmin(ca, R, step);
    p.visible = (fov0 < ca && ca < fov1) ? 1 : 0;
    const double ps = (p.vis / kTwoPi) * (double)R;
    p.start = (int)trunc((double)p.t - ps / 2.0);
    p.end = (int)trunc((double)p.t + ps / 2.0);
    return p;
}

// Indices of range(R)[a:b] (Python slice semantics), as a half-open range.
ABM_HD void py_slice(int a, int b, int R, int* lo, int* hi) {
    if (a < 0) { a += R; if (a < 0) a = 0; }
    if (a > R) a = R;
    if (b < 0) { b += R; if (b < 0) b = 0; }
    if (b > R) b = R;
    *lo = a; *hi = b > a ? b : a;
}

struct Rec {
    int valid;        // visible record (obstacle passed the FOV test)
    int social;
    int order;        // position in the reference's obstacle list
    int start, end;   // int(t -+ proj_size/2)
    int sx, ex;       // after exclusion
    double dist;
    double vis;
};

// Paint one record with Python slice semantics: wrap pieces get `wrap_code`,
// the main slice `main_code` (agent.py:577-590).
__device__ inline void paint_record(uint8_t* V, const Rec& rc, int R, uint8_t wrap_code,
                                    uint8_t main_code) {
    int s = rc.sx, e = rc.ex, lo, hi;
    if (s < 0) {
        py_slice(R + s, R, R, &lo, &hi);
        for (int r = lo; r < hi; ++r) V[r] = wrap_code;
        s = 0;
    }
    if (e >= R) {
        py_slice(0, e - R, R, &lo, &hi);
        for (int r = lo; r < hi; ++r) V[r] = wrap_code;
        e = R - 1;
    }
    py_slice(s, e, R, &lo, &hi);
    for (int r = lo; r < hi; ++r) V[r] = main_code;
}

// Per-replica constants in device memory.
struct FGRep {
    int32_t agent_offset, n_agents, n_rays, words, visual_exclusion, patchwise, tau, pad_;
    int32_t keep_lo, keep_hi;   // soc_v_field indices the FOV mask keeps (a contiguous range)
    int64_t field_offset;
    double fov0, fov1, width, height, pad, vision_range, step;
    double T_w, Eps_w, g_w, B_w, w_max, T_u, Eps_u, g_u, B_u, u_max, S_wu, S_uw, F_N, F_R;
    double exp_vel_max, exp_theta_min, exp_theta_max, reloc_theta_max, exp_stop_ratio;
};

__device__ inline int get_mode(int overriding, double w, double T_w) {
    // agent.py:659-669
    if (overriding >= 0) return overriding;
    return w > T_w ? ABM_MODE_RELOCATE : ABM_MODE_EXPLORE;
}

struct FGSmem {
    Focal* focal;   // step kernel: focal geometry of the next two agents, by parity
    double *x, *y, *th, *v, *w, *u, *cr, *crb, *nov, *rad;
    int *mode, *over, *env, *pid, *cls;
    Rec* rec;
    int* sorted;
    int* lst;       // step kernel: obstacles needing records, two lists of maxN by parity
    int* cls2;      // step kernel: classes for the agent after next (cls holds the next one's)
    double* uni;    // step kernel: the step's uniforms (or pairs of words), staged
    uint32_t* mtk;  // step kernel: the replica's generator key (device generators)
    uint8_t* V;
    int* cnt;       // step kernel: [2p] total, [2p+1] left half by parity; [4 + p] list sizes
    double* lastd;  // keep_distance: distance of the last processed obstacle
    double* spec;   // step kernel: [12 p ..] an agent's headings after a walk turn or none, with sin and
                    // cos, by parity p; [24 + p] uniforms drawn before an agent of parity p
};

__device__ inline FGSmem fg_carve(void* base, int maxN, int maxR) {
    FGSmem s;
    char* p = reinterpret_cast<char*>(base);
    s.focal = reinterpret_cast<Focal*>(p); p += 128;
    double** dptrs[] = {&s.x, &s.y, &s.th, &s.v, &s.w, &s.u, &s.cr, &s.crb, &s.nov, &s.rad};
    for (double** d : dptrs) { *d = reinterpret_cast<double*>(p); p += sizeof(double) * maxN; }
    s.lastd = reinterpret_cast<double*>(p); p += sizeof(double) * 2;
    s.spec = reinterpret_cast<double*>(p); p += sizeof(double) * 28;
    s.uni = reinterpret_cast<double*>(p); p += sizeof(double) * maxN;
    s.rec = reinterpret_cast<Rec*>(p); p += sizeof(Rec) * maxN;
    int** iptrs[] = {&s.mode, &s.over, &s.env, &s.pid, &s.cls};
    for (int** q : iptrs) { *q = reinterpret_cast<int*>(p); p += sizeof(int) * maxN; }
    s.sorted = reinterpret_cast<int*>(p); p += sizeof(int) * maxN;
    s.lst = reinterpret_cast<int*>(p); p += sizeof(int) * 2 * maxN;
    s.cls2 = reinterpret_cast<int*>(p); p += sizeof(int) * maxN;
    s.cnt = reinterpret_cast<int*>(p); p += sizeof(int) * 8;
    s.mtk = reinterpret_cast<uint32_t*>(p); p += sizeof(uint32_t) * 624;
    s.V = reinterpret_cast<uint8_t*>(p);
    return s;
}

static_assert(sizeof(Focal) <= 64, "two Focal slots of 64 bytes");

size_t fg_lds_bytes(int maxN, int maxR) {
    return 128 + sizeof(double) * ((size_t)11 * maxN + 30) + sizeof(Rec) * (size_t)maxN +
           sizeof(int) * ((size_t)9 * maxN + 8) + sizeof(uint32_t) * 624 + (size_t)maxR + 16;
}

// Records of one focal agent against the obstacle set marked in S.cls
// (kNone = not an obstacle), visual exclusion, and the raster into S.V.
// Every thread of the block calls it; it ends synchronised.
__device__ void project_focal(const FGSmem& S, int N, int R, double step, double fov0, double fov1,
                              bool exclusion, bool with_nonsocial, const Focal& f,
                              bool keep_distance = false) {
#pragma clang fp contract(off)
    const int tid = threadIdx.x, nthr = blockDim.x;
    for (int r = tid; r < R; r += nthr) S.V[r] = 0;
    for (int j = tid; j < N; j += nthr) {
        Rec rc;
        rc.valid = 0; rc.social = 0; rc.order = 0; rc.start = rc.end = rc.sx = rc.ex = 0;
        rc.dist = 0.0;
        rc.vis = 0.0;
        const int c = S.cls[j];
        if (c == kSocial || (with_nonsocial && (c == kNonExpl || c == kSamePatch))) {
            const PairFG p = pair_forage_exact(f, S.x[j], S.y[j], R, step, fov0, fov1);
            if (!p.skipped && p.visible) {
                rc.valid = 1;
                rc.social = c == kSocial;
                rc.order = c * N + j;
                rc.start = rc.sx = p.start;
                rc.end = rc.ex = p.end;
                rc.dist = p.dist;
                rc.vis = p.vis;
            }
        }
        S.rec[j] = rc;
    }
    __syncthreads();
    if (exclusion) {
        // rank = position in the stable ascending sort by distance
        for (int j = tid; j < N; j += nthr) {
            const Rec rf = S.rec[j];
            if (!rf.valid) continue;
            int rank = 0;
            for (int i = 0; i < N; ++i) {
                const Rec ri = S.rec[i];
                if (ri.valid && (ri.dist < rf.dist || (ri.dist == rf.dist && ri.order < rf.order)))
                    ++rank;
            }
            S.sorted[rank] = j;
        }
        __syncthreads();
        for (int j = tid; j < N; j += nthr) {
            Rec rf = S.rec[j];
            if (!rf.valid) continue;
            // walk the nearer records in rank order; rank 0 keeps its interval
            for (int q = 0; q < N; ++q) {
                const int i = S.sorted[q];
                if (i == j) break;
                const Rec ri = S.rec[i];
                if (ri.dist < rf.dist) {
                    if (rf.sx <= ri.start && ri.start <= rf.ex) rf.ex = ri.start;
                    if (rf.sx <= ri.end && ri.end <= rf.ex) rf.sx = ri.end;
                    if (ri.start <= rf.sx && ri.end >= rf.ex) { rf.sx = 0; rf.ex = 0; }
                }
            }
            S.rec[j].sx = rf.sx;
            S.rec[j].ex = rf.ex;
        }
        __syncthreads();
    }
    if (!keep_distance) {
        // every record paints 1, so the order of the records does not matter
        for (int j = tid; j < N; j += nthr) {
            const Rec rc = S.rec[j];
            if (!rc.valid || !rc.social) continue;
            paint_record(S.V, rc, R, 1, 1);
        }
    } else if (tid == 0) {
        // keep_distance_info: wrap pieces paint 1 and main slices the distance
        // value (code 2); later records overwrite, in descending vis_angle
        // order with ties in obstacle order (agent.py:567, 569-590)
        int last_vis_idx = -1;
        for (int n = 0; n < N; ++n) {
            int best = -1;
            for (int j = 0; j < N; ++j) {
                const Rec rc = S.rec[j];
                if (!rc.valid || !rc.social) continue;
                if (last_vis_idx >= 0) {
                    const Rec lr = S.rec[last_vis_idx];
                    const bool after = rc.vis < lr.vis || (rc.vis == lr.vis && rc.order > lr.order);
                    if (!after) continue;
                }
                if (best < 0) { best = j; continue; }
                const Rec br = S.rec[best];
                if (rc.vis > br.vis || (rc.vis == br.vis && rc.order < br.order)) best = j;
            }
            if (best < 0) break;
            paint_record(S.V, S.rec[best], R, 1, 2);
            last_vis_idx = best;
        }
    }
    __syncthreads();
}

// soc_v_field[k] = V[R-1-k] unless linspace_k is outside [fov0, fov1].
__device__ inline int soc_bit(const uint8_t* V, int k, int R, double step, double fov0, double fov1) {
    const double ph = linspace_at(k, R, step);
    if (ph < fov0 || ph > fov1) return 0;
    return V[R - 1 - k];
}

// Cue class of agent j for focal agent f (agent.py:396-413): in range by
// supcalc.distance; exploiting agents of another patch are the cues, those
// of the focal's own patch occlude (patchwise exclusion), exploiting agents
// without a patch are dropped; the rest in range (the focal included) occlude.
__device__ inline int cue_class(const FGSmem& S, const FGRep& P, int j, int f, double cfx, double cfy,
                                int pid_f) {
#pragma clang fp contract(off)
    const double dx = (S.x[j] + S.rad[j]) - cfx, dy = (S.y[j] + S.rad[j]) - cfy;
    const bool in_range = norm2(dx, dy) <= P.vision_range;
    const bool expl = in_range && j != f && get_mode(S.over[j], S.w[j], P.T_w) == ABM_MODE_EXPLOIT;
    int c = kNone;
    if (expl) {
        if (P.patchwise && S.pid[j] == pid_f) c = kSamePatch;
        else if (S.pid[j] != -1) c = kSocial;
    } else if (in_range) {
        c = kNonExpl;
    }
    return c;
}

// Per-replica float32 constants of the guarded record.
struct FastRec {
    float inv_step;   // bins of linspace(-pi, pi, R) per radian
    float hs;         // R / (2 pi): proj_size / 2 per radian of atan(r / d)
    float g_bins;     // bin-tie guard in bins (angle guard + float32 rounding of the coordinate)
    float fov0, fov1;
};

__device__ inline FastRec fast_rec_const(int R, double step, double fov0, double fov1) {
    FastRec q;
    q.inv_step = (float)(1.0 / step);
    q.hs = (float)((double)R / kTwoPi);
    q.g_bins = (float)(f32::kAngleGuardF / step + 1.5e-7 * R);
    q.fov0 = (float)fov0;
    q.fov1 = (float)fov1;
    return q;
}

// The exact record (rare): visible, start, end.  Out of line, or its constants
// (acos, atan) would be held in registers over every caller's loop.
__device__ __attribute__((noinline)) int4 record_exact(double ox, double oy, double px, double py, double radius,
                                                       double u1x, double u1y, int R, double step, double fov0,
                                                       double fov1) {
    Focal f;
    f.px = px; f.py = py; f.radius = radius;
    f.cx = px + radius; f.cy = py + radius;
    f.u1x = u1x; f.u1y = u1y;
    const PairFG p = pair_forage_exact(f, ox, oy, R, step, fov0, fov1);
    return make_int4(!p.skipped && p.visible, p.start, p.end, 0);
}

// Record of obstacle j (class c) for focal geometry f.  The bin, the
// interval and the FOV test come from a float32 decision when it is outside
// every guard band, else from the exact float64 record (agent.py:501-556):
//  * the centre difference (focal radius for both centres) in float64,
//    rounded once, and the focal's float64 unit heading: with atan2_f32 the
//    signed angle a from heading to object is within 1e-6 rad of the exact
//    one, and the reference's acos-based angle within 5e-8 rad of that;
//  * the reference's closed angle is -a for 0 < |a| < pi (a' = a mod 2 pi,
//    ca = -a' or 2 pi - a'); a = 0 gives 2 pi and |a| = pi gives pi: 4e-6 rad
//    bands around 0 and pi, and around the strict FOV ends;
//  * t = nearest bin of ca (bin-tie band as in the flocking kernels);
//  * start / end = int(t -+ proj_size / 2), truncated toward zero: with half
//    = proj_size / 2 outside a 4e-6 relative band around an integer, start =
//    t - floor(half) - 1 when that stays positive, else t - floor(half),
//    and end = t + floor(half).
// The float64 distance, which only visual exclusion ranks by, is exact.
__device__ inline Rec record_at(double ox, double oy, int c, int order, const Focal& f, int R, double step,
                                double fov0, double fov1, const FastRec& FR, bool need_dist) {
#pragma clang fp contract(off)
    Rec rc;
    rc.valid = 0; rc.social = 0; rc.order = 0; rc.start = rc.end = rc.sx = rc.ex = 0;
    rc.dist = 0.0; rc.vis = 0.0;
    if (ox == f.px && oy == f.py) return rc;                 // skipped (agent.py:502)
    const double v2x = (ox + f.radius) - f.cx, v2y = (oy + f.radius) - f.cy;
    {
        const float dx = (float)v2x, dy = (float)v2y;
        const float u1x = (float)f.u1x, u1y = (float)f.u1y;
        const float d2 = fmaf(dy, dy, dx * dx);
        const float a = f32::atan2_f32(fmaf(u1x, dy, -u1y * dx), fmaf(u1x, dx, u1y * dy));
        const float aa = fabsf(a);
        const float ca = -a;
        const float xb = (f32::kPiF - a) * FR.inv_step;     // bin coordinate of ca
        const float tr = rintf(xb);
        const float dfr = xb - tr;
        const float half = f32::atan_pos_f32((float)f.radius, __builtin_amdgcn_sqrtf(d2)) * FR.hs;
        const float hfl = floorf(half);
        const float hfrac = half - hfl;
        const float hg = 4e-6f * half + 1e-6f;
        const float g = f32::kAngleGuardF;
        const bool ok = (d2 > 1e-30f) & (aa > g) & (aa < f32::kPiF - g) &
                        (fabsf(dfr) <= 0.5f - FR.g_bins) & (hfrac >= hg) & (hfrac <= 1.0f - hg) &
                        (fabsf(ca - FR.fov0) >= g) & (fabsf(ca - FR.fov1) >= g);
        if (ok) {
            if (FR.fov0 < ca && ca < FR.fov1) {
                const int t = (int)tr, h = (int)hfl;
                rc.valid = 1;
                rc.social = c == kSocial;
                rc.order = order;
                rc.start = rc.sx = t - h >= 1 ? t - h - 1 : t - h;
                rc.end = rc.ex = t + h;
                if (need_dist) rc.dist = norm2(v2x, v2y);
            }
            return rc;
        }
    }
    const int4 p = record_exact(ox, oy, f.px, f.py, f.radius, f.u1x, f.u1y, R, step, fov0, fov1);
    if (p.x) {
        rc.valid = 1;
        rc.social = c == kSocial;
        rc.order = order;
        rc.start = rc.sx = p.y;
        rc.end = rc.ex = p.z;
        if (need_dist) rc.dist = norm2(v2x, v2y);
    }
    return rc;
}

__device__ inline Rec record_of(const FGSmem& S, int j, int c, int N, const Focal& f, int R, double step,
                                double fov0, double fov1, const FastRec& FR, bool need_dist) {
    return record_at(S.x[j], S.y[j], c, c * N + j, f, R, step, fov0, fov1, FR, need_dist);
}

// Classes of the agents j != skip for focal agent f into S.cls; those in
// range (agent.py:415-419) are appended to lst (in any order: records are
// kept per agent and ranked by (distance, list position)).  Thread t0 of
// `stride` threads, both multiples of 64 apart per wave.
__device__ void classify(const FGSmem& S, const FGRep& P, int N, int f, int skip1, int skip2, int* cls,
                         int* lst, int* lst_n, int t0, int stride) {
    const double cfx = S.x[f] + S.rad[f], cfy = S.y[f] + S.rad[f];
    const int pid_f = S.pid[f];
    const int lane = t0 & 63;
    for (int base = t0 - lane; base < N; base += stride) {
        const int j = base + lane;
        bool need = false;
        if (j < N && j != skip1 && j != skip2) {
            const int c = cue_class(S, P, j, f, cfx, cfy, pid_f);
            cls[j] = c;
            need = c != kNone;
        }
        const uint64_t m = __ballot(need);
        if (m) {
            int at = 0;
            if (lane == 0) at = atomicAdd(lst_n, (int)__popcll(m));
            at = __builtin_amdgcn_readfirstlane(at);
            if (need) lst[at + (int)__popcll(m & ((1ull << lane) - 1ull))] = j;
        }
    }
}

// sin and cos (out of line for the same reason).
__device__ __attribute__((noinline)) double2 sin_cos(double th) {
    double sn, cs;
    sincos(th, &sn, &cs);
    return make_double2(sn, cs);
}

// make_focal with one sincos for the heading (the same values as cos, sin).
__device__ inline Focal focal_at(double px, double py, double sn, double cs, double radius) {
#pragma clang fp contract(off)
    Focal f;
    f.px = px; f.py = py; f.radius = radius;
    f.cx = px + radius;
    f.cy = py + radius;
    const double ex = px + (1.0 + cs) * radius;
    const double ey = py + (1.0 - sn) * radius;
    const double v1x = ex - f.cx, v1y = ey - f.cy;
    const double n1 = norm2(v1x, v1y);
    f.u1x = v1x / n1;
    f.u1y = v1y / n1;
    return f;
}
__device__ inline Focal focal_at(double px, double py, double th, double radius) {
    double sn, cs;
    sincos(th, &sn, &cs);
    return focal_at(px, py, sn, cs, radius);
}
__device__ inline Focal focal_of(const FGSmem& S, int k) { return focal_at(S.x[k], S.y[k], S.th[k], S.rad[k]); }

// The heading agent f takes after a random-walk turn drawn from uniform
// d + c (c = 0, 1) or after no turn (c = 2), with its sin and cos, into
// buf[3c .. 3c + 2] (agent.py:187-200, 595-603: prove_orientation of the
// turned heading, then cos and sin for the move); buf[9] = d.  The same
// arithmetic as the move, computed by a spare wave before agent f's
// decision: the walk's draw index is d or d + 1 (the agent before draws at
// most one uniform), so the decision only picks a slot.
__device__ inline void spec_heading(const FGSmem& S, const FGRep& P, int N, int f, int d, int c, double* buf) {
#pragma clang fp contract(off)
    double dth = 0.0;
    if (c < 2) {
        const double uu = d + c < N ? S.uni[d + c] : 0.0;
        dth = P.exp_theta_min + (P.exp_theta_max - P.exp_theta_min) * uu;
    }
    const double th = prove_orientation(S.th[f] + dth);
    double sn, cs;
    sincos(th, &sn, &cs);
    buf[3 * c] = th;
    buf[3 * c + 1] = sn;
    buf[3 * c + 2] = cs;
    if (c == 0) buf[9] = (double)d;
}

// Set bits [lo, hi) of a bit-packed field.
__device__ inline void or_range(uint32_t* Vb, int lo, int hi) {
    while (lo < hi) {
        const int w = lo >> 5, b0 = lo & 31;
        const int end = min(hi, (w + 1) * 32);
        const int nb = end - lo;
        atomicOr(&Vb[w], nb == 32 ? 0xffffffffu : ((1u << nb) - 1u) << b0);
        lo = end;
    }
}

// paint_record for the step kernel's bit-packed raw field: every social
// record paints 1, so the pieces are ORed in any order (agent.py:577-590).
__device__ inline void paint_bits(uint32_t* Vb, const Rec& rc, int R) {
    int s = rc.sx, e = rc.ex, lo, hi;
    if (s < 0) {
        py_slice(R + s, R, R, &lo, &hi);
        or_range(Vb, lo, hi);
        s = 0;
    }
    if (e >= R) {
        py_slice(0, e - R, R, &lo, &hi);
        or_range(Vb, lo, hi);
        e = R - 1;
    }
    py_slice(s, e, R, &lo, &hi);
    or_range(Vb, lo, hi);
}

// Bits of word w inside the inclusive index range [a, b].
__device__ inline uint32_t word_range_mask(int w, int a, int b) {
    const int lo = max(a, w * 32), hi = min(b, w * 32 + 31);
    if (lo > hi) return 0u;
    const int nb = hi - lo + 1;
    return nb == 32 ? 0xffffffffu : ((1u << nb) - 1u) << (lo & 31);
}

// Visual exclusion (agent.py:421-445) over the listed records, then their
// raster (agent.py:569-590) into the bit-packed raw field S.V (uint32
// words, bit r = V[r]).  Every thread; ends synchronised.
__device__ void raster_list(const FGSmem& S, int R, const int* lst, int n0, int extra) {
    const int tid = threadIdx.x, nthr = blockDim.x;
    // the listed records, and one more (extra >= 0) kept outside the list
    const int n = n0 + (extra >= 0 ? 1 : 0);
    auto item = [&](int q) { return q < n0 ? lst[q] : extra; };
    // rank = position in the stable ascending sort by distance.  Both loops wait on
    // LDS: records are loaded four ahead, a walk's next item with the record before it
    // (2 replicas of 257 agents 20.3 -> 17.0 ms a step, one of 512 76.8 -> 64.4)
    for (int q = tid; q < n; q += nthr) {
        const int j = item(q);
        const Rec rf = S.rec[j];
        if (!rf.valid) continue;
        int rank = 0;
#pragma unroll 4
        for (int p = 0; p < n; ++p) {
            const Rec ri = S.rec[item(p)];
            if (ri.valid && (ri.dist < rf.dist || (ri.dist == rf.dist && ri.order < rf.order))) ++rank;
        }
        S.sorted[rank] = j;
    }
    __syncthreads();
    for (int q = tid; q < n; q += nthr) {
        const int j = item(q);
        Rec rf = S.rec[j];
        if (!rf.valid) continue;
        // walk the nearer records in rank order; rank 0 keeps its interval
        int i = S.sorted[0];
        for (int p = 0; p < n && i != j; ++p) {
            const Rec ri = S.rec[i];
            i = S.sorted[min(p + 1, n - 1)];
            if (ri.dist < rf.dist) {
                if (rf.sx <= ri.start && ri.start <= rf.ex) rf.ex = ri.start;
                if (rf.sx <= ri.end && ri.end <= rf.ex) rf.sx = ri.end;
                if (ri.start <= rf.sx && ri.end >= rf.ex) { rf.sx = 0; rf.ex = 0; }
            }
        }
        S.rec[j].sx = rf.sx;
        S.rec[j].ex = rf.ex;
    }
    __syncthreads();
    uint32_t* Vb = reinterpret_cast<uint32_t*>(S.V);
    for (int q = tid; q < n; q += nthr) {
        const Rec rc = S.rec[item(q)];
        if (rc.valid && rc.social) paint_bits(Vb, rc, R);
    }
    __syncthreads();
}

// Sum over the 64 lanes of wave 0 with DPP moves (no LDS round trips):
// prefix sums inside each row of 16 lanes (row_shr 1, 2, 4, 8), then row
// 15's and row 31's lane carried into the rows above (row_bcast 15, 31), so
// lane 63 holds the total.  Lanes a move has no source for add 0.
__device__ inline int wave_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return __builtin_amdgcn_readlane(v, 63);
}

__device__ inline void fg_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The returned field of agent k: counts for mean() and the left/right
// halves into cnt; soc_v_field[r] = V[R-1-r] on the rays the FOV mask keeps.
__device__ void count_field(const FGSmem& S, const FGRep& P, int R, int* cnt, uint32_t* bits_out, int k) {
    const int tid = threadIdx.x, nthr = blockDim.x, nl = R / 2, W = P.words;
    const uint32_t* Vb = reinterpret_cast<const uint32_t*>(S.V);
    // soc_v_field[q] = V[R-1-q] for keep_lo <= q <= keep_hi: raw indices
    // [R-1-keep_hi, R-1-keep_lo]; the left half q < R/2 is raw r >= R - R/2
    const int ta = R - 1 - P.keep_hi, tb = R - 1 - P.keep_lo, la = max(R - nl, ta);
    for (int w = tid; w < W; w += nthr) {
        const uint32_t bits = Vb[w];
        const int tot = __popc(bits & word_range_mask(w, ta, tb));
        const int left = __popc(bits & word_range_mask(w, la, tb));
        if (tot) atomicAdd(&cnt[0], tot);
        if (left) atomicAdd(&cnt[1], left);
    }
    if (bits_out) {
        uint32_t* dst = bits_out + P.field_offset + (int64_t)k * W;
        for (int wd = tid; wd < W; wd += nthr) {
            uint32_t m = 0;
            for (int b = 0; b < 32; ++b) {
                const int q = wd * 32 + b, r = R - 1 - q;
                if (q >= P.keep_lo && q <= P.keep_hi && ((Vb[r >> 5] >> (r & 31)) & 1u)) m |= 1u << b;
            }
            dst[wd] = m;
        }
    }
}

// ---- numpy's legacy MT19937 on the device (the published generator of
// Matsumoto and Nishimura, in numpy's mt19937_state layout: 624 key words and
// a position; numpy twists lazily, when a word is drawn at position 624)
constexpr int kMtN = 624, kMtM = 397;

__device__ inline uint32_t mt_temper(uint32_t y) {
    y ^= y >> 11;
    y ^= (y << 7) & 0x9d2c5680u;
    y ^= (y << 15) & 0xefc60000u;
    y ^= y >> 18;
    return y;
}

__device__ inline uint32_t mt_twist_word(uint32_t cur, uint32_t nxt, uint32_t far) {
    const uint32_t y = (cur & 0x80000000u) | (nxt & 0x7fffffffu);
    return far ^ (y >> 1) ^ ((y & 1u) ? 0x9908b0dfu : 0u);
}

// key[i] for i = 0..623 in order, in place, by one wave: in the chunks [0, 227),
// [227, 454), [454, 623) and {623} every element reads key[i + 1] not yet
// rewritten and key[(i + 397) % 624] already final, so each chunk is read in
// full, then written.
__device__ inline void mt_twist_wave(uint32_t* key) {
    const int lane = threadIdx.x & 63;
    constexpr int lo[4] = {0, kMtN - kMtM, 2 * (kMtN - kMtM), kMtN - 1};
    constexpr int hi[4] = {kMtN - kMtM, 2 * (kMtN - kMtM), kMtN - 1, kMtN};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        uint32_t v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int i = lo[c] + lane + 64 * t;
            const int far = i + kMtM < kMtN ? i + kMtM : i + kMtM - kMtN;
            v[t] = i < hi[c] ? mt_twist_word(key[i], key[i + 1 < kMtN ? i + 1 : 0], key[far]) : 0u;
        }
        fg_wave_sync();
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int i = lo[c] + lane + 64 * t;
            if (i < hi[c]) key[i] = v[t];
        }
        fg_wave_sync();
    }
}

// The same by a block of at least 227 threads, all of which call it.
__device__ inline void mt_twist_block(uint32_t* key) {
    const int tid = threadIdx.x;
    constexpr int lo[4] = {0, kMtN - kMtM, 2 * (kMtN - kMtM), kMtN - 1};
    constexpr int hi[4] = {kMtN - kMtM, 2 * (kMtN - kMtM), kMtN - 1, kMtN};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int i = lo[c] + tid;
        const bool mine = i < hi[c];
        uint32_t v = 0u;
        if (mine) {
            const int far = i + kMtM < kMtN ? i + kMtM : i + kMtM - kMtN;
            v = mt_twist_word(key[i], key[i + 1 < kMtN ? i + 1 : 0], key[far]);
        }
        __syncthreads();
        if (mine) key[i] = v;
        __syncthreads();
    }
}

// Draws from a generator state held in LDS, by one wave (every lane the same
// draw); never runs out.
struct MtCursor {
    uint32_t* key;
    int pos, used;
    bool out;
    __device__ uint32_t next() {
        if (pos >= kMtN) {
            mt_twist_wave(key);
            pos = 0;
        }
        ++used;
        return mt_temper(key[pos++]);
    }
};

// Status of a replica between the interaction kernel and the update.
constexpr int kWorldReady = 3;

// numpy's legacy random_sample from two raw MT19937 outputs (mt19937_next_double).
__device__ inline double words_to_double(uint32_t w0, uint32_t w1) {
    const uint32_t a = w0 >> 5, b = w1 >> 6;
    return ((double)a * 67108864.0 + (double)b) / 9007199254740992.0;
}

// The random walk's uniforms come either as doubles (uniforms) or as raw
// 32-bit outputs (words, two per draw, starting after the words the resource
// loop consumed: u_used[b] on entry).  With status, only replicas marked
// kWorldReady are updated, and they are marked ABM_WORLD_DONE.  FIELDS false:
// a step that writes no fields (bits_out is ignored).  The replicas of this
// kernel have visual exclusion: every agent in range, as it stands in its
// turn, occludes, so the agents are updated one after another.  It takes those
// with more agents than forage_occlude_kernel holds in registers.
template <bool FIELDS>
__global__ void __launch_bounds__(512)
forage_step_kernel(const FGRep* __restrict__ reps, abm_forage_state st,
                   const double* __restrict__ uniforms, const uint32_t* __restrict__ words,
                   const int64_t* __restrict__ u_off, const int32_t* __restrict__ u_cnt,
                   int32_t* __restrict__ u_used, int32_t* __restrict__ status,
                   uint32_t* __restrict__ bits_out, const int32_t* __restrict__ order,
                   abm_mt19937_state* __restrict__ mt, int maxN, int maxR) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) double smem[];
    if (!FIELDS) bits_out = nullptr;
    // blocks take the replicas largest first, so the longest id-order chains
    // start at once and the small replicas fill in behind them
    const int rb = order[blockIdx.x];
    if (status && status[rb] != kWorldReady) return;   // uniform over the block
    const int tid = threadIdx.x, nthr = blockDim.x;
    // the replica's parameters in LDS: read where used, rather than held in
    // scalar registers over the whole agent loop (which spills them)
    __shared__ FGRep sP;
    static_assert(sizeof(FGRep) % 8 == 0 && sizeof(FGRep) / 8 <= 64, "FGRep copy");
    if (tid < (int)(sizeof(FGRep) / 8))
        reinterpret_cast<uint64_t*>(&sP)[tid] = reinterpret_cast<const uint64_t*>(reps + rb)[tid];
    __syncthreads();
    const FGRep& P = sP;
    const int N = P.n_agents, R = P.n_rays, a0 = P.agent_offset;
    FGSmem S = fg_carve(smem, maxN, maxR);
    for (int i = tid; i < N; i += nthr) {
        const int g = a0 + i;
        S.x[i] = st.x[g]; S.y[i] = st.y[g]; S.th[i] = st.theta[g]; S.v[i] = st.v[g];
        S.w[i] = st.w[g]; S.u[i] = st.u[g]; S.cr[i] = st.collected_r[g];
        S.crb[i] = st.collected_r_before[g];
        double m = st.novelty[(int64_t)g * P.tau];
        for (int q = 1; q < P.tau; ++q) m = fmax(m, st.novelty[(int64_t)g * P.tau + q]);
        S.nov[i] = m;
        S.rad[i] = (double)st.radius[g];
        S.mode[i] = st.mode[g]; S.over[i] = st.overriding_mode[g];
        S.env[i] = st.env_status[g]; S.pid[i] = st.exploited_patch_id[g];
    }
    // the step's uniforms, staged in LDS: agent i's draw is the i-th (at most
    // one per agent); doubles, or pairs of words after those the resource
    // loop used (u_used[b] on entry); NaN past the end of the buffer
    const int ucount = mt ? 0 : u_cnt[rb];
    const int used0 = (words || mt) ? u_used[rb] : 0;
    int mt_pos0 = 0;
    if (mt) {
        // the replica's generator on the device: its next 2N words (a copy of
        // the key twisted in LDS as needed), as N uniforms
        for (int i = tid; i < kMtN; i += nthr) S.mtk[i] = mt[rb].key[i];
        mt_pos0 = mt[rb].pos;
        __syncthreads();
        uint32_t* wb = reinterpret_cast<uint32_t*>(S.uni);
        int made = 0, p = mt_pos0;
        while (made < 2 * N) {
            if (p >= kMtN) {
                mt_twist_block(S.mtk);
                p = 0;
            }
            const int take = min(kMtN - p, 2 * N - made);
            for (int j = tid; j < take; j += nthr) wb[made + j] = mt_temper(S.mtk[p + j]);
            made += take;
            p += take;
        }
        __syncthreads();
        for (int i = tid; i < N; i += nthr) {   // each thread rewrites its own 8 bytes
            const uint32_t w0 = wb[2 * i], w1 = wb[2 * i + 1];
            S.uni[i] = words_to_double(w0, w1);
        }
    } else {
        for (int i = tid; i < N; i += nthr) {
            double uu = NAN;
            if (words) {
                const uint32_t* wb = words + u_off[rb];
                const int at = used0 + 2 * i;
                if (at + 2 <= ucount) uu = words_to_double(wb[at], wb[at + 1]);
            } else if (i < ucount) {
                uu = uniforms[u_off[rb] + i];
            }
            S.uni[i] = uu;
        }
    }
    int draws = 0;   // meaningful in thread 0
    const int nl = R / 2;
    const FastRec FR = fast_rec_const(R, P.step, P.fov0, P.fov1);
    int* const lst[2] = {S.lst, S.lst + maxN};
    int* const clsb[2] = {S.cls, S.cls2};
    int* const lst_n = S.cnt + 4;
    // Pipeline over the agents in id order.  Agent m's field depends on the
    // agents moved before it only through their records.  So while thread 0
    // moves agent k and then adds agent k's class (and record) for agent
    // k+1, wave 1 builds agent k+1's records of every other obstacle, and
    // the other waves classify agent k+2's obstacles but k and k+1; one of
    // them then builds agent k+1's speculative headings and the next agent
    // k+2's focal geometry (agents move only in their own turn, so it is the
    // start-of-step pose).  After one barrier come exclusion, raster and
    // counts of agent k+1, during which wave 2 adds agent k's class for
    // agent k+2.
    // Classes, lists, focal geometry and counts alternate between two
    // buffers by parity of the focal agent.
    const int rbase = 64, cbase = 128, cstride = nthr - 128;   // blockDim 512
    if (tid == 0) {
        for (int q = 0; q < 8; ++q) S.cnt[q] = 0;
    }
    for (int w = tid; w < P.words; w += nthr) reinterpret_cast<uint32_t*>(S.V)[w] = 0u;
    __syncthreads();
    // ---- agent 0's field; agent 1's classes but agent 0's; agent 0's
    // speculative headings (slot 0, draw index 0)
    // two waves that classify once per focal agent also build the
    // speculative headings and the focal geometry: waves 4 and 5 of eight
    // (waves 2 and 3 classify twice for 512 agents)
    const int spec_tid = 256, focal_tid = spec_tid + 64;
    if (tid >= spec_tid && tid < spec_tid + 3) spec_heading(S, P, N, 0, 0, tid - spec_tid, S.spec);
    if (tid == 0) S.spec[24] = 0.0;    // uniforms drawn before agent 0
    if (tid == 0) S.focal[0] = focal_of(S, 0);
    if (tid == cbase && N > 1) S.focal[1] = focal_of(S, 1);
    classify(S, P, N, 0, -1, -1, clsb[0], lst[0], &lst_n[0], tid, nthr);
    if (N > 1) classify(S, P, N, 1, 0, -1, clsb[1], lst[1], &lst_n[1], tid, nthr);
    __syncthreads();
    for (int q = tid; q < lst_n[0]; q += nthr) {
        const int j = lst[0][q];
        S.rec[j] = record_of(S, j, clsb[0][j], N, S.focal[0], R, P.step, P.fov0, P.fov1, FR, true);
    }
    __syncthreads();
    raster_list(S, R, lst[0], lst_n[0], -1);
    if (tid == 0) lst_n[0] = 0;   // rebuilt for agent 2
    count_field(S, P, R, S.cnt, bits_out, 0);
    __syncthreads();

    // wave 0 carries the chain of moves: first issue on its SIMD
    if (tid < 64) __builtin_amdgcn_s_setprio(3);
    for (int k = 0; k < N; ++k) {
        const int f1 = k + 1, par = f1 & 1, f2 = k + 2, par2 = par ^ 1;
        const int n_set = S.cnt[2 * (k & 1)], n_left = S.cnt[2 * (k & 1) + 1];
        // ---- decision and motion (agent.py:168-283)
        if (tid == 0) {
            // every LDS operand first, in one batch: the replica's constants
            // and agent k's state (the loads then wait once, not in turn)
            const double T_w = P.T_w, Eps_w = P.Eps_w, g_w = P.g_w, B_w = P.B_w, w_max = P.w_max;
            const double T_u = P.T_u, Eps_u = P.Eps_u, g_u = P.g_u, B_u = P.B_u, u_max = P.u_max;
            const double S_wu = P.S_wu, S_uw = P.S_uw, F_N = P.F_N, F_R = P.F_R;
            const double vmax = P.exp_vel_max, rtmax = P.reloc_theta_max, stop = P.exp_stop_ratio;
            const double pad = P.pad, width = P.width, height = P.height;
            double w = S.w[k], u = S.u[k];
            const double vel0 = S.v[k], cr = S.cr[k], crb = S.crb[k], nov = S.nov[k];
            const double x0 = S.x[k], y0 = S.y[k], th0 = S.th[k], rad = S.rad[k];
            int over = S.over[k], mode = S.mode[k];
            const int env = S.env[k];
            const double* spec = S.spec + 12 * (k & 1);
            const double spec_d = spec[9];
            asm volatile("" ::: "memory");
            const double count = (double)n_set, cleft = (double)n_left;
            const double collected = cr - crb;
            const double ipriv = F_N * nov + F_R * collected;
            const double w_p = w > T_w ? w : 0.0;
            const double u_p = u > T_u ? u : 0.0;
            const double mean = count / (double)R;
            const double dw = Eps_w * mean - g_w * (w - B_w) - u_p * S_uw;
            const double du = Eps_u * ipriv - g_u * (u - B_u) - w_p * S_wu;
            w = w + dw;
            u = u + du;
            if (w > w_max) w = w_max;
            if (w < -w_max) w = -w_max;
            if (u > u_max) u = u_max;
            if (u < -u_max) u = -u_max;
            double dvel = 0.0, dth = 0.0;
            int slot = 2;   // speculative heading: 2 = no turn, 0 / 1 = walk, -1 = relocation
            const bool tw = w > T_w, tu = u > T_w;   // tr_u compares with T_w
            auto walk = [&]() {
                slot = draws - (int)spec_d;   // the uniform drawn: S.uni[draws]
                ++draws;
                dvel = vmax;
                over = -1; mode = ABM_MODE_EXPLORE;
            };
            auto reloc = [&]() {
                const double lm = cleft / (double)nl;
                const double rm = (count - cleft) / (double)(R - nl);
                dvel = vmax - vel0;
                dth = (lm - rm) * rtmax;
                slot = -1;
                over = -1; mode = ABM_MODE_RELOCATE;
            };
            auto exploit = [&]() {
                over = ABM_MODE_EXPLOIT; mode = ABM_MODE_EXPLOIT;
                dvel = -vel0 * stop;
                dth = 0.0;
            };
            if (over != ABM_MODE_COLLIDE) {   // get_mode() == "collide" only via the override
                if (!tw && !tu) walk();
                else if (tw && tu) { if (env == 1) exploit(); else reloc(); }
                else if (tw && !tu) reloc();
                else { if (env == 1) exploit(); else walk(); }
            }
            Pose p{x0, y0, th0, vel0};
            double sn, cs;
            if (slot < 0) {
                p.theta = prove_orientation(p.theta + dth);
                sincos(p.theta, &sn, &cs);
            } else {   // prove_orientation(theta + turn) and its sin, cos from the spare wave
                p.theta = spec[3 * slot];
                sn = spec[3 * slot + 1];
                cs = spec[3 * slot + 2];
            }
            p.v = p.v + dvel;
            // prove_velocity (agent.py:612-620): only in explore mode
            if (get_mode(over, w, T_w) == ABM_MODE_EXPLORE && fabs(p.v) > 1.0) p.v = vmax;
            p.x = p.x + p.v * cs;
            p.y = p.y - p.v * sn;
            p = reflect_walls(p, rad, pad, width, height);
            S.x[k] = p.x; S.y[k] = p.y; S.th[k] = p.theta; S.v[k] = p.v;
            S.w[k] = w; S.u[k] = u; S.over[k] = over; S.mode[k] = mode;
            S.crb[k] = cr;
            S.nov[k] = ipriv;   // read only by agent k's decision: now its I_priv
            S.spec[24 + (f1 & 1)] = (double)draws;   // uniforms drawn before agent k+1
        }
        // ---- thread 0, after the move: agent k's class and record for agent k+1
        if (tid == 0 && f1 < N) {
            const double cfx = S.x[f1] + S.rad[f1], cfy = S.y[f1] + S.rad[f1];
            const int c = cue_class(S, P, k, f1, cfx, cfy, S.pid[f1]);
            if (c != kNone) S.rec[k] = record_of(S, k, c, N, S.focal[par], R, P.step, P.fov0, P.fov1, FR, true);
            S.cnt[6] = c != kNone ? k : -1;
            S.cnt[2 * par] = 0; S.cnt[2 * par + 1] = 0;   // agent k+1's counts (last read by k-1)
        }
        // ---- wave 1: agent k+1's records but agent k's
        if (f1 < N && tid >= rbase && tid < cbase) {
            uint32_t* Vb = reinterpret_cast<uint32_t*>(S.V);
            for (int w = tid - rbase; w < P.words; w += 64) Vb[w] = 0u;
            const Focal f = S.focal[par];
            const int n = lst_n[par];
            for (int q = tid - rbase; q < n; q += 64) {
                const int j = lst[par][q];
                S.rec[j] = record_of(S, j, clsb[par][j], N, f, R, P.step, P.fov0, P.fov1, FR, true);
            }
        }
        // ---- waves 2 to 7: agent k+2's classes but agent k's and k+1's
        if (f2 < N && tid >= cbase)
            classify(S, P, N, f2, k, f1, clsb[par2], lst[par2], &lst_n[par2], tid - cbase, cstride);
        // ---- one classifying wave, then: agent k+1's speculative headings,
        // from the uniforms drawn before agent k
        if (f1 < N && tid >= spec_tid && tid < spec_tid + 3)
            spec_heading(S, P, N, f1, (int)S.spec[24 + (k & 1)], tid - spec_tid, S.spec + 12 * par);
        // ---- the next wave, then: agent k+2's focal geometry (its
        // start-of-step pose: agents move only in their own turn); that
        // buffer was last read for agent k
        if (tid == focal_tid && f2 < N) S.focal[par2] = focal_of(S, f2);
        __syncthreads();
        if (f1 >= N) break;
        // ---- exclusion, raster and counts of agent k+1; meanwhile wave 2
        // adds agent k's class for agent k+2
        raster_list(S, R, lst[par], lst_n[par], S.cnt[6]);
        if (tid == 0) lst_n[par] = 0;   // rebuilt for agent k+3
        if (tid == cbase && f2 < N) {   // agent k's class for agent k+2; its record comes with the others
            const double gx = S.x[f2] + S.rad[f2], gy = S.y[f2] + S.rad[f2];
            const int c2 = cue_class(S, P, k, f2, gx, gy, S.pid[f2]);
            clsb[par2][k] = c2;
            if (c2 != kNone) {
                lst[par2][lst_n[par2]] = k;
                lst_n[par2] += 1;
            }
        }
        count_field(S, P, R, S.cnt + 2 * par, bits_out, f1);
        __syncthreads();
    }
    for (int i = tid; i < N; i += nthr) {
        const int g = a0 + i;
        st.x[g] = S.x[i]; st.y[g] = S.y[i]; st.theta[g] = S.th[i]; st.v[g] = S.v[i];
        st.w[g] = S.w[i]; st.u[g] = S.u[i]; st.collected_r_before[g] = S.crb[i];
        st.mode[g] = S.mode[i]; st.overriding_mode[g] = S.over[i];
        st.I_priv[g] = S.nov[i];
    }
    if (tid == 0 && u_used) u_used[rb] = used0 + (words || mt ? 2 : 1) * draws;
    if (tid == 0 && status) status[rb] = ABM_WORLD_DONE;
    if (mt) {
        // advance the generator by the 2 * draws words used: numpy's state
        // after them is the key twisted v times at position pos0 + c - 624 v
        if (tid == 0) S.cnt[7] = draws;
        __syncthreads();
        const int c = 2 * S.cnt[7];
        int v = 0, pos = mt_pos0 + c;
        if (pos > kMtN) {
            v = (pos - 1) / kMtN;
            pos -= kMtN * v;
        }
        if (v > 0) {
            for (int i = tid; i < kMtN; i += nthr) S.mtk[i] = mt[rb].key[i];
            __syncthreads();
            for (int t = 0; t < v; ++t) mt_twist_block(S.mtk);
            for (int i = tid; i < kMtN; i += nthr) mt[rb].key[i] = S.mtk[i];
        }
        if (tid == 0) mt[rb].pos = pos;
    }
}

// ------------------------------------------------ update without visual exclusion
// Agent.update in id order (sims.py:861) without visual exclusion needs no
// id-order chain.  Agent k reads the agents before it (already moved) and
// after it (not yet) only as social cues, and what makes agent j a cue -- its
// overriding mode exploit, its patch id and its position -- does not depend on
// j's own field: the update leaves j exploiting exactly when u' > T_w with
// env_status 1 (agent.py:215-283: the exploit branches; u' comes from I_priv,
// u and the old w, agent.py:168-199), its patch id is never changed, and an
// exploiting agent keeps its heading and slows by a fixed ratio.  So every
// agent's moved cue is known before any field is, and all fields of a replica
// are built at once: agent k's from the cues j < k as moved and j > k as they
// started.  Only the walks' draw indices follow the id order (a scan of
// flags).  A collide override (kept by the update) is never a cue.

// u and I_priv after the update (agent.py:168-199), and whether the update
// leaves the agent exploiting.
struct Drive {
    double u, ipriv;
    bool exploit;
};
__device__ inline Drive drive_of(const FGRep& P, double w, double u, double nov, double cr, double crb,
                                 int over, int env) {
#pragma clang fp contract(off)
    Drive q;
    const double collected = cr - crb;
    q.ipriv = P.F_N * nov + P.F_R * collected;
    const double w_p = w > P.T_w ? w : 0.0;
    const double du = P.Eps_u * q.ipriv - P.g_u * (u - P.B_u) - w_p * P.S_wu;
    u = u + du;
    if (u > P.u_max) u = P.u_max;
    if (u < -P.u_max) u = -P.u_max;
    q.u = u;
    q.exploit = over != ABM_MODE_COLLIDE && u > P.T_w && env == 1;   // tr_u compares with T_w
    return q;
}

// The decision of an agent (agent.py:168-283): its new w, modes, speed and
// heading increments; kind 0 draws a walk turn.
struct Choice {
    double w, dth, dvel;
    int over, mode, kind;
};
__device__ inline Choice choose(const FGRep& P, int R, int n_set, int n_left, double w, double u0, double u1,
                                double vel0, int over, int mode, int env) {
#pragma clang fp contract(off)
    Choice c;
    const int nl = R / 2;
    const double count = (double)n_set, cleft = (double)n_left;
    const double u_p = u0 > P.T_u ? u0 : 0.0;
    const double mean = count / (double)R;
    const double dw = P.Eps_w * mean - P.g_w * (w - P.B_w) - u_p * P.S_uw;
    w = w + dw;
    if (w > P.w_max) w = P.w_max;
    if (w < -P.w_max) w = -P.w_max;
    c.w = w; c.dth = 0.0; c.dvel = 0.0; c.over = over; c.mode = mode; c.kind = 1;
    if (over == ABM_MODE_COLLIDE) return c;   // get_mode() == "collide" only via the override
    const bool tw = w > P.T_w, tu = u1 > P.T_w;   // tr_u compares with T_w
    if (tu && env == 1) {
        c.over = ABM_MODE_EXPLOIT; c.mode = ABM_MODE_EXPLOIT;
        c.dvel = -vel0 * P.exp_stop_ratio;
    } else if (tw) {   // relocation towards the fuller half of the field
        const double lm = cleft / (double)nl;
        const double rm = (count - cleft) / (double)(R - nl);
        c.dvel = P.exp_vel_max - vel0;
        c.dth = (lm - rm) * P.reloc_theta_max;
        c.over = -1; c.mode = ABM_MODE_RELOCATE;
    } else {
        c.dvel = P.exp_vel_max;
        c.over = -1; c.mode = ABM_MODE_EXPLORE; c.kind = 0;
    }
    return c;
}

// The move (agent.py:200-283, 595-620): heading turned by dth, speed by
// dvel, limited in explore mode only, one Euler step, the walls.
__device__ inline Pose fg_move(const FGRep& P, Pose p, double dth, double dvel, int over, double w, double rad) {
#pragma clang fp contract(off)
    p.theta = prove_orientation(p.theta + dth);
    double sn, cs;
    sincos(p.theta, &sn, &cs);
    p.v = p.v + dvel;
    if (get_mode(over, w, P.T_w) == ABM_MODE_EXPLORE && fabs(p.v) > 1.0) p.v = P.exp_vel_max;
    p.x = p.x + p.v * cs;
    p.y = p.y - p.v * sn;
    return reflect_walls(p, rad, P.pad, P.width, P.height);
}

// supcalc.distance <= vision_range of two centres: decided on the squared
// distance outside a band far wider than its rounding, else by the norm.
struct RangeTest {
    double vr, lo, hi;
};
__device__ inline RangeTest range_test(double vr) {
    RangeTest t;
    t.vr = vr;
    t.lo = vr > 0.0 ? vr * vr * (1.0 - 1e-9) : -1.0;
    t.hi = vr > 0.0 ? vr * vr * (1.0 + 1e-9) : HUGE_VAL;
    return t;
}
__device__ inline bool in_range(const RangeTest& t, double dx, double dy) {
#pragma clang fp contract(off)
    const double d2 = dx * dx + dy * dy;
    if (d2 <= t.lo) return true;
    if (d2 >= t.hi) return false;
    return norm2(dx, dy) <= t.vr;
}

// Raw bits V[lo .. lo + 31] of a field of W words (zero outside it).
__device__ inline uint32_t raw_window(const uint32_t* V, int W, int lo) {
    const int w = lo >> 5, sh = lo & 31;
    const uint32_t a = w >= 0 && w < W ? V[w] : 0u;
    if (sh == 0) return a;
    const uint32_t b = w + 1 >= 0 && w + 1 < W ? V[w + 1] : 0u;
    return (a >> sh) | (b << (32 - sh));
}

// Counts of a wave's raw field on the kept rays and on their left half, to
// every lane, and (dst not null) the returned field: soc_v_field[q] =
// V[R - 1 - q] on the kept rays (agent.py:593-595), a word of it being a raw
// window reversed.
__device__ inline void wave_counts(const uint32_t* V, int R, int W, int keep_lo, int keep_hi, uint32_t* dst,
                                   int* n_set, int* n_left) {
    const int lane = threadIdx.x & 63;
    const int nl = R / 2, ta = R - 1 - keep_hi, tb = R - 1 - keep_lo, la = max(R - nl, ta);
    int tot = 0, left = 0;
    for (int w = lane; w < W; w += 64) {
        const uint32_t bits = V[w];
        tot += __popc(bits & word_range_mask(w, ta, tb));
        left += __popc(bits & word_range_mask(w, la, tb));
        if (dst) dst[w] = __brev(raw_window(V, W, R - 32 - 32 * w)) & word_range_mask(w, keep_lo, keep_hi);
    }
    if (R < 32768) {   // one sum of both counts
        const int both = wave_sum(tot << 16 | left);
        *n_set = both >> 16;
        *n_left = both & 0xffff;
    } else {
        *n_set = wave_sum(tot);
        *n_left = wave_sum(left);
    }
}

// LDS of the update kernel: the replica's agents at the step's start, their
// moved poses where they are cues, and one raw field per wave.
struct UpdSmem {
    double *x, *y, *th, *v, *w, *u0, *u1, *ip, *cr, *u1x, *u1y, *xm, *ym;
    int *rad, *pid, *over, *mode, *env, *flag, *cue, *nset, *nleft, *idx;
    uint32_t *words, *key, *field;
    int *wtot, *ctl;
};
constexpr int kUpdDoubles = 13, kUpdInts = 10, kUpdWaves = 16;

__device__ inline UpdSmem upd_carve(void* base, int maxN) {
    UpdSmem s;
    char* p = reinterpret_cast<char*>(base);
    double** d[] = {&s.x, &s.y, &s.th, &s.v, &s.w, &s.u0, &s.u1, &s.ip, &s.cr, &s.u1x, &s.u1y, &s.xm, &s.ym};
    for (double** a : d) { *a = reinterpret_cast<double*>(p); p += sizeof(double) * maxN; }
    s.words = reinterpret_cast<uint32_t*>(p); p += sizeof(uint32_t) * 2 * maxN;
    int** i[] = {&s.rad, &s.pid, &s.over, &s.mode, &s.env, &s.flag, &s.cue, &s.nset, &s.nleft, &s.idx};
    for (int** a : i) { *a = reinterpret_cast<int*>(p); p += sizeof(int) * maxN; }
    s.key = reinterpret_cast<uint32_t*>(p); p += sizeof(uint32_t) * kMtN;
    s.wtot = reinterpret_cast<int*>(p); p += sizeof(int) * 2 * kUpdWaves;
    s.ctl = reinterpret_cast<int*>(p); p += sizeof(int) * 4;
    s.field = reinterpret_cast<uint32_t*>(p);
    return s;
}

size_t upd_lds_bytes(int maxN, int maxR, int waves) {
    return (size_t)maxN * (8 * kUpdDoubles + 8 + 4 * kUpdInts) + 4 * (kMtN + 2 * kUpdWaves + 4) +
           sizeof(uint32_t) * (size_t)waves * ((maxR + 31) / 32) + 16;
}

// What an agent is as a cue (UpdSmem.flag): where it started, and once moved.
constexpr int kCueStart = 1, kCueMoved = 2;

// One workgroup per replica, largest first.  Threads over agents: the drive,
// the focal geometry and the moved pose of every cue; one wave per agent: its
// cues' records (64 at a time, one per lane) ORed into the wave's raw field
// (each interval is a few words: LDS atomics) and the counts; threads over
// agents: the choice, the draw indices (a scan), the walk's words, the move.
// Bound by the waves' records and their raster (64 cues at a time) for large
// replicas, by the phases' latency for small ones.  Against the id-order chain
// (one agent at a time, its cues' intervals spread over the lanes one by one):
// 1000 replicas of 8 to 512 agents, a tenth of them cues, 3.95 ms -> 0.102 ms;
// one replica of 10 agents 26.6 us -> 9.1 us.
template <bool FIELDS>
__global__ void __launch_bounds__(1024)
forage_update_kernel(const FGRep* __restrict__ reps, abm_forage_state st,
                     const double* __restrict__ uniforms, const uint32_t* __restrict__ words,
                     const int64_t* __restrict__ u_off, const int32_t* __restrict__ u_cnt,
                     int32_t* __restrict__ u_used, int32_t* __restrict__ status,
                     uint32_t* __restrict__ bits_out, const int32_t* __restrict__ order,
                     abm_mt19937_state* __restrict__ mt, int maxN) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) double smem[];
    const int rb = order[blockIdx.x];
    if (status && status[rb] != kWorldReady) return;   // uniform over the block
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = nthr >> 6;
    __shared__ FGRep sP;
    if (tid < (int)(sizeof(FGRep) / 8))
        reinterpret_cast<uint64_t*>(&sP)[tid] = reinterpret_cast<const uint64_t*>(reps + rb)[tid];
    const UpdSmem S = upd_carve(smem, maxN);
    if (tid == 0) S.ctl[0] = 0;
    int mt_pos0 = 0;
    if (mt) {
        for (int i = tid; i < kMtN; i += nthr) S.key[i] = mt[rb].key[i];
        mt_pos0 = mt[rb].pos;
    }
    const int ucount = mt ? 0 : u_cnt[rb];
    const int used0 = (words || mt) ? u_used[rb] : 0;
    __syncthreads();
    const FGRep& P = sP;
    const int N = P.n_agents, R = P.n_rays, W = P.words, a0 = P.agent_offset, tau = P.tau;
    // ---- the agents, their drives and the cues
    for (int base = tid - lane; base < N; base += nthr) {
        const int i = base + lane;
        int flag = 0;
        if (i < N) {
            const int g = a0 + i;
            const double x = st.x[g], y = st.y[g], th = st.theta[g], v = st.v[g], w = st.w[g], u = st.u[g];
            const double cr = st.collected_r[g], crb = st.collected_r_before[g];
            const int rad = st.radius[g], over = st.overriding_mode[g], mode = st.mode[g];
            const int env = st.env_status[g], pid = st.exploited_patch_id[g];
            double m = st.novelty[(int64_t)g * tau];
            for (int q = 1; q < tau; ++q) m = fmax(m, st.novelty[(int64_t)g * tau + q]);
            const Drive d = drive_of(P, w, u, m, cr, crb, over, env);
            S.x[i] = x; S.y[i] = y; S.th[i] = th; S.v[i] = v; S.w[i] = w; S.u0[i] = u; S.u1[i] = d.u;
            S.ip[i] = d.ipriv; S.cr[i] = cr; S.rad[i] = rad; S.pid[i] = pid; S.over[i] = over;
            S.mode[i] = mode; S.env[i] = env;
            const Focal f = focal_at(x, y, th, (double)rad);
            S.u1x[i] = f.u1x; S.u1y[i] = f.u1y;
            if (pid != -1) {
                if (over == ABM_MODE_EXPLOIT) flag |= kCueStart;
                if (d.exploit) {
                    flag |= kCueMoved;
                    const Pose p = fg_move(P, Pose{x, y, th, v}, 0.0, -v * P.exp_stop_ratio, ABM_MODE_EXPLOIT,
                                           w, (double)rad);
                    S.xm[i] = p.x; S.ym[i] = p.y;
                }
            }
            S.flag[i] = flag;
        }
        const uint64_t m = __ballot(flag != 0);
        if (m) {
            int at = 0;
            if (lane == 0) at = atomicAdd(&S.ctl[0], (int)__popcll(m));
            at = __builtin_amdgcn_readfirstlane(at);
            if (flag) S.cue[at + (int)__popcll(m & ((1ull << lane) - 1ull))] = i;
        }
    }
    __syncthreads();
    // ---- the fields
    const int n_cue = S.ctl[0];
    {
        const FastRec FR = fast_rec_const(R, P.step, P.fov0, P.fov1);
        const RangeTest rt = range_test(P.vision_range);
        const int keep_lo = P.keep_lo, keep_hi = P.keep_hi, patchwise = P.patchwise;
        const double step = P.step, fov0 = P.fov0, fov1 = P.fov1;
        uint32_t* V = S.field + wave * W;
        for (int k = wave; k < N; k += nw) {
            int n_set = 0, n_left = 0;
            if (n_cue > 0) {
                for (int w = lane; w < W; w += 64) V[w] = 0u;
                fg_wave_sync();
                Focal f;
                f.radius = (double)S.rad[k];
                f.px = S.x[k]; f.py = S.y[k];
                f.cx = f.px + f.radius;
                f.cy = f.py + f.radius;
                f.u1x = S.u1x[k]; f.u1y = S.u1y[k];
                const int pid_k = S.pid[k];
                for (int q = lane; q < n_cue; q += 64) {
                    const int j = S.cue[q];
                    const int pid = S.pid[j];
                    const bool moved = j < k;
                    // agent.py:396-413: an exploiting agent in range with a
                    // patch other than the focal's own (patchwise exclusion)
                    if (j == k || !(S.flag[j] & (moved ? kCueMoved : kCueStart)) || (patchwise && pid == pid_k))
                        continue;
                    const double ox = moved ? S.xm[j] : S.x[j], oy = moved ? S.ym[j] : S.y[j];
                    const double rj = (double)S.rad[j];
                    if (!in_range(rt, (ox + rj) - f.cx, (oy + rj) - f.cy)) continue;
                    const Rec rc = record_at(ox, oy, kSocial, j, f, R, step, fov0, fov1, FR, false);
                    if (rc.valid) paint_bits(V, rc, R);
                }
                fg_wave_sync();
                wave_counts(V, R, W, keep_lo, keep_hi, FIELDS ? bits_out + P.field_offset + (int64_t)k * W : nullptr,
                            &n_set, &n_left);
                fg_wave_sync();
            } else if (FIELDS) {
                uint32_t* dst = bits_out + P.field_offset + (int64_t)k * W;
                for (int w = lane; w < W; w += 64) dst[w] = 0u;
            }
            if (lane == 0) { S.nset[k] = n_set; S.nleft[k] = n_left; }
        }
    }
    __syncthreads();
    // ---- the walks' draw indices, in id order
    int draws = 0;
    for (int c0 = 0, par = 0; c0 < N; c0 += nthr, par ^= 1) {
        const int k = c0 + tid;
        int kind = 1;
        if (k < N)
            kind = choose(P, R, S.nset[k], S.nleft[k], S.w[k], S.u0[k], S.u1[k], S.v[k], S.over[k], S.mode[k],
                          S.env[k]).kind;
        const uint64_t m = __ballot(kind == 0);
        if (lane == 0) S.wtot[kUpdWaves * par + wave] = (int)__popcll(m);
        __syncthreads();   // a half of wtot is rewritten two chunks later, after this chunk's barrier
        int d = draws + (int)__popcll(m & ((1ull << lane) - 1ull));
        for (int w = 0; w < nw; ++w) {
            const int t = S.wtot[kUpdWaves * par + w];
            if (w < wave) d += t;
            draws += t;
        }
        if (k < N) S.idx[k] = d;
    }
    // ---- the walks' words from the replica's device generator: exactly the
    // 2 * draws it consumes, so the key left is numpy's (which twists lazily,
    // when a word is drawn at position 624)
    if (mt) {
        int made = 0, p = mt_pos0, twists = 0;
        while (made < 2 * draws) {
            if (p >= kMtN) {
                mt_twist_block(S.key);
                ++twists;
                p = 0;
            }
            const int take = min(kMtN - p, 2 * draws - made);
            for (int j = tid; j < take; j += nthr) S.words[made + j] = mt_temper(S.key[p + j]);
            made += take;
            p += take;
        }
        __syncthreads();
        if (twists > 0)
            for (int i = tid; i < kMtN; i += nthr) mt[rb].key[i] = S.key[i];
        if (tid == 0) mt[rb].pos = p;
    }
    // ---- the moves (each thread its own agents of the scan)
    for (int k = tid; k < N; k += nthr) {
        const int g = a0 + k;
        const double vel0 = S.v[k];
        const Choice c = choose(P, R, S.nset[k], S.nleft[k], S.w[k], S.u0[k], S.u1[k], vel0, S.over[k], S.mode[k],
                                S.env[k]);
        double dth = c.dth;
        if (c.kind == 0) {
            // agent k's draw: doubles, or pairs of words after those the
            // resource loop used; NaN past the end of the buffer
            const int d = S.idx[k];
            double uu = NAN;
            if (mt) {
                uu = words_to_double(S.words[2 * d], S.words[2 * d + 1]);
            } else if (words) {
                const uint32_t* wb = words + u_off[rb];
                const int at = used0 + 2 * d;
                if (at + 2 <= ucount) uu = words_to_double(wb[at], wb[at + 1]);
            } else if (d < ucount) {
                uu = uniforms[u_off[rb] + d];
            }
            dth = P.exp_theta_min + (P.exp_theta_max - P.exp_theta_min) * uu;
        }
        const Pose p = fg_move(P, Pose{S.x[k], S.y[k], S.th[k], vel0}, dth, c.dvel, c.over, c.w, (double)S.rad[k]);
        st.x[g] = p.x; st.y[g] = p.y; st.theta[g] = p.theta; st.v[g] = p.v;
        st.w[g] = c.w; st.u[g] = S.u1[k]; st.collected_r_before[g] = S.cr[k];
        st.mode[g] = c.mode; st.overriding_mode[g] = c.over;
        st.I_priv[g] = S.ip[k];
    }
    if (tid == 0 && u_used) u_used[rb] = used0 + (words || mt ? 2 : 1) * draws;
    if (tid == 0 && status) status[rb] = ABM_WORLD_DONE;
}

// ------------------------------------------------ update with visual exclusion
// Agent.update in id order (sims.py:861) with visual exclusion: every agent in
// range, as it stands in agent k's turn, may occlude the others, so agent k + 1's
// field waits for agent k's move.  But only for the one record of agent k: the
// rest of the field is known a turn earlier.  Wave 0 carries the chain alone
// (decide and move agent k, its record in agent k + 1's view, what it occludes,
// the counts of agent k + 1's field) and the other H = 7 waves prepare the fields,
// each that of every 7th agent over the 7 turns before its own:
//   turn 0      the focal geometry and the records of the agents that will
//               not move before the focal agent does (a lane each)
//   turns 1, 2  how many of them are nearer than each
//   turns 3, 4  which nearer ones overlap each; the headings after a walk turn
//   turn 5      the records of the agents moved meanwhile, one by one
//   turn 6      the last but one's, the visible intervals, the field: to wave 0
// One barrier a turn.  A record's visible interval is cut by the nearer records
// in the order of their distance (agent.py:421-445); one that does not overlap it
// cuts nothing, so the walk goes over the others alone (few: the agents along
// one line of sight), and agent k's record changes only the intervals it overlaps.
// Bound by the chain's latency (about 4.0 thousand cycles a turn of 5.7 with 40
// agents: 1.9 decision and move, 1.0 record, 0.5 cuts, 0.5 counts), beyond 64
// agents by the preparing waves (12 thousand a turn with 80).  Against one
// kernel that ranked and cut all records between two agents' moves (still the one
// beyond 256 agents, where K would not fit in registers), ms a step: 200 replicas
// of 10 to 40 agents at R = 600 0.72 -> 0.134, 1000 of 10 to 64 1.68 -> 0.226,
// 700 of 80 5.23 -> 0.87, 20 of 250 24.3 -> 4.0, one of 10 0.085 -> 0.040.
// K <= 2 is held to 128 registers, so that two workgroups share a CU (700 of 80:
// 1.15 with one; 50 of 80 then take 0.495 instead of 0.472).
constexpr int kOcclMaxAgents = 256;   // K = 1, 2 or 4 records per lane

// A focal agent's records, K per lane (record j in lane j & 63, slot j >> 6):
// bins, distance, place in the reference's obstacle list, rank by distance
// (equal ones by place) and the nearer records that overlap it, a bit each.
// A record that a nearer one covers from end to end is hidden, whatever else
// cuts it (its interval only shrinks): its set is not needed.
template <int K>
struct Seen {
    int start[K], end[K], ord[K];   // ord: place, negative: no record
    int rank[K];                    // place by (distance, ord)
    int below[K];                   // nearer records
    int hid[K];                     // negative: hidden
    double dist[K];                 // no record: NaN, neither nearer nor as near as any
    uint32_t over[K][2 * K];        // [slot of the record][32 of the nearer ones]
};
struct OcclRec {                    // a record as the other records meet it
    double dist;
    int ord, start, end;
};

// LDS of the kernel: the agents, and by parity of the focal agent the records
// handed to wave 0.
struct OcclSmem {
    double *x, *y, *rad, *th, *v, *w, *u0, *u1, *ip, *uni;
    double* spec;      // [kOcclSpec q ..]: prepared headings, by agent mod 4; [4 kOcclSpec + p]: uniforms drawn before
    double* dist;      // the handed records, by rank: [64 K p ..]
    uint64_t* over;    // [64 K K p + 64 K c ..]: nearer records of rank 64 c .. that overlap
    int2 *span, *cut;  // [64 K p ..]: bins, and after exclusion
    int* ord;          // [64 K p ..]: place, + kOrdHidden
    int4* rec;         // [64 K h ..]: preparing wave h's records of its focal's first turn: below, start, end, ord
    double* rdist;     // [64 K h ..]: their distances
    int* rank;         // [64 K h ..]: their ranks when handed over
    Focal* focal;      // [wave]
    int *pid, *mode_over, *mode, *env, *kept;
    uint32_t* key;
    uint32_t* field;   // [4][W]: raw fields by focal agent mod 4
};
constexpr int kOcclDoubles = 10, kOcclInts = 4;
constexpr int kOrdHidden = 1 << 30;
constexpr int kOcclSpec = 16;   // four turns' headings and none's (each with sin, cos), the first's draw
constexpr int kOcclWaves = 8, kOcclPrep = kOcclWaves - 1;

__device__ inline OcclSmem occl_carve(void* base, int maxN, int K) {
    OcclSmem s;
    const int L = 128 * K;
    char* p = reinterpret_cast<char*>(base);
    s.focal = reinterpret_cast<Focal*>(p); p += 64 * kOcclWaves;
    s.rec = reinterpret_cast<int4*>(p); p += sizeof(int4) * 64 * K * kOcclPrep;
    s.rdist = reinterpret_cast<double*>(p); p += sizeof(double) * 64 * K * kOcclPrep;
    double** d[] = {&s.x, &s.y, &s.rad, &s.th, &s.v, &s.w, &s.u0, &s.u1, &s.ip, &s.uni};
    for (double** a : d) { *a = reinterpret_cast<double*>(p); p += sizeof(double) * maxN; }
    s.spec = reinterpret_cast<double*>(p); p += sizeof(double) * (4 * kOcclSpec + 2);
    s.dist = reinterpret_cast<double*>(p); p += sizeof(double) * L;
    s.over = reinterpret_cast<uint64_t*>(p); p += sizeof(uint64_t) * L * K;
    s.span = reinterpret_cast<int2*>(p); p += sizeof(int2) * L;
    s.cut = reinterpret_cast<int2*>(p); p += sizeof(int2) * L;
    s.ord = reinterpret_cast<int*>(p); p += sizeof(int) * L;
    s.rank = reinterpret_cast<int*>(p); p += sizeof(int) * 64 * K * kOcclPrep;
    int** i[] = {&s.pid, &s.mode_over, &s.mode, &s.env};
    for (int** a : i) { *a = reinterpret_cast<int*>(p); p += sizeof(int) * maxN; }
    s.kept = reinterpret_cast<int*>(p); p += sizeof(int) * 2;
    s.key = reinterpret_cast<uint32_t*>(p); p += sizeof(uint32_t) * kMtN;
    s.field = reinterpret_cast<uint32_t*>(p);
    return s;
}

size_t occl_lds_bytes(int maxN, int maxR, int K) {
    return 64 * (size_t)kOcclWaves + (size_t)maxN * (8 * kOcclDoubles + 4 * kOcclInts) + 8 * (4 * kOcclSpec + 2) +
           (size_t)128 * K * (8 + 8 * K + 8 + 8 + 4) + (size_t)64 * K * kOcclPrep * (16 + 8 + 4) +
           4 * (kMtN + 2) + 4 * sizeof(uint32_t) * (size_t)((maxR + 31) / 32);
}

__device__ inline int occl_class(const OcclSmem& S, int patchwise, const RangeTest& rt, int j, double cfx, double cfy,
                                 int pid_f) {
    if (!in_range(rt, (S.x[j] + S.rad[j]) - cfx, (S.y[j] + S.rad[j]) - cfy)) return kNone;
    if (S.mode_over[j] != ABM_MODE_EXPLOIT) return kNonExpl;   // get_mode() == "exploit" only via the override
    if (patchwise && S.pid[j] == pid_f) return kSamePatch;
    return S.pid[j] != -1 ? kSocial : kNone;
}

// A record's visible interval after nearer ones (agent.py:421-445): those of
// rank 64 c + (bit of m), nearest first.
struct Interval {
    int s, e;
};
__device__ inline bool cut_by(Interval& v, int2 i) {   // false: nothing is left to cut
    if (v.s <= i.x && i.x <= v.e) v.e = i.x;
    if (v.s <= i.y && i.y <= v.e) v.s = i.y;
    const bool covered = i.x <= v.s && i.y >= v.e;
    if (covered) v.s = v.e = 0;   // (no record moves an interval from there)
    return !covered;
}
__device__ inline bool cut_by_all(Interval& v, uint64_t m, const int2* span) {
    if (!m) return true;
    int2 i = span[__builtin_ctzll(m)];
    for (m &= m - 1; m; m &= m - 1) {
        const int2 next = span[__builtin_ctzll(m)];
        if (!cut_by(v, i)) return false;
        i = next;
    }
    return cut_by(v, i);
}

__device__ inline void paint_cut(uint32_t* V, Interval cut, int R) {
    Rec rc;
    rc.sx = cut.s; rc.ex = cut.e;
    paint_bits(V, rc, R);
}

template <int K, bool FIELDS>
__global__ void __launch_bounds__(64 * kOcclWaves) __attribute__((amdgpu_waves_per_eu(K < 4 ? 4 : 2)))
forage_occlude_kernel(const FGRep* __restrict__ reps, abm_forage_state st,
                      const double* __restrict__ uniforms, const uint32_t* __restrict__ words,
                      const int64_t* __restrict__ u_off, const int32_t* __restrict__ u_cnt,
                      int32_t* __restrict__ u_used, int32_t* __restrict__ status,
                      uint32_t* __restrict__ bits_out, const int32_t* __restrict__ order,
                      abm_mt19937_state* __restrict__ mt, int maxN) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) double smem[];
    const int rb = order[blockIdx.x];
    if (status && status[rb] != kWorldReady) return;   // uniform over the block
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int H = kOcclPrep;
    __shared__ FGRep sP;
    if (tid < (int)(sizeof(FGRep) / 8))
        reinterpret_cast<uint64_t*>(&sP)[tid] = reinterpret_cast<const uint64_t*>(reps + rb)[tid];
    __syncthreads();
    const FGRep& P = sP;
    const int N = P.n_agents, R = P.n_rays, W = P.words, a0 = P.agent_offset, tau = P.tau;
    const OcclSmem S = occl_carve(smem, maxN, K);
    for (int i = tid; i < N; i += nthr) {
        const int g = a0 + i;
        const double w = st.w[g], u = st.u[g], cr = st.collected_r[g], crb = st.collected_r_before[g];
        const int over = st.overriding_mode[g], env = st.env_status[g];
        double m = st.novelty[(int64_t)g * tau];
        for (int q = 1; q < tau; ++q) m = fmax(m, st.novelty[(int64_t)g * tau + q]);
        const Drive d = drive_of(P, w, u, m, cr, crb, over, env);
        S.x[i] = st.x[g]; S.y[i] = st.y[g]; S.th[i] = st.theta[g]; S.v[i] = st.v[g];
        S.w[i] = w; S.u0[i] = u; S.u1[i] = d.u; S.ip[i] = d.ipriv; S.rad[i] = (double)st.radius[g];
        S.pid[i] = st.exploited_patch_id[g]; S.mode_over[i] = over; S.mode[i] = st.mode[g]; S.env[i] = env;
        st.collected_r_before[g] = cr;
    }
    // the step's uniforms: agent i's draw is the i-th at the latest (at most
    // one per agent); doubles, or pairs of words after those the resource
    // loop used (u_used[b] on entry); NaN past the end of the buffer
    const int ucount = mt ? 0 : u_cnt[rb];
    const int used0 = (words || mt) ? u_used[rb] : 0;
    int mt_pos0 = 0;
    if (mt) {
        for (int i = tid; i < kMtN; i += nthr) S.key[i] = mt[rb].key[i];
        mt_pos0 = mt[rb].pos;
        __syncthreads();
        uint32_t* wb = reinterpret_cast<uint32_t*>(S.uni);
        int made = 0, p = mt_pos0;
        while (made < 2 * N) {
            if (p >= kMtN) {
                mt_twist_block(S.key);
                p = 0;
            }
            const int take = min(kMtN - p, 2 * N - made);
            for (int j = tid; j < take; j += nthr) wb[made + j] = mt_temper(S.key[p + j]);
            made += take;
            p += take;
        }
        __syncthreads();
        for (int i = tid; i < N; i += nthr) {   // each thread rewrites its own 8 bytes
            const uint32_t w0 = wb[2 * i], w1 = wb[2 * i + 1];
            S.uni[i] = words_to_double(w0, w1);
        }
    } else {
        for (int i = tid; i < N; i += nthr) {
            double uu = NAN;
            if (words) {
                const uint32_t* wb = words + u_off[rb];
                const int at = used0 + 2 * i;
                if (at + 2 <= ucount) uu = words_to_double(wb[at], wb[at + 1]);
            } else if (i < ucount) {
                uu = uniforms[u_off[rb] + i];
            }
            S.uni[i] = uu;
        }
    }
    if (tid < 2) S.spec[4 * kOcclSpec + tid] = 0.0;
    const FastRec FR = fast_rec_const(R, P.step, P.fov0, P.fov1);
    const RangeTest rt = range_test(P.vision_range);
    const double step = P.step, fov0 = P.fov0, fov1 = P.fov1;
    const int patchwise = P.patchwise;
    constexpr int L = 64 * K;
    __syncthreads();

    const int h = wave - 1;   // the preparing wave's number (wave 0: none)
    Seen<K> seen;
    // ---- the pieces of a focal agent's preparation (a whole wave each)
    auto record = [&](int j, int f, const Focal& fo) {
        Rec rc;
        rc.valid = 0;
        const int c = occl_class(S, patchwise, rt, j, fo.cx, fo.cy, S.pid[f]);
        if (c != kNone) rc = record_at(S.x[j], S.y[j], c, c * N + j, fo, R, step, fov0, fov1, FR, true);
        return rc;
    };
    auto begin = [&](int f, int lo) {   // every record but those of agents lo .. f
        const double2 sc = sin_cos(S.th[f]);
        const Focal fo = focal_at(S.x[f], S.y[f], sc.x, sc.y, S.rad[f]);
        if (lane == 0) S.focal[wave] = fo;
#pragma unroll
        for (int c = 0; c < K; ++c) {
            const int j = 64 * c + lane;
            seen.ord[c] = -1; seen.start[c] = seen.end[c] = seen.rank[c] = seen.below[c] = seen.hid[c] = 0;
            seen.dist[c] = NAN;
#pragma unroll
            for (int b = 0; b < 2 * K; ++b) seen.over[c][b] = 0;
            if (j < N && (j < lo || j > f)) {
                const Rec rc = record(j, f, fo);
                if (rc.valid) { seen.start[c] = rc.start; seen.end[c] = rc.end; seen.ord[c] = rc.order; seen.dist[c] = rc.dist; }
            }
            S.rdist[L * h + j] = seen.dist[c];
        }
        fg_wave_sync();
    };
    // whether a record (distance d, bins [s, e]) is nearer than this lane's
    // record in slot c and overlaps it
    auto cuts = [&](const OcclRec& r, int c) {
        return (r.dist < seen.dist[c]) & (r.start <= seen.end[c]) & (r.end >= seen.start[c]);
    };
    auto hides = [&](const OcclRec& r, int c) {
        return (r.dist < seen.dist[c]) & (r.start <= seen.start[c]) & (r.end >= seen.end[c]);
    };
    auto before = [&](const OcclRec& r, int c) {
        return (r.dist < seen.dist[c]) | ((r.dist == seen.dist[c]) & (r.ord < seen.ord[c]));
    };
    // the first turn's records against each other, in two passes over j0 ..
    // j1 - 1: how many are nearer than each, then which of them overlap or hide it.
    // (Vector operations only: sign bits, and carries into the counts.)
    int same[K];
    auto count_nearer = [&](int j0, int j1) {
        const double* q = S.rdist + L * h;
        for (int j = j0; j < j1; j += 4) {
            double d[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) d[i] = j + i < j1 ? q[min(j + i, L - 1)] : NAN;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < K; ++c) {
                    seen.below[c] += d[i] < seen.dist[c] ? 1 : 0;
                    same[c] += d[i] == seen.dist[c] ? 1 : 0;
                }
        }
    };
    auto end_count = [&]() {   // places, ties in the obstacle list's order (rare); the records for the second pass
        bool tie = false;
#pragma unroll
        for (int c = 0; c < K; ++c) {
            seen.rank[c] = seen.below[c];
            tie |= same[c] > 1;
            S.rec[L * h + 64 * c + lane] = make_int4(seen.ord[c] < 0 ? 1 << 30 : seen.below[c], seen.start[c],
                                                     seen.end[c], seen.ord[c]);
        }
        fg_wave_sync();
        if (__ballot(tie) != 0)
            for (int j = 0; j < N; ++j) {
                const double d = S.rdist[L * h + j];
                const int o = S.rec[L * h + j].w;
#pragma unroll
                for (int c = 0; c < K; ++c) seen.rank[c] += (d == seen.dist[c]) & (o < seen.ord[c]) ? 1 : 0;
            }
    };
    auto overlaps = [&](int j0, int j1) {
        const int4* q = S.rec + L * h;
#pragma unroll
        for (int b = 0; b < 2 * K; ++b) {
            const int e = min(j1, 32 * b + 32);
            for (int j = max(j0, 32 * b); j < e; j += 4) {   // (records past e are met again: the same bits)
                int4 r[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) r[i] = q[min(j + i, 32 * b + 31)];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t bit = 1u << (min(j + i, 32 * b + 31) & 31);
#pragma unroll
                    for (int c = 0; c < K; ++c) {
                        const int nearer = r[i].x - seen.below[c];
                        seen.over[c][b] |= (uint32_t)((nearer & (r[i].y - seen.end[c] - 1) & (seen.start[c] - r[i].z - 1)) >> 31) & bit;
                        seen.hid[c] |= nearer & (r[i].y - seen.start[c] - 1) & (seen.end[c] - r[i].z - 1);
                    }
                }
            }
        }
    };
    // a record more, of agent j: the ranks and sets it enters, and its own
    auto enter = [&](int j, const OcclRec& r) {
        const int cj = j >> 6, lj = j & 63;
        const uint32_t bit = 1u << (j & 31);
        int rank = 0, below = 0;
        uint64_t on[K], hidden = 0;
#pragma unroll
        for (int c = 0; c < K; ++c) {
            const bool after = before(r, c), nearer = seen.dist[c] < r.dist;
            rank += (int)__popcll(__ballot((seen.ord[c] >= 0) & !after));
            below += (int)__popcll(__ballot(nearer));
            seen.rank[c] += after ? 1 : 0;
            seen.below[c] += r.dist < seen.dist[c] ? 1 : 0;
            const bool by = cuts(r, c);
            seen.hid[c] |= hides(r, c) ? -1 : 0;
#pragma unroll
            for (int b = 0; b < 2 * K; ++b)
                if (b == j >> 5) seen.over[c][b] |= by ? bit : 0u;
            on[c] = __ballot(nearer & (seen.start[c] <= r.end) & (seen.end[c] >= r.start));
            hidden |= __ballot(nearer & (seen.start[c] <= r.start) & (seen.end[c] >= r.end));
        }
#pragma unroll
        for (int c = 0; c < K; ++c)
            if (c == cj && lane == lj) {
                seen.start[c] = r.start; seen.end[c] = r.end; seen.ord[c] = r.ord; seen.dist[c] = r.dist;
                seen.rank[c] = rank; seen.below[c] = below; seen.hid[c] = hidden != 0 ? -1 : 0;
#pragma unroll
                for (int b = 0; b < K; ++b) {
                    seen.over[c][2 * b] = (uint32_t)on[b];
                    seen.over[c][2 * b + 1] = (uint32_t)(on[b] >> 32);
                }
            }
    };
    auto insert = [&](int f, int j0, int j1) {   // the records of agents j0 .. j1 - 1 (at most 64), which have moved
        Rec rc;
        rc.valid = 0;
        const Focal fo = S.focal[wave];
        if (j0 + lane < j1) rc = record(j0 + lane, f, fo);
        const long long db = __double_as_longlong(rc.valid ? rc.dist : 0.0);
        for (uint64_t t = __ballot(rc.valid != 0); t; t &= t - 1) {
            const int l = __builtin_ctzll(t);
            OcclRec r;
            const uint32_t dl = (uint32_t)__builtin_amdgcn_readlane((int)db, l);
            const uint32_t dh = (uint32_t)__builtin_amdgcn_readlane((int)(db >> 32), l);
            r.dist = __longlong_as_double((long long)((uint64_t)dh << 32 | dl));
            r.ord = __builtin_amdgcn_readlane(rc.order, l);
            r.start = __builtin_amdgcn_readlane(rc.start, l);
            r.end = __builtin_amdgcn_readlane(rc.end, l);
            enter(j0 + l, r);
        }
    };
    // the headings after a walk turn by uniform d .. d + 3, or none
    // (agent.py:187-200, 595-603), d uniforms drawn before agent f - 3
    auto headings = [&](int f, int d) {
        if (lane < 5) {
            double dth = 0.0;
            if (lane < 4) dth = P.exp_theta_min + (P.exp_theta_max - P.exp_theta_min) * (d + lane < N ? S.uni[d + lane] : 0.0);
            const double th = prove_orientation(S.th[f] + dth);
            const double2 sc = sin_cos(th);
            double* q = S.spec + kOcclSpec * (f & 3) + 3 * lane;
            q[0] = th; q[1] = sc.x; q[2] = sc.y;
            if (lane == 0) S.spec[kOcclSpec * (f & 3) + 15] = (double)d;
        }
    };
    auto publish = [&](int f) {   // to wave 0, by rank, with the field of these records
        const int p = f & 1;
        double* dist = S.dist + L * p;
        int2 *span = S.span + L * p, *cut = S.cut + L * p;
        int* ord = S.ord + L * p;
        int* rank = S.rank + L * h;
        uint32_t* V = S.field + (f & 3) * W;
        for (int w = lane; w < W; w += 64) V[w] = 0u;
        int n = 0;
#pragma unroll
        for (int c = 0; c < K; ++c) n += (int)__popcll(__ballot(seen.ord[c] >= 0));
#pragma unroll
        for (int c = 0; c < K; ++c) {
            const int j = 64 * c + lane;
            if (j >= n) { dist[j] = NAN; ord[j] = -1; }
            if (seen.ord[c] >= 0) {
                const int r = seen.rank[c];
                rank[j] = r;
                dist[r] = seen.dist[c];
                span[r] = make_int2(seen.start[c], seen.end[c]);
                ord[r] = seen.ord[c] | (seen.hid[c] < 0 ? kOrdHidden : 0);
            }
        }
        fg_wave_sync();
#pragma unroll
        for (int c = 0; c < K; ++c) {
            // the cues lead the obstacle list; only they are painted
            if ((unsigned)seen.ord[c] >= (unsigned)N || seen.hid[c] < 0) continue;
            uint64_t m[K];
#pragma unroll
            for (int b = 0; b < K; ++b) m[b] = 0;
#pragma unroll
            for (int b = 0; b < 2 * K; ++b)
                for (uint32_t t = seen.over[c][b]; t; t &= t - 1) {
                    const int r = rank[32 * b + __builtin_ctz(t)];
#pragma unroll
                    for (int a = 0; a < K; ++a) m[a] |= r >> 6 == a ? 1ull << (r & 63) : 0ull;
                }
            Interval v{seen.start[c], seen.end[c]};
            bool on = true;
#pragma unroll
            for (int b = 0; b < K; ++b)
                if (on) on = cut_by_all(v, m[b], span + 64 * b);
            paint_cut(V, v, R);
            const int r = seen.rank[c];
            cut[r] = make_int2(v.s, v.e);
#pragma unroll
            for (int b = 0; b < K; ++b) S.over[(size_t)L * (K * p + b) + r] = m[b];
        }
    };
    auto output = [&](int f) {   // soc_v_field[q] = V[R - 1 - q] on the kept rays (agent.py:593-595)
        const uint32_t* V = S.field + (f & 3) * W;
        const int lo = P.keep_lo, hi = P.keep_hi;
        uint32_t* dst = bits_out + P.field_offset + (int64_t)f * W;
        for (int w = lane; w < W; w += 64) dst[w] = __brev(raw_window(V, W, R - 32 - 32 * w)) & word_range_mask(w, lo, hi);
    };

    // ---- before the first turn: agents 0 .. H - 1 begun, agent 0's field
    if (wave > 0 && h < N) {
        begin(h, 0);
#pragma unroll
        for (int c = 0; c < K; ++c) same[c] = 0;
        count_nearer(0, N);
        end_count();
        overlaps(0, N);
        if (h == 0) publish(0);
        if (h < 3) headings(h, 0);
    }
    __syncthreads();
    int draws = 0, n_set = 0, n_left = 0;   // wave 0
    if (wave == 0) {
        wave_counts(S.field, R, W, P.keep_lo, P.keep_hi, nullptr, &n_set, &n_left);
        __builtin_amdgcn_s_setprio(3);   // the chain issues first
    }
    for (int k = 0; k < N; ++k) {
        const int f1 = k + 1;
        Rec rc;
        rc.valid = 0;
        if (wave == 0) {
            // ---- agent k's decision and move (agent.py:168-283), on every lane
            const int fn = min(f1, N - 1), pid_k = S.pid[k], pid_f = S.pid[fn];
            const Focal fo = S.focal[1 + fn % H];
            const double w0 = S.w[k], u0 = S.u0[k], u1 = S.u1[k], vel0 = S.v[k];
            const double x0 = S.x[k], y0 = S.y[k], th0 = S.th[k], rad = S.rad[k];
            const int env = S.env[k];
            const double* spec = S.spec + kOcclSpec * (k & 3);
            const int spec_d = (int)spec[15];
            const Choice c = choose(P, R, n_set, n_left, w0, u0, u1, vel0, S.mode_over[k], S.mode[k], env);
            Pose p{x0, y0, th0, vel0};
            double sn, cs;
            if (c.mode == ABM_MODE_RELOCATE && c.over == -1) {
                p.theta = prove_orientation(p.theta + c.dth);
                const double2 sc = sin_cos(p.theta);
                sn = sc.x; cs = sc.y;
            } else {   // prepared: prove_orientation(theta + turn) and its sin, cos
                const double* q = spec + 3 * (c.kind == 0 ? draws - spec_d : 4);
                p.theta = q[0]; sn = q[1]; cs = q[2];
                draws += c.kind == 0 ? 1 : 0;
            }
            p.v = p.v + c.dvel;
            // prove_velocity (agent.py:612-620): only in explore mode
            if (get_mode(c.over, c.w, P.T_w) == ABM_MODE_EXPLORE && fabs(p.v) > 1.0) p.v = P.exp_vel_max;
            p.x = p.x + p.v * cs;
            p.y = p.y - p.v * sn;
            p = reflect_walls(p, rad, P.pad, P.width, P.height);
            if (lane == 0) {
                S.x[k] = p.x; S.y[k] = p.y; S.th[k] = p.theta; S.v[k] = p.v;
                S.w[k] = c.w; S.mode_over[k] = c.over; S.mode[k] = c.mode;
                S.spec[4 * kOcclSpec + (f1 & 1)] = (double)draws;
            }
            // ---- its record in agent k + 1's view
            if (f1 < N && in_range(rt, (p.x + rad) - fo.cx, (p.y + rad) - fo.cy)) {
                const int cls = c.over != ABM_MODE_EXPLOIT ? kNonExpl
                                : patchwise && pid_k == pid_f ? kSamePatch : pid_k != -1 ? kSocial : kNone;
                if (cls != kNone) rc = record_at(p.x, p.y, cls, cls * N + k, fo, R, step, fov0, fov1, FR, true);
            }
        } else {
            const int f = f1 + (((h - f1) % H) + H) % H, s = k + H - f;   // turns since f's first
            if (FIELDS && k >= 1 && (k - 1) % H == h) output(k - 1);
            if (f < N) {
                if (s == 0) {
                    begin(f, k);
#pragma unroll
                    for (int c = 0; c < K; ++c) same[c] = 0;
                } else if (s <= 2) {
                    if (f >= H) count_nearer(N * (s - 1) / 2, N * s / 2);
                    if (f >= H && s == 2) end_count();
                } else if (s <= H - 3) {
                    if (f >= H) overlaps(N * (s - 3) / (H - 5), N * (s - 2) / (H - 5));
                    if (s == H - 3) headings(f, (int)S.spec[4 * kOcclSpec + (k & 1)]);
                } else if (s == H - 2) {
                    insert(f, max(f - H, 0), k);
                } else if (k >= 1) {
                    insert(f, k - 1, k);
                }
                if (s == H - 1) publish(f);
            }
        }
        __syncthreads();
        if (f1 >= N) break;
        if (wave == 0) {
            // ---- agent k + 1's field: the prepared one, with agent k's record
            const int p = f1 & 1;
            double* dist = S.dist + L * p;
            int2 *span = S.span + L * p, *cut = S.cut + L * p;
            int* ord = S.ord + L * p;
            uint32_t* V = S.field + (f1 & 3) * W;
            if (rc.valid) {
                const OcclRec r{rc.dist, rc.order, rc.start, rc.end};
                bool walk[K], any = false;
                uint64_t on[K], hidden = 0;
                int at = 0;   // its rank
#pragma unroll
                for (int c = 0; c < K; ++c) {
                    const int q = 64 * c + lane;
                    seen.dist[c] = dist[q];
                    const int o = ord[q];
                    seen.ord[c] = o < 0 ? o : o & ~kOrdHidden;
                    seen.hid[c] = o < 0 || (o & kOrdHidden) != 0 || seen.ord[c] >= N;   // hidden, no cue or no record
                    const int2 b = span[q];
                    seen.start[c] = b.x; seen.end[c] = b.y;
                    at += (int)__popcll(__ballot((o >= 0) & !before(r, c)));
                    walk[c] = !seen.hid[c] & cuts(r, c);   // a cue, cut by the record
                    any |= walk[c];
                    const bool nearer = seen.dist[c] < r.dist;
                    on[c] = __ballot(nearer & (b.x <= r.end) & (b.y >= r.start));
                    hidden |= __ballot(nearer & (b.x <= r.start) & (b.y >= r.end));
                }
                const bool repaint = __ballot(any) != 0;
                if (repaint) {
                    for (int w = lane; w < W; w += 64) V[w] = 0u;
                    fg_wave_sync();
#pragma unroll
                    for (int c = 0; c < K; ++c) {
                        const int q = 64 * c + lane;
                        if (seen.hid[c]) continue;
                        const int2 had = cut[q];
                        Interval v{had.x, had.y};
                        if (walk[c]) {
                            v = Interval{seen.start[c], seen.end[c]};
                            bool open = true;
#pragma unroll
                            for (int b = 0; b < K; ++b) {   // the nearer ones before it, itself, those after it
                                const uint64_t m = S.over[(size_t)L * (K * p + b) + q];
                                const int l = min(max(at - 64 * b, 0), 64);
                                const uint64_t low = l == 64 ? ~0ull : (1ull << l) - 1ull;
                                if (open) open = cut_by_all(v, m & low, span + 64 * b);
                                if (open && at >= 64 * b && (at < 64 * b + 64 || b == K - 1)) open = cut_by(v, make_int2(r.start, r.end));
                                if (open) open = cut_by_all(v, m & ~low, span + 64 * b);
                            }
                        }
                        paint_cut(V, v, R);
                    }
                }
                if (rc.social && hidden == 0) {
                    Interval v{r.start, r.end};
                    bool open = true;
#pragma unroll
                    for (int b = 0; b < K; ++b)
                        if (open) open = cut_by_all(v, on[b], span + 64 * b);
                    if (lane == 0) paint_cut(V, v, R);
                }
                fg_wave_sync();
            }
            wave_counts(V, R, W, P.keep_lo, P.keep_hi, nullptr, &n_set, &n_left);
        }
    }
    if (FIELDS && wave > 0 && (N - 1) % H == h) output(N - 1);
    for (int i = tid; i < N; i += nthr) {
        const int g = a0 + i;
        st.x[g] = S.x[i]; st.y[g] = S.y[i]; st.theta[g] = S.th[i]; st.v[g] = S.v[i];
        st.w[g] = S.w[i]; st.u[g] = S.u1[i];
        st.mode[g] = S.mode[i]; st.overriding_mode[g] = S.mode_over[i];
        st.I_priv[g] = S.ip[i];
    }
    if (tid == 0) S.kept[0] = draws;
    __syncthreads();
    draws = S.kept[0];
    if (tid == 0 && u_used) u_used[rb] = used0 + (words || mt ? 2 : 1) * draws;
    if (tid == 0 && status) status[rb] = ABM_WORLD_DONE;
    if (mt) {
        // advance the generator by the 2 * draws words used: numpy's state
        // after them is the key twisted v times at position pos0 + c - 624 v
        const int c = 2 * draws;
        int v = 0, pos = mt_pos0 + c;
        if (pos > kMtN) {
            v = (pos - 1) / kMtN;
            pos -= kMtN * v;
        }
        if (v > 0) {
            for (int i = tid; i < kMtN; i += nthr) S.key[i] = mt[rb].key[i];
            __syncthreads();
            for (int t = 0; t < v; ++t) mt_twist_block(S.key);
            for (int i = tid; i < kMtN; i += nthr) mt[rb].key[i] = S.key[i];
        }
        if (tid == 0) mt[rb].pos = pos;
    }
}

// ------------------------------------------------ replicas over the whole GPU
// The same update for replicas beyond one workgroup's LDS, and for large ones:
// three launches over the agents of all of them, 64 (a chunk) to a wave in the
// first and last, one to a wave in the middle, with the cues in global memory.
// No host round trip, so a caller may capture the step.  Its predecessor swept
// all agents until a fixed point (three sweeps a step, checked on the host):
// one replica of 8192 agents with 100 to 700 cues took 0.41 ms in the sweeps,
// 0.04 ms now.
struct WideRep {
    int32_t rb, chunk0;   // the replica, its first chunk
    int64_t keys;         // its twisted keys in WideMem.keys, in words
};
struct WideCue {
    double x, y, xm, ym;         // at the step's start, and moved
    int32_t rad, j, pid, flag;   // flag: kCueStart, kCueMoved
};
// Agent k of a replica is entry 64 * chunk0 + k of every array.
struct WideMem {
    const WideRep* rep;          // the replicas
    const int32_t* of;           // [chunk]: which of them
    WideCue* cue;                // from the replica's first entry on
    double *u1, *ip, *u1x, *u1y;
    int32_t *nset, *nleft;
    uint32_t *uni;               // the next 2N words of a device generator
    uint32_t* keys;              // its key after each twist
    uint8_t* walk;               // 1: the agent draws a walk turn
    int32_t* ctl;                // [replica][kWdWords]
    int32_t* updates;            // [replica]: made so far
};
constexpr int kWdCues = 0, kWdSkip = 1, kWdUsed0 = 2, kWdWords = 4;

// Control words of new scratch.
__global__ void __launch_bounds__(256)
wide_clear_kernel(int32_t* __restrict__ ctl, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) ctl[i] = 0;
}

// One thread per agent: the drive, the focal geometry, the cues.
__global__ void __launch_bounds__(256)
wide_drive_kernel(const FGRep* __restrict__ reps, int n_chunks, abm_forage_state st,
                  const int32_t* __restrict__ status, const int32_t* __restrict__ u_used, int words_or_mt,
                  WideMem M) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const int chunk = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (chunk >= n_chunks) return;
    const int q = M.of[chunk], rb = M.rep[q].rb, chunk0 = M.rep[q].chunk0;
    int32_t* const ctl = M.ctl + kWdWords * q;
    const bool skip = status && status[rb] != kWorldReady;
    if (chunk == chunk0 && lane == 0) {
        ctl[kWdSkip] = skip;
        ctl[kWdUsed0] = words_or_mt ? u_used[rb] : 0;
    }
    if (skip) return;
    const FGRep& P = reps[rb];
    const int i = (chunk - chunk0) * 64 + lane, e = chunk * 64 + lane;
    int flag = 0;
    WideCue c;
    if (i < P.n_agents) {
        const int g = P.agent_offset + i, tau = P.tau;
        const double th = st.theta[g], v = st.v[g], w = st.w[g];
        c.x = st.x[g]; c.y = st.y[g]; c.rad = st.radius[g]; c.pid = st.exploited_patch_id[g]; c.j = i;
        const int over = st.overriding_mode[g];
        double m = st.novelty[(int64_t)g * tau];
        for (int q = 1; q < tau; ++q) m = fmax(m, st.novelty[(int64_t)g * tau + q]);
        const Drive d = drive_of(P, w, st.u[g], m, st.collected_r[g], st.collected_r_before[g], over,
                                 st.env_status[g]);
        const Focal f = focal_at(c.x, c.y, th, (double)c.rad);
        M.u1[e] = d.u; M.ip[e] = d.ipriv; M.u1x[e] = f.u1x; M.u1y[e] = f.u1y;
        c.xm = c.x; c.ym = c.y;
        if (c.pid != -1) {
            if (over == ABM_MODE_EXPLOIT) flag |= kCueStart;
            if (d.exploit) {
                flag |= kCueMoved;
                const Pose p = fg_move(P, Pose{c.x, c.y, th, v}, 0.0, -v * P.exp_stop_ratio, ABM_MODE_EXPLOIT, w,
                                       (double)c.rad);
                c.xm = p.x; c.ym = p.y;
            }
        }
        c.flag = flag;
    }
    const uint64_t m = __ballot(flag != 0);
    if (m) {
        int at = 0;
        if (lane == 0) at = atomicAdd(&ctl[kWdCues], (int)__popcll(m));
        at = __builtin_amdgcn_readfirstlane(at) + 64 * chunk0;
        if (flag) M.cue[at + (int)__popcll(m & ((1ull << lane) - 1ull))] = c;
    }
}

// One wave per agent, sixteen blocks per chunk from first_chunk on: its field
// from the cues, the counts and whether it walks.  With device generators the
// first n_reps blocks make each replica's next 2N words meanwhile.
template <bool FIELDS>
__global__ void __launch_bounds__(256)
wide_field_kernel(const FGRep* __restrict__ reps, int n_reps, int first_chunk, abm_forage_state st, WideMem M,
                  const abm_mt19937_state* __restrict__ mt, uint32_t* __restrict__ bits_out) {
#pragma clang fp contract(off)
    extern __shared__ uint32_t lds_u[];
    const int tid = threadIdx.x;
    int block = blockIdx.x;
    if (mt) {
        if (block < n_reps) {
            if (M.ctl[kWdWords * block + kWdSkip]) return;   // uniform over the block
            const int rb = M.rep[block].rb, N = reps[rb].n_agents;
            uint32_t* const keys = M.keys + M.rep[block].keys;
            uint32_t* const uni = M.uni + 128 * (int64_t)M.rep[block].chunk0;
            for (int i = tid; i < kMtN; i += 256) lds_u[i] = mt[rb].key[i];
            __syncthreads();
            int made = 0, p = mt[rb].pos, twists = 0;
            while (made < 2 * N) {
                if (p >= kMtN) {
                    mt_twist_block(lds_u);
                    for (int i = tid; i < kMtN; i += 256) keys[(int64_t)twists * kMtN + i] = lds_u[i];
                    ++twists;
                    p = 0;
                }
                const int take = min(kMtN - p, 2 * N - made);
                for (int j = tid; j < take; j += 256) uni[made + j] = mt_temper(lds_u[p + j]);
                made += take;
                p += take;
                __syncthreads();
            }
            return;
        }
        block -= n_reps;
    }
    const int chunk = first_chunk + (block >> 4), q = M.of[chunk], chunk0 = M.rep[q].chunk0;
    const int32_t* const ctl = M.ctl + kWdWords * q;
    if (ctl[kWdSkip]) return;
    const FGRep& P = reps[M.rep[q].rb];
    const int N = P.n_agents, R = P.n_rays, W = P.words, a0 = P.agent_offset;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int k = (chunk - chunk0) * 64 + (block & 15) * 4 + wave, e = chunk0 * 64 + k;
    if (k >= N) return;   // uniform over the wave; no block barrier below
    const int gk = a0 + k;
    uint32_t* V = lds_u + wave * W;
    for (int w = lane; w < W; w += 64) V[w] = 0u;
    Focal f;
    f.radius = (double)st.radius[gk];
    f.px = st.x[gk]; f.py = st.y[gk];
    f.cx = f.px + f.radius;
    f.cy = f.py + f.radius;
    f.u1x = M.u1x[e]; f.u1y = M.u1y[e];
    const int pid_k = st.exploited_patch_id[gk], patchwise = P.patchwise;
    const FastRec FR = fast_rec_const(R, P.step, P.fov0, P.fov1);
    const RangeTest rt = range_test(P.vision_range);
    const double step = P.step, fov0 = P.fov0, fov1 = P.fov1;
    const int n_cue = ctl[kWdCues];
    const WideCue* const cues = M.cue + 64 * (int64_t)chunk0;
    fg_wave_sync();
    for (int i = lane; i < n_cue; i += 64) {
        const WideCue c = cues[i];
        const bool moved = c.j < k;
        // agent.py:396-413, as the update kernel
        if (c.j == k || !(c.flag & (moved ? kCueMoved : kCueStart)) || (patchwise && c.pid == pid_k)) continue;
        const double ox = moved ? c.xm : c.x, oy = moved ? c.ym : c.y, rj = (double)c.rad;
        if (!in_range(rt, (ox + rj) - f.cx, (oy + rj) - f.cy)) continue;
        const Rec rc = record_at(ox, oy, kSocial, c.j, f, R, step, fov0, fov1, FR, false);
        if (rc.valid) paint_bits(V, rc, R);
    }
    fg_wave_sync();
    int n_set, n_left;
    wave_counts(V, R, W, P.keep_lo, P.keep_hi, FIELDS ? bits_out + P.field_offset + (int64_t)k * W : nullptr,
                &n_set, &n_left);
    if (lane == 0) {
        M.nset[e] = n_set; M.nleft[e] = n_left;
        M.walk[e] = choose(P, R, n_set, n_left, st.w[gk], st.u[gk], M.u1[e], st.v[gk], st.overriding_mode[gk],
                           st.mode[gk], st.env_status[gk]).kind == 0;
    }
}

// One thread per agent: the walk's draw index (the flags of every agent
// before it), the choice and the move, written to the state.  A replica's
// first chunk also leaves the words used, the status and the device generator
// advanced by them.
__global__ void __launch_bounds__(256)
wide_move_kernel(const FGRep* __restrict__ reps, int n_chunks, abm_forage_state st,
                 const double* __restrict__ uniforms, const uint32_t* __restrict__ words,
                 const int64_t* __restrict__ u_off, const int32_t* __restrict__ u_cnt,
                 int32_t* __restrict__ u_used, int32_t* __restrict__ status,
                 abm_mt19937_state* __restrict__ mt, WideMem M) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const int chunk = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (chunk >= n_chunks) return;
    const int q = M.of[chunk], rb = M.rep[q].rb, chunk0 = M.rep[q].chunk0;
    int32_t* const ctl = M.ctl + kWdWords * q;
    if (ctl[kWdSkip]) return;
    const FGRep& P = reps[rb];
    const int N = P.n_agents, R = P.n_rays, a0 = P.agent_offset;
    const bool first = chunk == chunk0;
    // walks before this chunk (the first: in all), sixteen flags at a time
    const uint8_t* const walk = M.walk + 64 * (int64_t)chunk0;
    const int upto = first ? N : (chunk - chunk0) * 64;
    int n = 0;
    for (int i = lane * 16; i < upto; i += 1024) {
        const uint4 f = *reinterpret_cast<const uint4*>(walk + i);
        const uint32_t four[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int left = upto - i - 4 * t;   // flags of this word that count
            n += __popc(left >= 4 ? four[t] : (left <= 0 ? 0u : four[t] & ((1u << (8 * left)) - 1u)));
        }
    }
    const int total = wave_sum(n);
    const int k = (chunk - chunk0) * 64 + lane, e = chunk * 64 + lane;
    const bool walks = k < N && M.walk[e] != 0;
    const uint64_t m = __ballot(walks);
    const int d = (first ? 0 : total) + (int)__popcll(m & ((1ull << lane) - 1ull));
    const int used0 = ctl[kWdUsed0];
    if (k < N) {
        const int g = a0 + k;
        const double vel0 = st.v[g];
        const Choice c = choose(P, R, M.nset[e], M.nleft[e], st.w[g], st.u[g], M.u1[e], vel0,
                                st.overriding_mode[g], st.mode[g], st.env_status[g]);
        double dth = c.dth;
        if (walks) {
            double uu = NAN;   // past the end of the buffer
            if (mt) {
                const uint32_t* uni = M.uni + 128 * (int64_t)chunk0;
                uu = words_to_double(uni[2 * d], uni[2 * d + 1]);
            } else if (words) {
                const uint32_t* wb = words + u_off[rb];
                const int at = used0 + 2 * d;
                if (at + 2 <= u_cnt[rb]) uu = words_to_double(wb[at], wb[at + 1]);
            } else if (d < u_cnt[rb]) {
                uu = uniforms[u_off[rb] + d];
            }
            dth = P.exp_theta_min + (P.exp_theta_max - P.exp_theta_min) * uu;
        }
        const Pose p = fg_move(P, Pose{st.x[g], st.y[g], st.theta[g], vel0}, dth, c.dvel, c.over, c.w,
                               (double)st.radius[g]);
        st.x[g] = p.x; st.y[g] = p.y; st.theta[g] = p.theta; st.v[g] = p.v;
        st.w[g] = c.w; st.u[g] = M.u1[e]; st.I_priv[g] = M.ip[e];
        st.collected_r_before[g] = st.collected_r[g];
        st.mode[g] = c.mode; st.overriding_mode[g] = c.over;
    }
    if (!first) return;
    if (mt) {
        // numpy's state after the 2 * total words: the key twisted v times at
        // position pos0 + c - 624 v (it twists lazily, when a word is drawn)
        int v = 0, pos = mt[rb].pos + 2 * total;
        if (pos > kMtN) {
            v = (pos - 1) / kMtN;
            pos -= kMtN * v;
            const uint32_t* const key = M.keys + M.rep[q].keys + (int64_t)(v - 1) * kMtN;
            for (int i = lane; i < kMtN; i += 64) mt[rb].key[i] = key[i];
        }
        if (lane == 0) mt[rb].pos = pos;
    }
    if (lane == 0) {
        ctl[kWdCues] = 0;   // for the next step's drive kernel
        atomicAdd(&M.updates[q], 1);
        if (u_used) u_used[rb] = used0 + (words || mt ? 2 : 1) * total;
        if (status) status[rb] = ABM_WORLD_DONE;
    }
}

// ------------------------------------------------ agent-resource interaction
constexpr int kMaxPatches = 64;     // patches per replica (one 64-bit membership word)
constexpr int kMaxRetries = 10000;  // add_new_resource_patch's max_retries (sims.py:335)

// Pending patch placements of a replica, kept between a phase that ran out of
// words and its resume.
constexpr int kPendNone = 0, kPendKill = 1, kPendFill = 2;

// Per-replica world constants on the device.
struct WRep {
    int32_t n_patches, patch_radius, pooling_time, regenerate, teleport, collide, ghost, n_agents;
    int64_t patch_offset;
    int64_t x_lo, x_hi, y_lo, y_hi, units_lo, units_hi;   // randint bounds [lo, hi)
    double consumption, q_lo, q_hi;
};

// Raw MT19937 outputs of one replica; reading past the end sets `out`.
struct WordCursor {
    const uint32_t* w;
    int used, limit;
    bool out;
    __device__ uint32_t next() {
        if (used >= limit) { out = true; return 0u; }
        return w[used++];
    }
};

// RandomState.randint(lo, hi) for a range below 2^32 - 1: numpy draws
// next_uint32 & mask until the value is <= hi - 1 - lo, mask being the
// smallest all-ones word covering it (random_bounded_uint64_fill with
// use_masked; no draw when the range holds one value).
template <typename Cursor>
__device__ inline int64_t np_randint(Cursor& c, int64_t lo, int64_t hi) {
    const uint32_t rng = (uint32_t)(hi - 1 - lo);
    if (rng == 0u) return lo;
    uint32_t mask = rng;
    mask |= mask >> 1; mask |= mask >> 2; mask |= mask >> 4; mask |= mask >> 8; mask |= mask >> 16;
    uint32_t v;
    do { v = c.next() & mask; } while (v > rng && !c.out);
    return lo + (int64_t)v;
}

// RandomState.uniform(lo, hi) = lo + (hi - lo) * random_sample.
template <typename Cursor>
__device__ inline double np_uniform(Cursor& c, double lo, double hi) {
#pragma clang fp contract(off)
    const uint32_t w0 = c.next(), w1 = c.next();
    return lo + (hi - lo) * words_to_double(w0, w1);
}

// Python's float x % (2*pi) (and numpy's remainder): fmod, shifted into
// [0, 2*pi) when negative, +0 for a zero.
__device__ inline double py_mod_2pi(double x) {
#pragma clang fp contract(off)
    double m = fmod(x, kTwoPi);
    if (m != 0.0) {
        if (m < 0.0) m = m + kTwoPi;
    } else {
        m = 0.0;
    }
    return m;
}

// notify_agent (sims.py:29-42): env status, novelty ring, pool_success, patch id.
__device__ inline void notify(const abm_forage_state& st, int32_t* pool_success, int tau, int g,
                              int status, int patch_id) {
    const int before = st.env_status[g];
    st.env_status[g] = status;
    double* nov = st.novelty + (int64_t)g * tau;
    // np.roll(novelty, 1), eight entries at a time from the top: a chunk's
    // loads are all issued before its stores, and read below what it writes
    for (int top = tau - 1; top > 0; top -= 8) {
        double v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (top - i > 0) v[i] = nov[top - i - 1];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (top - i > 0) nov[top - i] = v[i];
    }
    nov[0] = (status - before) > 0 ? 1.0 : 0.0;
    pool_success[g] = 1;
    st.exploited_patch_id[g] = patch_id;
}

// The condition under which the loop notifies an agent (sims.py:816-817, 852).
__device__ inline bool pooled(int mode, int pool_success, int pooling_time) {
    return ((mode == ABM_MODE_POOL || mode == ABM_MODE_RELOCATE) && pool_success) || pooling_time == 0;
}

// pygame.sprite.collide_circle of two patches: integer rect centres,
// squared distance <= (r1 + r2)^2.
__device__ inline bool patches_collide(int64_t cx1, int64_t cy1, int64_t r1, int64_t cx2, int64_t cy2,
                                       int64_t r2) {
    const int64_t dx = cx1 - cx2, dy = cy1 - cy2, rr = r1 + r2;
    return dx * dx + dy * dy <= rr * rr;
}

struct FreshPatch {
    int32_t id;
    int64_t x, y;
    double units, quality;
};

// Place the replica's pending patches (regenerations of the patches killed
// this step, in kill order, or create_resources' new patches) from the word
// buffer, then compact the list: live patches in order, new ones appended.
// One wave, lane t holding patch t and new patch t (at most 64 of each): the
// draws are the same on every lane, the overlap tests one patch per lane.
// Commits nothing unless every placement fits in the buffer.
static_assert(kMaxPatches == 64, "a lane per patch");
template <typename Cursor>
__device__ int place_patches(const WRep& W, const abm_patch_state& ps, int b, int kind, int n_pending,
                             const int32_t* __restrict__ pend_id, int32_t* __restrict__ kill_rank, Cursor& cur) {
    const int64_t po = W.patch_offset;
    const int lane = threadIdx.x & 63, count = ps.count[b];
    int n_new = 0;
    if (kind == kPendKill) n_new = W.regenerate ? n_pending : 0;
    else if (kind == kPendFill) n_new = W.n_patches - count;
    const int64_t r = W.patch_radius, s = po + lane;
    const bool held = lane < count;
    double px = 0.0, py = 0.0, pr = 0.0, units = 0.0, left = 0.0, quality = 0.0;
    int32_t id = 0, rank = -1, pend = 0;
    if (held) {
        px = ps.x[s]; py = ps.y[s]; pr = ps.radius[s]; units = ps.units[s]; left = ps.left[s];
        quality = ps.quality[s]; id = ps.id[s]; rank = kill_rank[s];
    }
    if (kind == kPendKill && lane < n_new) pend = pend_id[s];   // force_id: the killed patch's id
    const int64_t pcx = (int64_t)trunc(px + pr), pcy = (int64_t)trunc(py + pr), pri = (int64_t)pr;
    int32_t top = held ? id : INT32_MIN;   // the largest id, for create_resources
    for (int d = 1; d < 64; d <<= 1) top = max(top, __shfl_xor(top, d, 64));
    if (count == 0) top = 0;
    FreshPatch mine{0, 0, 0, 0.0, 0.0};
    for (int k = 0; k < n_new; ++k) {
        for (int retries = 0;; ++retries) {
            if (retries > kMaxRetries) return ABM_WORLD_TIMEOUT;
            const int64_t x = np_randint(cur, W.x_lo, W.x_hi);
            const int64_t y = np_randint(cur, W.y_lo, W.y_hi);
            const int64_t u = np_randint(cur, W.units_lo, W.units_hi);
            const double q = np_uniform(cur, W.q_lo, W.q_hi);
            if (cur.out) return ABM_WORLD_NEED_WORDS;
            const int64_t cx = x + r, cy = y + r;
            // the Group at the time: live patches, those killed later this
            // step, and the ones placed before this one
            bool hit = held && !(rank >= 0 && rank <= k) && patches_collide(pcx, pcy, pri, cx, cy, r);
            hit = hit || (lane < k && patches_collide(mine.x + r, mine.y + r, r, cx, cy, r));
            if (__ballot(hit)) continue;
            if (lane == k) {
                mine.id = kind == kPendKill ? pend : top + 1 + k;
                mine.x = x; mine.y = y; mine.units = (double)u; mine.quality = q;
            }
            break;
        }
    }
    // commit: drop the killed patches, keep the order, append the new ones
    const bool stays = held && rank < 0;
    const uint64_t m = __ballot(stays);
    const int kept = (int)__popcll(m);
    if (held && rank >= 0) kill_rank[s] = -1;
    if (stays) {
        const int64_t d = po + (int)__popcll(m & ((1ull << lane) - 1ull));
        ps.id[d] = id; ps.x[d] = px; ps.y[d] = py; ps.radius[d] = pr; ps.units[d] = units; ps.left[d] = left;
        ps.quality[d] = quality;
    }
    if (lane < n_new) {
        const int64_t d = po + kept + lane;
        ps.id[d] = mine.id; ps.x[d] = (double)mine.x; ps.y[d] = (double)mine.y; ps.radius[d] = (double)r;
        ps.units[d] = mine.units; ps.left[d] = mine.units; ps.quality[d] = mine.quality;
    }
    if (lane == 0) ps.count[b] = kept + n_new;
    return ABM_WORLD_DONE;
}

// ------------------------------------------------ agent-agent collisions
constexpr int kCollideMaxAgents = 2048;   // replicas with collisions on
constexpr int kCollideMaxNear = 256;      // agents within 2 r + 20 of a colliding agent

size_t collide_lds_bytes(int maxN, int maxR) {
    return ((sizeof(int32_t) * 5 * (size_t)maxN + sizeof(int32_t) * kCollideMaxNear + 15) & ~(size_t)15) +
           fg_lds_bytes(kCollideMaxNear, maxR) + 16;
}

// numpy's pairwise float64 sum (np.add.reduce of a contiguous array,
// pairwise_sum in numpy/_core/src/umath/loops_utils.h.src): fewer than 8
// elements in sequence from 0.0; up to 128 in eight strided partial sums
// combined as ((r0 + r1) + (r2 + r3)) + ((r4 + r5) + (r6 + r7)), then the
// remainder in sequence; longer runs split at n / 2 rounded down to a multiple
// of 8, each half summed the same way.  val(i) is element i.
template <class Val>
__device__ double np_block_sum(const Val& val, int lo, int n) {
#pragma clang fp contract(off)
    if (n < 8) {
        double res = 0.0;
        for (int i = 0; i < n; ++i) res += val(lo + i);
        return res;
    }
    double r[8];
    for (int j = 0; j < 8; ++j) r[j] = val(lo + j);
    int i = 8;
    for (; i < n - (n % 8); i += 8)
        for (int j = 0; j < 8; ++j) r[j] += val(lo + i + j);
    double res = ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
    for (; i < n; ++i) res += val(lo + i);
    return res;
}

template <class Val>
__device__ double np_pairwise_sum(const Val& val, int lo, int n) {
#pragma clang fp contract(off)
    // post-order walk of the split tree on an explicit stack
    int s_lo[32], s_n[32], s_state[32];
    double s_left[32];
    int sp = 0;
    s_lo[0] = lo; s_n[0] = n; s_state[0] = 0;
    for (;;) {
        if (s_n[sp] > 128) {
            const int n2 = s_n[sp] / 2 - (s_n[sp] / 2) % 8;
            s_state[sp] = 1;
            s_lo[sp + 1] = s_lo[sp]; s_n[sp + 1] = n2; s_state[sp + 1] = 0;
            ++sp;
            continue;
        }
        double ret = np_block_sum(val, s_lo[sp], s_n[sp]);
        for (;;) {
            if (sp == 0) return ret;   // the node just finished is the root
            --sp;
            if (s_state[sp] == 1) {    // its left half: start the right half
                const int n2 = s_n[sp] / 2 - (s_n[sp] / 2) % 8;
                s_left[sp] = ret;
                s_state[sp] = 2;
                s_lo[sp + 1] = s_lo[sp] + n2; s_n[sp + 1] = s_n[sp] - n2; s_state[sp + 1] = 0;
                ++sp;
                break;
            }
            ret = s_left[sp] + ret;    // its right half: this node is done
        }
    }
}

// Agent-agent collisions of the loop body (sims.py:736-787), one block per
// replica before the resource loop.  Collisions are those of
// pygame.sprite.groupcollide(agents, agents, ..., within_group_collision)
// with every radius grown by 2 (sims.py:738-747): collide_circle on the rect
// centres, int(position) + radius (the rect holds int() of the position and
// is 2 r wide), squared integer distance <= (r1 + 2 + r2 + 2)^2.  Each agent2
// of a colliding pair (agent1, agent2) takes the proximity response of
// agent_agent_collision_proximity (sims.py:421-467) once per partner agent1
// that passes the ghost-mode test; the response reads only agent2's own
// heading and everyone's positions, which it does not change, so the agents
// are handled one at a time with their responses in sequence.  Then the
// collided list (sims.py:760-777) ends or notifies the collide modes
// (sims.py:779-784).  A replica with an agent beyond kCollideMaxNear
// neighbours within 2 r + 20 is reported ABM_WORLD_CROWDED and not touched.
__global__ void __launch_bounds__(256)
forage_collide_kernel(const FGRep* __restrict__ reps, const WRep* __restrict__ wreps,
                      abm_forage_state st, int32_t* __restrict__ pool_success,
                      const int32_t* __restrict__ pend, int32_t* __restrict__ status) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) double smem[];
    const int b = blockIdx.x, tid = threadIdx.x, nthr = blockDim.x;
    const FGRep& P = reps[b];
    const WRep& W = wreps[b];
    if (!W.collide || pend[2 * b] != kPendNone) return;   // uniform over the block
    const int N = P.n_agents, a0 = P.agent_offset, R = P.n_rays;
    char* base = reinterpret_cast<char*>(smem);
    int32_t* cx = reinterpret_cast<int32_t*>(base);
    int32_t* cy = cx + N;
    int32_t* rr = cy + N;
    int32_t* cnt = rr + N;     // responses of each agent as agent2
    int32_t* flag = cnt + N;   // bit 0 collided, bit 1 exploiting
    int32_t* near = flag + N;
    FGSmem S = fg_carve(base + ((sizeof(int32_t) * 5 * (size_t)N + sizeof(int32_t) * kCollideMaxNear + 15) &
                                ~(size_t)15),
                        kCollideMaxNear, R);
    __shared__ int s_crowded, s_nn;
    if (tid == 0) s_crowded = 0;
    for (int j = tid; j < N; j += nthr) {
        const int g = a0 + j;
        const int r = st.radius[g];
        cx[j] = (int)trunc(st.x[g]) + r;
        cy[j] = (int)trunc(st.y[g]) + r;
        rr[j] = r;
        flag[j] = get_mode(st.overriding_mode[g], st.w[g], P.T_w) == ABM_MODE_EXPLOIT ? 2 : 0;
    }
    __syncthreads();
    // ---- pairs, responses per agent and the collided list
    for (int j = tid; j < N; j += nthr) {
        const bool ex_j = flag[j] & 2;
        int n_resp = 0;
        bool any = false, both = false;
        for (int i = 0; i < N; ++i) {
            if (i == j) continue;
            const long dx = cx[i] - cx[j], dy = cy[i] - cy[j], rs = rr[i] + rr[j] + 4;
            if (dx * dx + dy * dy > rs * rs) continue;
            const bool ne = !(flag[i] & 2) && !ex_j;
            any = true;
            both = both || ne;
            if (!W.ghost || ne) ++n_resp;
        }
        // sims.py:760-777: collided agents (the exploiting status never changes here)
        const bool collided = W.teleport ? (any && !ex_j) : (!W.ghost ? any : both);
        cnt[j] = n_resp;
        flag[j] |= collided ? 1 : 0;
        if (n_resp > 0) {
            // neighbours within 2 r + 20 (supcalc.distance, each agent's own radius)
            const int g = a0 + j;
            const double rj = (double)rr[j];
            const double cxj = st.x[g] + rj, cyj = st.y[g] + rj;
            int nn = 0;
            for (int i = 0; i < N; ++i) {
                if (i == j) continue;
                const int gi = a0 + i;
                const double ri = (double)rr[i];
                if (norm2((st.x[gi] + ri) - cxj, (st.y[gi] + ri) - cyj) < 2.0 * rj + 20.0) ++nn;
            }
            if (nn > kCollideMaxNear) s_crowded = 1;   // benign race: every writer stores 1
        }
    }
    __syncthreads();
    if (s_crowded) {
        if (tid == 0) status[b] = ABM_WORLD_CROWDED;
        return;   // uniform over the block
    }
    // ---- the proximity responses, agent by agent
    const double fov0 = -kPi, fov1 = kPi;
    for (int j = 0; j < N; ++j) {
        if (cnt[j] == 0) continue;   // uniform over the block
        const int g = a0 + j;
        const bool ex_j = flag[j] & 2;
        const double rj = (double)rr[j];
        const double pxj = st.x[g], pyj = st.y[g];
        if (tid == 0) {
            if (!ex_j) { st.overriding_mode[g] = ABM_MODE_COLLIDE; st.mode[g] = ABM_MODE_COLLIDE; }
            // the agents within 2 r + 20, in id order
            int nn = 0;
            for (int i = 0; i < N; ++i) {
                if (i == j) continue;
                const int gi = a0 + i;
                const double ri = (double)rr[i];
                if (norm2((st.x[gi] + ri) - (pxj + rj), (st.y[gi] + ri) - (pyj + rj)) < 2.0 * rj + 20.0) {
                    if (nn < kCollideMaxNear) near[nn] = gi;   // the count was checked above
                    ++nn;
                }
            }
            s_nn = nn < kCollideMaxNear ? nn : kCollideMaxNear;
        }
        __syncthreads();
        const int nn = s_nn;
        for (int q = tid; q < nn; q += nthr) {
            S.x[q] = st.x[near[q]];
            S.y[q] = st.y[near[q]];
            S.cls[q] = kSocial;
        }
        __syncthreads();
        for (int c = 0; c < cnt[j]; ++c) {
            const Focal f = make_focal(pxj, pyj, st.theta[g], rj);
            if (tid == 0) {
                // the distance left in projection_field's loop variable: its
                // last non-coincident obstacle (agent.py:501-556)
                S.lastd[0] = 0.0;
                for (int q = nn - 1; q >= 0; --q) {
                    const PairFG p = pair_forage_exact(f, S.x[q], S.y[q], R, P.step, fov0, fov1);
                    if (!p.skipped) { S.lastd[0] = p.dist; break; }
                }
            }
            project_focal(S, nn, R, P.step, fov0, fov1, P.visual_exclusion != 0, false, f, true);
            if (tid == 0) {
                // left / right excitation and the front (sims.py:444-462)
                const double val2 = 1.0 - S.lastd[0] / P.vision_range;
                auto val = [&](int r) {
                    const int code = soc_bit(S.V, r, R, P.step, fov0, fov1);
                    return code == 0 ? 0.0 : (code == 2 ? val2 : 1.0);
                };
                const int h = R / 2;
                const double left = np_pairwise_sum(val, 0, h) / (double)h;
                const double right = np_pairwise_sum(val, h, R - h) / (double)(R - h);
                const double D = left > right ? 1.0 : -1.0;   // np.sign, 0 taken as -1
                int lo, hi;
                py_slice(h - 100, h + 100, R, &lo, &hi);
                const bool front = hi > lo && np_pairwise_sum(val, lo, hi - lo) / (double)(hi - lo) > 0.0;
                if (!ex_j) st.theta[g] = st.theta[g] - D * 0.2;
                if (front) st.v[g] = 0.0;
                else if (!ex_j) st.v[g] = P.exp_vel_max;
            }
            __syncthreads();
        }
    }
    // ---- collide modes ended, or notified (sims.py:779-784)
    for (int j = tid; j < N; j += nthr) {
        const int g = a0 + j;
        if (get_mode(st.overriding_mode[g], st.w[g], P.T_w) != ABM_MODE_COLLIDE) continue;
        if (!(flag[j] & 1)) {
            st.overriding_mode[g] = -1;
            st.mode[g] = ABM_MODE_EXPLORE;
        } else {
            notify(st, pool_success, P.tau, g, -1, -1);
        }
    }
    if (tid == 0) status[b] = kWorldReady;
}

// Replicas above this many agents take the resource loop over the whole GPU
// (one workgroup spent about 0.2 of its 0.26 ms on testing 8192 agents against
// 64 patches on one CU).  At or below it a replica has one thread per agent of
// a single workgroup.
constexpr int kWorldBlockAgents = 1024;

// An agent's part of the resource loop that depends on nobody else: the patch
// its centre lies on (supcalc.distance(resc, agent) < resc.radius).  The norm
// (a sqrt) is taken only where both centre differences are within the radius,
// with a margin far above the rounding of the norm, so no pair inside is
// skipped.  each(p, in) sees every patch in order.
struct PatchLds {
    double pr[kMaxPatches], cx[kMaxPatches], cy[kMaxPatches];   // radius, resc.center
    double pq[kMaxPatches], pl[kMaxPatches];                    // quality, units left
    int32_t pid[kMaxPatches];
};
template <class Each>
__device__ inline void patch_tests(const PatchLds& L, int p0, int p1, bool live, double cx, double cy,
                                   const Each& each) {
#pragma unroll 4
    for (int p = p0; p < p1; ++p) {
        const double pr = L.pr[p], dx = cx - L.cx[p], dy = cy - L.cy[p];
        const double lim = pr * 1.0000001;
        bool in = false;
        if (live && fabs(dx) <= lim && fabs(dy) <= lim) in = norm2(dx, dy) < pr;
        each(p, in);
    }
}

// bias_agent_towards_res_center (sims.py:544-552) for the patch's centre.
__device__ inline double biased_heading(double th, double cx, double cy, double pcx, double pcy) {
#pragma clang fp contract(off)
    const double cl = py_mod_2pi(atan2(pcy - cy, pcx - cx) + th);
    return th + (cl - kPi) * 0.02;
}

// Rescource.deplete (rescource.py:118-133) by n exploiting agents in turn:
// every one up to the last served takes `units`, the last takes `last` (what
// is left, when that is less); the one that empties the patch is the last
// served and destroys it.
struct Depletion {
    double left, units, last;
    int served;
    bool destroyed;
};
__device__ inline Depletion deplete(double consumption, double quality, double left, int n) {
#pragma clang fp contract(off)
    Depletion d;
    d.units = consumption > quality ? quality : consumption;
    d.last = 0.0; d.served = 0; d.destroyed = false;
    while (d.served < n && !d.destroyed) {
        if (left >= d.units) { left = left - d.units; d.last = d.units; }
        else { d.last = left; left = 0.0; }
        d.destroyed = !(left > 0.0);
        ++d.served;
    }
    d.left = left;
    return d;
}

// What the agents need of a patch after its depletion.
struct PatchAfter {
    double units, last;
    int32_t served, destroyer;   // destroyer: its agent, or n_agents
};

// Index of the n-th set bit (n from 0) of m.
__device__ inline int nth_bit(uint64_t m, int n) {
    for (; n > 0; --n) m &= m - 1;
    return __builtin_ctzll(m);
}

// The depletions of np_ patches by their exploiting agents in id order,
// word(p, c) being those of patch p in the 64-agent chunk c of C.  The waves of
// the block (nw, at most 16) share the chunks out, a patch per lane; one lane
// per patch then runs its subtractions.  base(p, c, n) takes the number of a
// patch's exploiting agents before chunk c.  Every thread; ends synchronised.
template <class Word, class Base>
__device__ inline void deplete_patches(const Word& word, const Base& base, int np_, int C, int N, int nw,
                                       double consumption, PatchLds& L, int (*seg)[kMaxPatches],
                                       PatchAfter* after) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int per = (C + nw - 1) / nw, c0 = wave * per, c1 = min(C, c0 + per);
    int cnt = 0;
    if (lane < np_)
        for (int c = c0; c < c1; ++c) cnt += (int)__popcll(word(lane, c));
    seg[wave][lane] = cnt;
    __syncthreads();
    int before = 0, n = 0;
    for (int w = 0; w < nw; ++w) {
        const int t = seg[w][lane];
        if (w < wave) before += t;
        n += t;
    }
    if (lane < np_) {
        int run = before;
        for (int c = c0; c < c1; ++c) {
            base(lane, c, run);
            run += (int)__popcll(word(lane, c));
        }
        if (wave == 0) {
            const Depletion d = deplete(consumption, L.pq[lane], L.pl[lane], n);
            L.pl[lane] = d.left;
            after[lane] = PatchAfter{d.units, d.last, d.served, d.destroyed ? -1 : N};
        }
    }
    __syncthreads();
    if (lane < np_ && after[lane].destroyer < N) {   // whose wave holds the last agent served
        int r = after[lane].served - 1 - before;
        if (r >= 0 && r < cnt)
            for (int c = c0; c < c1; ++c) {
                const uint64_t m = word(lane, c);
                const int t = (int)__popcll(m);
                if (r < t) {
                    after[lane].destroyer = c * 64 + nth_bit(m, r);
                    break;
                }
                r -= t;
            }
    }
    __syncthreads();
}

// The agent's share of the walk over its patch (sims.py:803-845), everything
// the walk does to agent j of patch p: its heading, what it takes (rank: its
// place among the patch's exploiting agents), the notify of its own turn (a
// pooled agent up to the destroyer hears of the patch, and teleports), the
// destroyer's notify-all, and for agents after the destroyer the notify of
// their own turn.
__device__ inline void walk_agent(const abm_forage_state& st, int32_t* pool_success, const WRep& W, int tau, int g,
                                  int j, double theta, bool exploits, int rank, bool pool, const PatchAfter& a,
                                  int32_t pid, double pcx, double pcy) {
#pragma clang fp contract(off)
    st.theta[g] = theta;
    if (exploits && rank < a.served) {
        const double cr = st.collected_r[g];
        st.collected_r_before[g] = cr;
        st.collected_r[g] = cr + (rank == a.served - 1 ? a.last : a.units);
    }
    const int d = a.destroyer, N = W.n_agents;
    if (j <= d && pool) {
        notify(st, pool_success, tau, g, 1, pid);
        if (W.teleport) {
            const double ra = (double)st.radius[g];
            st.x[g] = pcx - ra;
            st.y[g] = pcy - ra;
        }
    }
    if (d < N) notify(st, pool_success, tau, g, -1, -1);   // the destroyer's notify-all
    if (j > d) notify(st, pool_success, tau, g, -1, -1);   // its own turn after it
}

// Scratch of the resource loop over the whole GPU.  Replica q of rep[] has
// its 64-agent chunks from chunk0 on; agent j is entry 64 * chunk0 + j.
struct WideWorldRep {
    int32_t b, chunk0;
};
struct WideWorldBlock {
    int32_t q, agent0;         // 64 agents of replica rep[q]
};
struct WideWorld {
    const WideWorldRep* rep;
    const WideWorldBlock* block;
    uint64_t *member, *expl;   // [chunk][64 patches]: agents on the patch; those exploiting
    int32_t* before;           // [chunk][64 patches]: exploiting agents of earlier chunks
    double* theta;             // the biased headings
    uint8_t *patch, *flag;     // the agent's patch (255: none), kExploits | kPools
    PatchAfter* after;         // [replica][64]
    PatchLds* geo;             // [replica]: the patches before any placement
    int32_t* ctl;              // [replica][kWwWords]
};
constexpr int kExploits = 1, kPools = 2;
constexpr int kWwGo = 0, kWwMulti = 1, kWwWords = 2;

__device__ inline void stage_patches(PatchLds& L, const abm_patch_state& ps, int64_t po, int np_, int tid, int nthr) {
    for (int p = tid; p < np_; p += nthr) {
        const int64_t s = po + p;
        const double pr = ps.radius[s];
        L.pr[p] = pr; L.cx[p] = ps.x[s] + pr; L.cy[p] = ps.y[s] + pr;
        L.pq[p] = ps.quality[s]; L.pl[p] = ps.left[s]; L.pid[p] = ps.id[s];
    }
}

// The agents' own parts of the loop (a replica above kWorldBlockAgents), 64
// agents per block: its four waves test a quarter of the patches each (128
// blocks of one wave left 8192 agents waiting on their tests' LDS reads).
// Membership words, headings, flags.
__global__ void __launch_bounds__(256)
wide_member_kernel(const FGRep* __restrict__ reps, const WRep* __restrict__ wreps, abm_forage_state st,
                   const int32_t* __restrict__ pool_success, abm_patch_state ps, WideWorld ww) {
#pragma clang fp contract(off)
    __shared__ PatchLds L;
    __shared__ uint64_t words[kMaxPatches];
    __shared__ int s_on[64], s_times[64];
    const WideWorldBlock B = ww.block[blockIdx.x];
    const int b = ww.rep[B.q].b, chunk0 = ww.rep[B.q].chunk0;
    const FGRep& P = reps[b];
    const WRep& W = wreps[b];
    const int N = P.n_agents, np_ = ps.count[b], tid = threadIdx.x, lane = tid & 63;
    if (np_ < 0 || np_ > W.n_patches) return;   // reported by the world kernel
    stage_patches(L, ps, W.patch_offset, np_, tid, blockDim.x);
    if (tid < 64) { words[tid] = 0ull; s_on[tid] = kMaxPatches; s_times[tid] = 0; }
    const int j = B.agent0 + lane, g = P.agent_offset + j;
    const bool live = j < N;
    double cx = 0.0, cy = 0.0;
    if (live) {
        const double ra = (double)st.radius[g];
        cx = st.x[g] + ra;
        cy = st.y[g] + ra;
    }
    __syncthreads();
    const int wave = tid >> 6, per = (np_ + 3) / 4;
    int on = kMaxPatches, times = 0;
    patch_tests(L, wave * per, min(np_, wave * per + per), live, cx, cy, [&](int p, bool in) {
        const uint64_t m = __ballot(in);
        if (lane == 0) words[p] = m;
        if (in) { on = min(on, p); ++times; }
    });
    if (times) { atomicMin(&s_on[lane], on); atomicAdd(&s_times[lane], times); }
    __syncthreads();
    if (wave != 0) return;
    on = s_on[lane];
    int flag = 0;
    if (live) {
        const int mode = get_mode(st.overriding_mode[g], st.w[g], P.T_w);
        flag = (mode == ABM_MODE_EXPLOIT ? kExploits : 0) | (pooled(mode, pool_success[g], W.pooling_time) ? kPools : 0);
    }
    const uint64_t ex = __ballot((flag & kExploits) != 0);
    const int64_t chunk = chunk0 + (B.agent0 >> 6), at = chunk * kMaxPatches + lane, e = chunk * 64 + lane;
    ww.member[at] = words[lane];
    ww.expl[at] = words[lane] & ex;
    if (__ballot(s_times[lane] > 1) && lane == 0) atomicOr(&ww.ctl[kWwWords * B.q + kWwMulti], 1);
    if (!live) return;
    ww.patch[e] = on < kMaxPatches ? (uint8_t)on : 255;
    ww.flag[e] = (uint8_t)flag;
    if (on < kMaxPatches) ww.theta[e] = biased_heading(st.theta[g], cx, cy, L.cx[on], L.cy[on]);
}

// The walk's effects on each agent, after the world kernel's depletions.
__global__ void __launch_bounds__(64)
wide_notify_kernel(const FGRep* __restrict__ reps, const WRep* __restrict__ wreps, abm_forage_state st,
                   int32_t* __restrict__ pool_success, WideWorld ww) {
    const WideWorldBlock B = ww.block[blockIdx.x];
    if (!ww.ctl[kWwWords * B.q + kWwGo]) return;
    const int b = ww.rep[B.q].b;
    const FGRep& P = reps[b];
    const int j = B.agent0 + threadIdx.x;
    if (j >= P.n_agents) return;
    const int64_t e = 64 * (int64_t)ww.rep[B.q].chunk0 + j;
    const int g = P.agent_offset + j, p = ww.patch[e], flag = ww.flag[e];
    if (p == 255) {   // agents on no patch (sims.py:847-855)
        if (flag) notify(st, pool_success, P.tau, g, -1, -1);
        return;
    }
    const int64_t at = (e >> 6) * kMaxPatches + p;
    const PatchLds& geo = ww.geo[B.q];
    const int rank = ww.before[at] + (int)__popcll(ww.expl[at] & ((1ull << (j & 63)) - 1ull));
    walk_agent(st, pool_success, wreps[b], P.tau, g, j, ww.theta[e], (flag & kExploits) != 0, rank,
               (flag & kPools) != 0, ww.after[kMaxPatches * B.q + p], geo.pid[p], geo.cx[p], geo.cy[p]);
}

// STEP: agent-resource interaction (sims.py:789-855) then the placement of
// regenerated patches; FILL: create_resources; RESUME: the placements a
// previous phase left pending.  One replica per block, one thread per agent;
// WIDE: the replicas above kWorldBlockAgents, whose agents' own parts come from
// wide_member_kernel and go to wide_notify_kernel.
// An agent's centre lies on at most one patch (patches never overlap), so of
// the walk over the patches and their agents in id order only each patch's
// depletion is sequential, a count of its exploiting agents and as many
// subtractions; each agent then takes its share by its rank.  Patches a caller
// loaded that overlap take the walk itself, in the reference's order, on one
// lane.  Waves that neither hold an agent nor are among the first four end at
// once (a barrier waits for those that live).  Bound by latency: the loads
// (each agent's in one batch), the notify's round trip, the barriers, and in
// steps that regenerate patches the placements' draws.  Against passes over the
// agents one after another, a lane per patch walking its agents' records in
// global memory and one thread twisting, drawing and compacting: 1000 replicas
// of 8 to 512 agents with ten patches 46 -> 31 us, one replica of 10 agents
// 10.2 -> 8.2, 8192 agents with 64 patches 261 -> 29 in three launches (7 us
// membership, 16 here, 6 notify).
template <bool WIDE>
__global__ void __launch_bounds__(1024)
forage_world_kernel(const FGRep* __restrict__ reps, const WRep* __restrict__ wreps, int phase,
                    abm_forage_state st, int32_t* __restrict__ pool_success, abm_patch_state ps,
                    int32_t* __restrict__ kill_rank, int32_t* __restrict__ pend,
                    int32_t* __restrict__ pend_id, const uint32_t* __restrict__ words,
                    const int64_t* __restrict__ w_off, const int32_t* __restrict__ w_cnt,
                    int32_t* __restrict__ w_used, int32_t* __restrict__ status,
                    abm_mt19937_state* __restrict__ mt, WideWorld ww) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) uint64_t member_lds[];   // [patch][chunk], then the exploiting ones
    __shared__ uint32_t mkey[kMtN];
    __shared__ int s_kind, s_pending, s_pos, s_multi;
    __shared__ PatchLds L;
    __shared__ PatchAfter s_after[kMaxPatches];
    __shared__ int s_seg[16][kMaxPatches];
    const int b = WIDE ? ww.rep[blockIdx.x].b : blockIdx.x, tid = threadIdx.x;
    const int nthr = WIDE ? 1024 : min((int)blockDim.x, max(256, (reps[b].n_agents + 63) & ~63));
    if (tid >= nthr) return;   // uniform over the wave
    const int64_t chunk0 = WIDE ? ww.rep[blockIdx.x].chunk0 : 0;
    int32_t* const wctl = WIDE ? ww.ctl + kWwWords * blockIdx.x : nullptr;
    // the replica's parameters in LDS, read where used
    __shared__ FGRep sP;
    __shared__ WRep sW;
    static_assert(sizeof(WRep) % 8 == 0 && sizeof(WRep) / 8 <= 64, "WRep copy");
    if (tid < (int)(sizeof(FGRep) / 8))
        reinterpret_cast<uint64_t*>(&sP)[tid] = reinterpret_cast<const uint64_t*>(reps + b)[tid];
    else if (tid >= 64 && tid < 64 + (int)(sizeof(WRep) / 8))
        reinterpret_cast<uint64_t*>(&sW)[tid - 64] = reinterpret_cast<const uint64_t*>(wreps + b)[tid - 64];
    int kind = pend[2 * b], n_pending = pend[2 * b + 1];
    const int n_live = ps.count[b], status0 = status[b];
    if (tid == 0) {
        // taken and cleared in one operation: a plain read of this uniform
        // address is a scalar load, which the clearing store may overtake
        s_multi = WIDE ? atomicExch(&wctl[kWwMulti], 0) : 0;
        if (WIDE) wctl[kWwGo] = 0;
    }
    __syncthreads();
    const FGRep& P = sP;
    const WRep& W = sW;
    const int N = P.n_agents, a0 = P.agent_offset, C = (N + 63) / 64;
    const int64_t po = W.patch_offset;
    if (!WIDE && phase == ABM_WORLD_STEP && N > kWorldBlockAgents) return;   // the WIDE launch's
    if (n_live < 0 || n_live > W.n_patches) {
        if (tid == 0) { w_used[b] = 0; status[b] = ABM_WORLD_BAD_COUNT; }
        return;
    }
    if (phase == ABM_WORLD_RESUME) {
        if (status0 != ABM_WORLD_NEED_WORDS || kind == kPendNone) {
            if (tid == 0) w_used[b] = 0;
            return;
        }
    } else if (kind != kPendNone) {
        // placements of an earlier phase still wait for words: resume first
        if (tid == 0) { w_used[b] = 0; status[b] = ABM_WORLD_NEED_WORDS; }
        return;
    }
    if (phase == ABM_WORLD_STEP) {
        // a replica the collision kernel found crowded is left as it is
        if (W.collide && status0 == ABM_WORLD_CROWDED) {
            if (tid == 0) w_used[b] = 0;
            return;
        }
        const int np_ = n_live, lane = tid & 63, g = a0 + tid;
        uint64_t* const member = member_lds;
        uint64_t* const expl = member_lds + (size_t)np_ * C;
        auto member_word = [&](int p, int c) {
            return WIDE ? ww.member[(chunk0 + c) * kMaxPatches + p] : member[p * C + c];
        };
        // the live patches' geometry, quality and units staged in LDS, and
        // (one thread per agent) the agent's own part
        stage_patches(L, ps, po, np_, tid, nthr);
        const bool live = !WIDE && tid < N;
        double cx = 0.0, cy = 0.0, th = 0.0;
        int flag = 0;
        if (live) {
            const double ra = (double)st.radius[g];
            cx = st.x[g] + ra;
            cy = st.y[g] + ra;
            th = st.theta[g];
            const int mode = get_mode(st.overriding_mode[g], st.w[g], P.T_w);
            flag = (mode == ABM_MODE_EXPLOIT ? kExploits : 0) |
                   (pooled(mode, pool_success[g], W.pooling_time) ? kPools : 0);
        }
        __syncthreads();
        int on = -1;
        if (!WIDE && (tid & ~63) < N) {
            const uint64_t ex = __ballot((flag & kExploits) != 0);
            int times = 0;
            patch_tests(L, 0, np_, live, cx, cy, [&](int p, bool in) {
                const uint64_t m = __ballot(in);
                if (lane == 0) { member[p * C + (tid >> 6)] = m; expl[p * C + (tid >> 6)] = m & ex; }
                if (in) { if (on < 0) on = p; ++times; }
            });
            if (__ballot(times > 1) && lane == 0) s_multi = 1;   // every writer stores 1
        }
        if (WIDE)
            for (int p = tid; p < np_; p += nthr) {
                PatchLds& geo = ww.geo[blockIdx.x];
                geo.cx[p] = L.cx[p]; geo.cy[p] = L.cy[p]; geo.pid[p] = L.pid[p];
            }
        __syncthreads();
        const bool multi = s_multi != 0;
        if (multi) {
            // patches loaded by the caller that overlap: the walk in the
            // reference's order, in one thread
            if (tid == 0) {
                int n_kill = 0;
                for (int p = 0; p < np_; ++p) {
                    const int64_t s = po + p;
                    const double pcx = L.cx[p], pcy = L.cy[p];   // resc.center
                    const int32_t pid = L.pid[p];
                    bool destroy = false;
                    for (int c = 0; c < C; ++c) {
                        uint64_t m = member_word(p, c);
                        while (m) {
                            const int gi = a0 + c * 64 + __builtin_ctzll(m);
                            m &= m - 1;
                            const double ra = (double)st.radius[gi];
                            st.theta[gi] = biased_heading(st.theta[gi], st.x[gi] + ra, st.y[gi] + ra, pcx, pcy);
                            if (destroy) {
                                notify(st, pool_success, P.tau, gi, -1, -1);
                                continue;
                            }
                            const int mode = get_mode(st.overriding_mode[gi], st.w[gi], P.T_w);
                            if (pooled(mode, pool_success[gi], W.pooling_time)) {
                                notify(st, pool_success, P.tau, gi, 1, pid);
                                if (W.teleport) {
                                    st.x[gi] = pcx - ra;
                                    st.y[gi] = pcy - ra;
                                }
                            }
                            if (mode == ABM_MODE_EXPLOIT) {
                                const Depletion d = deplete(W.consumption, L.pq[p], L.pl[p], 1);
                                L.pl[p] = d.left;
                                ps.left[s] = d.left;
                                destroy = d.destroyed;
                                const double cr = st.collected_r[gi];
                                st.collected_r_before[gi] = cr;
                                st.collected_r[gi] = cr + d.last;
                                if (destroy) {
                                    // every agent of the group hears of it
                                    for (int c2 = 0; c2 < C; ++c2) {
                                        uint64_t m2 = member_word(p, c2);
                                        while (m2) {
                                            const int g2 = a0 + c2 * 64 + __builtin_ctzll(m2);
                                            m2 &= m2 - 1;
                                            notify(st, pool_success, P.tau, g2, -1, -1);
                                        }
                                    }
                                }
                            }
                        }
                    }
                    if (destroy) {
                        kill_rank[s] = n_kill;
                        pend_id[po + n_kill] = pid;
                        ++n_kill;
                    }
                }
                // agents on no patch (sims.py:847-855)
                for (int j = 0; j < N; ++j) {
                    uint64_t any = 0ull;
                    for (int p = 0; p < np_; ++p) any |= member_word(p, j >> 6);
                    if ((any >> (j & 63)) & 1ull) continue;
                    const int mode = get_mode(st.overriding_mode[a0 + j], st.w[a0 + j], P.T_w);
                    if (pooled(mode, pool_success[a0 + j], W.pooling_time) || mode == ABM_MODE_EXPLOIT)
                        notify(st, pool_success, P.tau, a0 + j, -1, -1);
                }
                kind = n_kill ? kPendKill : kPendNone;
                n_pending = n_kill;
            }
        } else {
            deplete_patches([&](int p, int c) { return WIDE ? ww.expl[(chunk0 + c) * kMaxPatches + p] : expl[p * C + c]; },
                            [&](int p, int c, int n) { if (WIDE) ww.before[(chunk0 + c) * kMaxPatches + p] = n; }, np_, C,
                            N, nthr >> 6, W.consumption, L, s_seg, s_after);
            for (int p = tid; p < np_; p += nthr) {
                ps.left[po + p] = L.pl[p];
                if (WIDE) ww.after[kMaxPatches * blockIdx.x + p] = s_after[p];
            }
            if (WIDE && tid == 0) wctl[kWwGo] = 1;
            if (live) {
                if (on < 0) {
                    if (flag) notify(st, pool_success, P.tau, g, -1, -1);   // agents on no patch (sims.py:847-855)
                } else {
                    int rank = (int)__popcll(expl[on * C + (tid >> 6)] & ((1ull << lane) - 1ull));
                    for (int c = 0; c < tid >> 6; ++c) rank += (int)__popcll(expl[on * C + c]);
                    walk_agent(st, pool_success, W, P.tau, g, tid, biased_heading(th, cx, cy, L.cx[on], L.cy[on]),
                               (flag & kExploits) != 0, rank, (flag & kPools) != 0, s_after[on], L.pid[on], L.cx[on],
                               L.cy[on]);
                }
            }
            if (tid < 64) {   // the destroyed patches, in Group order
                const bool dead = tid < np_ && s_after[tid].destroyer < N;
                const uint64_t m = __ballot(dead);
                if (dead) {
                    const int k = (int)__popcll(m & ((1ull << tid) - 1ull));
                    kill_rank[po + tid] = k;
                    pend_id[po + k] = L.pid[tid];
                }
                kind = m ? kPendKill : kPendNone;
                n_pending = (int)__popcll(m);
            }
        }
    } else if (phase == ABM_WORLD_FILL) {
        kind = kPendFill;
        n_pending = 0;
    }
    // ---- placements, by the first wave: from the words the caller drew
    // ahead, but for those of the random walk of the update that follows, or
    // from the replica's generator on the device, its key in LDS meanwhile
    if (tid == 0) { s_kind = kind; s_pending = n_pending; }
    __syncthreads();
    kind = s_kind;
    n_pending = s_pending;
    const bool update_follows = kind != kPendFill;
    if (kind == kPendNone) {
        if (tid == 0) {
            pend[2 * b] = kPendNone; pend[2 * b + 1] = 0;
            w_used[b] = 0;
            status[b] = kWorldReady;
        }
        return;
    }
    if (mt) {
        for (int i = tid; i < kMtN; i += nthr) mkey[i] = mt[b].key[i];
        if (tid == 0) s_pos = mt[b].pos;
        __syncthreads();
    }
    if (tid < 64) {
        int rc, used;
        if (mt) {
            MtCursor cur{mkey, s_pos, 0, false};
            rc = place_patches(W, ps, b, kind, n_pending, pend_id, kill_rank, cur);
            used = cur.used;
            // a timeout: the generator stays where it was
            if (tid == 0) s_pos = rc == ABM_WORLD_DONE ? cur.pos : -1;
        } else {
            const int limit = w_cnt ? max(0, w_cnt[b] - (update_follows ? 2 * N : 0)) : 0;
            WordCursor cur{words ? words + w_off[b] : nullptr, 0, words ? limit : 0, false};
            rc = place_patches(W, ps, b, kind, n_pending, pend_id, kill_rank, cur);
            used = rc == ABM_WORLD_NEED_WORDS ? 0 : cur.used;   // nothing placed, nothing drawn
        }
        if (tid == 0) {
            w_used[b] = used;
            if (rc == ABM_WORLD_DONE) {
                pend[2 * b] = kPendNone; pend[2 * b + 1] = 0;
                status[b] = update_follows ? kWorldReady : ABM_WORLD_DONE;
            } else {
                // out of words (the kill ranks stay for the resume), or too
                // many retries: the reference raises
                pend[2 * b] = kind; pend[2 * b + 1] = n_pending;
                status[b] = rc;
            }
        }
    }
    if (!mt) return;
    __syncthreads();
    if (s_pos >= 0) {
        for (int i = tid; i < kMtN; i += nthr) mt[b].key[i] = mkey[i];
        if (tid == 0) mt[b].pos = s_pos;
    }
}

// Agent.projection_field of one focal agent: obstacles [0, n_social) are the
// social cues, [n_social, n) the non-social occluders (when n_nonsocial >= 0).
__global__ void __launch_bounds__(256)
forage_projection_kernel(int R, double step, double fov0, double fov1, int exclusion,
                         double vision_range, int keep_distance, double fx, double fy,
                         double fth, double fr, const double* __restrict__ ox,
                         const double* __restrict__ oy, int n_social, int n_nonsocial,
                         double* __restrict__ out, int maxN) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) double smem[];
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int N = n_social + (n_nonsocial > 0 ? n_nonsocial : 0);
    FGSmem S = fg_carve(smem, maxN, R);
    for (int i = tid; i < N; i += nthr) {
        S.x[i] = ox[i]; S.y[i] = oy[i];
        S.cls[i] = i < n_social ? kSocial : kNonExpl;
    }
    if (tid == 0) S.lastd[0] = 0.0;
    __syncthreads();
    const Focal f = make_focal(fx, fy, fth, fr);
    // the distance left in the reference's loop variable: last non-coincident obstacle
    if (tid == 0 && keep_distance) {
        for (int i = N - 1; i >= 0; --i) {
            const PairFG p = pair_forage_exact(f, S.x[i], S.y[i], R, step, fov0, fov1);
            if (!p.skipped) { S.lastd[0] = p.dist; break; }
        }
    }
    project_focal(S, N, R, step, fov0, fov1, exclusion != 0, n_nonsocial >= 0, f, keep_distance != 0);
    const double val = 1.0 - S.lastd[0] / vision_range;
    for (int r = tid; r < R; r += nthr) {
        const int b = soc_bit(S.V, r, R, step, fov0, fov1);
        out[r] = b == 0 ? 0.0 : (b == 2 ? val : 1.0);
    }
}

}  // namespace
}  // namespace abm

using namespace abm;

namespace {

constexpr int kForageMaxAgents = 65536;
constexpr int kWideMaxRays = 8192;   // of the update over the whole GPU
constexpr int kWideMinAgents = 64, kWideMaxPerCu = 96;   // where it is the better one (plan_classes)

// Generator keys a step may twist to while making 2M words.
int wide_key_slots(int M) { return (2 * M + kMtN) / kMtN + 1; }

// Device memory of the update over the whole GPU for so many replicas, chunks
// and twisted key words; with base null only its size is found.
size_t wide_carve(void* base, size_t reps, size_t chunks, size_t key_words, WideMem* m) {
    const size_t n = 64 * chunks;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        char* p = reinterpret_cast<char*>(base) + at;
        at += (bytes + 255) & ~(size_t)255;
        return p;
    };
    m->rep = reinterpret_cast<WideRep*>(take(sizeof(WideRep) * reps));
    m->of = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * chunks));
    m->cue = reinterpret_cast<WideCue*>(take(sizeof(WideCue) * n));
    for (double** d : {&m->u1, &m->ip, &m->u1x, &m->u1y}) *d = reinterpret_cast<double*>(take(sizeof(double) * n));
    for (int32_t** i : {&m->nset, &m->nleft}) *i = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * n));
    m->uni = reinterpret_cast<uint32_t*>(take(sizeof(uint32_t) * 2 * n));
    m->keys = reinterpret_cast<uint32_t*>(take(sizeof(uint32_t) * key_words));
    m->walk = reinterpret_cast<uint8_t*>(take(n));
    m->ctl = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * kWdWords * reps));
    m->updates = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * reps));
    return at;
}

WideMem wide_mem(const WidePlan& w) {
    WideMem m;
    wide_carve(w.mem, w.reps.size(), (size_t)w.chunks, (size_t)w.keys, &m);
    return m;
}

// Updates the wide replicas' move kernels have made.
int wide_updates(const abm_forage_batch* bt, int64_t* total) {
    *total = 0;
    for (const WidePlan& w : bt->wide) {
        if (!w.mem) continue;
        std::vector<int32_t> made(w.reps.size());
        if (int rc = check_hip(hipDeviceSynchronize(), "hipDeviceSynchronize")) return rc;
        if (int rc = check_hip(hipMemcpy(made.data(), wide_mem(w).updates, sizeof(int32_t) * made.size(),
                                         hipMemcpyDeviceToHost), "read update counts"))
            return rc;
        for (int32_t n : made) *total += n;
    }
    return ABM_OK;
}

// The scratch of a plan, made whole before the plan has it.
int make_wide(abm_forage_batch* bt, WidePlan& w) {
    if (w.mem || w.reps.empty()) return ABM_OK;
    if (!bt->wide_done)
        if (int rc = check_hip(hipEventCreateWithFlags(&bt->wide_done, hipEventDisableTiming), "hipEventCreate")) return rc;
    std::vector<WideRep> rep;
    std::vector<int32_t> of;
    int64_t keys = 0;
    for (int b : w.reps) {
        rep.push_back(WideRep{b, (int32_t)of.size(), keys});
        of.insert(of.end(), (bt->rep_n[b] + 63) / 64, (int32_t)rep.size() - 1);
        keys += (int64_t)kMtN * wide_key_slots(bt->rep_n[b]);
    }
    WidePlan made = w;
    made.chunks = (int32_t)of.size();
    made.keys = keys;
    WideMem m;
    const size_t bytes = wide_carve(nullptr, rep.size(), of.size(), (size_t)keys, &m);
    if (int rc = check_hip(hipMalloc(&made.mem, bytes), "hipMalloc(wide update)")) return rc;
    m = wide_mem(made);
    int rc = check_hip(hipMemcpy(const_cast<WideRep*>(m.rep), rep.data(), sizeof(WideRep) * rep.size(),
                                 hipMemcpyHostToDevice), "upload wide replicas");
    if (!rc) rc = check_hip(hipMemcpy(const_cast<int32_t*>(m.of), of.data(), sizeof(int32_t) * of.size(),
                                      hipMemcpyHostToDevice), "upload wide chunks");
    if (!rc) rc = check_hip(hipMemset(m.ctl, 0, sizeof(int32_t) * kWdWords * rep.size()), "clear wide control");
    if (!rc) rc = check_hip(hipMemset(m.updates, 0, sizeof(int32_t) * rep.size()), "clear update counts");
    if (!rc) rc = check_hip(hipDeviceSynchronize(), "plan wide update");
    if (rc) {
        (void)hipFree(made.mem);
        return rc;
    }
    made.clean = true;
    w = std::move(made);
    return ABM_OK;
}

// Device memory of the resource loop over the whole GPU; with base null only
// its size is found.
size_t wide_world_carve(void* base, const abm_forage_world* w, WideWorld* m) {
    const size_t reps = (size_t)w->wide_reps, chunks = (size_t)w->wide_chunks, agents = 64 * chunks;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        char* p = reinterpret_cast<char*>(base) + at;
        at += (bytes + 255) & ~(size_t)255;
        return p;
    };
    m->rep = reinterpret_cast<WideWorldRep*>(take(sizeof(WideWorldRep) * reps));
    m->block = reinterpret_cast<WideWorldBlock*>(take(sizeof(WideWorldBlock) * (size_t)w->wide_blocks));
    m->member = reinterpret_cast<uint64_t*>(take(sizeof(uint64_t) * chunks * kMaxPatches));
    m->expl = reinterpret_cast<uint64_t*>(take(sizeof(uint64_t) * chunks * kMaxPatches));
    m->before = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * chunks * kMaxPatches));
    m->theta = reinterpret_cast<double*>(take(sizeof(double) * agents));
    m->patch = reinterpret_cast<uint8_t*>(take(agents));
    m->flag = reinterpret_cast<uint8_t*>(take(agents));
    m->after = reinterpret_cast<PatchAfter*>(take(sizeof(PatchAfter) * reps * kMaxPatches));
    m->geo = reinterpret_cast<PatchLds*>(take(sizeof(PatchLds) * reps));
    m->ctl = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * kWwWords * reps));
    return at;
}

// Which kernel updates which replica: the update kernel those without visual
// exclusion that fit one workgroup's LDS, the step kernel those with it, and
// the wide launches those beyond one workgroup's LDS, or every replica without
// visual exclusion: on request (ABM_FORAGE_PATH_SWEEP), or when the batch's
// agents are too few to fill the GPU a workgroup per replica and some replica
// has work for more than one CU (ms a step, wide against a workgroup each: one
// replica of 512 agents 0.039 and 0.090, of 128 0.029 and 0.037, of 60 0.026
// both, of 10 0.025 and 0.020; 30 of 512 0.067 and 0.132, 50 of 300 0.066 and
// 0.093, 100 of 8 to 512 0.064 and 0.113; 300 of 100 0.085 and 0.074, 1000 of 8
// to 512 0.226 and 0.148).  A kernel's blocks take their replicas
// largest first (the cost grows with the agents; rays add to each agent's).
// The lists are made once: a captured step keeps order_dev's address, and its
// replays take the same replicas whatever path is chosen later.
int plan_classes(abm_forage_batch* bt) {
    const int n = bt->n_replicas;
    std::vector<int32_t> plain, narrow, occl, crowd, big, spread;
    int64_t agents = 0;
    int largest = 0;
    for (int b = 0; b < n; ++b) {
        const bool wideable = !bt->exclusion[b] && bt->rep_r[b] <= kWideMaxRays;
        if (wideable) {
            agents += bt->rep_n[b];
            largest = std::max(largest, bt->rep_n[b]);
        }
        if (bt->too_big[b]) big.push_back(b);
        else if (bt->exclusion[b]) (bt->rep_n[b] <= kOcclMaxAgents ? occl : crowd).push_back(b);
        else plain.push_back(b);
        if (!bt->too_big[b] && !bt->exclusion[b] && !wideable) narrow.push_back(b);
        if (bt->too_big[b] || wideable) spread.push_back(b);
    }
    bt->spread_auto = largest >= kWideMinAgents && agents <= (int64_t)kWideMaxPerCu * bt->cus;
    auto cost = [&](int b) { return (double)bt->rep_n[b] * (64.0 + bt->rep_r[b] / 32.0); };
    std::vector<int32_t> order;
    auto add = [&](std::vector<int32_t>& v, ForageClass& c) {
        std::stable_sort(v.begin(), v.end(), [&](int a, int d) { return cost(a) > cost(d); });
        c.first = (int32_t)order.size();
        c.count = (int32_t)v.size();
        for (int b : v) {
            c.max_agents = std::max(c.max_agents, bt->rep_n[b]);
            c.max_rays = std::max(c.max_rays, bt->rep_r[b]);
        }
        order.insert(order.end(), v.begin(), v.end());
    };
    add(plain, bt->plain);
    add(narrow, bt->narrow);
    add(occl, bt->occl);
    add(crowd, bt->crowd);
    bt->wide[0].reps = big;
    bt->wide[1].reps = spread;
    for (WidePlan& w : bt->wide)
        for (int b : w.reps) w.max_rays = std::max(w.max_rays, bt->rep_r[b]);
    const size_t bytes = sizeof(int32_t) * order.size();
    if (int rc = check_hip(hipMalloc(&bt->order_dev, std::max(bytes, sizeof(int32_t))), "hipMalloc(forage order)")) return rc;
    return check_hip(hipMemcpy(bt->order_dev, order.data(), bytes, hipMemcpyHostToDevice), "upload forage order");
}

// Takes a path, with the scratch it needs; a failure leaves the one in use.
int take_path(abm_forage_batch* bt, int path) {
    std::lock_guard<std::mutex> guard(bt->wide_lock);
    const bool spread = path == ABM_FORAGE_PATH_SWEEP || bt->spread_auto;
    if (int rc = make_wide(bt, bt->wide[spread])) return rc;
    bt->path = path;
    bt->spread = spread;
    return ABM_OK;
}

// Waves of the update kernel's workgroups: sixteen, so that a large replica's
// agents share a CU's four SIMDs (1000 replicas of 8 to 512 agents: 0.140 ms a
// step with sixteen, 0.161 with eight, 0.237 with four; 300 of 300 agents:
// 0.126, 0.126, 0.179); four where more workgroups than two per CU queue and no
// replica has work for more (1000 replicas of 10 agents: 0.048 ms with four,
// 0.070 with sixteen; of 50: 0.068, 0.090; of 128: 0.121, 0.137).  Fewer too
// where the waves' fields would not fit in LDS, or a launch would have 2^32 threads.
int upd_waves(const ForageClass& c, int cus) {
    int waves = c.count > 2 * cus && c.max_agents <= 128 ? 4 : 16;
    while (waves > 4 && (upd_lds_bytes(c.max_agents, c.max_rays, waves) > (size_t)163840 - sizeof(FGRep) ||
                         ((int64_t)c.count * 64 * waves) >> 32 != 0))
        waves /= 2;
    return waves;
}

int check_state(const abm_forage_state* st, const char* who) {
    const void* req[] = {st->x, st->y, st->theta, st->v, st->w, st->u, st->I_priv, st->collected_r,
                         st->collected_r_before, st->novelty, st->mode, st->overriding_mode,
                         st->env_status, st->exploited_patch_id, st->radius};
    for (const void* p : req)
        if (!p) return set_error(ABM_ERR_INVALID, "%s: every state array is required", who);
    return ABM_OK;
}

// A launch has fewer than 2^32 threads: 64-agent chunks per field launch (2^30
// threads, beside one workgroup per replica).
constexpr int kFieldChunks = 1 << 18;

// Agent.update of a plan's replicas (see wide_drive_kernel) on scratch m.
int wide_launches(const abm_forage_batch* b, const WidePlan& plan, const WideMem& m, const abm_forage_state* st,
                  const double* uniforms, const uint32_t* words, const int64_t* offset, const int32_t* count,
                  int32_t* used, int32_t* status, uint32_t* field_bits, hipStream_t s, abm_mt19937_state* mt) {
    const int n = (int)plan.reps.size(), chunks = plan.chunks, W = (plan.max_rays + 31) / 32;
    const FGRep* reps = (const FGRep*)b->reps_dev;
    const int blocks = (chunks + 3) / 4;
    hipLaunchKernelGGL(wide_drive_kernel, dim3(blocks), dim3(256), 0, s, reps, chunks, *st, status, used,
                       (words || mt) ? 1 : 0, m);
    if (int rc = check_hip(hipGetLastError(), "wide_drive_kernel launch")) return rc;
    const size_t lds = sizeof(uint32_t) * (size_t)std::max(kMtN, 4 * W);
    for (int c = 0; c < chunks; c += kFieldChunks) {
        const abm_mt19937_state* gen = c == 0 ? mt : nullptr;
        hipLaunchKernelGGL(field_bits ? wide_field_kernel<true> : wide_field_kernel<false>,
                           dim3(16 * std::min(kFieldChunks, chunks - c) + (gen ? n : 0)), dim3(256), lds, s, reps, n, c,
                           *st, m, gen, field_bits);
        if (int rc = check_hip(hipGetLastError(), "wide_field_kernel launch")) return rc;
    }
    hipLaunchKernelGGL(wide_move_kernel, dim3(blocks), dim3(256), 0, s, reps, chunks, *st, uniforms, words, offset,
                       count, used, status, mt, m);
    if (int rc = check_hip(hipGetLastError(), "wide_move_kernel launch")) return rc;
    return ABM_OK;
}

int wide_clear(const WidePlan& plan, const WideMem& m, hipStream_t s) {
    const int n = kWdWords * (int)plan.reps.size();
    hipLaunchKernelGGL(wide_clear_kernel, dim3((n + 255) / 256), dim3(256), 0, s, m.ctl, n);
    return check_hip(hipGetLastError(), "wide_clear_kernel launch");
}

// A scratch other than the null stream's, allocated (also while a stream is
// captured: in relaxed mode) by the first step that needs it and freed with the
// batch.
constexpr int kMaxCaptures = 1024;
int other_scratch(abm_forage_batch* b, int plan, unsigned long long capture, hipStream_t s, WideMem* m,
                  WideScratch** out) {
    const WidePlan& w = b->wide[plan];
    const WideMem base = wide_mem(w);
    WideScratch* c = b->scratch;
    while (c && !(c->plan == plan && c->capture == capture && c->stream == s)) c = c->next;
    if (!c) {
        if (capture && b->n_captures >= kMaxCaptures)
            return set_error(ABM_ERR_UNSUPPORTED, "forage update over the whole GPU: %d captures of this batch hold "
                             "scratch until it is destroyed", kMaxCaptures);
        c = new (std::nothrow) WideScratch;
        if (!c) return set_error(ABM_ERR_HIP, "forage update over the whole GPU: out of host memory");
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        int rc = check_hip(hipThreadExchangeStreamCaptureMode(&mode), "capture mode");
        if (!rc) {
            rc = check_hip(hipMalloc(&c->mem, wide_carve(nullptr, w.reps.size(), (size_t)w.chunks, (size_t)w.keys, m)),
                           "hipMalloc(wide update)");
            (void)hipThreadExchangeStreamCaptureMode(&mode);
        }
        if (rc) {
            delete c;
            return rc;
        }
        c->plan = plan; c->capture = capture; c->stream = s;
        c->next = b->scratch;
        b->scratch = c;
        b->n_captures += capture != 0;
    }
    wide_carve(c->mem, w.reps.size(), (size_t)w.chunks, (size_t)w.keys, m);
    m->rep = base.rep; m->of = base.of; m->updates = base.updates;
    *out = c;
    return ABM_OK;
}

// Agent.update of the wide replicas.  Calls on one batch may come from several
// streams and threads, each with its own state, and may not share scratch while
// they run.  The null stream has its own: its calls are in order, it cannot be
// destroyed, and an event after each call would cost 3 us (8192 agents 63.4 ->
// 66.4 us a step).  The other streams share one, each call behind an event of the
// one before.  A captured step cannot wait for calls outside its graph, nor they
// for its replays: its capture has scratch of its own.
int launch_wide(abm_forage_batch* b, int plan, const abm_forage_state* st, const double* uniforms,
                const uint32_t* words, const int64_t* offset, const int32_t* count, int32_t* used,
                int32_t* status, uint32_t* field_bits, hipStream_t s, abm_mt19937_state* mt) {
    std::lock_guard<std::mutex> guard(b->wide_lock);
    WidePlan& w = b->wide[plan];
    if (!w.mem) return set_error(ABM_ERR_HIP, "forage update over the whole GPU: no scratch");
    WideMem m = wide_mem(w);
    bool* clean = &w.clean;
    hipStreamCaptureStatus state = hipStreamCaptureStatusNone;
    unsigned long long capture = 0;
    if (s)
        if (int rc = check_hip(hipStreamGetCaptureInfo(s, &state, &capture), "hipStreamGetCaptureInfo")) return rc;
    const bool captured = state != hipStreamCaptureStatusNone;
    if (s) {
        WideScratch* c = nullptr;
        if (int rc = other_scratch(b, plan, captured ? capture : 0, captured ? s : nullptr, &m, &c)) return rc;
        clean = &c->clean;
        if (!captured)
            if (int rc = check_hip(hipStreamWaitEvent(s, b->wide_done, 0), "hipStreamWaitEvent")) return rc;
    }
    // The last launch of a step leaves the cue counts 0.  After a call that failed
    // before it, and on new scratch (a graph's first replay), they are cleared first.
    int rc = captured || !*clean ? wide_clear(w, m, s) : ABM_OK;
    *clean = false;
    if (!rc) rc = wide_launches(b, w, m, st, uniforms, words, offset, count, used, status, field_bits, s, mt);
    *clean = rc == ABM_OK && !captured;
    if (!s || captured) return rc;
    const int done = check_hip(hipEventRecord(b->wide_done, s), "hipEventRecord");
    if (done) (void)hipDeviceSynchronize();   // no event to wait for: nothing may be left
    return rc ? rc : done;
}

// Agent.update for every replica (all, or those a status array marks ready).
int launch_forage_step(abm_forage_batch* b, const abm_forage_state* st, const double* uniforms,
                       const uint32_t* words, const int64_t* offset, const int32_t* count,
                       int32_t* used, int32_t* status, uint32_t* field_bits, void* stream,
                       abm_mt19937_state* mt = nullptr) {
    const int32_t* const order = (const int32_t*)b->order_dev;
    const bool spread = b->spread;
    if (const ForageClass& c = spread ? b->narrow : b->plain; c.count > 0) {
        const int waves = upd_waves(c, b->cus);
        const size_t lds = upd_lds_bytes(c.max_agents, c.max_rays, waves);
        auto kern = field_bits ? forage_update_kernel<true> : forage_update_kernel<false>;
        if (lds > 65536) {
            if (int rc = check_hip(hipFuncSetAttribute((const void*)kern,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                                   "hipFuncSetAttribute"))
                return rc;
        }
        hipLaunchKernelGGL(kern, dim3(c.count), dim3(64 * waves), lds, (hipStream_t)stream,
                           (const FGRep*)b->reps_dev, *st, uniforms, words, offset, count, used, status,
                           field_bits, order + c.first, mt, c.max_agents);
        if (int rc = check_hip(hipGetLastError(), "forage_update_kernel launch")) return rc;
    }
    if (const ForageClass& c = b->occl; c.count > 0) {
        const int K = c.max_agents <= 64 ? 1 : (c.max_agents <= 128 ? 2 : 4);
        const size_t lds = occl_lds_bytes(c.max_agents, c.max_rays, K);
        auto kern = field_bits ? (K == 1 ? forage_occlude_kernel<1, true>
                                         : (K == 2 ? forage_occlude_kernel<2, true> : forage_occlude_kernel<4, true>))
                               : (K == 1 ? forage_occlude_kernel<1, false>
                                         : (K == 2 ? forage_occlude_kernel<2, false> : forage_occlude_kernel<4, false>));
        if (lds > 65536) {
            if (int rc = check_hip(hipFuncSetAttribute((const void*)kern,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                                   "hipFuncSetAttribute"))
                return rc;
        }
        hipLaunchKernelGGL(kern, dim3(c.count), dim3(64 * kOcclWaves), lds, (hipStream_t)stream,
                           (const FGRep*)b->reps_dev, *st, uniforms, words, offset, count, used, status,
                           field_bits, order + c.first, mt, c.max_agents);
        if (int rc = check_hip(hipGetLastError(), "forage_occlude_kernel launch")) return rc;
    }
    if (const ForageClass& c = b->crowd; c.count > 0) {   // visual exclusion beyond its registers
        const size_t lds = fg_lds_bytes(c.max_agents, c.max_rays);
        auto kern = field_bits ? forage_step_kernel<true> : forage_step_kernel<false>;
        if (lds > 65536) {
            if (int rc = check_hip(hipFuncSetAttribute((const void*)kern,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                                   "hipFuncSetAttribute"))
                return rc;
        }
        hipLaunchKernelGGL(kern, dim3(c.count), dim3(512), lds, (hipStream_t)stream,
                           (const FGRep*)b->reps_dev, *st, uniforms, words, offset, count, used, status,
                           field_bits, order + c.first, mt, c.max_agents, c.max_rays);
        if (int rc = check_hip(hipGetLastError(), "forage_step_kernel launch")) return rc;
    }
    if (!b->wide[spread].reps.empty())
        return launch_wide(b, spread, st, uniforms, words, offset, count, used, status, field_bits, (hipStream_t)stream, mt);
    return ABM_OK;
}

}  // namespace

extern "C" {

int abm_forage_batch_create(const abm_forage_replica* reps, int32_t n, abm_forage_batch** out) {
    if (!out) return set_error(ABM_ERR_INVALID, "abm_forage_batch_create: out is NULL");
    *out = nullptr;
    if (!reps || n <= 0) return set_error(ABM_ERR_INVALID, "abm_forage_batch_create: no replicas");
    std::vector<FGRep> host(n);
    int64_t agents = 0, words = 0;
    int max_n = 0, max_r = 0;
    for (int b = 0; b < n; ++b) {
        const abm_forage_replica& r = reps[b];
        if (r.n_agents < 1 || r.n_agents > kForageMaxAgents)
            return set_error(ABM_ERR_INVALID, "forage replica %d: n_agents=%d out of range [1, %d]", b,
                             r.n_agents, kForageMaxAgents);
        if (r.n_rays < 2 || r.n_rays > (1 << 16))
            return set_error(ABM_ERR_INVALID, "forage replica %d: n_rays=%d out of range", b, r.n_rays);
        if (r.tau < 1 || r.tau > 4096)
            return set_error(ABM_ERR_INVALID, "forage replica %d: tau=%d out of range", b, r.tau);
        FGRep& d = host[b];
        std::memset(&d, 0, sizeof(d));
        d.agent_offset = (int32_t)agents; d.n_agents = r.n_agents; d.n_rays = r.n_rays;
        d.words = (r.n_rays + 31) / 32; d.visual_exclusion = r.visual_exclusion ? 1 : 0;
        d.patchwise = r.patchwise_exclusion ? 1 : 0; d.tau = r.tau; d.field_offset = words;
        d.fov0 = r.fov0; d.fov1 = r.fov1; d.width = r.width; d.height = r.height;
        d.pad = r.window_pad; d.vision_range = r.vision_range; d.step = linspace_step(r.n_rays);
        d.T_w = r.T_w; d.Eps_w = r.Eps_w; d.g_w = r.g_w; d.B_w = r.B_w; d.w_max = r.w_max;
        d.T_u = r.T_u; d.Eps_u = r.Eps_u; d.g_u = r.g_u; d.B_u = r.B_u; d.u_max = r.u_max;
        d.S_wu = r.S_wu; d.S_uw = r.S_uw; d.F_N = r.F_N; d.F_R = r.F_R;
        d.exp_vel_max = r.exp_vel_max; d.exp_theta_min = r.exp_theta_min;
        d.exp_theta_max = r.exp_theta_max; d.reloc_theta_max = r.reloc_theta_max;
        d.exp_stop_ratio = r.exp_stop_ratio;
        // soc_v_field[k] survives the FOV mask unless linspace_k < fov0 or
        // > fov1 (agent.py:593-595); linspace is monotonic, so the kept
        // indices form one range
        int lo = r.n_rays, hi = -1, kept = 0;
        for (int k = 0; k < r.n_rays; ++k) {
            const double ph = linspace_at(k, r.n_rays, d.step);
            if (ph < r.fov0 || ph > r.fov1) continue;
            if (lo == r.n_rays) lo = k;
            hi = k;
            ++kept;
        }
        if (kept != (hi >= lo ? hi - lo + 1 : 0))
            return set_error(ABM_ERR_INVALID, "forage replica %d: the FOV keeps no single ray range", b);
        d.keep_lo = lo; d.keep_hi = hi;
        agents += r.n_agents;
        words += (int64_t)r.n_agents * d.words;
        max_n = std::max(max_n, r.n_agents);
        max_r = std::max(max_r, r.n_rays);
    }
    abm_forage_batch* bt = new abm_forage_batch();
    bt->n_replicas = n; bt->n_agents_total = (int32_t)agents; bt->field_words = words;
    bt->max_agents = max_n; bt->max_rays = max_r;
    int rc = check_hip(hipGetDevice(&bt->device), "hipGetDevice");
    if (!rc) rc = check_hip(hipDeviceGetAttribute(&bt->cus, hipDeviceAttributeMultiprocessorCount, bt->device),
                            "hipDeviceGetAttribute");
    int dev_max = 0;
    if (!rc) rc = check_hip(hipDeviceGetAttribute(&dev_max, hipDeviceAttributeMaxSharedMemoryPerBlock,
                                                  bt->device), "hipDeviceGetAttribute");
    // a replica beyond one workgroup's LDS is updated over the whole GPU,
    // without visual exclusion and with at most 8192 rays.  One measure for all:
    // the step kernel's layout, the largest (172 bytes an agent and a byte a ray,
    // where the update kernel needs 152 and its waves' fields), so what a batch
    // accepts does not depend on the kernel that takes a replica
    bt->too_big.assign(n, 0);
    bt->exclusion.assign(n, 0);
    for (int b = 0; !rc && b < n; ++b) {
        const size_t need = fg_lds_bytes(host[b].n_agents, host[b].n_rays) + sizeof(FGRep);
        bt->too_big[b] = need > (size_t)dev_max;
        bt->exclusion[b] = host[b].visual_exclusion != 0;
        if (bt->too_big[b] && (host[b].visual_exclusion || host[b].n_rays > kWideMaxRays))
            rc = set_error(ABM_ERR_UNSUPPORTED, "forage replica %d: %d agents x %d rays need %zu B of LDS "
                           "(one workgroup has %d B); replicas that large are updated over the whole GPU, which "
                           "supports neither visual exclusion nor more than %d rays", b, host[b].n_agents,
                           host[b].n_rays, need, dev_max, kWideMaxRays);
    }
    bt->rep_n.resize(n);
    bt->rep_r.resize(n);
    for (int b = 0; b < n; ++b) { bt->rep_n[b] = host[b].n_agents; bt->rep_r[b] = host[b].n_rays; }
    if (!rc) rc = check_hip(hipMalloc(&bt->reps_dev, sizeof(FGRep) * n), "hipMalloc(forage replicas)");
    if (!rc) rc = check_hip(hipMemcpy(bt->reps_dev, host.data(), sizeof(FGRep) * n, hipMemcpyHostToDevice),
                           "upload forage replicas");
    if (!rc) rc = plan_classes(bt);
    if (!rc) rc = take_path(bt, ABM_FORAGE_PATH_AUTO);
    if (rc) { abm_forage_batch_destroy(bt); return rc; }
    bt->agent_offset_host = new int32_t[n + 1];
    bt->field_offset_host = new int64_t[n + 1];
    for (int b = 0; b < n; ++b) {
        bt->agent_offset_host[b] = host[b].agent_offset;
        bt->field_offset_host[b] = host[b].field_offset;
    }
    bt->agent_offset_host[n] = (int32_t)agents;
    bt->field_offset_host[n] = words;
    *out = bt;
    return ABM_OK;
}

int abm_forage_batch_destroy(abm_forage_batch* b) {
    if (!b) return ABM_OK;
    if (b->reps_dev) (void)hipFree(b->reps_dev);
    if (b->order_dev) (void)hipFree(b->order_dev);
    for (const WidePlan& w : b->wide)
        if (w.mem) (void)hipFree(w.mem);
    if (b->wide_done) (void)hipEventDestroy(b->wide_done);
    while (WideScratch* c = b->scratch) {
        b->scratch = c->next;
        (void)hipFree(c->mem);
        delete c;
    }
    delete[] b->agent_offset_host;
    delete[] b->field_offset_host;
    delete b;
    return ABM_OK;
}

int abm_forage_batch_get_info(const abm_forage_batch* b, abm_batch_info* out) {
    if (!b || !out) return set_error(ABM_ERR_INVALID, "abm_forage_batch_get_info: NULL argument");
    out->n_replicas = b->n_replicas; out->n_agents_total = b->n_agents_total;
    out->field_words = b->field_words; out->max_agents = b->max_agents; out->max_rays = b->max_rays;
    return ABM_OK;
}

int abm_forage_batch_get_offsets(const abm_forage_batch* b, int32_t* agent_offset, int64_t* field_offset) {
    if (!b) return set_error(ABM_ERR_INVALID, "abm_forage_batch_get_offsets: NULL batch");
    if (agent_offset) std::copy(b->agent_offset_host, b->agent_offset_host + b->n_replicas + 1, agent_offset);
    if (field_offset) std::copy(b->field_offset_host, b->field_offset_host + b->n_replicas + 1, field_offset);
    return ABM_OK;
}


int abm_forage_sweep_counts(const abm_forage_batch* b, int64_t* updates, int64_t* sweeps) {
    if (!b || !updates || !sweeps) return set_error(ABM_ERR_INVALID, "abm_forage_sweep_counts: NULL argument");
    int64_t made = 0;
    std::lock_guard<std::mutex> guard(b->wide_lock);
    if (int rc = wide_updates(b, &made)) return rc;
    *updates = *sweeps = made;
    return ABM_OK;
}

int abm_forage_set_path(abm_forage_batch* b, int32_t path) {
    if (!b) return set_error(ABM_ERR_INVALID, "abm_forage_set_path: NULL batch");
    if (path != ABM_FORAGE_PATH_AUTO && path != ABM_FORAGE_PATH_SWEEP)
        return set_error(ABM_ERR_INVALID, "abm_forage_set_path: unknown path %d", path);
    return take_path(b, path);
}

int abm_forage_step_f64(abm_forage_batch* b, const abm_forage_state* st, const double* uniforms,
                        const int64_t* uniform_offset, const int32_t* uniform_count,
                        int32_t* uniforms_used, uint32_t* field_bits, void* stream) {
    if (!b || !st) return set_error(ABM_ERR_INVALID, "abm_forage_step_f64: NULL batch or state");
    if (int rc = check_state(st, "abm_forage_step_f64")) return rc;
    if (!uniforms || !uniform_offset || !uniform_count)
        return set_error(ABM_ERR_INVALID, "abm_forage_step_f64: the uniform buffer is required");
    return launch_forage_step(b, st, uniforms, nullptr, uniform_offset, uniform_count, uniforms_used,
                              nullptr, field_bits, stream);
}

int abm_forage_world_create(abm_forage_batch* b, const abm_forage_world_params* params,
                            abm_forage_world** out) {
    if (!out) return set_error(ABM_ERR_INVALID, "abm_forage_world_create: out is NULL");
    *out = nullptr;
    if (!b || !params) return set_error(ABM_ERR_INVALID, "abm_forage_world_create: NULL batch or params");
    const int n = b->n_replicas;
    std::vector<FGRep> reps(n);
    if (int rc = check_hip(hipMemcpy(reps.data(), b->reps_dev, sizeof(FGRep) * n, hipMemcpyDeviceToHost),
                           "download forage replicas"))
        return rc;
    std::vector<WRep> host(n);
    int64_t total = 0;
    size_t lds = 8, collide_lds = 0;
    const int64_t kRange = 0xFFFFFFFEll;   // randint ranges up to 2^32 - 2 values
    for (int i = 0; i < n; ++i) {
        const abm_forage_world_params& q = params[i];
        WRep& w = host[i];
        std::memset(&w, 0, sizeof(w));
        if (q.n_patches < 0 || q.n_patches > kMaxPatches)
            return set_error(ABM_ERR_INVALID, "forage world %d: n_patches=%d out of range [0, %d]", i,
                             q.n_patches, kMaxPatches);
        if (q.patch_radius < 0)
            return set_error(ABM_ERR_INVALID, "forage world %d: negative patch radius", i);
        w.n_patches = q.n_patches; w.patch_radius = q.patch_radius; w.pooling_time = q.pooling_time;
        w.regenerate = q.regenerate ? 1 : 0; w.teleport = q.teleport_exploit ? 1 : 0;
        w.collide = q.collide_agents ? 1 : 0; w.ghost = q.ghost_mode ? 1 : 0;
        if (w.collide && reps[i].n_agents > kCollideMaxAgents)
            return set_error(ABM_ERR_UNSUPPORTED, "forage world %d: agent-agent collisions for up to %d "
                             "agents per replica (got %d)", i, kCollideMaxAgents, reps[i].n_agents);
        if (w.collide)
            collide_lds = std::max(collide_lds, collide_lds_bytes(reps[i].n_agents, reps[i].n_rays));
        w.n_agents = reps[i].n_agents;
        w.patch_offset = total;
        // the bounds numpy sees: int() of the Python expressions (sims.py:349-356)
        const double r = (double)q.patch_radius, pad = reps[i].pad;
        const double W = reps[i].width, H = reps[i].height;
        if (q.allow_border_overlap) {
            w.x_lo = (int64_t)trunc(pad - r); w.x_hi = (int64_t)trunc(W + pad - r);
            w.y_lo = (int64_t)trunc(pad - r); w.y_hi = (int64_t)trunc(H + pad - r);
        } else {
            w.x_lo = (int64_t)trunc(pad); w.x_hi = (int64_t)trunc(W + pad - 2.0 * r);
            w.y_lo = (int64_t)trunc(pad); w.y_hi = (int64_t)trunc(H + pad - 2.0 * r);
        }
        w.units_lo = q.min_units; w.units_hi = q.max_units;
        const int64_t lo[] = {w.x_lo, w.y_lo, w.units_lo}, hi[] = {w.x_hi, w.y_hi, w.units_hi};
        for (int k = 0; k < 3; ++k)
            if (q.n_patches > 0 && (hi[k] <= lo[k] || hi[k] - 1 - lo[k] > kRange))
                return set_error(ABM_ERR_INVALID, "forage world %d: randint(%lld, %lld) has no values "
                                 "(numpy raises low >= high) or too many", i, (long long)lo[k],
                                 (long long)hi[k]);
        w.consumption = q.consumption; w.q_lo = q.min_quality; w.q_hi = q.max_quality;
        if (!std::isfinite(q.max_quality - q.min_quality))
            return set_error(ABM_ERR_INVALID, "forage world %d: quality range is not finite", i);
        total += q.n_patches;
        lds = std::max(lds, sizeof(uint64_t) * (size_t)q.n_patches * (size_t)((reps[i].n_agents + 63) / 64));
    }
    abm_forage_world* wd = new abm_forage_world();
    wd->batch = b; wd->n_replicas = n; wd->patch_total = total; wd->member_lds = lds;
    wd->collide_lds = collide_lds;
    // the world kernel's workgroups: a thread per agent of the replicas that
    // take one workgroup, membership words of every patch and of its
    // exploiting agents; the larger replicas' blocks and chunks
    std::vector<WideWorldRep> wide;
    std::vector<WideWorldBlock> blocks;
    int64_t chunks = 0;
    int threads = 256;
    for (int i = 0; i < n; ++i) {
        const int N = reps[i].n_agents;
        if (N > kWorldBlockAgents) {
            for (int a = 0; a < N; a += 64) blocks.push_back(WideWorldBlock{(int32_t)wide.size(), a});
            wide.push_back(WideWorldRep{i, (int32_t)chunks});
            chunks += (N + 63) / 64;
        } else {
            while (threads < N) threads *= 2;
            wd->world_lds = std::max(wd->world_lds, 2 * sizeof(uint64_t) * (size_t)host[i].n_patches *
                                                        (size_t)((N + 63) / 64));
        }
    }
    wd->threads = threads;
    wd->wide_reps = (int32_t)wide.size();
    wd->wide_blocks = (int32_t)blocks.size();
    wd->wide_chunks = chunks;
    if (collide_lds > (size_t)163840) {
        delete wd;
        return set_error(ABM_ERR_UNSUPPORTED, "forage world: the collision kernel needs %zu B of LDS",
                         collide_lds);
    }
    const size_t slots = (size_t)std::max<int64_t>(total, 1);
    int rc = check_hip(hipMalloc(&wd->wreps_dev, sizeof(WRep) * n), "hipMalloc(world replicas)");
    if (!rc) rc = check_hip(hipMalloc(&wd->kill_rank, sizeof(int32_t) * slots), "hipMalloc(kill ranks)");
    if (!rc) rc = check_hip(hipMalloc(&wd->pend, sizeof(int32_t) * 2 * n), "hipMalloc(pending)");
    if (!rc) rc = check_hip(hipMalloc(&wd->pend_id, sizeof(int32_t) * slots), "hipMalloc(pending ids)");
    if (!rc) rc = check_hip(hipMemcpy(wd->wreps_dev, host.data(), sizeof(WRep) * n, hipMemcpyHostToDevice),
                           "upload world replicas");
    if (!rc) rc = check_hip(hipMemset(wd->kill_rank, 0xff, sizeof(int32_t) * slots), "clear kill ranks");
    if (!rc) rc = check_hip(hipMemset(wd->pend, 0, sizeof(int32_t) * 2 * n), "clear pending");
    if (!rc && wd->wide_reps > 0) {
        WideWorld ww;
        const size_t bytes = wide_world_carve(nullptr, wd, &ww);
        rc = check_hip(hipMalloc(&wd->wide_mem, bytes), "hipMalloc(wide world)");
        if (!rc) {
            wide_world_carve(wd->wide_mem, wd, &ww);
            rc = check_hip(hipMemset(ww.ctl, 0, sizeof(int32_t) * kWwWords * wide.size()), "clear wide world control");
        }
        if (!rc) rc = check_hip(hipMemcpy(const_cast<WideWorldRep*>(ww.rep), wide.data(),
                                          sizeof(WideWorldRep) * wide.size(), hipMemcpyHostToDevice),
                                "upload wide world replicas");
        if (!rc) rc = check_hip(hipMemcpy(const_cast<WideWorldBlock*>(ww.block), blocks.data(),
                                          sizeof(WideWorldBlock) * blocks.size(), hipMemcpyHostToDevice),
                                "upload wide world blocks");
    }
    if (!rc) rc = check_hip(hipDeviceSynchronize(), "world create");
    if (rc) { abm_forage_world_destroy(wd); return rc; }
    wd->patch_offset_host = new int64_t[n + 1];
    for (int i = 0; i < n; ++i) wd->patch_offset_host[i] = host[i].patch_offset;
    wd->patch_offset_host[n] = total;
    *out = wd;
    return ABM_OK;
}

int abm_forage_world_destroy(abm_forage_world* w) {
    if (!w) return ABM_OK;
    if (w->wreps_dev) (void)hipFree(w->wreps_dev);
    if (w->kill_rank) (void)hipFree(w->kill_rank);
    if (w->pend) (void)hipFree(w->pend);
    if (w->pend_id) (void)hipFree(w->pend_id);
    if (w->wide_mem) (void)hipFree(w->wide_mem);
    delete[] w->patch_offset_host;
    delete w;
    return ABM_OK;
}

int abm_forage_world_get_offsets(const abm_forage_world* w, int64_t* patch_offset) {
    if (!w || !patch_offset) return set_error(ABM_ERR_INVALID, "abm_forage_world_get_offsets: NULL argument");
    std::copy(w->patch_offset_host, w->patch_offset_host + w->n_replicas + 1, patch_offset);
    return ABM_OK;
}

}  // extern "C"

namespace {

// One phase of the resource loop; the placements and the walk draw from a
// word buffer (words) or from device generators (mt).
int world_run(abm_forage_world* w, int32_t phase, const abm_forage_state* st, int32_t* pool_success,
              const abm_patch_state* ps, const uint32_t* words, const int64_t* word_offset,
              const int32_t* word_count, int32_t* words_used, int32_t* status, uint32_t* field_bits,
              void* stream, abm_mt19937_state* mt, const char* who) {
    if (!w || !st || !ps) return set_error(ABM_ERR_INVALID, "%s: NULL world, state or patches", who);
    if (int rc = check_state(st, who)) return rc;
    if (!pool_success || !words_used || !status)
        return set_error(ABM_ERR_INVALID, "%s: pool_success, words_used and status are required", who);
    if (w->patch_total > 0 && (!ps->count || !ps->id || !ps->x || !ps->y || !ps->radius || !ps->units ||
                               !ps->left || !ps->quality))
        return set_error(ABM_ERR_INVALID, "%s: every patch array is required", who);
    if (!ps->count) return set_error(ABM_ERR_INVALID, "%s: patch count array is required", who);
    abm_forage_batch* b = w->batch;
    // (the masks of replicas above kWorldBlockAgents lie in global memory, which
    // does not need this limit; worlds beyond it are untested and refused)
    if (w->member_lds > 65536)
        return set_error(ABM_ERR_UNSUPPORTED, "%s: %zu B of membership masks", who, w->member_lds);
    if (phase == ABM_WORLD_STEP && w->collide_lds > 0) {
        // agent-agent collisions first (sims.py:736-787)
        if (w->collide_lds > 65536) {
            if (int rc = check_hip(hipFuncSetAttribute((const void*)forage_collide_kernel,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       (int)w->collide_lds), "hipFuncSetAttribute"))
                return rc;
        }
        hipLaunchKernelGGL(forage_collide_kernel, dim3(b->n_replicas), dim3(256), w->collide_lds,
                           (hipStream_t)stream, (const FGRep*)b->reps_dev, (const WRep*)w->wreps_dev, *st,
                           pool_success, w->pend, status);
        if (int rc = check_hip(hipGetLastError(), "forage_collide_kernel launch")) return rc;
    }
    const bool wide = phase == ABM_WORLD_STEP && w->wide_reps > 0;
    const FGRep* reps = (const FGRep*)b->reps_dev;
    const WRep* wreps = (const WRep*)w->wreps_dev;
    WideWorld ww{};
    if (!wide || w->wide_reps < b->n_replicas) {
        hipLaunchKernelGGL(forage_world_kernel<false>, dim3(b->n_replicas), dim3(w->threads), w->world_lds,
                           (hipStream_t)stream, reps, wreps, (int)phase, *st, pool_success, *ps, w->kill_rank,
                           w->pend, w->pend_id, words, word_offset, word_count, words_used, status, mt, ww);
        if (int rc = check_hip(hipGetLastError(), "forage_world_kernel launch")) return rc;
    }
    if (wide) {
        wide_world_carve(w->wide_mem, w, &ww);
        hipLaunchKernelGGL(wide_member_kernel, dim3(w->wide_blocks), dim3(256), 0, (hipStream_t)stream, reps, wreps,
                           *st, pool_success, *ps, ww);
        if (int rc = check_hip(hipGetLastError(), "wide_member_kernel launch")) return rc;
        hipLaunchKernelGGL(forage_world_kernel<true>, dim3(w->wide_reps), dim3(1024), 0, (hipStream_t)stream, reps,
                           wreps, (int)phase, *st, pool_success, *ps, w->kill_rank, w->pend, w->pend_id, words,
                           word_offset, word_count, words_used, status, mt, ww);
        if (int rc = check_hip(hipGetLastError(), "forage_world_kernel launch")) return rc;
        hipLaunchKernelGGL(wide_notify_kernel, dim3(w->wide_blocks), dim3(64), 0, (hipStream_t)stream, reps, wreps,
                           *st, pool_success, ww);
        if (int rc = check_hip(hipGetLastError(), "wide_notify_kernel launch")) return rc;
    }
    if (phase == ABM_WORLD_FILL) return ABM_OK;
    // the update draws its walk after the placements
    return launch_forage_step(b, st, nullptr, words, word_offset, word_count, words_used, status,
                              field_bits, stream, mt);
}

}  // namespace

extern "C" {

int abm_forage_world_run(abm_forage_world* w, int32_t phase, const abm_forage_state* st,
                         int32_t* pool_success, const abm_patch_state* ps, const uint32_t* words,
                         const int64_t* word_offset, const int32_t* word_count, int32_t* words_used,
                         int32_t* status, uint32_t* field_bits, void* stream) {
    if (phase != ABM_WORLD_STEP && phase != ABM_WORLD_RESUME && phase != ABM_WORLD_FILL)
        return set_error(ABM_ERR_INVALID, "abm_forage_world_run: unknown phase %d", phase);
    if (!words || !word_offset || !word_count)
        return set_error(ABM_ERR_INVALID, "abm_forage_world_run: the word buffer is required");
    return world_run(w, phase, st, pool_success, ps, words, word_offset, word_count, words_used, status,
                     field_bits, stream, nullptr, "abm_forage_world_run");
}

int abm_forage_world_run_dev(abm_forage_world* w, int32_t phase, const abm_forage_state* st,
                             int32_t* pool_success, const abm_patch_state* ps, abm_mt19937_state* mt,
                             int32_t* words_used, int32_t* status, uint32_t* field_bits, void* stream) {
    if (phase != ABM_WORLD_STEP && phase != ABM_WORLD_FILL)
        return set_error(ABM_ERR_INVALID, "abm_forage_world_run_dev: phase %d (STEP or FILL)", phase);
    if (!mt) return set_error(ABM_ERR_INVALID, "abm_forage_world_run_dev: NULL generator states");
    return world_run(w, phase, st, pool_success, ps, nullptr, nullptr, nullptr, words_used, status,
                     field_bits, stream, mt, "abm_forage_world_run_dev");
}

int abm_forage_projection(int32_t R, double fov0, double fov1, int32_t visual_exclusion,
                          double vision_range, int32_t keep_distance, double fx, double fy,
                          double ftheta, double fradius, const double* ox, const double* oy,
                          int32_t n_social, int32_t n_nonsocial, double* out_field, void* stream) {
    if (R < 2 || R > (1 << 16)) return set_error(ABM_ERR_INVALID, "abm_forage_projection: n_rays=%d", R);
    if (n_social < 0) return set_error(ABM_ERR_INVALID, "abm_forage_projection: n_social < 0");
    const int n = n_social + (n_nonsocial > 0 ? n_nonsocial : 0);
    if (n > 4096) return set_error(ABM_ERR_INVALID, "abm_forage_projection: more than 4096 obstacles");
    if (!out_field || (n > 0 && (!ox || !oy)))
        return set_error(ABM_ERR_INVALID, "abm_forage_projection: NULL array");
    const int maxN = n > 0 ? n : 1;
    const size_t lds = fg_lds_bytes(maxN, R);
    if (lds > 65536) {
        if (int rc = check_hip(hipFuncSetAttribute((const void*)forage_projection_kernel,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                               "hipFuncSetAttribute"))
            return rc;
    }
    hipLaunchKernelGGL(forage_projection_kernel, dim3(1), dim3(256), lds, (hipStream_t)stream, R,
                       linspace_step(R), fov0, fov1, visual_exclusion, vision_range, keep_distance,
                       fx, fy, ftheta, fradius, ox, oy, n_social, n_nonsocial, out_field, maxN);
    return check_hip(hipGetLastError(), "forage_projection_kernel launch");
}

}  // extern "C"
