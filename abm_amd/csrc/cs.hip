// cs.hip -- cooperative-signalling visual projections on the GPU.
//
// The cooperative-signalling agent (abm/projects/cooperative_signaling)
// perceives others through its own projection_field
// (cs_agent/cs_supcalc.py:204-295), which differs from the VSWRM one
// (vf_supcalc.py:20-138) in five ways:
//   * object centres and visual angles use the focal agent's radius;
//   * no periodic images;
//   * visibility is the closed-angle test fov0 <= ca <= fov1, not the pixel
//     test on start / end;
//   * an object whose projection size exceeds max_proj_size is not drawn
//     (:270, validate_projection_size :298-307);
//   * a drawn row is scaled by the object's meter (:286-287), and after the
//     flip the rays with phis < fov0 or phis > fov1 are zeroed (:291-294).
// CSAgent combines the rows two ways (cs_agent.py:83-131): the crowding
// density, rows summed over objects and divided by len(agents), and the
// signalling density, the maximum over rows.  This file computes the rows,
// the sum and the maximum for many focal agents at once, each with its own
// object list (CSR), in float64 with the reference's operation order, so the
// results equal the reference's bit for bit (up to the device libm's last ulp
// in acos / atan, which moves a decision only within an ulp of a tie).
//
// One wave per focal agent.  Lanes decide a chunk of objects; rows are written
// directly, and the two combines accumulate in the wave's LDS (see CSPath).
// The decisions are integers and comparisons (bin, half-width, field of view,
// size limit): float32 makes those it is certain of, outside guard bands, and
// the float64 code the others, so every output is the float64 one.
// Built with -ffp-contract=off.
#include <algorithm>

#include "vf_batch.hpp"
#include "vf_exact.hpp"
#include "vf_f32_common.hpp"

namespace abm {

namespace {

constexpr int kCSMaxRaysLDS = 7936;        // one wave's LDS (segments + accumulator) within 64 KB

// One object's row: not drawn (all zero), or the pieces of rays set to 1 and
// the row then multiplied by val (so 0 * val elsewhere, as numpy's row *=).
struct CSSeg {
    int a0, b0, a1, b1;
    int drawn;
    double val;
};

// A focal agent: position, centre, and its heading vector (cos th, -sin th) in
// float32 for the guarded decision.
struct CSFocal {
    double px, py, cx, cy, radius, theta;
    float ux, uy;
};

// Raster decision of one object for the cooperative-signalling field
// (cs_supcalc.py:238-287): its pieces, or x = -1 when it is not drawn.  Out of
// line: few objects take it, and inlined its registers halve the waves in
// flight.
__device__ __noinline__ int4 cs_segment(double px, double py, double radius, double theta, double ox, double oy,
                                        int R, double step, double fov0, double fov1, int has_max,
                                        double max_proj) {
#pragma clang fp contract(off)
    const int4 none = make_int4(-1, 0, 0, 0);
    const Focal f = make_focal(px, py, theta, radius);
    const double ocx = ox + f.radius;                         // focal radius (:244)
    const double ocy = oy + f.radius;
    const double v2x = ocx - f.cx;                            // :247
    const double v2y = ocy - f.cy;
    const double ca = closed_angle_vf(f, v2x, v2y, norm2(v2x, v2y));   // :250
    const double dist = norm2(ocx - f.cx, ocy - f.cy);       // :252
    const double vis = 2.0 * atan(f.radius / (1.0 * dist));  // :255
    const int t = linspace_argmin(ca, R, step);               // :258
    if (!(fov0 <= ca && ca <= fov1)) return none;             // :262
    const double ps = (vis / kTwoPi) * (double)R;             // :267
    if (has_max && !(ps <= max_proj)) return none;            // :270
    const int h = (int)floor(ps / 2.0);                       // :273-274
    int4 s;
    vf_pieces(t - h, t + h, R, &s.x, &s.y, &s.z, &s.w);      // :277-284
    return s;
}

// Per-launch float32 constants of the guarded decision.
struct CSFast {
    float inv_step, hs, g_bins, fov0, fov1, max_proj;
};
__device__ inline CSFast cs_fast(int R, double step, double fov0, double fov1, double max_proj) {
    CSFast q;
    q.inv_step = (float)(1.0 / step);
    q.hs = (float)((double)R / kTwoPi);
    q.g_bins = (float)(f32::kAngleGuardF / step + 1.5e-7 * R);
    q.fov0 = (float)fov0; q.fov1 = (float)fov1; q.max_proj = (float)max_proj;
    return q;
}

// The pieces of one object.  The centre difference is the float64 one and the
// heading vector a float64 one (within 1e-11), each rounded once, so the
// float32 closed angle is within 1e-6 rad of the exact one (vf_f32_common.hpp):
// bands of 4e-6 rad around the bin ties, the +-pi wrap and the two ends of the
// field of view, of 4e-6 relative + 1e-6 around an integer half-width, and the
// same around the size limit (of the whole projection, twice that) go to
// cs_segment.
__device__ inline CSSeg cs_segment_guarded(const CSFocal& f, double ox, double oy, double meter, int R,
                                           double step, double fov0, double fov1, int has_max,
                                           double max_proj, const CSFast& Q) {
#pragma clang fp contract(off)
    CSSeg s{0, 0, 0, 0, 0, 0.0};
    if (ox == f.px && oy == f.py) return s;                  // coincident (:240)
    const float dx = (float)((ox + f.radius) - f.cx), dy = (float)((oy + f.radius) - f.cy);
    const float d2 = fmaf(dy, dy, dx * dx);
    const float a = f32::atan2_f32(fmaf(f.ux, dy, -f.uy * dx), fmaf(f.ux, dx, f.uy * dy)), ca = -a;
    const float z = (float)f.radius * __builtin_amdgcn_rsqf(d2);
    const float xb = (f32::kPiF - a) * Q.inv_step, tr = rintf(xb), dfr = xb - tr;
    const float half = f32::atan_unit_f32(z) * Q.hs;
    const float hfl = floorf(half), hfrac = half - hfl, hg = 4e-6f * fabsf(half) + 1e-6f;
    const float g = f32::kAngleGuardF;
    const bool ok = (d2 > 1e-30f) & (fabsf(z) < 1.0f) & (fabsf(a) < f32::kPiF - g) &
                    (fabsf(dfr) <= 0.5f - Q.g_bins) & (hfrac >= hg) & (hfrac <= 1.0f - hg) &
                    (fabsf(ca - Q.fov0) >= g) & (fabsf(ca - Q.fov1) >= g) &
                    (!has_max | (fabsf(2.0f * half - Q.max_proj) >= 2.0f * hg));
    if (ok) {
        if (!(Q.fov0 <= ca && ca <= Q.fov1) || (has_max && !(2.0f * half <= Q.max_proj))) return s;
        const int t = (int)tr, h = (int)hfl;
        vf_pieces(t - h, t + h, R, &s.a0, &s.b0, &s.a1, &s.b1);  // :277-284
    } else {
        const int4 e = cs_segment(f.px, f.py, f.radius, f.theta, ox, oy, R, step, fov0, fov1, has_max, max_proj);
        if (e.x < 0) return s;
        s.a0 = e.x; s.b0 = e.y; s.a1 = e.z; s.b1 = e.w;
    }
    s.drawn = 1;
    s.val = meter;
    return s;
}

// A segment as the ordered fold keeps it in LDS (rays fit 16 bits).
struct CSPack {
    uint16_t a0, b0, a1, b1;
    double val;
};
static_assert(kCSMaxRaysLDS < 0xffff, "0xffff marks a segment that is not drawn");
__device__ inline CSPack cs_pack(const CSSeg& s) {
    return CSPack{(uint16_t)(s.drawn ? s.a0 : 0xffff), (uint16_t)s.b0, (uint16_t)s.a1, (uint16_t)s.b1, s.val};
}

// Value of the row at raw ray r.
__device__ inline double row_value(const CSPack& s, int r) {
#pragma clang fp contract(off)
    if (s.a0 == 0xffff) return 0.0;
    const bool on = (r >= s.a0 && r < s.b0) || (r >= s.a1 && r < s.b1);
    return (on ? 1.0 : 0.0) * s.val;
}

// numpy's maximum: NaN propagates.
__device__ inline double np_maximum(double a, double v) {
    if (a != a) return a;
    if (v != v) return v;
    return v > a ? v : a;
}

// Post positions [lo, hi] of the flipped field that the FOV mask keeps
// (cs_supcalc.py:291-294 zeroes phis < fov0 and phis > fov1; linspace is
// increasing, so the kept positions are one range, found from the same
// float64 linspace values).
ABM_HD void fov_keep_range(int R, double step, double fov0, double fov1, int* lo, int* hi) {
    int a = 0, b = R - 1;
    while (a < R && linspace_at(a, R, step) < fov0) ++a;
    while (b >= 0 && linspace_at(b, R, step) > fov1) --b;
    *lo = a;
    *hi = b;
}

// How a focal agent's rows are combined:
//   rows      every row written out;
//   count     SUM without meters: every row is 0/1, so the sum is a count per
//             ray, exact in any order -- a difference array (+1 at each
//             piece's start, -1 at its end, LDS atomics) and a prefix scan,
//             O(objects + R) instead of O(objects x R);
//   max bits  MAX when every meter is a non-negative number other than -0.0:
//             such doubles order like their bit patterns as unsigned
//             integers, so each object raises its covered rays with a 64-bit
//             LDS atomic max, O(covered rays);
//   ordered   otherwise (meters in a SUM, or a NaN / negative / -0.0 meter in
//             a MAX): per ray, the rows folded in object order as numpy's
//             reduce does.
__device__ inline bool plain_meter(double v) { return v >= 0.0 && !signbit(v); }

// LDS of the wave's lanes before the barrier visible to every lane after it.
__device__ inline void cs_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The launch's constants.  Post positions [keep_lo, keep_hi] of a field survive
// the mask; raw rays [k0, k0 + kn) are those, the only ones accumulated.
struct CSArgs {
    int R, has_max, n_focal, keep_lo, keep_hi, k0, kn;
    double step, fov0, fov1, max_proj;
    const double *focal, *obj, *meters, *norm;
    const int64_t* obj_offset;
    double* out;
};

__device__ inline CSFocal cs_focal(const CSArgs& A, int f) {
    const double* fp = A.focal + 4 * (int64_t)f;
    CSFocal F;
    F.px = fp[0]; F.py = fp[1]; F.radius = fp[2]; F.theta = fp[3];
    F.cx = F.px + F.radius;
    F.cy = F.py + F.radius;
    double sn, cs;
    if (!f32::sincos_f64_small(F.theta, &sn, &cs)) sincos(F.theta, &sn, &cs);
    F.ux = heading_kept(F.px, F.py, F.radius) ? (float)cs : NAN;   // NaN: no guard lets it through
    F.uy = -(float)sn;
    return F;
}

// A focal agent's rows written out (ROWS), or folded in object order into acc
// (kn doubles of the wave's LDS, raw ray k0 + i in acc[i]); seg: 64 segments.
template <bool ROWS, bool MAX>
__device__ void cs_ordered(const CSArgs& A, const CSFocal& F, const CSFast& Q, int64_t o0, int64_t o1, CSPack* seg,
                           double* acc) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, R = A.R;
    for (int64_t c = o0; c < o1; c += 64) {
        const int n = (int)(o1 - c < 64 ? o1 - c : 64);
        if (lane < n) {
            const int64_t i = c + lane;
            seg[lane] = cs_pack(cs_segment_guarded(F, A.obj[2 * i], A.obj[2 * i + 1], A.meters ? A.meters[i] : 1.0, R,
                                                   A.step, A.fov0, A.fov1, A.has_max, A.max_proj, Q));
        }
        cs_wave_sync();
        if (ROWS) {
            // row i, post position p <- raw ray R - 1 - p (flip), masked rays 0
            for (int i = 0; i < n; ++i) {
                double* row = A.out + (c + i) * R;
                for (int p = lane; p < R; p += 64)
                    row[p] = (p < A.keep_lo || p > A.keep_hi) ? 0.0 : row_value(seg[i], R - 1 - p);
            }
        } else {
            for (int q = lane; q < A.kn; q += 64) {
                // object order; numpy's reduce starts from the first row
                double a = c == o0 ? row_value(seg[0], A.k0 + q) : acc[q];
                for (int i = c == o0 ? 1 : 0; i < n; ++i) {
                    const double v = row_value(seg[i], A.k0 + q);
                    a = MAX ? np_maximum(a, v) : a + v;
                }
                acc[q] = a;
            }
        }
        cs_wave_sync();
    }
}

// The wave's focal agent, or -1 beyond the last (no workgroup barrier in any
// of the kernels).
__device__ inline int cs_wave_focal(const CSArgs& A) {
    const int f = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    return f < A.n_focal ? f : -1;
}

// Rows, or a sum of meter-scaled rows.
template <bool ROWS>
__global__ void __launch_bounds__(256)
cs_rows_kernel(CSArgs A) {
#pragma clang fp contract(off)
    extern __shared__ double smem[];
    const int f = cs_wave_focal(A), lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6, R = A.R;
    if (f < 0) return;
    CSPack* seg = reinterpret_cast<CSPack*>(smem) + 64 * wave;
    double* acc = smem + (sizeof(CSPack) * 64 * waves) / sizeof(double) + (size_t)A.kn * wave;
    const int64_t o0 = A.obj_offset[f], o1 = A.obj_offset[f + 1];
    const CSFast Q = cs_fast(R, A.step, A.fov0, A.fov1, A.max_proj);
    cs_ordered<ROWS, false>(A, cs_focal(A, f), Q, o0, o1, seg, acc);
    if (ROWS) return;
    const double dv = A.norm ? A.norm[f] : 1.0;
    double* dst = A.out + (int64_t)f * R;
    for (int p = lane; p < R; p += 64)
        dst[p] = (p < A.keep_lo || p > A.keep_hi || o1 <= o0 ? 0.0 : acc[A.keep_hi - p]) / dv;
}

// Sum of 0/1 rows: the counts per ray over norm.  The quotients of the counts
// below 64 are made once, one per lane (a float64 division a ray was a third of
// the launch).  Bound by the output, R doubles per focal agent: 50,000 agents of
// 49 objects at R = 1200, FOV 0.45, 480 MB in 195 us with every decision in
// float64 and every ray accumulated, 89 us now (5.4 TB/s; a fill reaches 6.9).
__global__ void __launch_bounds__(256)
cs_count_kernel(CSArgs A) {
#pragma clang fp contract(off)
    extern __shared__ double smem[];
    const int f = cs_wave_focal(A), lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6, R = A.R;
    if (f < 0) return;
    double* quot = smem + 64 * wave;
    int* cnt = reinterpret_cast<int*>(smem + 64 * waves) + (size_t)(A.kn + 1) * wave;
    for (int q = lane; q <= A.kn; q += 64) cnt[q] = 0;
    const double dv = A.norm ? A.norm[f] : 1.0;
    quot[lane] = (double)lane / dv;
    const CSFocal F = cs_focal(A, f);
    const CSFast Q = cs_fast(R, A.step, A.fov0, A.fov1, A.max_proj);
    const int64_t o0 = A.obj_offset[f], o1 = A.obj_offset[f + 1];
    cs_wave_sync();
    for (int64_t i = o0 + lane; i < o1; i += 64) {
        const CSSeg sg = cs_segment_guarded(F, A.obj[2 * i], A.obj[2 * i + 1], 1.0, R, A.step, A.fov0, A.fov1,
                                            A.has_max, A.max_proj, Q);
        if (!sg.drawn) continue;
        auto count = [&](int a, int b) {   // the kept part of a piece
            a = max(a - A.k0, 0);
            b = min(b - A.k0, A.kn);
            if (a < b) { atomicAdd(&cnt[a], 1); atomicAdd(&cnt[b], -1); }
        };
        count(sg.a0, sg.b0);
        count(sg.a1, sg.b1);
    }
    cs_wave_sync();
    // inclusive prefix sum of the difference array: each lane walks a
    // contiguous run of rays; the run totals are scanned across the wave
    const int per = ((A.kn + 63) / 64) | 1;   // odd: the lanes' words in different banks
    const int lo = min(lane * per, A.kn), hi = min(lo + per, A.kn);
    int local = 0;
    for (int r = lo; r < hi; ++r) local += cnt[r];
    int incl = local;
    for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
    }
    int run = incl - local;
    for (int r = lo; r < hi; ++r) {
        run += cnt[r];
        cnt[r] = run;
    }
    cs_wave_sync();
    double* dst = A.out + (int64_t)f * R;
    const bool small = o1 - o0 < 64;   // no count reaches 64
    for (int p = lane; p < R; p += 64) {
        const int c = (p < A.keep_lo || p > A.keep_hi) ? 0 : cnt[A.keep_hi - p];
        const double v = small ? quot[c] : (double)c / dv;
        __builtin_nontemporal_store(v, &dst[p]);
    }
}

// Raise the kept rays of the lanes' pieces [a, b) to their values: pieces up to
// kCSShort rays by their own lane, longer ones by the whole wave one after
// another (a lane's loop would hold the other 63 for the longest of them).
constexpr int kCSShort = 24;
__device__ inline void cs_raise(unsigned long long* m, bool any, int a, int b, unsigned long long v) {
    const int lane = threadIdx.x & 63, len = any ? b - a : 0;
    uint64_t wide = __ballot(len > kCSShort);
    if (len > 0 && len <= kCSShort)
        for (int r = a; r < b; ++r) atomicMax(&m[r], v);
    while (wide) {
        const int l = __builtin_ctzll(wide);
        wide &= wide - 1;
        const int from = __builtin_amdgcn_readlane(a, l), to = __builtin_amdgcn_readlane(b, l);
        const unsigned long long w = ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), l) << 32) |
                                     (uint32_t)__builtin_amdgcn_readlane((int)v, l);
        for (int r = from + lane; r < to; r += 64) atomicMax(&m[r], w);
    }
}

// Maximum of meter-scaled rows (1 without meters).  Bound by the output and the
// wave's LDS (a double per kept ray): the same agents with 100 objects each,
// 480 MB written and 120 MB read, 365 us with float64 decisions, every ray
// accumulated and each piece raised by its own lane, 118 us now (5.1 TB/s).
__global__ void __launch_bounds__(256)
cs_max_kernel(CSArgs A) {
#pragma clang fp contract(off)
    extern __shared__ double smem[];
    const int f = cs_wave_focal(A), lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6, R = A.R;
    if (f < 0) return;
    CSPack* seg = reinterpret_cast<CSPack*>(smem) + 64 * wave;
    double* acc = smem + (sizeof(CSPack) * 64 * waves) / sizeof(double) + (size_t)A.kn * wave;
    unsigned long long* m = reinterpret_cast<unsigned long long*>(acc);
    for (int q = lane; q < A.kn; q += 64) m[q] = 0ull;   // +0.0
    const int64_t o0 = A.obj_offset[f], o1 = A.obj_offset[f + 1];
    const CSFocal F = cs_focal(A, f);
    const CSFast Q = cs_fast(R, A.step, A.fov0, A.fov1, A.max_proj);
    bool plain = true;
    if (A.meters)
        for (int64_t i = o0 + lane; i < o1; i += 64) plain = plain && plain_meter(A.meters[i]);
    cs_wave_sync();
    if (__ballot(!plain) == 0ull) {
        for (int64_t c = o0; c < o1; c += 64) {
            const int64_t i = c + lane;
            CSSeg sg{0, 0, 0, 0, 0, 0.0};
            if (i < o1)
                sg = cs_segment_guarded(F, A.obj[2 * i], A.obj[2 * i + 1], A.meters ? A.meters[i] : 1.0, R, A.step,
                                        A.fov0, A.fov1, A.has_max, A.max_proj, Q);
            const unsigned long long v = (unsigned long long)__double_as_longlong(sg.val);
            const bool any = sg.drawn && v != 0ull;
            cs_raise(m, any, max(sg.a0 - A.k0, 0), min(sg.b0 - A.k0, A.kn), v);
            if (__ballot(any && sg.a1 < sg.b1)) cs_raise(m, any, max(sg.a1 - A.k0, 0), min(sg.b1 - A.k0, A.kn), v);
        }
    } else {
        cs_ordered<false, true>(A, F, Q, o0, o1, seg, acc);
    }
    cs_wave_sync();
    double* dst = A.out + (int64_t)f * R;
    for (int p = lane; p < R; p += 64) {
        const double v = (p < A.keep_lo || p > A.keep_hi) ? 0.0 : acc[A.keep_hi - p];
        __builtin_nontemporal_store(v, &dst[p]);
    }
}

}  // namespace

}  // namespace abm

extern "C" {

int abm_cs_projection(const abm_cs_params* prm, int32_t n_focal, const double* focal,
                      const int64_t* obj_offset, const double* obj, const double* meters,
                      const double* norm, int32_t mode, double* out, void* stream) {
    using namespace abm;
    if (!prm) return set_error(ABM_ERR_INVALID, "abm_cs_projection: NULL params");
    const int R = prm->n_rays;
    if (R < 2 || R > kCSMaxRaysLDS)
        return set_error(ABM_ERR_INVALID, "abm_cs_projection: n_rays=%d outside [2, %d]", R, kCSMaxRaysLDS);
    if (mode != ABM_CS_ROWS && mode != ABM_CS_SUM && mode != ABM_CS_MAX)
        return set_error(ABM_ERR_INVALID, "abm_cs_projection: mode=%d", mode);
    if (n_focal < 0) return set_error(ABM_ERR_INVALID, "abm_cs_projection: n_focal < 0");
    if (n_focal == 0) return ABM_OK;
    if (!focal || !obj_offset || !out)
        return set_error(ABM_ERR_INVALID, "abm_cs_projection: NULL focal, offset or output array");
    if (!(prm->fov0 == prm->fov0) || !(prm->fov1 == prm->fov1))
        return set_error(ABM_ERR_INVALID, "abm_cs_projection: NaN field of view");
    const double step = linspace_step(R);
    int keep_lo, keep_hi;
    fov_keep_range(R, step, prm->fov0, prm->fov1, &keep_lo, &keep_hi);
    const int kn = std::max(0, keep_hi - keep_lo + 1);
    const CSArgs A{R, prm->has_max_proj_size ? 1 : 0, (int)n_focal, keep_lo, keep_hi, R - 1 - keep_hi, kn, step, prm->fov0, prm->fov1,
                   prm->max_proj_size, focal, obj, meters, norm, obj_offset, out};
    // waves (focal agents) per workgroup: four, fewer when their LDS would
    // not fit in 64 KB
    const bool count = mode == ABM_CS_SUM && !meters;
    const size_t per_wave = count ? sizeof(double) * 64 + sizeof(int) * ((size_t)kn + 1)
                                  : sizeof(CSPack) * 64 + sizeof(double) * (size_t)kn;
    int waves = 4;
    while (waves > 1 && per_wave * waves > 65536) --waves;
    const int blocks = (n_focal + waves - 1) / waves;
    auto kern = count ? cs_count_kernel
                      : mode == ABM_CS_MAX ? cs_max_kernel
                                           : mode == ABM_CS_ROWS ? cs_rows_kernel<true> : cs_rows_kernel<false>;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * waves), per_wave * waves, (hipStream_t)stream, A);
    return check_hip(hipGetLastError(), "cooperative-signalling projection launch");
}

}  // extern "C"
