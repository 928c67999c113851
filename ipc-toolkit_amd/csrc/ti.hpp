// Tight-Inclusion continuous collision detection for one candidate, run by
// one lane with its level lists in LDS or by a whole workgroup with shared
// level lists, plus the IPC Toolkit strategy around it
// (tight_inclusion_ccd.cpp:33-336).
//
// Tight-Inclusion (v1.0.6, third party) is restated from its published
// algorithm (Wang, Ferguson, Schneider, Panozzo, ACM TOG 40(5) 2021):
// breadth-first bisection of the (t,u,v) box [0,1]^3, the corner inclusion
// of the multilinear F(t,u,v), the floating-point filter epsilon box, the
// per-level termination rule.  Within a level boxes are visited in
// increasing lower t, ties first-in first-out.
//
// GPU form: all boxes of a level share their widths (the split axis is a
// function of the widths only), so a box is its lower corner (t0,u0,v0) and
// a level is a sorted array.  A t-split level is built by merging the lower
// and upper halves (each already sorted); a u/v-split level is the children
// in push order.  The lower t of every box is dyadic, so all corners are
// exact and the corner evaluations reproduce the CPU restatement bit for
// bit.  `bound` hides outcomes >= bound (boxes starting at t >= bound are
// dropped), which leaves every outcome below bound unchanged because a
// level is visited in increasing t.
#pragma once

#include "common.hpp"
#include "geometry.hpp"

namespace ipcg {

struct TIBox {
    double t, u, v;
};

// TI_OVERFLOW: a level outgrew the lists; TI_DEEP: a box needs more
// halvings than the packed form holds (both: another tier searches again)
enum TIResult : int { TI_MISS = 0, TI_HIT = 1, TI_OVERFLOW = 2, TI_DEEP = 3 };

// Guards that keep every search finite on the GPU: a level cap (each level
// halves one width, so a search that resolves needs far fewer) and a cap on
// the no_zero_toi retries (the reference allows INT_MAX; both restatements
// stop after this many halvings).
constexpr int TI_MAX_LEVELS = 1024;
constexpr int TI_MAX_NO_ZERO_TOI_ITER = 64;

struct TIQuery {
    double s[12], d[12]; // positions at t=0, differences to t=1
    bool vf;
    double err[3];
    double tol[3];
    double itol[3]; // 1 / tol: widths are powers of two, so 2^-k / tol is itol scaled
};

// What the tolerances and the filter of a query need of its positions.
struct TIScale {
    double len3[3]; // 3 max |dF| along t, u, v over the cube's corners
    double mag[3];  // per axis, max(|x|, 1)
};

// F(t,u,v) along one axis, points in the order (ea0, ea1, eb0, eb1) or
// (p, t0, t1, t2):
//   edge-edge    (a1 - a0) u + a0 - ((b1 - b0) v + b0)
//   vertex-face  p - ((t1 - t0) u + (t2 - t0) v + t0)
// with every point x = d t + s.
template <bool VF>
IPCG_HD double ti_corner(const TIQuery& q, int k, double t, double u, double v)
{
    const double x0 = q.d[0 + k] * t + q.s[0 + k];
    const double x1 = q.d[3 + k] * t + q.s[3 + k];
    const double x2 = q.d[6 + k] * t + q.s[6 + k];
    const double x3 = q.d[9 + k] * t + q.s[9 + k];
    if (VF) {
        const double pt = (x2 - x1) * u + (x3 - x1) * v + x1;
        return x0 - pt;
    }
    const double va = (x1 - x0) * u + x0;
    const double vb = (x3 - x2) * v + x2;
    return va - vb;
}

// Smallest and largest F over the eight corners [t0,t1] x [u0,u1] x [v0,v1].
// u enters one product and v another, and every rounded operation is
// monotone in each operand, so the extremes over the corners of one t are
// the same chain of operations over the extremes of the products: the same
// doubles as the eight corners give, in about 55 operations an axis instead
// of 75.  Where the range is not finite (overflow, infinities, NaN) the corners
// are compared one by one; edges whose differences overflow to NaN at one t alone
// show the other t's range, where their filter, which grows with the cube of the
// coordinates, is infinite and takes the box either way.
template <bool VF>
IPCG_HD void ti_range(const TIQuery& q, int k, double t0, double t1, double u0, double u1,
                      double v0, double v1, double& mn, double& mx)
{
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const double t = j ? t1 : t0;
        const double x0 = q.d[0 + k] * t + q.s[0 + k];
        const double x1 = q.d[3 + k] * t + q.s[3 + k];
        const double x2 = q.d[6 + k] * t + q.s[6 + k];
        const double x3 = q.d[9 + k] * t + q.s[9 + k];
        double lo, hi;
        if (VF) {
            const double eu = x2 - x1, ev = x3 - x1;
            const double a = eu * u0, b = eu * u1, c = ev * v0, e = ev * v1;
            lo = x0 - (fmax(a, b) + fmax(c, e) + x1);
            hi = x0 - (fmin(a, b) + fmin(c, e) + x1);
        } else {
            const double ea = x1 - x0, eb = x3 - x2;
            const double a = ea * u0 + x0, b = ea * u1 + x0;
            const double c = eb * v0 + x2, e = eb * v1 + x2;
            lo = fmin(a, b) - fmax(c, e);
            hi = fmax(a, b) - fmin(c, e);
        }
        mn = j == 0 ? lo : fmin(mn, lo);
        mx = j == 0 ? hi : fmax(mx, hi);
    }
    if (!(mx - mn < INFINITY)) {
        for (int c = 0; c < 8; c++) {
            const double f =
                ti_corner<VF>(q, k, (c & 4) ? t1 : t0, (c & 2) ? u1 : u0, (c & 1) ? v1 : v0);
            mn = (c == 0 || f < mn) ? f : mn;
            mx = (c == 0 || f > mx) ? f : mx;
        }
    }
}

// s, e: 12 positions at t=0 / t=1.  One axis at a time: few values live at
// once.
IPCG_HD void ti_scale(const double* s, const double* e, bool vf, TIScale& c)
{
    double dl = 0, lu = 0, lv = 0;
    auto grow = [](double& m, double a, double b) {
        const double x = fabs(b - a);
        m = x > m ? x : m;
    };
#pragma unroll
    for (int k = 0; k < 3; k++) {
        double p[8];
        if (vf) {
            p[0] = s[k] - s[3 + k];
            p[1] = s[k] - s[9 + k];
            p[3] = s[k] - (s[6 + k] + s[9 + k] - s[3 + k]);
            p[2] = s[k] - s[6 + k];
            p[4] = e[k] - e[3 + k];
            p[5] = e[k] - e[9 + k];
            p[7] = e[k] - (e[6 + k] + e[9 + k] - e[3 + k]);
            p[6] = e[k] - e[6 + k];
        } else {
            p[0] = s[k] - s[6 + k];
            p[1] = s[k] - s[9 + k];
            p[3] = s[3 + k] - s[9 + k];
            p[2] = s[3 + k] - s[6 + k];
            p[4] = e[k] - e[6 + k];
            p[5] = e[k] - e[9 + k];
            p[7] = e[3 + k] - e[9 + k];
            p[6] = e[3 + k] - e[6 + k];
        }
        grow(dl, p[0], p[4]);
        grow(dl, p[1], p[5]);
        grow(dl, p[3], p[7]);
        grow(dl, p[2], p[6]);
        grow(lu, p[0], p[2]);
        grow(lu, p[4], p[6]);
        grow(lu, p[5], p[7]);
        grow(lu, p[1], p[3]);
        grow(lv, p[0], p[1]);
        grow(lv, p[4], p[5]);
        grow(lv, p[6], p[7]);
        grow(lv, p[2], p[3]);
        double m = fabs(s[k]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const double a = fabs(s[3 * i + k]), b = fabs(e[3 * i + k]);
            m = a > m ? a : m;
            m = b > m ? b : m;
        }
        c.mag[k] = m > 1 ? m : 1;
    }
    c.len3[0] = 3 * dl;
    c.len3[1] = 3 * lu;
    c.len3[2] = 3 * lv;
}

// Parameter tolerances delta / (3 max |dF| along t, u, v over cube corners)
IPCG_HD void ti_param_tol(TIQuery& q, const TIScale& c, double delta)
{
    for (int k = 0; k < 3; k++) {
        q.tol[k] = delta / c.len3[k];
        q.itol[k] = 1.0 / q.tol[k];
    }
}

// Published floating-point filter: max(|x|, 1)^3 * c per axis.
IPCG_HD void ti_filter(TIQuery& q, const TIScale& c, bool use_ms)
{
    const double f = q.vf ? (use_ms ? 7.549516567451064e-15 : 6.661338147750939e-15)
                          : (use_ms ? 7.105427357601002e-15 : 6.217248937900877e-15);
    for (int k = 0; k < 3; k++) q.err[k] = c.mag[k] * c.mag[k] * c.mag[k] * f;
}

// Inclusion of the origin in the corner box of F over [t,t+wt]x[u,u+wu]x
// [v,v+wv], inflated by err and ms.  The kind is a template argument so the
// evaluation of an axis is one straight block, not branches on q.vf.
template <bool VF>
IPCG_HD bool ti_inclusion_k(const TIQuery& q, const TIBox& b, double wt, double wu, double wv,
                            double ms, bool& box_in, double* width)
{
    box_in = true;
    const double t1 = b.t + wt, u1 = b.u + wu, v1 = b.v + wv;
    for (int d = 0; d < 3; d++) {
        double mn, mx;
        ti_range<VF>(q, d, b.t, t1, b.u, u1, b.v, v1, mn, mx);
        width[d] = mx - mn;
        const double eps = q.err[d];
        if (mn - ms > eps || mx + ms < -eps) return false;
        if (!(mn + ms >= -eps && mx - ms <= eps)) box_in = false;
    }
    return true;
}

IPCG_HD bool ti_inclusion(const TIQuery& q, const TIBox& b, double wt, double wu, double wv,
                          double ms, bool& box_in, double* width)
{
    return q.vf ? ti_inclusion_k<true>(q, b, wt, wu, wv, ms, box_in, width)
                : ti_inclusion_k<false>(q, b, wt, wu, wv, ms, box_in, width);
}

// The same test for a query in LDS, AXES axes at a time (3: shortest chain, 1:
// fewer registers); `tol` tells whether every width of the corner box is within co_tol (meaningful when the
// origin is included).
template <bool VF, int AXES>
__device__ __forceinline__ bool ti_inclusion_tol_k(const TIQuery& q, const TIBox& b, double wt,
                                                   double wu, double wv, double ms, double co_tol,
                                                   bool& box_in, bool& tol)
{
    box_in = tol = true;
    const double t1 = b.t + wt, u1 = b.u + wu, v1 = b.v + wv;
    bool zero = true;
#pragma unroll AXES
    for (int d = 0; d < 3; d++) {
        double mn, mx;
        ti_range<VF>(q, d, b.t, t1, b.u, u1, b.v, v1, mn, mx);
        const double eps = q.err[d];
        if (!(mx - mn <= co_tol)) tol = false;
        if (mn - ms > eps || mx + ms < -eps) zero = false;
        if (!(mn + ms >= -eps && mx - ms <= eps)) box_in = false;
    }
    return zero;
}

template <int AXES>
__device__ __forceinline__ bool ti_inclusion_tol(const TIQuery& q, const TIBox& b, double wt,
                                                 double wu, double wv, double ms, double co_tol,
                                                 bool& box_in, bool& tol)
{
    return q.vf ? ti_inclusion_tol_k<true, AXES>(q, b, wt, wu, wv, ms, co_tol, box_in, tol)
                : ti_inclusion_tol_k<false, AXES>(q, b, wt, wu, wv, ms, co_tol, box_in, tol);
}

// The axis a level is split along: the first with the largest width over
// tolerance among those wider than their tolerance.
__device__ __forceinline__ int ti_axis(const TIQuery& q, double wt, double wu, double wv)
{
    double best = -INFINITY;
    int axis = 0;
    const double w3[3] = { wt, wu, wv };
    for (int i = 0; i < 3; i++) {
        const double r = w3[i] > q.tol[i] ? w3[i] * q.itol[i] : -INFINITY;
        axis = r > best ? i : axis;
        best = r > best ? r : best;
    }
    return axis;
}

// Outcomes at or above max(scale * g, floor) are hidden, g the smaller of
// the running minimum *ptr and the expected minimum *expect (ptr null: no
// bound; expect null: the running minimum alone).
struct TIBound {
    const double* ptr;
    const double* expect;
    double scale, floor;
    __device__ double get() const
    {
        if (!ptr) return INFINITY;
        double g = __hip_atomic_load(ptr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (expect) {
            const double x = __hip_atomic_load(expect, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            g = x < g ? x : g;
        }
        const double b = g * scale;
        return b > floor ? b : floor;
    }
};

// ---------------------------------------------------------------------------
// Level lists in LDS.  Every box of a level is its lower corner counted in
// the level widths 2^-kt, 2^-ku, 2^-kv, so TI_LDS_BITS bits per axis hold
// it exactly while no axis has been halved more often than that; a search
// that needs more halvings returns TI_DEEP, one that needs more than `cap`
// boxes in a list TI_OVERFLOW (the caller hands it to another tier).  The
// decoded corners are the same doubles in every tier, so all tiers give the
// same outcome.
// ---------------------------------------------------------------------------
constexpr int TI_LDS_BITS = 21;
constexpr unsigned TI_LDS_MASK = (1u << TI_LDS_BITS) - 1;

struct TILdsLists {
    unsigned long long* base; // this lane's slot 0 of list 0
    int stride;               // elements between a lane's consecutive slots
    int cap;                  // boxes per list
    __device__ unsigned long long& at(int list, int j) const
    {
        return base[(list * cap + j) * stride];
    }
};

__device__ __forceinline__ unsigned long long ti_pack(unsigned it, unsigned iu, unsigned iv)
{
    return ((unsigned long long)it << (2 * TI_LDS_BITS)) |
           ((unsigned long long)iu << TI_LDS_BITS) | iv;
}

// Searches of more than `budget` boxes overflow too: the wave waits for its
// longest search, and the tiers above search long ones faster.
__device__ inline int ti_bfs_lds(const TIQuery& q, double co_tol, double ms, long max_itr,
                                 const TIBound& B, const TILdsLists& L, long budget, double& toi)
{
    double temp_toi = INFINITY;
    double toi_skip = 4;
    bool use_skip = false;
    long refine = 0;
    int kt = 0, ku = 0, kv = 0; // the level's widths are 2^-k
    int ncur = 1;
    L.at(0, 0) = 0;
    toi = INFINITY;
    // The running minimum only decreases; a value read once per search
    // hides a subset of what a fresher read hides, all at or above the final
    // minimum.
    const double bound = B.get();
    while (ncur > 0) {
        const double wt = ldexp(1.0, -kt), wu = ldexp(1.0, -ku), wv = ldexp(1.0, -kv);
        bool level_less_tol = true, level_root = false;
        const bool c1 = wt <= q.tol[0] && wu <= q.tol[1] && wv <= q.tol[2];
        const int axis = ti_axis(q, wt, wu, wv);
        const int nk = (axis == 0 ? kt : axis == 1 ? ku : kv) + 1;
        int nlo = 0, nhi = 0;
        for (int i = 0; i < ncur; i++) {
            const unsigned long long pb = L.at(0, i);
            const unsigned it = (unsigned)(pb >> (2 * TI_LDS_BITS));
            const unsigned iu = (unsigned)(pb >> TI_LDS_BITS) & TI_LDS_MASK;
            const unsigned iv = (unsigned)pb & TI_LDS_MASK;
            const TIBox b { ldexp((double)it, -kt), ldexp((double)iu, -ku),
                            ldexp((double)iv, -kv) };
            if (b.t >= toi_skip || b.t >= bound) continue;
            refine++;
            if (refine > budget) return TI_OVERFLOW;
            bool box_in;
            double tw[3];
            if (!ti_inclusion(q, b, wt, wu, wv, ms, box_in, tw)) continue;
            const bool tol_cond = tw[0] <= co_tol && tw[1] <= co_tol && tw[2] <= co_tol;
            const bool c2 = box_in && level_less_tol;
            if (!tol_cond) level_less_tol = false;
            if (c1 || c2 || level_less_tol) {
                toi = b.t;
                return TI_HIT;
            }
            if (max_itr > 0) {
                if (!level_root) {
                    temp_toi = b.t;
                    level_root = true;
                }
                if (refine > max_itr) {
                    toi = temp_toi;
                    return TI_HIT;
                }
            }
            if (tol_cond || box_in) {
                toi_skip = b.t < toi_skip ? b.t : toi_skip;
                use_skip = true;
                continue;
            }
            if (nk > TI_LDS_BITS) return TI_DEEP;
            if (axis == 0) {
                if (nlo >= L.cap || nhi >= L.cap) return TI_OVERFLOW;
                L.at(2, nhi++) = ti_pack(2 * it + 1, iu, iv);
                L.at(1, nlo++) = ti_pack(2 * it, iu, iv);
            } else {
                // upper half first, each kept when it can hold a point of the
                // triangle (vertex-face)
                const unsigned hu = axis == 1 ? 2 * iu + 1 : iu, hv = axis == 1 ? iv : 2 * iv + 1;
                const unsigned lu = axis == 1 ? 2 * iu : iu, lv = axis == 1 ? iv : 2 * iv;
                const int nku = axis == 1 ? nk : ku, nkv = axis == 1 ? kv : nk;
                if (!q.vf || ldexp((double)hu, -nku) + ldexp((double)hv, -nkv) <= 1) {
                    if (nlo >= L.cap) return TI_OVERFLOW;
                    L.at(1, nlo++) = ti_pack(it, hu, hv);
                }
                if (!q.vf || b.u + b.v <= 1) {
                    if (nlo >= L.cap) return TI_OVERFLOW;
                    L.at(1, nlo++) = ti_pack(it, lu, lv);
                }
            }
        }
        // next level
        if (axis == 0) {
            kt = nk;
            if (nlo + nhi > L.cap) return TI_OVERFLOW;
            int i = 0, j = 0, k = 0;
            while (i < nlo && j < nhi) {
                const unsigned long long a = L.at(1, i), h = L.at(2, j);
                if ((h >> (2 * TI_LDS_BITS)) <= (a >> (2 * TI_LDS_BITS))) {
                    L.at(0, k++) = h;
                    j++;
                } else {
                    L.at(0, k++) = a;
                    i++;
                }
            }
            while (i < nlo) L.at(0, k++) = L.at(1, i++);
            while (j < nhi) L.at(0, k++) = L.at(2, j++);
            ncur = k;
        } else {
            if (axis == 1) ku = nk;
            else kv = nk;
            for (int i = 0; i < nlo; i++) L.at(0, i) = L.at(1, i);
            ncur = nlo;
        }
    }
    if (use_skip) {
        toi = toi_skip;
        return TI_HIT;
    }
    return TI_MISS;
}

// ---------------------------------------------------------------------------
// A whole workgroup of NW waves per search: the boxes of a level are tested
// 64 NW at a time (the query q is in LDS), the sequential rules of a level (ti_bfs_lds) are resolved
// from the first lanes that match.  Levels are packed as above in two lists
// `cur`, `nxt` of `cap` boxes (LDS or global memory).
//
// Reading the rules in parallel: a level is sorted by t, so the boxes that
// are scanned (t below the bound and the earliest tolerance box) are a
// prefix of it, box i is the (i + 1)-th scanned of the level, and the scan
// ends at the first zero box that is within tolerance or inside the eps box
// (any zero box once the level's widths are within tolerance, c1): the
// search ends there if that is the level's first zero box, else it becomes
// the earliest tolerance box.
//
// beam: a level that outgrows the lists keeps its first `cap` boxes (the
// earliest in t) and sets `cut`.  A hit found after that need not be the
// search's outcome but bounds it from above: the hit's box descends from
// boxes that the full search visits too, unless it ended at or before one
// of them, and at the hit's box it ends or sets its earliest tolerance box.
// ---------------------------------------------------------------------------
template <int NW> struct TIGroup {
    unsigned long long zero[2][NW], stop[2][NW], past[2][NW], hi[2][NW], lo[2][NW];
    unsigned tz[2][NW], ts[2][NW], live[2][NW];
    unsigned dead[2]; // per level parity
    double bound;
    unsigned long long* slab;
};

// Larger lists in global memory for searches that outgrow a workgroup's
// LDS: the first `count` claims of a launch get one (two lists of `cap`
// boxes).
struct TISlabs {
    unsigned long long* mem;
    unsigned long long* claimed; // zeroed before the launch
    int count, cap;
};

// What one chunk (64 NW boxes) of a level says to every lane of the group.
struct TIChunk {
    int zero, stop, past; // first lane of each kind in the chunk, -1: none
    unsigned tz, ts;      // t (in level widths) of the first zero / stop lane
    unsigned live;        // scanned boxes of the chunk
    unsigned before;      // children of lower lanes that come before `stop`
    unsigned total;       // children of the chunk that come before `stop`
};

template <int NW>
__device__ __forceinline__ TIChunk ti_chunk(TIGroup<NW>& G, int parity, bool live, bool zero,
                                            bool stop, bool past, bool hi, bool lo, unsigned it)
{
    const int lane = lane_id();
    const unsigned long long mz = __ballot(zero), ms = __ballot(stop), mp = __ballot(past),
                             mh = __ballot(hi), ml = __ballot(lo), mv = __ballot(live);
    const int fz = mz ? __ffsll((long long)mz) - 1 : 0, fs = ms ? __ffsll((long long)ms) - 1 : 0;
    const unsigned tz = (unsigned)__builtin_amdgcn_readlane((int)it, fz);
    const unsigned ts = (unsigned)__builtin_amdgcn_readlane((int)it, fs);
    auto below = [&](unsigned long long m) {
        return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                         __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
    };
    auto upto = [](unsigned long long m, int l) { // lanes below l
        return l >= WAVE ? m : m & ((1ull << l) - 1ull);
    };
    TIChunk c;
    if constexpr (NW == 1) {
        c.zero = mz ? fz : -1;
        c.stop = ms ? fs : -1;
        c.past = mp ? __ffsll((long long)mp) - 1 : -1;
        c.tz = tz;
        c.ts = ts;
        c.live = (unsigned)__popcll(mv);
        const int end = ms ? fs : WAVE;
        const unsigned long long h = upto(mh, end), l = upto(ml, end);
        c.before = below(h) + below(l);
        c.total = (unsigned)(__popcll(h) + __popcll(l));
        return c;
    } else {
        const int w = threadIdx.x / WAVE;
        if (lane == 0) {
            G.zero[parity][w] = mz;
            G.stop[parity][w] = ms;
            G.past[parity][w] = mp;
            G.hi[parity][w] = mh;
            G.lo[parity][w] = ml;
            G.tz[parity][w] = tz;
            G.ts[parity][w] = ts;
            G.live[parity][w] = (unsigned)__popcll(mv);
        }
        __syncthreads();
        // lane k < NW looks at wave k
        const bool in = lane < NW;
        const int k = in ? lane : 0;
        const unsigned long long az = in ? G.zero[parity][k] : 0, as = in ? G.stop[parity][k] : 0,
                                 ap = in ? G.past[parity][k] : 0;
        const unsigned long long wz = __ballot(az != 0), ws = __ballot(as != 0),
                                 wp = __ballot(ap != 0);
        auto first = [&](unsigned long long waves, const unsigned long long* m, int& wave) {
            if (!waves) return -1;
            wave = __builtin_amdgcn_readfirstlane(__ffsll((long long)waves) - 1);
            return wave * WAVE + (__ffsll((long long)m[wave]) - 1);
        };
        int iz = 0, is = NW, ip = 0;
        c.zero = first(wz, G.zero[parity], iz);
        c.stop = first(ws, G.stop[parity], is);
        c.past = first(wp, G.past[parity], ip);
        c.tz = G.tz[parity][wz ? iz : 0];
        c.ts = G.ts[parity][ws ? is : 0];
        // children of whole waves before the stop lane
        const int end = c.stop < 0 ? WAVE * NW : c.stop;
        unsigned n = 0;
        if (in) {
            const int e = end - k * WAVE; // lanes of wave k before the stop lane
            if (e > 0)
                n = (unsigned)(__popcll(upto(G.hi[parity][k], e)) + __popcll(upto(G.lo[parity][k], e)));
        }
        unsigned v = in ? G.live[parity][k] : 0;
        unsigned x = n;
#pragma unroll
        for (int o = 1; o < NW; o <<= 1) {
            const unsigned y = __shfl_up(x, o, WAVE);
            if (lane >= o) x += y;
        }
#pragma unroll
        for (int o = NW / 2; o > 0; o >>= 1) v += __shfl_down(v, o, WAVE);
        c.total = __shfl(x, NW - 1, WAVE);
        c.live = __shfl(v, 0, WAVE);
        const unsigned base = __shfl(x - n, w, WAVE);
        const int e = end - w * WAVE;
        c.before = base + (e > 0 ? below(upto(mh, e)) + below(upto(ml, e)) : 0u);
        return c;
    }
}

template <int NW>
__device__ inline int ti_bfs_group(const TIQuery& q, double co_tol, double ms, long max_itr,
                                   const TIBound& B, unsigned long long* cur,
                                   unsigned long long* nxt, int cap, TISlabs* slabs, bool beam,
                                   TIGroup<NW>& G, double& toi, bool& cut)
{
    constexpr int SIZE = NW * WAVE;
    const int tid = (int)threadIdx.x;
    double toi_skip = 4;
    bool use_skip = false;
    long refine = 0;
    int kt = 0, ku = 0, kv = 0; // the level's widths are 2^-k
    int ncur = 1;
    toi = INFINITY;
    double fresh = B.get();
    __syncthreads(); // the lists may still be read by the search before
    if (tid == 0) cur[0] = 0;
    // every level halves one axis and TI_LDS_BITS halvings of an axis end the
    // search, so there are at most 3 TI_LDS_BITS + 1 levels
    while (ncur > 0) {
        const double wt = ldexp(1.0, -kt), wu = ldexp(1.0, -ku), wv = ldexp(1.0, -kv);
        const bool c1 = wt <= q.tol[0] && wu <= q.tol[1] && wv <= q.tol[2];
        const int axis = ti_axis(q, wt, wu, wv);
        const int nk = (axis == 0 ? kt : axis == 1 ? ku : kv) + 1;
        double bound;
        const int lp = (kt + ku + kv) & 1;
        if constexpr (NW > 1) {
            if (tid == 0) { // one value for the whole group
                G.bound = fresh;
                G.dead[lp] = 0;
                if (slabs && 2 * ncur > cap) {
                    G.slab = nullptr;
                    const unsigned long long k = atomicAdd(slabs->claimed, 1ull);
                    if (k < (unsigned long long)slabs->count)
                        G.slab = slabs->mem + k * 2 * (unsigned long long)slabs->cap;
                }
            }
        }
        __syncthreads(); // the level's boxes (and bound) are written
        unsigned long long* spare = cur; // the list after next's
        if constexpr (NW == 1) {
            bound = fresh;
        } else {
            bound = G.bound;
            // a level that may outgrow the lists puts its children into a
            // slab, where the search stays
            if (slabs && 2 * ncur > cap) {
                if (G.slab) {
                    nxt = G.slab;
                    spare = nxt + slabs->cap;
                    cap = slabs->cap;
                }
                slabs = nullptr;
            }
        }
        // the running minimum as it is at the end of this level
        fresh = NW == 1 || tid == 0 ? B.get() : 0.0;
        bool seen_zero = false;
        double temp_toi = INFINITY;
        int n = 0; // t split: boxes that split (packed to the front of cur); else children
        bool more = true;
        for (int base = 0, parity = 0; base < ncur && more; base += SIZE, parity ^= 1) {
            const int i = base + tid;
            unsigned long long pb = 0;
            bool live = false, zero = false, tol = false, box_in = false;
            if (i < ncur) pb = cur[i];
            const unsigned it = (unsigned)(pb >> (2 * TI_LDS_BITS));
            const unsigned iu = (unsigned)(pb >> TI_LDS_BITS) & TI_LDS_MASK;
            const unsigned iv = (unsigned)pb & TI_LDS_MASK;
            const TIBox b { ldexp((double)it, -kt), ldexp((double)iu, -ku), ldexp((double)iv, -kv) };
            live = i < ncur && !(b.t >= toi_skip || b.t >= bound);
            if (live) zero = ti_inclusion_tol<3>(q, b, wt, wu, wv, ms, co_tol, box_in, tol);
            const bool stop = zero && (c1 || tol || box_in);
            const bool past = zero && max_itr > 0 && refine + i + 1 > max_itr;
            // children: both halves of t; the halves of u or v that can hold
            // a point of the triangle (vertex-face), upper half first
            const unsigned hu = axis == 1 ? 2 * iu + 1 : iu, hv = axis == 1 ? iv : 2 * iv + 1;
            const unsigned lu = axis == 1 ? 2 * iu : iu, lv = axis == 1 ? iv : 2 * iv;
            const int nku = axis == 1 ? nk : ku, nkv = axis == 1 ? kv : nk;
            const bool hi = zero && axis != 0
                && (!q.vf || ldexp((double)hu, -nku) + ldexp((double)hv, -nkv) <= 1);
            const bool lo = zero && (axis == 0 || !q.vf || b.u + b.v <= 1);
            const TIChunk c = ti_chunk<NW>(G, parity, live, zero, stop, past, hi, lo, it);
            if (c.zero >= 0 && !seen_zero) {
                seen_zero = true;
                temp_toi = ldexp((double)c.tz, -kt);
                if (c.stop == c.zero) {
                    toi = temp_toi;
                    return TI_HIT;
                }
            }
            if (c.past >= 0 && (c.stop < 0 || c.past <= c.stop)) { // iteration limit
                toi = temp_toi;
                return TI_HIT;
            }
            if (c.total > 0 && nk > TI_LDS_BITS) return TI_DEEP;
            if (c.stop >= 0) {
                const double t = ldexp((double)c.ts, -kt);
                toi_skip = t < toi_skip ? t : toi_skip;
                use_skip = true;
                more = false;
                refine += base + c.stop + 1;
            } else if (base + SIZE >= ncur || c.live < (unsigned)SIZE) {
                more = false; // what follows is not scanned
                refine += base + (int)c.live;
            }
            const bool keep = c.stop < 0 || tid < c.stop;
            const int at = n + (int)c.before;
            if (axis == 0) {
                // at <= i, and every lane of the chunk holds its box: the
                // slot's own box has been read
                if (lo && keep) cur[at] = pb;
            } else {
                if (hi && keep && at < cap) nxt[at] = ti_pack(it, hu, hv);
                const int al = at + (hi ? 1 : 0);
                if (lo && keep && al < cap) nxt[al] = ti_pack(it, lu, lv);
            }
            n += (int)c.total;
        }
        int children = n;
        if (axis == 0) {
            // Children of boxes r = 0 .. n-1 in order of t: a lower half keeps
            // t, an upper half adds half a width, so among the boxes [g0, g1)
            // of one t all lower halves come first: box r's lower half lands
            // at r + g0, its upper half at r + g1.  Upper halves at or past the
            // bound or the earliest tolerance box are the end of the list and
            // are left out.
            const double end = toi_skip < bound ? toi_skip : bound;
            int dead = 0;
            __syncthreads(); // the packed boxes are written
            for (int r0 = 0; r0 < n; r0 += SIZE) {
                const int r = r0 + tid;
                const bool in = r < n;
                const unsigned long long pb = in ? cur[r] : 0;
                const unsigned it = (unsigned)(pb >> (2 * TI_LDS_BITS));
                const unsigned uv_u = (unsigned)(pb >> TI_LDS_BITS) & TI_LDS_MASK;
                const unsigned uv_v = (unsigned)pb & TI_LDS_MASK;
                int g0, g1;
                if (NW == 1 && n <= WAVE) {
                    const unsigned prev = (unsigned)__shfl_up((int)it, 1, WAVE);
                    const unsigned long long st = __ballot(in && (tid == 0 || prev != it));
                    const unsigned long long le = st & (~0ull >> (WAVE - 1 - tid));
                    const unsigned long long gt = tid == WAVE - 1 ? 0 : st >> (tid + 1) << (tid + 1);
                    g0 = le ? 63 - __clzll((long long)le) : 0;
                    g1 = gt ? __ffsll((long long)gt) - 1 : n;
                } else {
                    int a = 0, z = in ? r : 0; // first box of this t
                    while (a < z) {
                        const int m = (a + z) >> 1;
                        if ((unsigned)(cur[m] >> (2 * TI_LDS_BITS)) < it) a = m + 1;
                        else z = m;
                    }
                    g0 = a;
                    a = in ? r + 1 : 0; // first box of a later t
                    z = in ? n : 0;
                    while (a < z) {
                        const int m = (a + z) >> 1;
                        if ((unsigned)(cur[m] >> (2 * TI_LDS_BITS)) <= it) a = m + 1;
                        else z = m;
                    }
                    g1 = a;
                }
                if (in) {
                    if (r + g0 < cap) nxt[r + g0] = ti_pack(2 * it, uv_u, uv_v);
                    if (r + g1 < cap) nxt[r + g1] = ti_pack(2 * it + 1, uv_u, uv_v);
                }
                const unsigned long long md =
                    __ballot(in && ldexp((double)(2 * it + 1), -nk) >= end);
                if constexpr (NW == 1) {
                    dead += __popcll(md);
                } else {
                    if (md && lane_id() == 0) atomicAdd(&G.dead[lp], (unsigned)__popcll(md));
                }
            }
            if constexpr (NW > 1) {
                __syncthreads();
                dead = (int)G.dead[lp];
            }
            children = 2 * n - dead;
            kt = nk;
        } else if (axis == 1) {
            ku = nk;
        } else {
            kv = nk;
        }
        if (children > cap) {
            if (!beam) return TI_OVERFLOW;
            cut = true;
            children = cap;
        }
        ncur = children;
        cur = nxt;
        nxt = spare;
    }
    if (use_skip) {
        toi = toi_skip;
        return TI_HIT;
    }
    return TI_MISS;
}

// ---------------------------------------------------------------------------
// W lanes of a wave per search (64 / W searches side by side), for searches
// of a few boxes a level; lists of `cap` boxes in LDS, the rules read from
// ballots as in ti_bfs_group.  Lanes of one search stay together, the
// searches of a wave may diverge.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void ti_wave_sync()
{
    // LDS operations of a wave execute in order: only the compiler must not
    // move them
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int W>
__device__ inline int ti_bfs_sub(const TIQuery& q, double co_tol, double ms, long max_itr,
                                 const TIBound& B, unsigned long long* cur,
                                 unsigned long long* nxt, int cap, double& toi)
{
    static_assert(W <= 32, "a search takes at most half a wave");
    const int g = lane_id() & (W - 1), g_base = lane_id() & ~(W - 1);
    auto vote = [&](bool p) { // the search's lanes only
        return (unsigned)(__ballot(p) >> g_base) & (unsigned)((1ull << W) - 1ull);
    };
    const unsigned below = (1u << g) - 1u;
    double toi_skip = 4;
    bool use_skip = false;
    long refine = 0;
    int kt = 0, ku = 0, kv = 0; // the level's widths are 2^-k
    int ncur = 1;
    toi = INFINITY;
    double fresh = B.get();
    if (g == 0) cur[0] = 0;
    // at most 3 TI_LDS_BITS + 1 levels, as in ti_bfs_group
    while (ncur > 0) {
        const double wt = ldexp(1.0, -kt), wu = ldexp(1.0, -ku), wv = ldexp(1.0, -kv);
        const bool c1 = wt <= q.tol[0] && wu <= q.tol[1] && wv <= q.tol[2];
        const int axis = ti_axis(q, wt, wu, wv);
        const int nk = (axis == 0 ? kt : axis == 1 ? ku : kv) + 1;
        const double bound = __shfl(fresh, g_base, WAVE); // one value per search
        fresh = B.get(); // for the next level
        ti_wave_sync();
        bool seen_zero = false;
        double temp_toi = INFINITY;
        int n = 0; // t split: boxes that split (packed to the front of cur); else children
        bool more = true;
        for (int base = 0; base < ncur && more; base += W) {
            const int i = base + g;
            const unsigned long long pb = i < ncur ? cur[i] : 0;
            const unsigned it = (unsigned)(pb >> (2 * TI_LDS_BITS));
            const unsigned iu = (unsigned)(pb >> TI_LDS_BITS) & TI_LDS_MASK;
            const unsigned iv = (unsigned)pb & TI_LDS_MASK;
            const TIBox b { ldexp((double)it, -kt), ldexp((double)iu, -ku), ldexp((double)iv, -kv) };
            const bool live = i < ncur && !(b.t >= toi_skip || b.t >= bound);
            bool zero = false, tol = false, box_in = false;
            if (live) zero = ti_inclusion_tol<1>(q, b, wt, wu, wv, ms, co_tol, box_in, tol);
            const bool past = zero && max_itr > 0 && refine + i + 1 > max_itr;
            const unsigned hu = axis == 1 ? 2 * iu + 1 : iu, hv = axis == 1 ? iv : 2 * iv + 1;
            const unsigned lu = axis == 1 ? 2 * iu : iu, lv = axis == 1 ? iv : 2 * iv;
            const int nku = axis == 1 ? nk : ku, nkv = axis == 1 ? kv : nk;
            const bool hi = zero && axis != 0
                && (!q.vf || ldexp((double)hu, -nku) + ldexp((double)hv, -nkv) <= 1);
            const bool lo = zero && (axis == 0 || !q.vf || b.u + b.v <= 1);
            const unsigned mz = vote(zero), mst = vote(zero && (c1 || tol || box_in)),
                           mp = vote(past), mv = vote(live);
            const int fs = mst ? __ffs((int)mst) - 1 : -1;
            if (mz && !seen_zero) {
                const int fz = __ffs((int)mz) - 1;
                seen_zero = true;
                temp_toi = ldexp((double)(unsigned)__shfl((int)it, g_base + fz, WAVE), -kt);
                if (fs == fz) {
                    toi = temp_toi;
                    return TI_HIT;
                }
            }
            if (mp && (fs < 0 || __ffs((int)mp) - 1 <= fs)) { // iteration limit
                toi = temp_toi;
                return TI_HIT;
            }
            // children before the stop lane
            const unsigned keep = fs < 0 ? ~0u : (1u << fs) - 1u;
            const unsigned mh = vote(hi) & keep, ml = vote(lo) & keep;
            if ((mh | ml) && nk > TI_LDS_BITS) return TI_DEEP;
            if (fs >= 0) {
                const double t = ldexp((double)(unsigned)__shfl((int)it, g_base + fs, WAVE), -kt);
                toi_skip = t < toi_skip ? t : toi_skip;
                use_skip = true;
                more = false;
                refine += base + fs + 1;
            } else if (base + W >= ncur || __popc(mv) < W) {
                more = false; // what follows is not scanned
                refine += base + __popc(mv);
            }
            const int at = n + __popc(mh & below) + __popc(ml & below);
            const bool put_hi = (mh >> g) & 1u, put_lo = (ml >> g) & 1u;
            if (axis == 0) {
                ti_wave_sync(); // the chunk has been read
                if (put_lo) cur[at] = pb;
            } else {
                if (put_hi && at < cap) nxt[at] = ti_pack(it, hu, hv);
                const int al = at + (put_hi ? 1 : 0);
                if (put_lo && al < cap) nxt[al] = ti_pack(it, lu, lv);
            }
            n += __popc(mh) + __popc(ml);
        }
        int children = n;
        if (axis == 0) { // positions as in ti_bfs_group
            const double end = toi_skip < bound ? toi_skip : bound;
            int dead = 0;
            ti_wave_sync();
            for (int r0 = 0; r0 < n; r0 += W) {
                const int r = r0 + g;
                const bool in = r < n;
                const unsigned long long pb = in ? cur[r] : 0;
                const unsigned it = (unsigned)(pb >> (2 * TI_LDS_BITS));
                const unsigned iu = (unsigned)(pb >> TI_LDS_BITS) & TI_LDS_MASK;
                const unsigned iv = (unsigned)pb & TI_LDS_MASK;
                int g0, g1;
                if (n <= W) {
                    const unsigned prev = (unsigned)__shfl_up((int)it, 1, WAVE);
                    const unsigned st = vote(in && (g == 0 || prev != it));
                    const unsigned le = st & (below | (1u << g)), gt = st & ~(below | (1u << g));
                    g0 = le ? 31 - __clz((int)le) : 0;
                    g1 = gt ? __ffs((int)gt) - 1 : n;
                } else {
                    int a = 0, z = in ? r : 0; // first box of this t
                    while (a < z) {
                        const int m = (a + z) >> 1;
                        if ((unsigned)(cur[m] >> (2 * TI_LDS_BITS)) < it) a = m + 1;
                        else z = m;
                    }
                    g0 = a;
                    a = in ? r + 1 : 0; // first box of a later t
                    z = in ? n : 0;
                    while (a < z) {
                        const int m = (a + z) >> 1;
                        if ((unsigned)(cur[m] >> (2 * TI_LDS_BITS)) <= it) a = m + 1;
                        else z = m;
                    }
                    g1 = a;
                }
                if (in) {
                    if (r + g0 < cap) nxt[r + g0] = ti_pack(2 * it, iu, iv);
                    if (r + g1 < cap) nxt[r + g1] = ti_pack(2 * it + 1, iu, iv);
                }
                dead += __popc(vote(in && ldexp((double)(2 * it + 1), -nk) >= end));
            }
            children = 2 * n - dead;
            kt = nk;
        } else if (axis == 1) {
            ku = nk;
        } else {
            kv = nk;
        }
        if (children > cap) return TI_OVERFLOW;
        ncur = children;
        unsigned long long* const x = cur;
        cur = nxt;
        nxt = x;
    }
    if (use_skip) {
        toi = toi_skip;
        return TI_HIT;
    }
    return TI_MISS;
}

} // namespace ipcg
