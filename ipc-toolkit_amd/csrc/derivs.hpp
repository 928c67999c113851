// Closed-form derivatives of the barrier energy of one collision stencil, in
// a translation-free orthonormal basis, with PSD projection.
//
// Every squared distance on the contact path is a function of point
// differences ("reduced variables", each P_plus - P_minus).  Derivatives are
// formed in those variables (quotient rule on d = N / D with N, D low-degree
// polynomials) and mapped into the n-1 dimensional subspace orthogonal to
// rigid translations, spanned by an orthonormal basis Q of the stencil's
// point space (Hadamard rows of 4 points).  The energy Hessian H_x of a
// stencil satisfies H_x = Q B Q^T with
// B = Q^T H_x Q (3(n-1) x 3(n-1)), and the translation directions are
// exact null vectors, so PSD(H_x) = Q PSD(B) Q^T: the eigen-problem of the
// reference's project_to_psd (eigen_ext.tpp:63-108) on 12x12 matrices is
// solved here on 9x9 ones (mollified edge pairs) or, in the frame of the
// closest points, on 5x5 ones (all others), in registers, with cyclic Jacobi.
#pragma once

#include "geometry.hpp"

namespace ipcg {

struct m33 {
    double a[9];
};

IPCG_HD m33 m33_zero()
{
    m33 r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.a[i] = 0;
    return r;
}
IPCG_HD m33 outer(const d3& u, const d3& v)
{
    return { { u.x * v.x, u.x * v.y, u.x * v.z, u.y * v.x, u.y * v.y, u.y * v.z,
               u.z * v.x, u.z * v.y, u.z * v.z } };
}
IPCG_HD m33 skew(const d3& c) // [c]x : [c]x w = c x w
{
    return { { 0, -c.z, c.y, c.z, 0, -c.x, -c.y, c.x, 0 } };
}
IPCG_HD m33 diag3(double s) { return { { s, 0, 0, 0, s, 0, 0, 0, s } }; }
IPCG_HD m33 transpose(const m33& m)
{
    return { { m.a[0], m.a[3], m.a[6], m.a[1], m.a[4], m.a[7], m.a[2], m.a[5], m.a[8] } };
}
IPCG_HD void axpy(m33& y, double s, const m33& x)
{
#pragma clang fp contract(fast)
#pragma unroll
    for (int i = 0; i < 9; i++) y.a[i] += s * x.a[i];
}
IPCG_HD d3 axpy3(const d3& y, double s, const d3& x)
{
#pragma clang fp contract(fast)
    return { y.x + s * x.x, y.y + s * x.y, y.z + s * x.z };
}

// Reduced derivatives of a scalar: value, R gradient blocks, upper Hessian
// blocks H[A][B] (A <= B) stored at tri(A,B).
template <int R> struct Red {
    static constexpr int NB = R * (R + 1) / 2;
    double v;
    d3 g[R];
    m33 H[NB];
    static IPCG_HD constexpr int tri(int a, int b) { return a * R - a * (a - 1) / 2 + (b - a); }
};

// d = N / D by the quotient rule.
template <int R>
IPCG_HD void quotient(const Red<R>& N, const Red<R>& D, Red<R>& out)
{
#pragma clang fp contract(fast)
    const double iD = 1.0 / D.v, iD2 = iD * iD, iD3 = iD2 * iD;
    out.v = N.v * iD;
#pragma unroll
    for (int a = 0; a < R; a++)
        out.g[a] = axpy3(scale(N.g[a], iD), -N.v * iD2, D.g[a]);
#pragma unroll
    for (int a = 0; a < R; a++)
#pragma unroll
        for (int b = a; b < R; b++) {
            const int t = Red<R>::tri(a, b);
            m33 h = N.H[t];
#pragma unroll
            for (int i = 0; i < 9; i++) h.a[i] = h.a[i] * iD - N.v * iD2 * D.H[t].a[i];
            axpy(h, -iD2, outer(N.g[a], D.g[b]));
            axpy(h, -iD2, outer(D.g[a], N.g[b]));
            axpy(h, 2 * N.v * iD3, outer(D.g[a], D.g[b]));
            out.H[t] = h;
        }
}

// |u x v|^2 over reduced (u, v)
IPCG_HD void cross2_derivs(const d3& u, const d3& v, Red<2>& X)
{
    const d3 n = cross(u, v);
    X.v = sqn(n);
    X.g[0] = scale(cross(v, n), 2.0);
    X.g[1] = scale(cross(n, u), 2.0);
    m33 uu = diag3(2 * sqn(v));
    axpy(uu, -2.0, outer(v, v));
    m33 vv = diag3(2 * sqn(u));
    axpy(vv, -2.0, outer(u, u));
    m33 uv = diag3(-2 * dot(u, v));
    axpy(uv, 2.0, outer(u, v));
    axpy(uv, -2.0, skew(n));
    X.H[Red<2>::tri(0, 0)] = uu;
    X.H[Red<2>::tri(0, 1)] = uv;
    X.H[Red<2>::tri(1, 1)] = vv;
}

// point-point: d = |delta|^2
IPCG_HD void pp_derivs(const d3& delta, Red<1>& out)
{
    out.v = sqn(delta);
    out.g[0] = scale(delta, 2.0);
    out.H[0] = diag3(2.0);
}

// point-line: a = e0 - p, b = e1 - p, d = |a x b|^2 / |b - a|^2
IPCG_HD void pl_derivs(const d3& a, const d3& b, Red<2>& out)
{
    Red<2> N, D;
    cross2_derivs(a, b, N);
    const d3 e = sub(b, a);
    D.v = sqn(e);
    D.g[0] = scale(e, -2.0);
    D.g[1] = scale(e, 2.0);
    D.H[0] = diag3(2.0);
    D.H[1] = diag3(-2.0);
    D.H[2] = diag3(2.0);
    quotient<2>(N, D, out);
}

// point-plane / line-line: s = w . (u x v), d = s^2 / |u x v|^2
IPCG_HD void triple_derivs(const d3& w, const d3& u, const d3& v, Red<3>& out)
{
    const d3 n = cross(u, v);
    const double s = dot(w, n);
    const d3 gs[3] = { n, cross(v, w), cross(w, u) };
    Red<3> N, D;
    N.v = s * s;
#pragma unroll
    for (int a = 0; a < 3; a++) N.g[a] = scale(gs[a], 2 * s);
    // Hessian of s: (w,u) = -[v]x, (w,v) = [u]x, (u,v) = -[w]x, diagonal 0
    m33 hs[6];
    hs[Red<3>::tri(0, 0)] = m33_zero();
    hs[Red<3>::tri(1, 1)] = m33_zero();
    hs[Red<3>::tri(2, 2)] = m33_zero();
    hs[Red<3>::tri(0, 1)] = skew(scale(v, -1.0));
    hs[Red<3>::tri(0, 2)] = skew(u);
    hs[Red<3>::tri(1, 2)] = skew(scale(w, -1.0));
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = a; b < 3; b++) {
            const int t = Red<3>::tri(a, b);
            m33 h = outer(gs[a], gs[b]);
#pragma unroll
            for (int i = 0; i < 9; i++) h.a[i] = 2 * h.a[i] + 2 * s * hs[t].a[i];
            N.H[t] = h;
        }
    Red<2> X;
    cross2_derivs(u, v, X);
    D.v = X.v;
    D.g[0] = { 0, 0, 0 };
    D.g[1] = X.g[0];
    D.g[2] = X.g[1];
    D.H[Red<3>::tri(0, 0)] = m33_zero();
    D.H[Red<3>::tri(0, 1)] = m33_zero();
    D.H[Red<3>::tri(0, 2)] = m33_zero();
    D.H[Red<3>::tri(1, 1)] = X.H[0];
    D.H[Red<3>::tri(1, 2)] = X.H[1];
    D.H[Red<3>::tri(2, 2)] = X.H[2];
    quotient<3>(N, D, out);
}

// ---------------------------------------------------------------------------
// Orthonormal translation-free basis Q (4 points x 3 columns; stencils of
// fewer points give the others weight 0)
// ---------------------------------------------------------------------------
template <int NP> struct QBasis;
template <> struct QBasis<4> {
    static IPCG_HD double q(int x, int k)
    {
        // rows of the 4x4 Hadamard matrix / 2 without the all-ones row
        const int s = (k == 0) ? (x & 1) : (k == 1 ? (x >> 1) : ((x ^ (x >> 1)) & 1));
        return s ? -0.5 : 0.5;
    }
};

// Packed symmetric N x N (lower), index of (i, j), i >= j
IPCG_HD constexpr int sp(int i, int j) { return i >= j ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i; }

// Q-space image of reduced derivatives: reduced variable i is
// P[plus[i]] - P[minus[i]], so S[i][k] = Q[plus][k] - Q[minus][k].
// gq = S^T g;  Hq += alpha * S^T H S  (packed 3K x 3K).
template <int NP, int R>
IPCG_HD void to_qspace(const Red<R>& d, const int* plus, const int* minus,
                       double alpha, d3* gq, double* Hq)
{
#pragma clang fp contract(fast)
    constexpr int K = NP - 1;
    double S[R][K];
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
        for (int k = 0; k < K; k++)
            S[i][k] = QBasis<NP>::q(plus[i], k) - QBasis<NP>::q(minus[i], k);
#pragma unroll
    for (int k = 0; k < K; k++) {
        d3 acc = { 0, 0, 0 };
#pragma unroll
        for (int i = 0; i < R; i++) acc = axpy3(acc, S[i][k], d.g[i]);
        gq[k] = acc;
    }
#pragma unroll
    for (int k = 0; k < K; k++)
#pragma unroll
        for (int l = k; l < K; l++) {
            m33 blk = m33_zero();
#pragma unroll
            for (int i = 0; i < R; i++)
#pragma unroll
                for (int j = 0; j < R; j++) {
                    const double c = alpha * S[i][k] * S[j][l];
                    const m33 h = i <= j ? d.H[Red<R>::tri(i, j)]
                                         : transpose(d.H[Red<R>::tri(j, i)]);
                    axpy(blk, c, h);
                }
#pragma unroll
            for (int r = 0; r < 3; r++)
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const int I = 3 * k + r, J = 3 * l + c;
                    if (k < l || I >= J) Hq[sp(I, J)] += blk.a[3 * r + c];
                }
        }
}

// point-space gradient: g[plus[i]] += alpha g_i, g[minus[i]] -= alpha g_i
// (gp holds NP points; every point is addressed by a compile-time index so
// the array stays in registers, each point updated in the same order)
template <int NP, int R>
IPCG_HD void to_points(const Red<R>& d, const int* plus, const int* minus,
                       double alpha, d3* gp)
{
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
        for (int j = 0; j < NP; j++) {
            if (plus[i] == j) gp[j] = axpy3(gp[j], alpha, d.g[i]);
            if (minus[i] == j) gp[j] = axpy3(gp[j], -alpha, d.g[i]);
        }
}

// Hq += alpha * (a b^T + b a^T) / (sym ? 2 : 1) on packed 3K storage, with
// a, b given as K blocks.
template <int K>
IPCG_HD void add_sym_outer(double* Hq, double alpha, const d3* a, const d3* b)
{
#pragma clang fp contract(fast)
    constexpr int N = 3 * K;
    double av[N], bv[N];
#pragma unroll
    for (int k = 0; k < K; k++) {
        av[3 * k] = a[k].x; av[3 * k + 1] = a[k].y; av[3 * k + 2] = a[k].z;
        bv[3 * k] = b[k].x; bv[3 * k + 1] = b[k].y; bv[3 * k + 2] = b[k].z;
    }
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int j = 0; j <= i; j++) Hq[sp(i, j)] += alpha * (av[i] * bv[j] + bv[i] * av[j]);
}

// ---------------------------------------------------------------------------
// 1/sqrt(x) and 1/x for normal x: the hardware estimate refined by two Newton
// steps (each squares the relative error), a few ulp from the correctly
// rounded ones at a fraction of their instructions.
// ---------------------------------------------------------------------------
IPCG_HD double rsqrt_nr(double x)
{
#ifdef __HIP_DEVICE_COMPILE__
    double r = __builtin_amdgcn_rsq(x);
    const double h = 0.5 * x;
    r = r * fma(-h * r, r, 1.5);
    return r * fma(-h * r, r, 1.5);
#else
    return 1.0 / sqrt(x);
#endif
}

IPCG_HD double rcp_nr(double x)
{
#ifdef __HIP_DEVICE_COMPILE__
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
#else
    return 1.0 / x;
#endif
}

// ---------------------------------------------------------------------------
// PSD projection (cyclic Jacobi, eigenvectors accumulated in registers).
// The tangent of a rotation, h / (|d| + sqrt(d^2 + h^2)) for h = 2 a_pq and
// d = a_qq - a_pp, may be a few ulp off: c and s are normalized to the
// tangent that was computed, and the entry set to 0 is off by as many ulp.
// (Rounded division and square root were two thirds of a rotation's
// instructions on a 5 x 5 matrix.)
// method: 0 none, 1 clamp, 2 abs (PSDProjectionMethod, eigen_ext.hpp:202-206)
// ---------------------------------------------------------------------------
template <int N>
IPCG_HD void project_psd(double* A /* packed N */, int method)
{
#pragma clang fp contract(fast)
    if (method == 0) return;
    double V[N][N];
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int j = 0; j < N; j++) V[i][j] = i == j ? 1.0 : 0.0;
    for (int sweep = 0; sweep < 16; sweep++) {
        double off = 0, tot = 0;
#pragma unroll
        for (int i = 0; i < N; i++) {
            tot += A[sp(i, i)] * A[sp(i, i)];
#pragma unroll
            for (int j = 0; j < i; j++) off += A[sp(i, j)] * A[sp(i, j)];
        }
        tot += 2 * off;
        if (!(off > 1e-30 * tot)) break;
#pragma unroll
        for (int p = 0; p < N; p++)
#pragma unroll
            for (int q = p + 1; q < N; q++) {
                const double apq = A[sp(p, q)];
                const double app = A[sp(p, p)], aqq = A[sp(q, q)];
                const double dd = aqq - app, h = 2 * apq, x = dd * dd + h * h;
                double t = h * rcp_nr(fabs(dd) + x * rsqrt_nr(x));
                t = dd < 0 ? -t : t;
                t = x >= 1e-290 ? t : 0.0; // (both entries vanish)
                const double c = rsqrt_nr(t * t + 1), s = t * c; // |t| <= 1
#pragma unroll
                for (int k = 0; k < N; k++) {
                    if (k == p || k == q) continue;
                    const double akp = A[sp(k, p)], akq = A[sp(k, q)];
                    A[sp(k, p)] = c * akp - s * akq;
                    A[sp(k, q)] = s * akp + c * akq;
                }
                A[sp(p, p)] = app - t * apq;
                A[sp(q, q)] = aqq + t * apq;
                A[sp(p, q)] = 0.0;
#pragma unroll
                for (int k = 0; k < N; k++) {
                    const double vkp = V[k][p], vkq = V[k][q];
                    V[k][p] = c * vkp - s * vkq;
                    V[k][q] = s * vkp + c * vkq;
                }
            }
    }
    double lam[N];
#pragma unroll
    for (int i = 0; i < N; i++) {
        const double l = A[sp(i, i)];
        lam[i] = l >= 0 ? l : (method == 1 ? 0.0 : -l);
    }
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int j = 0; j <= i; j++) {
            double acc = 0;
#pragma unroll
            for (int k = 0; k < N; k++) acc += V[i][k] * lam[k] * V[j][k];
            A[sp(i, j)] = acc;
        }
}

// ---------------------------------------------------------------------------
// Hessian of b(d) of an unmollified stencil in five coordinates.
//
// Let q be the vector between the closest points (points weighted by c, sum
// 0), n its direction and e1, e2 the other axes of an orthonormal frame:
//   plane (point-triangle, interior edge-edge): n normal to the plane,
//   line  (point-line): e1 along the line,
//   point (point-point): any e1, e2.
// With sigma = n . q, d = sigma^2 and rho_k the rotation of the frame about
// the closest points (linear in n . dx: the point weights r_k), the second
// derivative of d / 2 along dx is
//   (n . dq)^2 - 2 sum_k rho_k (e_k . dq) - sum_k rho_k^2 + sum_k y_k (e_k . dq)^2
// with y_k = 1 along the axes in which the nearest feature does not extend
// (rho_k = 0 there).  So the energy Hessian acts on n (x) R^3 and e_k (x) c
// only: five orthonormal coordinates z0..z2 = n (x) (c^, f1, f2) and
// e_k (x) c^, where it is
//   4 d b'' + 2 b' on the n . dq term, 2 b' on the others,
// and its projection is that of a 5 x 5 matrix.
// ---------------------------------------------------------------------------
struct ContactFrame {
    d3 n, e1, e2;
    double c[4], r1[4], r2[4]; // point weights
    double y1, y2;
};

// two axes completing the unit vector a (Duff et al., "Building an
// Orthonormal Basis, Revisited", JCGT 2017)
IPCG_HD void complement(const d3& a, d3& b, d3& c)
{
    const double sg = a.z < 0 ? -1.0 : 1.0;
    const double h = -1.0 / (sg + a.z), xy = a.x * a.y * h;
    b = { 1.0 + sg * a.x * a.x * h, sg * xy, -sg * a.x };
    c = { xy, sg + a.y * a.y * h, -a.y };
}

// 4-point weights to the Q basis
IPCG_HD d3 weights_q(const double* w)
{
    return { 0.5 * ((w[0] - w[1]) + (w[2] - w[3])), 0.5 * ((w[0] + w[1]) - (w[2] + w[3])),
             0.5 * ((w[0] - w[1]) - (w[2] - w[3])) };
}

// plane through the origin along u, v (weights U, V), w (weights W) to it
IPCG_HD void frame_plane(const d3& w, const d3& u, const d3& v, const double* W, const double* U,
                         const double* V, ContactFrame& f)
{
#pragma clang fp contract(fast)
    const double lu = sqrt(sqn(u)), iu = 1.0 / lu;
    f.e1 = scale(u, iu);
    const d3 m = cross(u, v);
    const double in = 1.0 / sqrt(sqn(m));
    f.n = scale(m, in);
    f.e2 = cross(f.n, f.e1);
    const double v1 = dot(v, f.e1), w2 = dot(w, f.e2);
    const double k2 = lu * in;
    const double b = w2 * k2, a = dot(w, f.e1) * iu - v1 * in * w2;
    const double sig = dot(w, f.n);
    const double su = sig * iu, s2u = -sig * v1 * in, s2v = sig * k2;
    f.y1 = f.y2 = 0;
#pragma unroll
    for (int x = 0; x < 4; x++) {
        f.c[x] = (W[x] - a * U[x]) - b * V[x];
        f.r1[x] = su * U[x];
        f.r2[x] = s2u * U[x] + s2v * V[x];
    }
}

// Line l0 l1, w0 and w1 from its ends to the point (weights W from l0, L
// along the line).  The direction off the line comes from w0 x w1, the
// vectors of the squared distance: a rounded unit vector along the line would
// turn it by |w| / |r| roundings.
IPCG_HD void frame_line(const d3& w, const d3& w1, const d3& e, const double* W, const double* L,
                        ContactFrame& f)
{
#pragma clang fp contract(fast)
    const double e2 = sqn(e), ie = 1.0 / sqrt(e2), ie2 = 1.0 / e2;
    f.e1 = scale(e, ie);
    const d3 m = cross(w1, w);
    const double m2 = sqn(m);
    d3 b, c;
    complement(f.e1, b, c);
    f.e2 = m2 > 0 ? scale(m, 1.0 / sqrt(m2)) : b;
    f.n = cross(f.e1, f.e2);
    const double a = dot(w, e) * ie2, s = sqrt(m2) * ie2;
    f.y1 = 0;
    f.y2 = 1;
#pragma unroll
    for (int x = 0; x < 4; x++) {
        f.c[x] = W[x] - a * L[x];
        f.r1[x] = s * L[x];
        f.r2[x] = 0;
    }
}

IPCG_HD void frame_point(const d3& w, const double* W, ContactFrame& f)
{
    const double w2 = sqn(w);
    f.n = w2 > 0 ? scale(w, 1.0 / sqrt(w2)) : d3 { 1, 0, 0 };
    complement(f.n, f.e1, f.e2);
    f.y1 = f.y2 = 1;
#pragma unroll
    for (int x = 0; x < 4; x++) {
        f.c[x] = W[x];
        f.r1[x] = f.r2[x] = 0;
    }
}

// Projected Hessian from the frame and the derivatives f1, f2 of the energy
// by d, as a record of FRAME_LEN values: n, c, M (packed 3 x 3), R (3 rows),
// T (packed 3 x 3), with the 3 x 3 block of the 4-point Q basis rows k, l
//   M_kl n n^T + c_k R_l n^T + c_l n R_k^T + c_k c_l T.
// The 5 x 5 matrix is scaled to entries of at most 1 for the projection.
constexpr int FRAME_LEN = 27;

IPCG_HD void frame_hessian(const ContactFrame& f, double d, double f1, double f2, int method,
                           double* o)
{
#pragma clang fp contract(fast)
    const d3 cq = weights_q(f.c), q1 = weights_q(f.r1), q2 = weights_q(f.r2);
    const double cl2 = sqn(cq), cl = sqrt(cl2);
    const d3 ch = scale(cq, 1.0 / cl);
    d3 g1, g2;
    complement(ch, g1, g2);
    const double a[3] = { dot(q1, ch), dot(q1, g1), dot(q1, g2) };
    const double b[3] = { dot(q2, ch), dot(q2, g1), dot(q2, g2) };
    const double k = 2 * f1, kc = -k * cl;
    double B[15];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j <= i; j++) B[sp(i, j)] = -k * (a[i] * a[j] + b[i] * b[j]);
    B[0] += (4 * d * f2 + k) * cl2;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        B[sp(3, j)] = kc * a[j];
        B[sp(4, j)] = kc * b[j];
    }
    B[sp(3, 3)] = k * cl2 * f.y1;
    B[sp(4, 4)] = k * cl2 * f.y2;
    B[sp(4, 3)] = 0;
    if (method != 0) {
        double mx = 0;
#pragma unroll
        for (int e = 0; e < 15; e++) mx = fmax(mx, fabs(B[e]));
        if (mx > 0) { // (a NaN stays in its entry)
            const double im = 1.0 / mx;
#pragma unroll
            for (int e = 0; e < 15; e++) B[e] *= im;
            project_psd<5>(B, method);
#pragma unroll
            for (int e = 0; e < 15; e++) B[e] *= mx;
        }
    }
    // M = F B_zz F^T over F = (c^, g1, g2), R = F B_zy (e1, e2)^T, and the
    // in-frame part T = sum B_yy e e^T
    const double F[3][3] = { { ch.x, g1.x, g2.x }, { ch.y, g1.y, g2.y }, { ch.z, g1.z, g2.z } };
    o[0] = f.n.x; o[1] = f.n.y; o[2] = f.n.z;
    o[3] = ch.x; o[4] = ch.y; o[5] = ch.z;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double t[3];
#pragma unroll
        for (int j = 0; j < 3; j++)
            t[j] = F[i][0] * B[sp(0, j)] + F[i][1] * B[sp(1, j)] + F[i][2] * B[sp(2, j)];
#pragma unroll
        for (int j = 0; j <= i; j++)
            o[6 + sp(i, j)] = t[0] * F[j][0] + t[1] * F[j][1] + t[2] * F[j][2];
        const double p = F[i][0] * B[sp(3, 0)] + F[i][1] * B[sp(3, 1)] + F[i][2] * B[sp(3, 2)];
        const double q = F[i][0] * B[sp(4, 0)] + F[i][1] * B[sp(4, 1)] + F[i][2] * B[sp(4, 2)];
        o[12 + 3 * i] = p * f.e1.x + q * f.e2.x;
        o[13 + 3 * i] = p * f.e1.y + q * f.e2.y;
        o[14 + 3 * i] = p * f.e1.z + q * f.e2.z;
    }
    const double u[3] = { f.e1.x, f.e1.y, f.e1.z }, v[3] = { f.e2.x, f.e2.y, f.e2.z };
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int t = 0; t <= r; t++)
            o[21 + sp(r, t)] = B[sp(3, 3)] * u[r] * u[t] + B[sp(4, 4)] * v[r] * v[t]
                + B[sp(4, 3)] * (u[r] * v[t] + v[r] * u[t]);
}

} // namespace ipcg
