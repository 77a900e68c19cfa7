// tri_dev.h -- triangular dislocation (Nikkhoo & Walter 2015) stress and
// displacement for one (receiver, source) pair per lane, two slips at once.
//
// Follows jdpmoore/unicycle fortran/3d/src/StrainInHalfSpace.c:42-173
// (straininhalfspace_: main + image + free-surface harmonic parts) and
// nikkhoo15.f90:120-163.  Each part's strain is the exact gradient, by
// forward-mode differentiation, of the same part's displacement field
// (DispInHalfSpace.c:153-616), evaluated in binary64.  Source-only geometry
// (frames, vertex angles, side transforms) is precomputed on the host with the C
// library (TriSource).
//
// The gradients are taken in the frame of each angular dislocation, where a
// coordinate's gradient is a unit vector: the number type carries which partial
// derivatives exist (D<mask>), so products with coordinates cost what they have
// to, and the 3 x 3 gradients are rotated once they are summed.  Taken in the
// source's frame, with every gradient full, a pair cost 21,680 flop, a third of
// them for a tensile component that unit strike and dip slip do not have.
// Quotients are products with reciprocals (3 per angular dislocation and 4 per
// harmonic term instead of some 20 and 36 divisions), sums of products are fused.
#pragma once
#include <hip/hip_runtime.h>

namespace ucy {

// products and sums fuse throughout: no bit of this arithmetic is the
// reference's, which differentiates by hand
#pragma clang fp contract(fast)

// 1/x by the hardware estimate and two Newton steps, within an ulp; NaN at 0
__device__ __forceinline__ double fast_rcp(double x)
{
    double q = __builtin_amdgcn_rcp(x);
    q = fma(fma(-x, q, 1.0), q, q);
    return fma(fma(-x, q, 1.0), q, q);
}
// Coordinates and lengths are rounded product by product, as the reference forms
// them: next to an edge, or to its extension, a rounding of these outweighs all
// later ones, and the differences r - z carry it on.
__device__ __forceinline__ double dot2(double a, double x, double b, double y)
{
#pragma clang fp contract(off)
    return a * x + b * y;
}
__device__ __forceinline__ double dot3(const double a[3], double x, double y, double z)
{
#pragma clang fp contract(off)
    return a[0] * x + a[1] * y + a[2] * z;
}

__device__ __forceinline__ double length3(double x, double y, double z)
{
#pragma clang fp contract(off)
    return sqrt(x * x + y * y + z * z);
}

// a value and those of its three partial derivatives that M names (bits 0, 1, 2);
// the others are zero and not held
template <int M>
struct D {
    double v, g[3];
};
__device__ __forceinline__ D<0> value(double v) { return {v, {0.0, 0.0, 0.0}}; }
// the coordinate along axis k, differentiated or not
template <bool GRAD, int K>
__device__ __forceinline__ auto coordinate(double v)
{
    if constexpr (GRAD) return D<1 << K>{v, {K == 0 ? 1.0 : 0.0, K == 1 ? 1.0 : 0.0, K == 2 ? 1.0 : 0.0}};
    else return value(v);
}
template <int A, class F>
__device__ __forceinline__ D<A> each(double v, F f)
{
    D<A> r;
    r.v = v;
#pragma unroll
    for (int k = 0; k < 3; k++) r.g[k] = A >> k & 1 ? f(k) : 0.0;
    return r;
}
template <int A>
__device__ __forceinline__ D<A> operator-(const D<A> &a)
{
    return each<A>(-a.v, [&](int k) { return -a.g[k]; });
}
template <int A, int B>
__device__ __forceinline__ D<A | B> operator+(const D<A> &a, const D<B> &b)
{
    return each<A | B>(a.v + b.v, [&](int k) {
        return !(A >> k & 1) ? b.g[k] : !(B >> k & 1) ? a.g[k] : a.g[k] + b.g[k];
    });
}
template <int A, int B>
__device__ __forceinline__ D<A | B> operator-(const D<A> &a, const D<B> &b)
{
    return each<A | B>(a.v - b.v, [&](int k) {
        return !(A >> k & 1) ? -b.g[k] : !(B >> k & 1) ? a.g[k] : a.g[k] - b.g[k];
    });
}
template <int A, int B>
__device__ __forceinline__ D<A | B> operator*(const D<A> &a, const D<B> &b)
{
    return each<A | B>(a.v * b.v, [&](int k) {
        return !(A >> k & 1) ? a.v * b.g[k] : !(B >> k & 1) ? a.g[k] * b.v
                                            : fma(a.g[k], b.v, a.v * b.g[k]);
    });
}
template <int A>
__device__ __forceinline__ D<A> operator+(const D<A> &a, double c)
{
    return each<A>(a.v + c, [&](int k) { return a.g[k]; });
}
template <int A>
__device__ __forceinline__ D<A> operator+(double c, const D<A> &a) { return a + c; }
template <int A>
__device__ __forceinline__ D<A> operator-(const D<A> &a, double c) { return a + (-c); }
template <int A>
__device__ __forceinline__ D<A> operator-(double c, const D<A> &a) { return (-a) + c; }
template <int A>
__device__ __forceinline__ D<A> operator*(double c, const D<A> &a)
{
    return each<A>(c * a.v, [&](int k) { return c * a.g[k]; });
}
template <int A>
__device__ __forceinline__ D<A> operator*(const D<A> &a, double c) { return c * a; }
// 1/a
template <int A>
__device__ __forceinline__ D<A> inverse(const D<A> &a)
{
    // the displacement's few terms keep the division
    const double q = A ? fast_rcp(a.v) : 1.0 / a.v, s = -(q * q);
    return each<A>(q, [&](int k) { return s * a.g[k]; });
}
// log a, of which 1/a is known
template <int A>
__device__ __forceinline__ D<A> log_of(const D<A> &a, const D<A> &ia)
{
    return each<A>(log(a.v), [&](int k) { return ia.v * a.g[k]; });
}
// the length of (x, y, z) and its reciprocal
template <int A, int B, int C>
__device__ __forceinline__ void length(const D<A> &x, const D<B> &y, const D<C> &z,
                                       D<A | B | C> &r, D<A | B | C> &ir)
{
    constexpr int M = A | B | C;
    const double s = length3(x.v, y.v, z.v), is = M != 0 ? fast_rcp(s) : 1.0 / s;
    r = each<A | B | C>(s, [&](int k) {
        double t = A >> k & 1 ? x.v * x.g[k] : 0.0;
        if (B >> k & 1) t = A >> k & 1 ? fma(y.v, y.g[k], t) : y.v * y.g[k];
        if (C >> k & 1) t = (A | B) >> k & 1 ? fma(z.v, z.g[k], t) : z.v * z.g[k];
        return t * is;
    });
    const double q = -(is * is);
    ir = each<A | B | C>(is, [&](int k) { return q * r.g[k]; });
}
// Sums of two slips in one frame: the three components of the displacement, or
// the strain of its gradient (xx, 2xy, 2xz, yy, 2yz, zz).
template <bool GRAD>
struct TwoSlips {
    static constexpr int n = GRAD ? 6 : 3;
    double s[2][n];
    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int i = 0; i < n; i++) s[0][i] = s[1][i] = 0.0;
    }
    // the displacement component i of slip k grows by c a
    template <int A>
    __device__ __forceinline__ void add(int k, int i, double c, const D<A> &a)
    {
        if constexpr (GRAD) {
            constexpr int at[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
#pragma unroll
            for (int j = 0; j < 3; j++)
                if (A >> j & 1) s[k][at[i][j]] = fma(c, a.g[j], s[k][at[i][j]]);
        } else {
            s[k][i] = fma(c, a.v, s[k][i]);
        }
    }
};

// full-space TD (main or image) geometry, DispInHalfSpace.c:153-240
struct TdFull {
    double A[3][3];       // rows: normal, strike, dip (TDCS axes in ENU)
    double P2[3];         // origin of the TDCS (second vertex)
    double p1y, p1z, p3y, p3z;
    double vy[3], vz[3];  // vertex y,z in the TDCS (p1, p2 = 0, p3)
    double s1[3][2];      // configuration I side vectors (y,z): -e13, e12, e23
    double s2[3][2];      // configuration II: e13, -e12, -e23
    double ca[3], sa[3];  // cos/sin(-pi + vertex angle)
};

// one TD side of the harmonic correction, DispInHalfSpace.c:462-539
struct TdSide {
    int skip;             // vertical side (beta ~ 0 or pi)
    int pad;
    double A[3][3];       // ADCS axes (ey1 ey2 ey3 as columns)
    double PA[3];
    double sA[3];         // side vector in ADCS
    double aA, aB;        // -PA_z, -PB_z
    double beta;
    double trig[2][5];    // for angle -pi+beta (conf. I) and beta: sin, cos, cot,
                          // cot(angle/2), 1/cos
};

struct TriSource {
    TdFull full[2];       // main, image
    TdSide side[3];
    double bfs[2][3];     // EFCS slip of the two computed directions (harmonic part)
    double btd[2][3];     // TDCS Burgers vectors (tensile, strike, dip) of the two
                          // directions; used by the general-slip form only
    int surface;          // all vertices at z = 0 (image yz/zz sign quirk)
    int pad;
};

struct TriMedium {
    double mu, lambda, nu;
};

// barycentric configuration choice, DispInHalfSpace.c:389-417
__device__ __forceinline__ int tri_mode_d(double x, double y, double z, double p1a, double p1b,
                                          double p3a, double p3b)
{
    const double p2a = 0.0, p2b = 0.0;
    const double den = (p2b - p3b) * (p1a - p3a) + (p3a - p2a) * (p1b - p3b);
    const double a = ((p2b - p3b) * (x - p3a) + (p3a - p2a) * (y - p3b)) / den;
    const double b = ((p3b - p1b) * (x - p3a) + (p1a - p3a) * (y - p3b)) / den;
    const double c = 1.0 - a - b;
    int m = 1;
    if (a <= 0.0 && b > c && c > a) m = -1;
    else if (b <= 0.0 && c > a && a > b) m = -1;
    else if (c <= 0.0 && a > b && b > c) m = -1;
    else if (a == 0.0 && b >= 0.0 && c >= 0.0) m = 0;
    else if (a >= 0.0 && b == 0.0 && c >= 0.0) m = 0;
    else if (a >= 0.0 && b >= 0.0 && c == 0.0) m = 0;
    if (m == 0 && z != 0.0) m = 1;
    return m;
}

// angular dislocation without the Burgers-function term (DispInHalfSpace.c:
// 541-571) at (x, y, z) of its frame, for the Burgers vectors b[slip]; without
// TENSILE their first component is zero
template <bool GRAD, bool TENSILE>
__device__ __forceinline__ void angdis(double X, double Y, double Z, double ca, double sa,
                                       double nu, const double b[2][3], TwoSlips<GRAD> &W)
{
    const auto x = coordinate<GRAD, 0>(X);
    const auto y = coordinate<GRAD, 1>(Y);
    const auto z = coordinate<GRAD, 2>(Z);
    auto eta = y * ca - z * sa, zeta = y * sa + z * ca;
    eta.v = dot2(ca, Y, -sa, Z);
    zeta.v = dot2(sa, Y, ca, Z);
    constexpr int F = GRAD ? 7 : 0;
    D<F> r, w;
    length(x, y, z, r, w);
    D<F> rz = r - z, rt = r - zeta;
    if (GRAD) {   // on or beyond the ends by a rounding: singular
        if (Z > r.v) rz.v = __builtin_nan("");
        if (zeta.v > r.v) rt.v = __builtin_nan("");
    } else {
        if (Z > r.v) rz.v = 0.0;
        if (zeta.v > r.v) rt.v = 0.0;
    }
    const auto irz = inverse(rz), b2 = inverse(rt);
    const auto lz = log_of(rz, irz), lt = log_of(rt, b2);
    const auto a1 = w * irz, a2 = w * b2;
    const double k = 1.0 / (8.0 * 3.14159265358979323846 * (1.0 - nu)), n12 = 1.0 - 2.0 * nu;
    W.clear();
    auto put = [&](int i, int j, const auto &B) {
        W.add(0, i, k * b[0][j], B);
        W.add(1, i, k * b[1][j], B);
    };
    const auto g = n12 * (ca * lt - lz);
    const auto yd = y * (ca * a2 - a1);   // shared by the second column
    put(0, 1, x * x * (ca * a2 - a1) - g);
    put(1, 1, x * (yd - (sa * ca) * b2));
    put(2, 1, x * (ca * (z * a2) - (ca * ca) * b2 + w));
    put(0, 2, sa * (n12 * lt - x * x * a2));
    put(1, 2, sa * (x * (sa * b2 - y * a2)));
    put(2, 2, sa * (x * (ca * b2 - z * a2)));
    if constexpr (TENSILE) {
        put(0, 0, x * (y * a1 - eta * a2));
        put(1, 0, sa * (eta * b2) - y * (eta * a2) + y * y * a1 + g);
        put(2, 0, ca * (eta * b2) - y * w - z * (eta * a2) - (n12 * sa) * lt);
    }
}

// gradient of the solid angle that the edge from a to b (seen from the point)
// contributes, a x b (|a| + |b|) / (|a| |b| (|a| |b| + a.b)); the difference is
// taken by the product with |a||b| - a.b, whose product with the sum is
// |a x b|^2, where it would cancel
__device__ __forceinline__ void edge_solid_angle(const double a[3], const double b[3], double na,
                                                 double ina, double nb, double inb, double g[3])
{
    const double c[3] = {fma(a[1], b[2], -a[2] * b[1]), fma(a[2], b[0], -a[0] * b[2]),
                         fma(a[0], b[1], -a[1] * b[0])};
    const double ab = fma(a[0], b[0], fma(a[1], b[1], a[2] * b[2])), nn = na * nb;
    const double cc = fma(c[0], c[0], fma(c[1], c[1], c[2] * c[2]));
    const double t = ab > 0.0 ? fast_rcp(nn + ab) : (nn - ab) * fast_rcp(cc);
    const double f = (ina + inb) * t;
#pragma unroll
    for (int k = 0; k < 3; k++) g[k] = fma(f, c[k], g[k]);
}

// full-space TD (main or image), DispInHalfSpace.c:153-300, at the point X of the
// source frame: the sums of the two slips (bt: tensile, strike, dip components in
// the TDCS) in the TDCS.  False on the triangle's plane exactly above a side:
// NaN in the reference.
template <bool GRAD, bool TENSILE>
__device__ __forceinline__ bool td_full(const TdFull &T, const double X[3], double nu,
                                        const double bt[2][3], TwoSlips<GRAD> &U)
{
    const double dX = X[0] - T.P2[0], dY = X[1] - T.P2[1], dZ = X[2] - T.P2[2];
    const double x = dot3(T.A[0], dX, dY, dZ), y = dot3(T.A[1], dX, dY, dZ),
                 z = dot3(T.A[2], dX, dY, dZ);
    const int mode = tri_mode_d(y, z, x, T.p1y, T.p1z, T.p3y, T.p3z);
    U.clear();
#pragma unroll 1
    for (int v = 0; v < 3; v++) {
        const double s1 = mode == 1 ? T.s1[v][0] : T.s2[v][0];
        const double s2 = mode == 1 ? T.s1[v][1] : T.s2[v][1];
        // TDSetupD (DispInHalfSpace.c:419-460)
        const double ty = y - T.vy[v], tz = z - T.vz[v];
        double b[2][3];
#pragma unroll
        for (int s = 0; s < 2; s++) {
            b[s][0] = bt[s][0];
            b[s][1] = s2 * bt[s][1] + (-s1) * bt[s][2];
            b[s][2] = s1 * bt[s][1] + s2 * bt[s][2];
        }
        TwoSlips<GRAD> W;
        angdis<GRAD, TENSILE>(x, dot2(s2, ty, -s1, tz), dot2(s1, ty, s2, tz), T.ca[v], T.sa[v], nu, b,
                              W);
        // back to the TDCS, a rotation about its first axis
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const double *q = W.s[k];
            double *u = U.s[k];
            if constexpr (GRAD) {
                const double m = s1 * s2, p = fma(s2, s2, -s1 * s1);
                const double d = m * (q[3] - q[5]), h = m * q[4];
                u[0] += q[0];
                u[1] = fma(s2, q[1], fma(s1, q[2], u[1]));
                u[2] = fma(s2, q[2], fma(-s1, q[1], u[2]));
                u[3] += fma(s2 * s2, q[3], fma(s1 * s1, q[5], h));
                u[4] += fma(p, q[4], -2.0 * d);
                u[5] += fma(s1 * s1, q[3], fma(s2 * s2, q[5], -h));
            } else {
                u[0] += q[0];
                u[1] += s2 * q[1] + s1 * q[2];
                u[2] += (-s1) * q[1] + s2 * q[2];
            }
        }
    }
    // Burgers function: -1/4pi times the triangle's solid angle
    // (DispInHalfSpace.c:276-290)
    const double a[3] = {-x, T.p1y - y, T.p1z - z}, b[3] = {-x, -y, -z},
                 c[3] = {-x, T.p3y - y, T.p3z - z};
    const double na = length3(a[0], a[1], a[2]), nb = length3(b[0], b[1], b[2]),
                 nc = length3(c[0], c[1], c[2]);
    const double k = 1.0 / (4.0 * 3.14159265358979323846);
    D<GRAD ? 7 : 0> f;
    if constexpr (GRAD) {
        const double ia = fast_rcp(na), ib = fast_rcp(nb), ic = fast_rcp(nc);
        double g[3] = {0.0, 0.0, 0.0};
        edge_solid_angle(a, b, na, ia, nb, ib, g);
        edge_solid_angle(b, c, nb, ib, nc, ic, g);
        edge_solid_angle(c, a, nc, ic, na, ia, g);
        f = each<7>(0.0, [&](int j) { return -k * g[j]; });
    } else {
        const double trip = a[0] * (b[1] * c[2] - b[2] * c[1]) - a[1] * (b[0] * c[2] - b[2] * c[0])
                            + a[2] * (b[0] * c[1] - b[1] * c[0]);
        const double den = na * nb * nc + (a[0] * b[0] + a[1] * b[1] + a[2] * b[2]) * nc
                           + (a[0] * c[0] + a[1] * c[1] + a[2] * c[2]) * nb
                           + (b[0] * c[0] + b[1] * c[1] + b[2] * c[2]) * na;
        f = value(-2.0 * k * atan2(trip, den));
    }
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (TENSILE || i > 0) U.add(s, i, bt[s][i], f);
    return mode != 0;
}

// harmonic correction of an angular dislocation at depth a (DispInHalfSpace.c:
// 577-606; Nikkhoo & Walter 2015) at (y1, y2, y3) of its frame: w += sign times
// the displacement sums for the Burgers vectors b[slip]
template <bool GRAD>
__device__ __forceinline__ void fsc_add(double Y1, double Y2, double Y3, const double tr[5],
                                        double nu, double a, double sign, const double b[2][3],
                                        TwoSlips<GRAD> &W)
{
    const double sb = tr[0], cb = tr[1], cot = tr[2], cth = tr[3], icb = tr[4];
    const double k = sign / (4.0 * 3.14159265358979323846 * (1.0 - nu)), N1 = 1.0 - 2.0 * nu,
                 nu1 = 1.0 - nu, c2 = cot * cot;
    auto put = [&](int i, int j, const auto &B) {
        W.add(0, i, k * b[0][j], B);
        W.add(1, i, k * b[1][j], B);
    };
    const auto y1 = coordinate<GRAD, 0>(Y1);
    const auto y2 = coordinate<GRAD, 1>(Y2);
    const auto y3b = coordinate<GRAD, 2>(Y3 + 2.0 * a);
    constexpr int F = GRAD ? 7 : 0;
    D<F> rb, irb;
    length(y1, y2, y3b, rb, irb);
    auto z1b = y1 * cb + y3b * sb, z3b = y3b * cb - y1 * sb;
    z1b.v = dot2(cb, Y1, sb, y3b.v);
    z3b.v = dot2(-sb, Y1, cb, y3b.v);
    const auto W6 = rb + y3b, W7 = rb + z3b;
    const auto iW6 = inverse(W6), iW7 = inverse(W7);
    const auto L6 = log_of(W6, iW6), L7 = log_of(W7, iW7);
    // 2 atan(-y2 / (y1 - W6 cot(beta/2)))
    const auto den = y1 - cth * W6;
    D<F> Fib;
    {
        const double s = fast_rcp(fma(den.v, den.v, Y2 * Y2));
        Fib = each<F>(GRAD ? 0.0 : 2.0 * atan(-Y2 / den.v), [&](int j) {
            const double t = Y2 * den.g[j];
            return 2.0 * s * (j == 1 ? t - den.v : t);
        });
    }
    const auto ya = y3b - a;
    const auto q = rb * cb + y3b, s1 = rb * sb - y1;
    const auto ar = a * irb, ir2 = irb * irb, ar2 = a * ir2, ir3 = ir2 * irb;
    const auto c1 = ar + cb, n1 = ar + nu, n2 = ar + 2.0 * nu, o1 = 1.0 + icb * ar;
    const auto y3r = a * (y3b * ir2), g7 = q * iW7, yr = ya * irb, y2r = y2 * yr, p6 = y1 * iW6;
    const auto t6 = y2 * iW6, t7 = y2 * iW7, z7 = z1b * iW7, ya6 = ya * iW6, ya7 = ya * iW7;
    const auto y2r7 = y2r * iW7, yy3 = a * (ya * ir3), g71 = g7 * c1;
    const auto qz = a * (z1b * (irb * q)), yir7 = irb * iW7;
    const auto y22 = y2 * y2;
    put(0, 0, (-2.0 * nu1 * N1 * c2) * Fib + N1 * (t6 * (cot * (N1 - ar) - p6 * n1))
                  + (N1 * cb * cot) * (t7 * c1) + cot * (y2 * yy3)
                  + y2r * iW6 * (p6 * n2 + a * (y1 * ir2) - N1 * cot)
                  + y2r7 * (cb * (iW7 * (cot * (q * (N1 * cb - ar)) + (2.0 * nu1 * cb) * s1))
                            - (cb * cot) * y3r));
    put(1, 0, (N1 * (2.0 * nu1 * c2 - nu)) * L6 - (N1 * (2.0 * nu1 * c2 + N1) * cb) * L7
                  - N1 * (iW6 * (cot * (y1 * (N1 - ar)) + nu * y3b - a + y2 * t6 * n1))
                  - (N1 * cot) * (z7 * c1) - cot * (y1 * yy3)
                  + ya6 * (irb * ((N1 * cot) * y1 - a) + y2 * t6 * irb * n2 + a * (y22 * ir3)
                           - 2.0 * nu)
                  + ya7 * (cb * cb - irb * ((N1 * cot) * z1b + a * cb)
                           + cot * (irb * (y3r * z1b)) - yir7 * ((cb * cb) * y22 - cot * qz)));
    put(2, 0, (2.0 * nu1 * N1 * cot) * Fib + (2.0 * nu1) * (t6 * n2 - cb * (t7 * c1))
                  + y2r * ((2.0 * nu) * iW6 + ar2) + cb * (y2r7 * (N1 - g71 - y3r)));
    put(0, 1, (N1 * (2.0 * nu1 * c2 + nu)) * L6 - (N1 * (2.0 * nu1 * c2 + 1.0) * cb) * L7
                  + N1 * (iW6 * (nu * y3b - (N1 * cot) * y1 - a + cot * (y1 * ar) + y1 * p6 * n1))
                  - (N1 * cot) * (iW7 * (cb * z1b - icb * (s1 * ar))) - cot * (y1 * yy3)
                  + ya6 * (irb * ((N1 * cot) * y1 + a) - y1 * p6 * irb * n2 - a * (y1 * y1 * ir3)
                           + 2.0 * nu)
                  + cot * (ya7 * (icb * (y1 * (irb * y3r)) + s1 * irb * (2.0 * nu1 * cb - g7 * o1)
                                  - cb * sb)));
    put(1, 1, (2.0 * nu1 * N1 * c2) * Fib + N1 * (t6 * (p6 * n1 - cot * (N1 - ar)))
                  - (N1 * cot) * (t7 * o1) - cot * (y2 * yy3)
                  + y2r * iW6 * (N1 * cot - (2.0 * nu) * p6 - y1 * ar * (irb + iW6))
                  + cot * (y2r7 * (g7 * o1 + icb * y3r - 2.0 * nu1 * cb)));
    put(2, 1, (-2.0 * nu1 * N1 * cot) * (L6 - cb * L7) - (2.0 * nu1) * (p6 * n2 - z7 * c1)
                  + yr * (N1 * cot - (2.0 * nu) * p6 - a * (y1 * ir2))
                  - ya7 * (cb * sb + cot * (q * irb * (2.0 * nu1 * cb - g7))
                           + ar * (sb - y3b * (z1b * ir2) - z7 * (q * irb))));
    put(0, 2, N1 * (t6 * (1.0 + ar) - cb * (t7 * c1)) - y2r * (ar2 + iW6)
                  + cb * (y2r7 * (g71 + y3r)));
    put(1, 2, N1 * (z7 * c1 - sb * L7 - p6 * (1.0 + ar)) + y1 * yr * (ar2 + iW6)
                  - ya7 * (sb * (cb - ar) + z1b * irb * (1.0 + y3r)
                           - yir7 * ((cb * sb) * y22 - qz)));
    put(2, 2, (2.0 * nu1) * (Fib + sb * (t7 * c1)) + sb * (y2r7 * (1.0 + g71 + y3r)));
}

// harmonic part of both slips (DispInHalfSpace.c:306-368, 462-539) at the point X
// of the source frame, in that frame
template <bool GRAD>
__device__ __forceinline__ void td_fsc(const TriSource &S, const double X[3], double nu,
                                       TwoSlips<GRAD> &U)
{
    U.clear();
    // each side's two ends in one loop, so that the term's code is there once
#pragma unroll 1
    for (int se = 0; se < 6; se++) {
        const TdSide &T = S.side[se >> 1];
        if (T.skip) continue;
        const bool end = se & 1;
        // the side's axes: horizontal (h0, h1), (h1, -h0), and down
        const double h0 = T.A[0][0], h1 = T.A[0][1];
        const double dx = X[0] - T.PA[0], dy = X[1] - T.PA[1], dz = X[2] - T.PA[2];
        double y[3] = {dot2(h0, dx, h1, dy), dot2(h1, dx, -h0, dy), -dz};
        const int cfg = (T.beta * y[0] >= 0.0) ? 0 : 1;
        if (end)
#pragma unroll
            for (int i = 0; i < 3; i++) y[i] -= T.sA[i];
        double b[2][3], tr[5];
#pragma unroll
        for (int s = 0; s < 2; s++) {
            b[s][0] = h0 * S.bfs[s][0] + h1 * S.bfs[s][1];
            b[s][1] = h1 * S.bfs[s][0] - h0 * S.bfs[s][1];
            b[s][2] = -S.bfs[s][2];
        }
#pragma unroll
        for (int i = 0; i < 5; i++) tr[i] = T.trig[cfg][i];
        TwoSlips<GRAD> W;
        W.clear();
        fsc_add<GRAD>(y[0], y[1], y[2], tr, nu, end ? T.aB : T.aA, end ? 1.0 : -1.0, b, W);
        // back to the source frame
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const double *q = W.s[k];
            double *u = U.s[k];
            if constexpr (GRAD) {
                const double m = h0 * h1, p = fma(h1, h1, -h0 * h0);
                const double d = m * (q[0] - q[3]), h = m * q[1];
                u[0] += fma(h0 * h0, q[0], fma(h1 * h1, q[3], h));
                u[1] += fma(p, q[1], 2.0 * d);
                u[2] -= fma(h0, q[2], h1 * q[4]);
                u[3] += fma(h1 * h1, q[0], fma(h0 * h0, q[3], -h));
                u[4] -= fma(h1, q[2], -h0 * q[4]);
                u[5] += q[5];
            } else {
                u[0] += h0 * q[0] + h1 * q[1];
                u[1] += h1 * q[0] - h0 * q[1];
                u[2] -= q[2];
            }
        }
    }
}

// a strain in the TDCS (rows of A) to the source frame
__device__ __forceinline__ void rotate_strain(const double A[3][3], const double t[6], double e[6])
{
    const double xy = 0.5 * t[1], xz = 0.5 * t[2], yz = 0.5 * t[4];
    const double m[3][3] = {{t[0], xy, xz}, {xy, t[3], yz}, {xz, yz, t[5]}};
    double p[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
            p[i][j] = fma(m[i][0], A[0][j], fma(m[i][1], A[1][j], m[i][2] * A[2][j]));
    int c = 0;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = i; j < 3; j++, c++)
            e[c] = fma(A[0][i], p[0][j], fma(A[1][i], p[1][j], A[2][i] * p[2][j]));
}

__device__ __forceinline__ void hooke6(const double e[6], double mu, double lambda, double s[6])
{
    const double tr = e[0] + e[3] + e[5];
    s[0] = 2.0 * mu * e[0] + lambda * tr;
    s[3] = 2.0 * mu * e[3] + lambda * tr;
    s[5] = 2.0 * mu * e[5] + lambda * tr;
    s[1] = 2.0 * mu * e[1];
    s[2] = 2.0 * mu * e[2];
    s[4] = 2.0 * mu * e[4];
}

// strains (ENU) of the three parts for the two slips, straininhalfspace_: e[0]
// main and harmonic parts, e[1] the image's, whose yz and zz change sign for a
// triangle with every vertex at the surface (StrainInHalfSpace.c:162-165)
template <bool GEN>
__device__ __forceinline__ void tri_strain2(const TriMedium &M, const TriSource &S,
                                            const double X[3], double e[2][2][6])
{
    // TDCS Burgers vectors (tensile, strike, dip): strike unit -> (0,1,0);
    // dip unit d=1 enters as Ds=-d (nikkhoo15.f90:142) -> (0,0,-1)
    const double unit[2][3] = {{0.0, 1.0, 0.0}, {0.0, 0.0, -1.0}};
    const double (*bt)[3] = GEN ? S.btd : unit;
    TwoSlips<true> U;
    // the longest part first, while the fewest sums are held
    td_fsc<true>(S, X, M.nu, U);
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int k = 0; k < 6; k++) e[0][s][k] = k == 0 || k == 3 || k == 5 ? U.s[s][k] : 0.5 * U.s[s][k];
#pragma unroll 1
    for (int part = 0; part < 2; part++) {
        const bool ok = td_full<true, GEN>(S.full[part], X, M.nu, bt, U);
#pragma unroll
        for (int s = 0; s < 2; s++) {
            double r[6];
            rotate_strain(S.full[part].A, U.s[s], r);
#pragma unroll
            for (int k = 0; k < 6; k++) {
                const double v = ok ? r[k] : __builtin_nan("");
                if (part == 0) e[0][s][k] += v;
                else e[1][s][k] = v;
            }
        }
    }
}

// NED stress (s11,s12,s13,s22,s23,s33) at NED point (x1,x2,x3) for two slip
// vectors of the source: straininhalfspace_ in ENU with the conversions of
// nikkhoo15.f90:130-161.  GEN = false: unit strike (Ss) and unit dip (Sd),
// with the Burgers vectors as compile-time constants; GEN = true: the two
// TDCS Burgers vectors stored in the source (any strike / dip / opening).
template <bool GEN = false>
__device__ __forceinline__ void tri_stress2(const TriMedium &M, const TriSource &S, double x1,
                                            double x2, double x3, double Ss[6], double Sd[6])
{
    const double X[3] = {x2, x1, -x3};
    double e[2][2][6];
    tri_strain2<GEN>(M, S, X, e);
    double *out[2] = {Ss, Sd};
#pragma unroll
    for (int k = 0; k < 2; k++) {
        double s[6], im[6];
        hooke6(e[0][k], M.mu, M.lambda, s);
        hooke6(e[1][k], M.mu, M.lambda, im);
        if (S.surface) {
            im[4] = -im[4];
            im[5] = -im[5];
        }
#pragma unroll
        for (int i = 0; i < 6; i++) s[i] += im[i];
        // ENU (xx,xy,xz,yy,yz,zz) -> NED (nikkhoo15.f90:156-161)
        out[k][0] = s[3];
        out[k][1] = s[1];
        out[k][2] = -s[4];
        out[k][3] = s[0];
        out[k][4] = -s[2];
        out[k][5] = s[5];
    }
}

// NED displacement at NED point (x1, x2, x3) for unit strike slip (us) and
// unit dip slip (ud): computeDisplacementNikkhoo15 (nikkhoo15.f90:324-367)
// over dispinhalfspace_ (DispInHalfSpace.c:42-152).  The main, harmonic and
// image parts are summed in that order; with every vertex at the surface the
// image part's vertical component and then the total change sign.
__device__ __forceinline__ void tri_disp2(const TriMedium &M, const TriSource &S, double x1,
                                          double x2, double x3, double us[3], double ud[3])
{
    const double X[3] = {x2, x1, -x3};
    const double unit[2][3] = {{0.0, 1.0, 0.0}, {0.0, 0.0, -1.0}};
    double w[2][3];
    TwoSlips<false> U, H;
    td_fsc<false>(S, X, M.nu, H);
#pragma unroll 1
    for (int part = 0; part < 2; part++) {
        const TdFull &T = S.full[part];
        const bool ok = td_full<false, false>(T, X, M.nu, unit, U);
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                double d = T.A[0][i] * U.s[s][0] + T.A[1][i] * U.s[s][1]
                           + T.A[2][i] * U.s[s][2];
                if (!ok) d = __builtin_nan("");
                if (part == 0) w[s][i] = d + H.s[s][i];
                else w[s][i] += S.surface && i == 2 ? -d : d;
                if (part == 1 && S.surface) w[s][i] = -w[s][i];
            }
    }
    // east, north, up -> north, east, down
    double *out[2] = {us, ud};
#pragma unroll
    for (int s = 0; s < 2; s++) {
        out[s][0] = w[s][1];
        out[s][1] = w[s][0];
        out[s][2] = -w[s][2];
    }
}

#pragma clang fp contract(off)

}  // namespace ucy
