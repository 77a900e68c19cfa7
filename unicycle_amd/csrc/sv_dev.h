// sv_dev.h -- strains of a vertical strain volume (Barbot, Moore & Lambert 2017)
// for the six unit eigenstrains, one (receiver, volume) pair per lane.
//
// The displacement J-integrals of sv_jint.h (strainvolume.f90:215-991) summed
// over the 8 corners and differentiated, with three things done on paper:
//
// - A term that depends on two of a corner's three coordinates cancels over the
//   third and is not formed: x3 atan2(x3, a), y2 atan2(-3 y2, a), u atan(u/w),
//   x3 log(a^2 + b^2) and so on.  With log(R2 - w) = log(u^2 + p^2) - log(R2 + w)
//   six logarithms and six angles per corner are left.  The quotients of J1113,
//   J1123 and their kin reduce to
//     Q = (x3 (R2 + y3) - k p R2) / (R2 (R2 + p)),  k = (nu - 1)(2 nu - 1),
//   and to x3 y3 (ab, bp, ap) / (R2 (a^2 + p^2)) or (b^2 + p^2): they have no pole
//   above a corner.  The rounding of the cancelled terms, x3 times an angle, next
//   to the sum's (size/distance)^3, is gone with them.
// - Logarithms and angles are multiplied by coefficients that are linear in the
//   coordinates, so their values enter a gradient times constants only: their
//   signed sums over the corners do.  A sum of logarithms is one logarithm of a
//   quotient of products, a sum of angles the argument of a product of complex
//   numbers with its turns counted: 12 functions per pair, not 96.
// - Strains need the symmetric part of the gradient: 36 sums, not 54.
//
// Differentiating the formula text of sv_jint.h in forward mode took 19.4
// thousand instructions per corner in three passes (155 KB of code, read again
// for each corner, past the instruction cache); this takes 1.8 thousand.  Against
// quadruple precision the median error falls 1.2 times (5 km away) to 12 times
// (200 km away); the largest ones, from 1 - (p/R2)^2 below a volume, are the same.
#pragma once
#include <hip/hip_runtime.h>

namespace ucy {

// products and sums fuse up to the end of this header
#pragma clang fp contract(fast)

// nu's polynomials, formed once on the host
struct SvMedium {
    double m14;            // 4 (nu-1)
    double m2, m22, m2s;   // 2nu-1, 2(2nu-1), 2(2nu-1)^2
    double k, k4;          // (nu-1)(2nu-1), 4k
    double c3, c5, c6, c7, c8, c9;
    double n4m2;           // 4 nu (2nu-1)
};

inline SvMedium sv_medium(double nu)
{
    const double m1 = nu - 1.0, m2 = 2.0 * nu - 1.0;
    SvMedium M;
    M.m14 = 4.0 * m1;
    M.m2 = m2;
    M.m22 = 2.0 * m2;
    M.m2s = 2.0 * m2 * m2;
    M.k = m1 * m2;
    M.k4 = 4.0 * m1 * m2;
    M.c3 = 4.0 * nu - 3.0;
    M.c5 = 5.0 + 4.0 * nu * (2.0 * nu - 3.0);
    M.c6 = 3.0 - 6.0 * nu + 4.0 * nu * nu;
    M.c7 = 4.0 * nu * nu - 2.0 * nu - 1.0;
    M.c8 = 7.0 + 8.0 * (nu - 2.0) * nu;
    M.c9 = 1.0 + 8.0 * m1 * nu;
    M.n4m2 = 4.0 * nu * m2;
    return M;
}

// 1/x and 1/sqrt(x) by the hardware estimates and Newton steps; x > 0 here
__device__ __forceinline__ double sv_rcp(double x)
{
    double q = __builtin_amdgcn_rcp(x);
    q = fma(fma(-x, q, 1.0), q, q);
    return fma(fma(-x, q, 1.0), q, q);
}
__device__ __forceinline__ double sv_rsqrt(double x)
{
    double q = __builtin_amdgcn_rsq(x);
    q = fma(q * 0.5, fma(-x * q, q, 1.0), q);
    return fma(q * 0.5, fma(-x * q, q, 1.0), q);
}

// The image distance and 1/(1 - (p/R2)^2), the slope of acoth(p/R2), rounded as the
// formula text has them: far below a volume the difference loses digits, and
// results keep the ones that they had
__device__ __forceinline__ double sv_length(double a2, double b2, double p2)
{
#pragma clang fp contract(off)
    return sqrt(a2 + b2 + p2);
}
__device__ __forceinline__ double sv_acoth_slope(double p, double R)
{
#pragma clang fp contract(off)
    const double X = p / R;
    return sv_rcp(1.0 - X * X);
}

// The sum of signed angles atan2(y, x): the argument of the product of x + iy,
// and the turns by which the sum exceeds its principal value.  Adding an angle of
// [0, pi] to one of [0, pi] and landing below the axis is a turn, the signs of
// zeros included (pi + pi is a product of -0 imaginary part).
struct AngleSum {
    double x, y;
    int turns;
};
__device__ __forceinline__ int sign_bit(double v)
{
    return (int)((unsigned)__double2hiint(v) >> 31);
}
__device__ __forceinline__ void add_angle(AngleSum &P, double y, double x)
{
    const double nx = P.x * x - P.y * y, ny = P.x * y + P.y * x;
    const int a = sign_bit(y), b = sign_bit(P.y), c = sign_bit(ny);
    P.turns += (~(a | b) & c) - (a & b & ~c & 1);
    P.x = nx;
    P.y = ny;
}
__device__ __forceinline__ double value(const AngleSum &P)
{
    return atan2(P.y, P.x) + 6.283185307179586 * (double)P.turns;
}

// The sum of signed logarithms, positive ones in num
struct LogSum {
    double num, den;
};
__device__ __forceinline__ double value(const LogSum &P) { return log(P.num / P.den); }

// y = R + a, R^2 = a^2 + w, without cancellation for negative a; returns 1/y,
// given 1/w
__device__ __forceinline__ double sum_inverse(double R, double a, double w, double iw, double &y)
{
    const double t = R + fabs(a), it = sv_rcp(t);
    const bool up = a >= 0.0;
    y = up ? t : w * it;
    return up ? it : t * iw;
}

// Strain sums (11, 2 x 12, 2 x 13, 22, 2 x 23, 33 in the volume's frame) of the
// six slots of sv_jint.h's Grad; u(i) of slot k has gradient (g0, g1, g2)
struct SvSums {
    double s[6][6];
};
template <int I>
__device__ __forceinline__ void add_gradient(SvSums &A, int k, double g0, double g1, double g2)
{
    constexpr int at[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
    A.s[k][at[I][0]] += g0;
    A.s[k][at[I][1]] += g1;
    A.s[k][at[I][2]] += g2;
}

// running sums over the corners
struct SvAngles {
    AngleSum A1, B1, C1, A2, B2, C2;   // atan2(R a, b c), (R b, a c), (R c, a b)
};

// One corner: a, b, x3-y3, x3+y3 = x1'-y1, x2'-y2, c, p; sg its sign; S =
// 1/(a^2+b^2).  y: the arguments of its logarithms, R1 + a, b, c, R2 + a, b, p
__device__ __forceinline__ void sv_corner(const SvMedium &M, SvSums &A, SvAngles &F, double sg,
                                          double a, double b, double x3, double y3, double a2,
                                          double b2, double S, double y[6])
{
    const double c = x3 - y3, p = x3 + y3;
    {
        // the source point's terms
        const double c2 = c * c, ac2 = a2 + c2, bc2 = b2 + c2;
        const double rr = a2 + bc2, ir = sv_rsqrt(rr), R = rr * ir, r = sg * ir;
        const double T = sv_rcp(ac2), U = sv_rcp(bc2);
        const double la = r * sum_inverse(R, a, bc2, U, y[0]);
        const double lb = r * sum_inverse(R, b, ac2, T, y[1]);
        const double lc = r * sum_inverse(R, c, a2 + b2, S, y[2]);
        const double ir2 = ir * ir;
        add_angle(F.A1, sg * (a * ir), b * c * ir2);
        add_angle(F.B1, sg * (b * ir), a * c * ir2);
        add_angle(F.C1, sg * (c * ir), a * b * ir2);
        // gradients: LA (r, b la, c la), LB (a lb, r, c lb), LC (a lc, b lc, r)
        const double bcr = b * c * r, acr = a * c * r, abr = a * b * r;
        const double A10 = bcr * (S + T), A11 = -acr * S, A12 = -abr * T;
        const double B10 = -bcr * S, B11 = acr * (S + U), B12 = -abr * U;
        const double C10 = -bcr * T, C11 = -acr * U, C12 = abr * (T + U);
        const double LA1 = b * la, LA2 = c * la, LB0 = a * lb, LB2 = c * lb, LC0 = a * lc,
                     LC1 = b * lc;
        {
            const double x = -M.m22 * a, y = -M.c3 * b, z = -M.c3 * c;
            add_gradient<0>(A, 0, x * A10 + y * LC0 + z * LB0, x * A11 + y * LC1 + z * r,
                            x * A12 + y * r + z * LB2);
        }
        add_gradient<0>(A, 1, -b * LC0, -b * LC1, -b * r);
        add_gradient<0>(A, 2, -c * LB0, -c * r, -c * LB2);
        {
            const double x = -M.m14 * b, y = -M.m22 * a, z = -M.m14 * c;
            add_gradient<0>(A, 3, x * B10 + y * LC0 + z * r, x * B11 + y * LC1 + z * LA1,
                            x * B12 + y * r + z * LA2);
            // (0,4): a log(R+b), b log(R+a), c C1
            add_gradient<0>(A, 4, y * LB0 + x * r + z * C10, y * r + x * LA1 + z * C11,
                            y * LB2 + x * LA2 + z * C12);
        }
        const double R0 = -2.0 * a * r, R1 = -2.0 * b * r, R2 = -2.0 * c * r;
        add_gradient<0>(A, 5, R0, R1, R2);
        add_gradient<1>(A, 4, R0, R1, R2);
        add_gradient<2>(A, 3, R0, R1, R2);
        add_gradient<1>(A, 0, -a * LC0, -a * LC1, -a * r);
        {
            const double x = -M.m22 * b, y = -M.c3 * a, z = -M.c3 * c;
            add_gradient<1>(A, 1, x * B10 + y * LC0 + z * r, x * B11 + y * LC1 + z * LA1,
                            x * B12 + y * r + z * LA2);
        }
        add_gradient<1>(A, 2, -c * r, -c * LA1, -c * LA2);
        {
            const double x = -M.m14 * a, y = -M.m22 * b, z = -M.m14 * c;
            add_gradient<1>(A, 3, x * A10 + y * LC0 + z * LB0, x * A11 + y * LC1 + z * r,
                            x * A12 + y * r + z * LB2);
            add_gradient<1>(A, 5, y * r + x * LB0 + z * C10, y * LA1 + x * r + z * C11,
                            y * LA2 + x * LB2 + z * C12);
        }
        add_gradient<2>(A, 0, -a * LB0, -a * r, -a * LB2);
        add_gradient<2>(A, 1, -b * r, -b * LA1, -b * LA2);
        {
            const double x = -M.m22 * c, y = -M.c3 * a, z = -M.c3 * b;
            add_gradient<2>(A, 2, x * C10 + y * LB0 + z * r, x * C11 + y * r + z * LA1,
                            x * C12 + y * LB2 + z * LA2);
        }
        {
            const double x = -M.m14 * a, y = -M.m14 * b, z = -M.m22 * c;
            add_gradient<2>(A, 4, x * A10 + y * LC0 + z * LB0, x * A11 + y * LC1 + z * r,
                            x * A12 + y * r + z * LB2);
            add_gradient<2>(A, 5, y * B10 + x * LC0 + z * r, y * B11 + x * LC1 + z * LA1,
                            y * B12 + x * r + z * LA2);
        }
    }
    {
        // the image's terms
        const double p2 = p * p, ap2 = a2 + p2, bp2 = b2 + p2;
        const double R = sv_length(a2, b2, p2), ir = sv_rcp(R), r = sg * ir;
        const double T = sv_rcp(ap2), U = sv_rcp(bp2);
        const double la = r * sum_inverse(R, a, bp2, U, y[3]);
        const double lb = r * sum_inverse(R, b, ap2, T, y[4]);
        const double ip = sum_inverse(R, p, a2 + b2, S, y[5]), lp = r * ip;
        const double ir2 = ir * ir;
        add_angle(F.A2, sg * (a * ir), b * p * ir2);
        add_angle(F.B2, sg * (b * ir), a * p * ir2);
        add_angle(F.C2, sg * (p * ir), a * b * ir2);
        const double bpr = b * p * r, apr = a * p * r, abr = a * b * r;
        const double A20 = bpr * (S + T), A21 = -apr * S, A22 = -abr * T;
        const double B20 = -bpr * S, B21 = apr * (S + U), B22 = -abr * U;
        const double C20 = -bpr * T, C21 = -apr * U, C22 = abr * (T + U);
        const double LA1 = b * la, LA2 = p * la, LB0 = a * lb, LB2 = p * lb, LP0 = a * lp,
                     LP1 = b * lp;
        // a Q and b Q
        const double x3ip = x3 * ip, pip = p * ip;
        const double Q = sg * (x3ip * (ir * y3 + 1.0) - M.k * pip);
        const double qR = r * (M.k * pip * ip - x3 * ir2 + x3ip * x3ip * ir + x3 * x3ip * ir2);
        const double q2 = p * qR
                          + sg * (M.k * (pip - 1.0) * ip + ir - 2.0 * x3ip * ir + x3ip * x3ip * ir);
        const double aq = a * qR, bq = b * qR;
        const double QA0 = Q + a * aq, QA1 = a * bq, QA2 = a * q2;
        const double QB0 = QA1, QB1 = Q + b * bq, QB2 = b * q2;
        // H1, M1 = x3 y3 (bp, ab) / (R2 (a^2+p^2)), H2, M2 with a and b exchanged
        const double xy = x3 * y3, t1 = r * T, t2 = r * U;
        const double f1 = ir2 + 2.0 * T, f2 = ir2 + 2.0 * U;
        const double g1 = xy * t1, g2 = xy * t2, y1t = y3 * t1, y2t = y3 * t2, px = p + x3;
        const double h1 = b * p * g1, m1 = a * b * g1, h2 = a * p * g2, m2 = a * b * g2;
        const double H10 = -a * f1 * h1, H11 = p * g1 - b * ir2 * h1, H12 = b * px * y1t - p * f1 * h1;
        const double M10 = b * g1 - a * f1 * m1, M11 = a * g1 - b * ir2 * m1,
                     M12 = a * b * y1t - p * f1 * m1;
        const double H20 = p * g2 - a * ir2 * h2, H21 = -b * f2 * h2, H22 = a * px * y2t - p * f2 * h2;
        const double M20 = b * g2 - a * ir2 * m2, M21 = a * g2 - b * f2 * m2,
                     M22 = a * b * y2t - p * f2 * m2;
        // x3 y3 / R2
        const double e = xy * r * ir2;
        const double E0 = -a * e, E1 = -b * e, E2 = y3 * r - p * e;
        const double R0 = a * r, R1 = b * r, R2 = p * r;
        // acoth(p/R2), 2 c3 x3 times it
        const double ac = 2.0 * M.c3 * x3 * sv_acoth_slope(p, R) * r * ir2;
        const double AC0 = -ac * p * a, AC1 = -ac * p * b, AC2 = ac * (a2 + b2);
        {
            const double x = -M.m2s * a, y = -M.c6 * b, z = 2.0 * x3 - M.c5 * p;
            add_gradient<0>(A, 0, 2.0 * (H10 - QB0) + x * A20 + y * LP0 + z * LB0,
                            2.0 * (H11 - QB1) + x * A21 + y * LP1 + z * r,
                            2.0 * (H12 - QB2) + x * A22 + y * r + z * LB2);
        }
        {
            const double y = -M.c7 * b;
            add_gradient<0>(A, 1, 2.0 * QB0 + y * LP0, 2.0 * QB1 + y * LP1, 2.0 * QB2 + y * r);
        }
        const double z2 = -(M.c8 * x3 + M.c9 * y3);
        {
            const double x = -M.k4 * a, y = -M.k4 * b;
            add_gradient<0>(A, 2, -2.0 * H10 + x * A20 + y * LP0 + z2 * LB0,
                            -2.0 * H11 + x * A21 + y * LP1 + z2 * r,
                            -2.0 * H12 + x * A22 + y * r + z2 * LB2);
            add_gradient<1>(A, 2, -2.0 * H20 + y * B20 + x * LP0 + z2 * r,
                            -2.0 * H21 + y * B21 + x * LP1 + z2 * LA1,
                            -2.0 * H22 + y * B22 + x * r + z2 * LA2);
        }
        const double ma = M.m14 * a, mb = M.m14 * b, mp = M.m14 * p, mx = -2.0 * M.m14 * x3;
        {
            const double y = -M.m2s * a;
            add_gradient<0>(A, 3, 4.0 * QA0 + mb * B20 + y * LP0 + mp * r,
                            4.0 * QA1 + mb * B21 + y * LP1 + mp * LA1,
                            4.0 * QA2 + mb * B22 + y * r + mp * LA2);
        }
        {
            const double y = -M.m2s * b;
            add_gradient<1>(A, 3, 4.0 * QB0 + ma * A20 + y * LP0 + mp * LB0,
                            4.0 * QB1 + ma * A21 + y * LP1 + mp * r,
                            4.0 * QB2 + ma * A22 + y * r + mp * LB2);
        }
        {
            const double y = M.m22 * a, z = M.m22 * b;
            add_gradient<0>(A, 4, 4.0 * M10 + mx * A20 + y * LB0 - mb * r - mp * C20,
                            4.0 * M11 + mx * A21 + y * r - mb * LA1 - mp * C21,
                            4.0 * M12 + mx * A22 + y * LB2 - mb * LA2 - mp * C22);
            add_gradient<1>(A, 5, 4.0 * M20 + mx * B20 + z * r - ma * LB0 - mp * C20,
                            4.0 * M21 + mx * B21 + z * LA1 - ma * r - mp * C21,
                            4.0 * M22 + mx * B22 + z * LA2 - ma * LB2 - mp * C22);
        }
        {
            const double x = 2.0 * M.c3, w = mx + x * x3;
            const double g0 = x * R0 - 4.0 * E0 + w * LP0 - AC0,
                         g1_ = x * R1 - 4.0 * E1 + w * LP1 - AC1,
                         g2_ = x * R2 - 4.0 * E2 + w * r - AC2;
            add_gradient<0>(A, 5, g0, g1_, g2_);
            add_gradient<1>(A, 4, g0, g1_, g2_);
        }
        {
            const double y = -M.c7 * a;
            add_gradient<1>(A, 0, 2.0 * QA0 + y * LP0, 2.0 * QA1 + y * LP1, 2.0 * QA2 + y * r);
        }
        {
            const double x = -M.m2s * b, y = -M.c6 * a, z = 2.0 * x3 - M.c5 * p;
            add_gradient<1>(A, 1, 2.0 * (H20 - QA0) + x * B20 + y * LP0 + z * r,
                            2.0 * (H21 - QA1) + x * B21 + y * LP1 + z * LA1,
                            2.0 * (H22 - QA2) + x * B22 + y * r + z * LA2);
        }
        {
            // y3 grad atan(b/a) = y3 S (-b, a, 0), and minus that of atan(a/b)
            const double v = -M.k4 * sg * y3 * S, w = -(M.n4m2 * x3 + M.k4 * y3);
            const double y = M.c9 * a, z = M.c9 * b;
            add_gradient<2>(A, 0, -2.0 * M10 - v * b + w * A20 + y * LB0,
                            -2.0 * M11 + v * a + w * A21 + y * r, -2.0 * M12 + w * A22 + y * LB2);
            add_gradient<2>(A, 1, -2.0 * M20 + v * b + w * B20 + z * r,
                            -2.0 * M21 - v * a + w * B21 + z * LA1, -2.0 * M22 + w * B22 + z * LA2);
            const double q = 2.0 * (w + 2.0 * M.c3 * x3);
            add_gradient<2>(A, 3, 2.0 * (M.c9 * R0 - AC0) + 4.0 * E0 + q * LP0,
                            2.0 * (M.c9 * R1 - AC1) + 4.0 * E1 + q * LP1,
                            2.0 * (M.c9 * R2 - AC2) + 4.0 * E2 + q * r);
        }
        {
            const double x = M.m2s * p, y = M.c5 * a, z = M.c5 * b;
            add_gradient<2>(A, 2, 2.0 * (M10 + M20) + x * C20 + y * LB0 + z * r,
                            2.0 * (M11 + M21) + x * C21 + y * r + z * LA1,
                            2.0 * (M12 + M22) + x * C22 + y * LB2 + z * LA2);
        }
        {
            const double z = M.m22 * c;
            add_gradient<2>(A, 4, 4.0 * H10 + ma * A20 + mb * LP0 + z * LB0,
                            4.0 * H11 + ma * A21 + mb * LP1 + z * r,
                            4.0 * H12 + ma * A22 + mb * r + z * LB2);
            add_gradient<2>(A, 5, 4.0 * H20 + mb * B20 + ma * LP0 + z * r,
                            4.0 * H21 + mb * B21 + ma * LP1 + z * LA1,
                            4.0 * H22 + mb * B22 + ma * r + z * LA2);
        }
    }
}

// the coefficients' own gradients times the sums of logarithms and angles
__device__ __forceinline__ void sv_values(const SvMedium &M, SvSums &A, const SvAngles &F,
                                          const LogSum G[6])
{
    const double A1 = value(F.A1), B1 = value(F.B1), C1 = value(F.C1);
    const double A2 = value(F.A2), B2 = value(F.B2), C2 = value(F.C2);
    const double LA = value(G[0]), LB = value(G[1]), LC = value(G[2]);
    const double LA2 = value(G[3]), LB2 = value(G[4]), LP = value(G[5]);
    const double m = M.m14, w = 2.0 - M.c5;
    const double lcp = -M.c3 * LC - M.c6 * LP, l7 = -LC - M.c7 * LP, kp = -M.k4 * LP;
    const double c12 = -m * (C1 + C2), l22 = -M.m22 * LC - M.m2s * LP, lp = -2.0 * m * LP;
    add_gradient<0>(A, 0, -M.m22 * A1 - M.m2s * A2, lcp, -M.c3 * LB + w * LB2);
    add_gradient<0>(A, 1, 0.0, l7, 0.0);
    add_gradient<0>(A, 2, -M.k4 * A2, kp, -LB - M.c8 * LB2);
    add_gradient<0>(A, 3, l22, m * (B2 - B1), m * (LA2 - LA));
    add_gradient<0>(A, 4, M.m22 * (LB2 - LB), -m * (LA + LA2), c12 - 2.0 * m * A2);
    add_gradient<0>(A, 5, 0.0, 0.0, lp);
    add_gradient<1>(A, 0, l7, 0.0, 0.0);
    add_gradient<1>(A, 1, lcp, -M.m22 * B1 - M.m2s * B2, -M.c3 * LA + w * LA2);
    add_gradient<1>(A, 2, kp, -M.k4 * B2, -LA - M.c8 * LA2);
    add_gradient<1>(A, 3, m * (A2 - A1), l22, m * (LB2 - LB));
    add_gradient<1>(A, 4, 0.0, 0.0, lp);
    add_gradient<1>(A, 5, -m * (LB + LB2), M.m22 * (LA2 - LA), c12 - 2.0 * m * B2);
    add_gradient<2>(A, 0, -LB + M.c9 * LB2, 0.0, -M.n4m2 * A2);
    add_gradient<2>(A, 1, 0.0, -LA + M.c9 * LA2, -M.n4m2 * B2);
    add_gradient<2>(A, 2, -M.c3 * LB + M.c5 * LB2, -M.c3 * LA + M.c5 * LA2,
                    M.m2s * C2 - M.m22 * C1);
    add_gradient<2>(A, 3, 0.0, 0.0, -2.0 * M.n4m2 * LP);
    add_gradient<2>(A, 4, m * (A2 - A1), m * (LP - LC), M.m22 * (LB2 - LB));
    add_gradient<2>(A, 5, m * (LP - LC), m * (B2 - B1), M.m22 * (LA2 - LA));
}

// The 36 sums at (x1p, x2p, x3) of the volume (y1 in {0, L}, y2 in {+-T/2}, y3 in
// {q3, q3 + W}); x1p and x2p not on a face's plane
__device__ __forceinline__ void sv_sums(const SvMedium &M, SvSums &A, double x1p, double x2p,
                                        double x3, double q3, double L, double Th, double W)
{
    for (int k = 0; k < 6; k++)
        for (int j = 0; j < 6; j++) A.s[k][j] = 0.0;
    const AngleSum one = {1.0, 0.0, 0};
    SvAngles F = {one, one, one, one, one, one};
    LogSum G[6];
    for (int k = 0; k < 6; k++) G[k] = {1.0, 1.0};
    const double h = Th / 2.0;
    // a corner's sign: that of y1 = L, of y2 = T/2 and of y3 = q3 + W, multiplied
#pragma unroll 1
    for (int n = 0; n < 4; n++) {
        const double a = n < 2 ? x1p - L : x1p, b = (n & 1) ? x2p + h : x2p - h;
        const bool plus = n == 0 || n == 3;
        const double sg = plus ? 1.0 : -1.0;
        const double a2 = a * a, b2 = b * b, S = sv_rcp(a2 + b2);
        double yd[6], yu[6];
        sv_corner(M, A, F, sg, a, b, x3, q3 + W, a2, b2, S, yd);
        sv_corner(M, A, F, -sg, a, b, x3, q3, a2, b2, S, yu);
        for (int k = 0; k < 6; k++) {
            G[k].num *= plus ? yd[k] : yu[k];
            G[k].den *= plus ? yu[k] : yd[k];
        }
    }
    sv_values(M, A, F, G);
}

// Stresses (NED 11 12 13 22 23 33) of the six unit eigenstrains from the sums:
// strain in the primed frame, rotation, eigenstrain removed inside the volume,
// Hooke (strainvolume.f90:1073-1138)
__device__ __forceinline__ void sv_stresses(const SvSums &A, double G, double nu, double lambda,
                                            double ct, double st, double inside, double out[6][6])
{
    const double K = 1.0 / (16.0 * 3.141592653589793115997963468544185161 * (1.0 - nu) * G);
    // slots: 11, 22, 33, 12, 13, 23; columns: 11, 12, 13, 22, 23, 33
    constexpr int slot[6] = {0, 3, 4, 1, 5, 2};
    double tr[6];
#pragma unroll
    for (int j = 0; j < 6; j++) tr[j] = lambda * (A.s[0][j] + A.s[1][j] + A.s[2][j]);
#pragma unroll
    for (int e = 0; e < 6; e++) {
        const bool diagonal = slot[e] < 3;
        double ep[6];
#pragma unroll
        for (int j = 0; j < 6; j++) {
            const double v = 2.0 * G * A.s[slot[e]][j];
            const double h = (j == 1 || j == 2 || j == 4) ? 0.5 * K : K;
            ep[j] = h * (diagonal ? v + tr[j] : v) - (e == j ? inside : 0.0);
        }
        const double e11 = (ct * ep[0] - st * ep[1]) * ct - (ct * ep[1] - st * ep[3]) * st;
        const double e12 = (ct * ep[0] - st * ep[1]) * st + (ct * ep[1] - st * ep[3]) * ct;
        const double e13 = ct * ep[2] - st * ep[4];
        const double e22 = (st * ep[0] + ct * ep[1]) * st + (st * ep[1] + ct * ep[3]) * ct;
        const double e23 = st * ep[2] + ct * ep[4];
        const double lk = lambda * (e11 + e22 + ep[5]);
        out[e][0] = lk + 2.0 * G * e11;
        out[e][1] = 2.0 * G * e12;
        out[e][2] = 2.0 * G * e13;
        out[e][3] = lk + 2.0 * G * e22;
        out[e][4] = 2.0 * G * e23;
        out[e][5] = lk + 2.0 * G * ep[5];
    }
}

#pragma clang fp contract(off)

}  // namespace ucy
