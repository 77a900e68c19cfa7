// ode_dev.h -- device functions of the single-instance integrator shared by the
// captured attempt (k_ode.hip) and the resident one (k_resident.hip): the
// per-element pre- and post-passes of odefun, the Cash-Karp stage inputs, the
// row dot products and the step control.  Both integrators call the same
// functions in the same order, so a run gives the same bits on either.
#pragma once
#include <hip/hip_runtime.h>
#include "ucy_internal.h"

namespace ucy {

// ratestate.f90:130 lg10=LOG(1.d1)
constexpr double kLg10 = 2.302585092994045684;

// Cash-Karp tableau (ode45.f90:126-134)
#define B21 0.2
#define B31 (3.0 / 40.0)
#define B32 (9.0 / 40.0)
#define B41 0.3
#define B42 (-0.9)
#define B43 1.2
#define B51 (-11.0 / 54.0)
#define B52 2.5
#define B53 (-70.0 / 27.0)
#define B54 (35.0 / 27.0)
#define B61 (1631.0 / 55296.0)
#define B62 (175.0 / 512.0)
#define B63 (575.0 / 13824.0)
#define B64 (44275.0 / 110592.0)
#define B65 (253.0 / 4096.0)
#define C1 (37.0 / 378.0)
#define C3 (250.0 / 621.0)
#define C4 (125.0 / 594.0)
#define C6 (512.0 / 1771.0)
#define DC1 (C1 - 2825.0 / 27648.0)
#define DC3 (C3 - 18575.0 / 48384.0)
#define DC4 (C4 - 13525.0 / 55296.0)
#define DC5 (-277.0 / 14336.0)
#define DC6 (C6 - 0.25)

__device__ __forceinline__ unsigned long long dbits(double x)
{
    return (unsigned long long)__double_as_longlong(x);
}

// ---------------------------------------------------------------------------
// pre-pass for one patch (ratestate.f90:683-702) and one volume
// (viscouscycles.f90:940-995)
// ---------------------------------------------------------------------------
// what the friction law needs of an element before its traction rate is known:
// d(log10 theta)/dt of the aging law (ratestate.f90:752) and the terms of
// d(log10 V)/dt (ratestate.f90:758-762)
struct FrictionTerms {
    double dtheta, evolution, direct, damping;
};
__device__ __forceinline__ FrictionTerms friction_terms(double theta, double velocity,
                                                        const Friction &f)
{
    FrictionTerms g;
    g.dtheta = (exp(-theta * kLg10) - velocity / f.L) / kLg10;
    g.evolution = f.b * f.sig * g.dtheta * kLg10;
    g.damping = f.damping * velocity;
    g.direct = f.a * f.sig + g.damping;
    return g;
}

// what the post-pass of a patch takes over from the pre-pass at the same state
struct PatchPre {
    double velocity, cr, sr;
};

__device__ __forceinline__ void patch_pre(double ts, double td, double logv, PatchPre &q)
{
    const double rake = atan2(td, ts);
    q.cr = cos(rake);
    q.sr = sin(rake);
    q.velocity = exp(logv * kLg10);
}

__device__ __forceinline__ double patch_prepass(const double *p, const Friction &f, double *dp,
                                                double *vp)
{
    PatchPre q;
    patch_pre(p[2], p[3], p[6], q);
    const double vs = q.velocity * q.cr, vd = q.velocity * q.sr;
    dp[0] = vs;
    dp[1] = vd;
    vp[0] = vs - f.vplc;
    vp[1] = vd - f.vpls;
    return q.velocity;
}

// 2-D antiplane patch (fortran/2d/antiplane/src/ratestate.f90:660-677): slip
// rate V, v = V - Vpl (vplc holds Vpl)
__device__ __forceinline__ double ap_prepass(const double *p, const Friction &f, double *dp,
                                             double *vp)
{
    const double velocity = exp(p[3] * kLg10);
    dp[0] = velocity;
    vp[0] = velocity - f.vplc;
    return velocity;
}

// ratestate.f90 (2-D antiplane):698-722
__device__ __forceinline__ void ap_post(double t, const FrictionTerms &g, double *dp)
{
    const double dtau = t;
    dp[2] = g.dtheta;
    dp[3] = (dtau - g.evolution) / g.direct / kLg10;
    dp[1] = dtau - g.damping * dp[3] * kLg10;
}

__device__ __forceinline__ void ap_postpass(const double *p, const Friction &f, double t,
                                            double *dp)
{
    ap_post(t, friction_terms(p[2], exp(p[3] * kLg10), f), dp);
}

// 2-D plane-strain patch (fortran/2d/planestrain/src/ratestate.f90:692-712):
// dip-slip rate V, v = V - Vpl (vplc holds Vpl)
__device__ __forceinline__ double ps_prepass(const double *p, const Friction &f, double *dp,
                                             double *vp)
{
    const double velocity = exp(p[4] * kLg10);
    dp[0] = velocity;
    vp[0] = velocity - f.vplc;
    return velocity;
}

// ratestate.f90 (2-D plane strain):723-750: the dip traction drives the
// friction law at the constant normal stress sig; the normal traction rate is
// integrated as is
__device__ __forceinline__ void ps_post(const double *t, const FrictionTerms &g, double *dp)
{
    const double dtau = t[0];
    dp[3] = g.dtheta;
    dp[4] = (dtau - g.evolution) / g.direct / kLg10;
    dp[1] = dtau - g.damping * dp[4] * kLg10;
    dp[2] = t[1];
}

__device__ __forceinline__ void ps_postpass(const double *p, const Friction &f, const double *t,
                                            double *dp)
{
    ps_post(t, friction_terms(p[3], exp(p[4] * kLg10), f), dp);
}

// 2-D antiplane volume (fortran/2d/antiplane/src/viscouscycles.f90:846-877):
// state [e12, e13, s12, s13]; strain rate eII s with
// eII = gammadot0 (sII/Gm)^(n-1) / Gm exp(-Q/(R To)), v = that less the
// background rate; returns the strain-rate norm (eMax of :869)
__device__ __forceinline__ double ap_volume_prepass(const double *q, const Rheology &r, double *dq,
                                                    double *vq)
{
    const double s12 = q[2], s13 = q[3];
    const double sII = sqrt(s12 * s12 + s13 * s13);
    const double eII = r.gammadot0 * pow(sII / r.Gm, r.npower - 1.0) / r.Gm * r.arr;
    const double e12 = eII * s12, e13 = eII * s13;
    dq[0] = e12;
    dq[1] = e13;
    vq[0] = e12 - r.ebg[1];
    vq[1] = e13 - r.ebg[2];
    return sqrt(e12 * e12 + e13 * e13);
}

// 2-D plane-strain volume (fortran/2d/planestrain/src/viscouscycles.f90:
// 929-967): state [e22, e23, e33, s22, s23, s33]; with the 2-D deviatoric
// stress s' (p = (s22 + s33) / 2), strain rate eII s' with
// eII = gammadot0 sII^(n-1) exp(-Q/(R To)); v = (that - the background
// rate) 1e3, as K's volume columns are strains of 1e-3; returns the
// strain-rate norm (eMax of :962)
__device__ __forceinline__ double ps_volume_prepass(const double *q, const Rheology &r, double *dq,
                                                    double *vq)
{
    const double s22 = q[3], s23 = q[4], s33 = q[5];
    const double p = (s22 + s33) / 2.0;
    const double s22p = s22 - p, s33p = s33 - p;
    const double sII = sqrt((s22p * s22p + 2.0 * (s23 * s23) + s33p * s33p) / 2.0);
    const double eII = r.gammadot0 * pow(sII, r.npower - 1.0) * r.arr;
    const double e22 = eII * s22p, e23 = eII * s23, e33 = eII * s33p;
    dq[0] = e22;
    dq[1] = e23;
    dq[2] = e33;
    vq[0] = (e22 - r.ebg[3]) * 1e3;
    vq[1] = (e23 - r.ebg[4]) * 1e3;
    vq[2] = (e33 - r.ebg[5]) * 1e3;
    return sqrt((e22 * e22 + 2.0 * (e23 * e23) + e33 * e33) / 2.0);
}

__device__ __forceinline__ void volume_prepass(const double *q, const Rheology &r, double *dq,
                                               double *vq)
{
    double s11 = q[6], s12 = q[7], s13 = q[8], s22 = q[9], s23 = q[10], s33 = q[11];
    const double p = (s11 + s22 + s33) / 3.0;
    s11 = s11 - p;
    s22 = s22 - p;
    s33 = s33 - p;
    const double sII = sqrt((s11 * s11 + 2.0 * (s12 * s12) + 2.0 * (s13 * s13) + s22 * s22
                             + 2.0 * (s23 * s23) + s33 * s33) / 2.0);
    const double eII = r.gammadot0 * pow(sII, r.npower - 1.0);
    const double e[6] = {0.0 + eII * s11, 0.0 + eII * s12, 0.0 + eII * s13,
                         0.0 + eII * s22, 0.0 + eII * s23, 0.0 + eII * s33};
#pragma unroll
    for (int k = 0; k < 6; k++) {
        dq[k] = e[k];
        vq[k] = e[k] - r.ebg[k];
    }
}

// post-pass for one patch (ratestate.f90:747-771): dp[2..4] and dp[6] from the
// traction rates t, the pre-pass and its friction terms at the same state
__device__ __forceinline__ void patch_post(const double *t, const PatchPre &q,
                                           const FrictionTerms &g, double *dp)
{
    const double dtau = t[0] * q.cr + t[1] * q.sr;
    dp[5] = g.dtheta;
    dp[6] = (dtau - g.evolution) / g.direct / kLg10;
    const double correction = g.damping * dp[6] * kLg10;
    dp[2] = t[0] - correction * q.cr;
    dp[3] = t[1] - correction * q.sr;
    dp[4] = t[2];
}

__device__ __forceinline__ void patch_postpass(const double *p, const Friction &f, const double *t,
                                               double *dp)
{
    PatchPre q;
    patch_pre(p[2], p[3], p[6], q);
    patch_post(t, q, friction_terms(p[5], q.velocity, f), dp);
}

__device__ __forceinline__ int elem_state_off(const PlainDims &d, int e)
{
    if (d.ps) return e < d.np ? 5 * e : 5 * d.np + 6 * (e - d.np);
    if (d.ap) return 4 * e;
    return e < d.np ? 7 * e : 7 * d.np + 12 * (e - d.np);
}
__device__ __forceinline__ int elem_v_off(const PlainDims &d, int e)
{
    if (d.ps) return e < d.np ? e : d.np + 3 * (e - d.np);
    if (d.ap) return e < d.np ? e : d.np + 2 * (e - d.np);
    return e < d.np ? 2 * e : 2 * d.np + 6 * (e - d.np);
}
__device__ __forceinline__ int elem_row_off(const PlainDims &d, int e)
{
    if (d.ps) return e < d.np ? 2 * e : 2 * d.np + 3 * (e - d.np);
    if (d.ap) return e < d.np ? e : d.np + 2 * (e - d.np);
    return e < d.np ? 3 * e : 3 * d.np + 6 * (e - d.np);
}
// state entries and slip-rate entries of element e
__device__ __forceinline__ int elem_nstate(const PlainDims &d, int e)
{
    return d.ps ? (e < d.np ? 5 : 6) : d.ap ? 4 : (e < d.np ? 7 : 12);
}
__device__ __forceinline__ int elem_nv(const PlainDims &d, int e)
{
    return d.ps ? (e < d.np ? 1 : 3) : d.ap ? (e < d.np ? 1 : 2) : (e < d.np ? 2 : 6);
}

// a butterfly over the wavefront, partners at distance 32, 16, 8, 4, 2, 1 (the
// order of an xor shuffle; f commutes, so both partners get the same bits),
// every lane active.  The swaps and DPP moves stay in the vector unit: an xor
// shuffle is a trip through the LDS crossbar per step and half, some 60 cycles
// against 8, six steps in a row at the end of every row of K.
template <int CTRL>
__device__ __forceinline__ unsigned long long dpp64(unsigned long long b)
{
    const unsigned lo = __builtin_amdgcn_update_dpp(0u, (unsigned)b, CTRL, 0xf, 0xf, true);
    const unsigned hi = __builtin_amdgcn_update_dpp(0u, (unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
    return (unsigned long long)hi << 32 | lo;
}
template <class F>
__device__ __forceinline__ unsigned long long wave_butterfly(unsigned long long b, F f)
{
    // both halves' (rows') values in every lane: the sum of the two is each
    // lane's sum with its partner
    auto l = __builtin_amdgcn_permlane32_swap((unsigned)b, (unsigned)b, false, false);
    auto h = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
    b = f((unsigned long long)h[0] << 32 | l[0], (unsigned long long)h[1] << 32 | l[1]);
    l = __builtin_amdgcn_permlane16_swap((unsigned)b, (unsigned)b, false, false);
    h = __builtin_amdgcn_permlane16_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
    b = f((unsigned long long)h[0] << 32 | l[0], (unsigned long long)h[1] << 32 | l[1]);
    b = f(b, dpp64<0x128>(b));   // row_ror:8
    b = f(b, dpp64<0x124>(b));   // row_ror:4, equal at distance 8 by now
    b = f(b, dpp64<0x4E>(b));    // quad_perm [2,3,0,1]
    b = f(b, dpp64<0xB1>(b));    // quad_perm [1,0,3,2]
    return b;
}
__device__ __forceinline__ double wave_sum(double a)
{
    return __longlong_as_double((long long)wave_butterfly(
        dbits(a), [](unsigned long long x, unsigned long long y) {
            return dbits(__longlong_as_double((long long)x) + __longlong_as_double((long long)y));
        }));
}

// ---------------------------------------------------------------------------
// wave-level dot products of NR rows of K with v; one wavefront per element
// ---------------------------------------------------------------------------
// K is streamed once per RHS: non-temporal loads keep it from evicting v and
// the state from the caches
typedef double f64x2 __attribute__((ext_vector_type(2)));

template <int NR, bool NT = true>
__device__ __forceinline__ void wave_rows_dot(const double *__restrict__ K, int64_t row0, int n,
                                              const double *__restrict__ v, int lane, double acc[NR])
{
#pragma unroll
    for (int r = 0; r < NR; r++) acc[r] = 0.0;
    const int n2 = n >> 1;
    const double2 *v2 = reinterpret_cast<const double2 *>(v);
    const f64x2 *kr[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) kr[r] = reinterpret_cast<const f64x2 *>(K + (row0 + r) * (int64_t)n);
    int j = lane;
    for (; j + 192 < n2; j += 256) {
        double2 vv[4];
        f64x2 kk[NR][4];
#pragma unroll
        for (int u = 0; u < 4; u++) vv[u] = v2[j + 64 * u];
#pragma unroll
        for (int r = 0; r < NR; r++)
#pragma unroll
            for (int u = 0; u < 4; u++)
                kk[r][u] = NT ? __builtin_nontemporal_load(kr[r] + j + 64 * u) : kr[r][j + 64 * u];
#pragma unroll
        for (int r = 0; r < NR; r++)
#pragma unroll
            for (int u = 0; u < 4; u++) {
                acc[r] = fma(kk[r][u].x, vv[u].x, acc[r]);
                acc[r] = fma(kk[r][u].y, vv[u].y, acc[r]);
            }
    }
    for (; j < n2; j += 64) {
        const double2 vv = v2[j];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const f64x2 kk = kr[r][j];
            acc[r] = fma(kk.x, vv.x, acc[r]);
            acc[r] = fma(kk.y, vv.y, acc[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < NR; r++) {
        acc[r] = wave_sum(acc[r]);
    }
}

// the same with the packed split-bf16 K: entry = (hi + lo) * rs[row], each
// pair decoded exactly to binary64 and accumulated in binary64 (the GEMV is
// bound by HBM at 4 bytes per entry, so the wider arithmetic is free)
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ double split_entry(uint32_t w)
{
    return (double)__uint_as_float(w & 0xFFFF0000u) + (double)__uint_as_float(w << 16);
}

template <int NR>
__device__ __forceinline__ void wave_rows_dot_split(const uint32_t *__restrict__ Kp,
                                                    const double *__restrict__ rs, int64_t row0,
                                                    int n, const double *__restrict__ v, int lane,
                                                    double acc[NR])
{
#pragma unroll
    for (int r = 0; r < NR; r++) acc[r] = 0.0;
    const int n2 = n >> 1;
    const double2 *v2 = reinterpret_cast<const double2 *>(v);
    const u32x2 *kr[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) kr[r] = reinterpret_cast<const u32x2 *>(Kp + (row0 + r) * (int64_t)n);
    int j = lane;
    for (; j + 192 < n2; j += 256) {
        double2 vv[4];
        u32x2 kk[NR][4];
#pragma unroll
        for (int u = 0; u < 4; u++) vv[u] = v2[j + 64 * u];
#pragma unroll
        for (int r = 0; r < NR; r++)
#pragma unroll
            for (int u = 0; u < 4; u++) kk[r][u] = __builtin_nontemporal_load(kr[r] + j + 64 * u);
#pragma unroll
        for (int r = 0; r < NR; r++)
#pragma unroll
            for (int u = 0; u < 4; u++) {
                acc[r] = fma(split_entry(kk[r][u].x), vv[u].x, acc[r]);
                acc[r] = fma(split_entry(kk[r][u].y), vv[u].y, acc[r]);
            }
    }
    for (; j < n2; j += 64) {
        const double2 vv = v2[j];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const u32x2 kk = kr[r][j];
            acc[r] = fma(split_entry(kk.x), vv.x, acc[r]);
            acc[r] = fma(split_entry(kk.y), vv.y, acc[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < NR; r++) {
        acc[r] = wave_sum(acc[r]) * rs[row0 + r];
    }
}

// intermediate state of stage s (ode45.f90:137-180), BLAS-1 order kept:
// yrkck = B_s1*dydt; yrkck += B_sj*AKj; ytmp = yin + h*yrkck
__device__ __forceinline__ double stage_value(int stage, double h, double y0, double k1, double k2,
                                              double k3, double k4, double k5)
{
    double yr;
    switch (stage) {
    case 2:
        return y0 + (h * B21) * k1;
    case 3:
        yr = B31 * k1;
        yr = yr + B32 * k2;
        return y0 + h * yr;
    case 4:
        yr = B41 * k1;
        yr = yr + B42 * k2;
        yr = yr + B43 * k3;
        return y0 + h * yr;
    case 5:
        yr = B51 * k1;
        yr = yr + B52 * k2;
        yr = yr + B53 * k3;
        yr = yr + B54 * k4;
        return y0 + h * yr;
    default:
        yr = B61 * k1;
        yr = yr + B62 * k2;
        yr = yr + B63 * k3;
        yr = yr + B64 * k4;
        yr = yr + B65 * k5;
        return y0 + h * yr;
    }
}

// max of the bit patterns of a wavefront's non-negative values (NaN bits
// order above +inf), every lane active
__device__ __forceinline__ unsigned long long wave_max_bits(unsigned long long b)
{
    return wave_butterfly(b, [](unsigned long long x, unsigned long long y) {
        return x > y ? x : y;
    });
}

// step control of RKQSm (ode45.f90:70-105) and the time update / exit test of
// the main loop (ratestate.f90:317-326).  RKQSm is called with t0 = 0
// (ratestate.f90:317), so its underflow test is h == 0.  log: write the step
// log (one of several blocks that take the same decision does).
__device__ __forceinline__ void controller_step(const RkBuffers &b, Control *ctl, bool log)
{
    if (ctl->done) return;
    const double SAFETY = 0.7, PGROW = -0.2, PSHRNK = -0.15, ERRCON = 1.89e-4;
    ctl->attempts += 1;
    ctl->rhs_evals += ctl->need_rhs ? 6 : 5;
    const double raw = __longlong_as_double((long long)ctl->errmax_bits);
    if (!(raw == raw) || raw > 1.7976931348623157e308) {
        ctl->error = 2;
        ctl->done = 1;
        ctl->accepted = 0;
        return;
    }
    const double errmax = raw / ctl->epsilon;
    double h = ctl->h;
    if (errmax > 1.0) {
        h = h * SAFETY * pow(errmax, PSHRNK);
        ctl->h = h;
        ctl->need_rhs = 0;
        ctl->accepted = 0;
        ctl->step_rejects += 1;
        if (0.0 + h == 0.0) {
            ctl->error = 1;
            ctl->done = 1;
        }
        return;
    }
    double hnext = errmax > ERRCON ? SAFETY * h * pow(errmax, PGROW) : 10.0 * h;
    if (hnext > ctl->max_step) hnext = ctl->max_step;
    ctl->hdid = h;
    ctl->hnext = hnext;
    ctl->time = ctl->time + h;
    ctl->steps += 1;
    if (ctl->log_count < ctl->log_cap) {
        if (log) {
            b.tlog[ctl->log_count] = ctl->time;
            b.dtlog[ctl->log_count] = h;
            b.vlog[ctl->log_count] = ctl->vmax;
            if (b.elog) {
                b.elog[ctl->log_count] = errmax;
                b.rlog[ctl->log_count] = (double)ctl->step_rejects;
            }
            if (b.emlog) b.emlog[ctl->log_count] = ctl->emax;
        }
        ctl->log_count += 1;
    }
    ctl->step_rejects = 0;
    ctl->last_vmax = ctl->vmax;
    ctl->vmax = 0.0;
    ctl->emax = 0.0;
    ctl->accepted = 1;
    ctl->obs_pending = 1;
    ctl->need_rhs = 1;
    ctl->h = hnext;
    if (ctl->interval <= ctl->time || ctl->steps >= ctl->max_steps) ctl->done = 1;
}

}  // namespace ucy
