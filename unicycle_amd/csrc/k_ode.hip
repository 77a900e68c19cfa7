// k_ode.hip -- rate-and-state right-hand side, the traction matvec and the
// Cash-Karp RK45 attempt, device-resident for graph capture.
//
// Reference: jdpmoore/unicycle fortran/3d/src
//   ratestate.f90:624-778   odefun (pre-pass, DGEMV, post-pass)
//   viscouscycles.f90:933-1080  volume branch of odefun
//   ode45.f90:51-202        RKQSm / RKCKm
//   ratestate.f90:307-328   main loop (yscal, time, exit test)
//
// Every kernel of the attempt reads the Control block first and returns when
// the run is done, so a captured attempt can be replayed any number of times.
#include <hip/hip_runtime.h>
#include "../../include/ucy.h"
#include "ode_dev.h"

namespace ucy {

__global__ void __launch_bounds__(256) matvec_split_kernel(const uint32_t *__restrict__ Kp,
                                                           const double *__restrict__ rs, int m,
                                                           int n, const double *__restrict__ v,
                                                           double *__restrict__ t)
{
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= m) return;
    double acc[1];
    wave_rows_dot_split<1>(Kp, rs, row, n, v, lane, acc);
    if (lane == 0) t[row] = acc[0];
}

void launch_matvec_split(hipStream_t st, const uint32_t *Kp, const double *rs, int m, int n,
                         const double *v, double *t)
{
    hipLaunchKernelGGL(matvec_split_kernel, dim3((m + 3) / 4), dim3(256), 0, st, Kp, rs, m, n, v, t);
}

// generic t = K v (m rows), one wavefront per row
__global__ void __launch_bounds__(256) matvec_kernel(const double *__restrict__ K, int m, int n,
                                                     const double *__restrict__ v,
                                                     double *__restrict__ t)
{
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= m) return;
    double acc[1];
    wave_rows_dot<1>(K, row, n, v, lane, acc);
    if (lane == 0) t[row] = acc[0];
}

void launch_matvec(hipStream_t st, const double *K, int m, int n, const double *v, double *t)
{
    hipLaunchKernelGGL(matvec_kernel, dim3((m + 3) / 4), dim3(256), 0, st, K, m, n, v, t);
}

// ---------------------------------------------------------------------------
// standalone odefun pieces (ucy_odefun)
// ---------------------------------------------------------------------------
__global__ void prepass_kernel(PlainDims d, const Friction *__restrict__ fr,
                               const Rheology *__restrict__ rh, const double *__restrict__ y,
                               double *__restrict__ dydt, double *__restrict__ v, double *vmax)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= d.np + d.nv) return;
    const int so = elem_state_off(d, e), vo = elem_v_off(d, e);
    if (d.ps && e >= d.np) {
        dydt[so + 3] = dydt[so + 4] = dydt[so + 5] = 0.0;
        ps_volume_prepass(y + so, rh[e - d.np], dydt + so, v + vo);
    } else if (d.ps) {
        for (int k = 1; k < 5; k++) dydt[so + k] = 0.0;
        const double vel = ps_prepass(y + so, fr[e], dydt + so, v + vo);
        if (vmax) atomicMax(reinterpret_cast<unsigned long long *>(vmax), dbits(vel));
    } else if (d.ap && e >= d.np) {
        dydt[so + 2] = dydt[so + 3] = 0.0;
        ap_volume_prepass(y + so, rh[e - d.np], dydt + so, v + vo);
    } else if (d.ap) {
        for (int k = 1; k < 4; k++) dydt[so + k] = 0.0;
        const double vel = ap_prepass(y + so, fr[e], dydt + so, v + vo);
        if (vmax) atomicMax(reinterpret_cast<unsigned long long *>(vmax), dbits(vel));
    } else if (e < d.np) {
        for (int k = 2; k < 7; k++) dydt[so + k] = 0.0;
        const double vel = patch_prepass(y + so, fr[e], dydt + so, v + vo);
        if (vmax) atomicMax(reinterpret_cast<unsigned long long *>(vmax), dbits(vel));
    } else {
        volume_prepass(y + so, rh[e - d.np], dydt + so, v + vo);
    }
}

void launch_prepass(hipStream_t st, const PlainDims &d, const Friction *fr, const Rheology *rh,
                    const double *y, double *dydt, double *v, double *vmax_out)
{
    const int ne = d.np + d.nv;
    hipLaunchKernelGGL(prepass_kernel, dim3((ne + 255) / 256), dim3(256), 0, st, d, fr, rh, y,
                       dydt, v, vmax_out);
}

// matvec modes of the RHS: binary64 K v; binary64 K v kept as t0 (step start
// of the mixed path); split K v kept as t0 (step start of the split path);
// t0 + split K dv (stages of both reduced paths, v holding v - v0)
enum { DOT_F64 = 0, DOT_F64_T0 = 1, DOT_SPLIT_T0 = 2, DOT_SPLIT_INC = 3 };

template <int NR, int MODE>
__device__ __forceinline__ void elem_rows(const KOperand &K, int64_t ro, int n,
                                          const double *__restrict__ v, double *t0, int lane,
                                          double acc[NR])
{
    if (MODE <= DOT_F64_T0) wave_rows_dot<NR>(K.K, ro, n, v, lane, acc);
    else wave_rows_dot_split<NR>(K.Kp, K.rs, ro, n, v, lane, acc);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < NR; r++) {
            if (MODE == DOT_F64_T0 || MODE == DOT_SPLIT_T0) t0[ro + r] = acc[r];
            if (MODE == DOT_SPLIT_INC) acc[r] += t0[ro + r];
        }
    }
}

// K v for the rows of element e, then that element's post-pass.  One
// wavefront per element; 4 elements per 256-thread block.
template <int MODE>
__device__ __forceinline__ void elem_gemv_post(const PlainDims &d, const KOperand &K,
                                               const Friction *__restrict__ fr,
                                               const double *__restrict__ y,
                                               const double *__restrict__ v,
                                               double *__restrict__ dydt, double *t_out, int e,
                                               int lane, const double *yscal_h, double *yscal,
                                               double *t0)
{
    const int so = elem_state_off(d, e);
    const int64_t ro = elem_row_off(d, e);
    if (d.ps && e >= d.np) {
        double acc[3];
        elem_rows<3, MODE>(K, ro, d.n, v, t0, lane, acc);
        if (lane == 0) {
            for (int k = 0; k < 3; k++) {
                if (t_out) t_out[ro + k] = acc[k];
                dydt[so + 3 + k] = acc[k];  // viscouscycles.f90 (2-D plane strain):1048-1053
            }
            if (yscal) {
                const double h = *yscal_h;
                for (int k = 0; k < 6; k++)
                    yscal[so + k] = fabs(y[so + k]) + fabs(h * dydt[so + k]) + 1.0e-30;
            }
        }
    } else if (d.ps) {
        double acc[2];
        elem_rows<2, MODE>(K, ro, d.n, v, t0, lane, acc);
        if (lane == 0) {
            if (t_out) { t_out[ro] = acc[0]; t_out[ro + 1] = acc[1]; }
            ps_postpass(y + so, fr[e], acc, dydt + so);
            if (yscal) {
                const double h = *yscal_h;
                for (int k = 0; k < 5; k++)
                    yscal[so + k] = fabs(y[so + k]) + fabs(h * dydt[so + k]) + 1.0e-30;
            }
        }
    } else if (d.ap && e >= d.np) {
        double acc[2];
        elem_rows<2, MODE>(K, ro, d.n, v, t0, lane, acc);
        if (lane == 0) {
            if (t_out) { t_out[ro] = acc[0]; t_out[ro + 1] = acc[1]; }
            dydt[so + 2] = acc[0];  // viscouscycles.f90 (2-D antiplane):939-942
            dydt[so + 3] = acc[1];
            if (yscal) {
                const double h = *yscal_h;
                for (int k = 0; k < 4; k++)
                    yscal[so + k] = fabs(y[so + k]) + fabs(h * dydt[so + k]) + 1.0e-30;
            }
        }
    } else if (d.ap) {
        double acc[1];
        elem_rows<1, MODE>(K, ro, d.n, v, t0, lane, acc);
        if (lane == 0) {
            if (t_out) t_out[ro] = acc[0];
            ap_postpass(y + so, fr[e], acc[0], dydt + so);
            if (yscal) {
                const double h = *yscal_h;
                for (int k = 0; k < 4; k++)
                    yscal[so + k] = fabs(y[so + k]) + fabs(h * dydt[so + k]) + 1.0e-30;
            }
        }
    } else if (e < d.np) {
        double acc[3];
        elem_rows<3, MODE>(K, ro, d.n, v, t0, lane, acc);
        if (lane == 0) {
            if (t_out) { t_out[ro] = acc[0]; t_out[ro + 1] = acc[1]; t_out[ro + 2] = acc[2]; }
            patch_postpass(y + so, fr[e], acc, dydt + so);
            if (yscal) {
                const double h = *yscal_h;
                for (int k = 0; k < 7; k++)
                    yscal[so + k] = fabs(y[so + k]) + fabs(h * dydt[so + k]) + 1.0e-30;
            }
        }
    } else {
        double acc[6];
        elem_rows<6, MODE>(K, ro, d.n, v, t0, lane, acc);
        if (lane == 0) {
            for (int k = 0; k < 6; k++) {
                if (t_out) t_out[ro + k] = acc[k];
                dydt[so + 6 + k] = acc[k];  // viscouscycles.f90:1075-1080
            }
            if (yscal) {
                const double h = *yscal_h;
                for (int k = 0; k < 12; k++)
                    yscal[so + k] = fabs(y[so + k]) + fabs(h * dydt[so + k]) + 1.0e-30;
            }
        }
    }
}

__global__ void __launch_bounds__(256) gemv_post_kernel(PlainDims d, const double *__restrict__ K,
                                                        const Friction *__restrict__ fr,
                                                        const double *__restrict__ y,
                                                        const double *__restrict__ v,
                                                        double *__restrict__ dydt, double *t_out)
{
    const int lane = threadIdx.x & 63;
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= d.np + d.nv) return;
    const KOperand k{K, nullptr, nullptr, 0};
    elem_gemv_post<DOT_F64>(d, k, fr, y, v, dydt, t_out, e, lane, nullptr, nullptr, nullptr);
}

// a stage RHS of the reduced paths alone (t0 + split K dv, post-pass), for timing
__global__ void __launch_bounds__(256) gemv_post_inc_kernel(PlainDims d, KOperand K,
                                                            const Friction *__restrict__ fr,
                                                            const double *__restrict__ y,
                                                            const double *__restrict__ v,
                                                            double *__restrict__ dydt, double *t0)
{
    const int lane = threadIdx.x & 63;
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= d.np + d.nv) return;
    elem_gemv_post<DOT_SPLIT_INC>(d, K, fr, y, v, dydt, nullptr, e, lane, nullptr, nullptr, t0);
}

void launch_gemv_post_inc(hipStream_t st, const PlainDims &d, const KOperand &K, const Friction *fr,
                          const double *y, const double *v, double *dydt, double *t0)
{
    const int ne = d.np + d.nv;
    hipLaunchKernelGGL(gemv_post_inc_kernel, dim3((ne + 3) / 4), dim3(256), 0, st, d, K, fr, y, v,
                       dydt, t0);
}

void launch_gemv_post(hipStream_t st, const PlainDims &d, const double *K, const Friction *fr,
                      const double *y, const double *v, double *dydt, double *t_out)
{
    const int ne = d.np + d.nv;
    hipLaunchKernelGGL(gemv_post_kernel, dim3((ne + 3) / 4), dim3(256), 0, st, d, K, fr, y, v,
                       dydt, t_out);
}

// ---------------------------------------------------------------------------
// one RK45 attempt as 8 graph-capturable kernels:
//   start        commit of the previous accepted step (y = ycand,
//                ode45.f90:103) and the step-start pre-pass at y
//                (ratestate.f90:309, odefun :667-707), thread per element
//   rhs_stage 1  K v + post-pass at y (dydt, yscal of ratestate.f90:315),
//                then the input of stage 2 and its pre-pass, wave per element
//   rhs_stage s  K v + post-pass of stage s (2..5), then stage s+1's input
//   rhs_finish   K v + post-pass of stage 6, the 5th-order solution and the
//                embedded error (ode45.f90:185-200), max |yerr/yscal| (:75)
//   controller   RKQSm's decision and the main loop's time update
// The slip-rate vector is double-buffered (odd stages read v, even stages
// v2) because a wave writes the next stage's entries of its element while
// other waves still read the current ones.  A run ends with one commit.
// ---------------------------------------------------------------------------
__global__ void start_kernel(PlainDims d, const Friction *__restrict__ fr,
                             const Rheology *__restrict__ rh, RkBuffers b, Control *ctl)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e == 0) ctl->obs_pending = 0;
    const bool live = e < d.np + d.nv;
    // the step-start vMax and eMax, reduced over the wavefront and then
    // folded in with one atomic per wave (one per element would serialise
    // on the two addresses)
    double vel = 0.0, en = 0.0;
    if (live) {
        const int so = elem_state_off(d, e), vo = elem_v_off(d, e);
        if (ctl->accepted) {
            const int ns = elem_nstate(d, e);
            for (int k = 0; k < ns; k++) b.y[so + k] = b.ycand[so + k];
        }
        // ctl->vmax was cleared by the controller that accepted the previous step
        if (!ctl->done && ctl->need_rhs) {
            if (d.ps && e >= d.np) {
                // eMax of the step-start odefun (viscouscycles.f90 (2-D plane strain):962)
                en = ps_volume_prepass(b.y + so, rh[e - d.np], b.dydt + so, b.v + vo);
            } else if (d.ps) {
                vel = ps_prepass(b.y + so, fr[e], b.dydt + so, b.v + vo);
            } else if (d.ap && e >= d.np) {
                // eMax of the step-start odefun (viscouscycles.f90 (2-D antiplane):869)
                en = ap_volume_prepass(b.y + so, rh[e - d.np], b.dydt + so, b.v + vo);
            } else if (d.ap) {
                vel = ap_prepass(b.y + so, fr[e], b.dydt + so, b.v + vo);
            } else if (e < d.np) {
                // vMax of the step-start odefun (ratestate.f90:693), as exported every step
                vel = patch_prepass(b.y + so, fr[e], b.dydt + so, b.v + vo);
            } else {
                volume_prepass(b.y + so, rh[e - d.np], b.dydt + so, b.v + vo);
                // eMax of the step-start odefun (viscouscycles.f90:986), printed by export
                const double *r = b.dydt + so;
                en = sqrt((r[0] * r[0] + 2.0 * (r[1] * r[1]) + 2.0 * (r[2] * r[2]) +
                           r[3] * r[3] + 2.0 * (r[4] * r[4]) + r[5] * r[5]) / 2.0);
            }
            if (b.v0) {
                const int nvk = elem_nv(d, e);
                for (int k = 0; k < nvk; k++) b.v0[vo + k] = b.v[vo + k];
            }
        }
    }
    const unsigned long long bv = wave_max_bits(dbits(vel)), be = wave_max_bits(dbits(en));
    if ((threadIdx.x & 63) == 0) {
        if (bv) atomicMax(reinterpret_cast<unsigned long long *>(&ctl->vmax), bv);
        if (be) atomicMax(reinterpret_cast<unsigned long long *>(&ctl->emax), be);
    }
}

void launch_start(hipStream_t st, const PlainDims &d, const Friction *fr, const Rheology *rh,
                  const RkBuffers &b, Control *ctl)
{
    const int ne = d.np + d.nv;
    hipLaunchKernelGGL(start_kernel, dim3((ne + 255) / 256), dim3(256), 0, st, d, fr, rh, b, ctl);
}

// the N state entries from so on of the input of stage `stage`.  All loads before
// the stores, which may alias them: entry by entry each waited for the last one's
// memory (a stage of 945 patches 12.9 us at best, so 11.3).
template <int N>
__device__ __forceinline__ void stage_entries(const RkBuffers &b, double h, int so, int stage)
{
    double v[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int i = so + k;
        v[k] = stage_value(stage, h, b.y[i], b.dydt[i], b.ak[2][i], b.ak[3][i], b.ak[4][i],
                           b.ak[5][i]);
    }
#pragma unroll
    for (int k = 0; k < N; k++) b.ytmp[so + k] = v[k];
}

// the input of stage `stage` (2..6) for element e and its pre-pass; the
// slip-rate entries go to vout (less v0 in the reduced paths)
__device__ __forceinline__ void stage_elem(const PlainDims &d, const Friction *__restrict__ fr,
                                           const Rheology *__restrict__ rh, const RkBuffers &b,
                                           double h, int e, int stage, double *vout)
{
    const int so = elem_state_off(d, e), vo = elem_v_off(d, e);
    switch (elem_nstate(d, e)) {
    case 4: stage_entries<4>(b, h, so, stage); break;
    case 5: stage_entries<5>(b, h, so, stage); break;
    case 6: stage_entries<6>(b, h, so, stage); break;
    case 7: stage_entries<7>(b, h, so, stage); break;
    default: stage_entries<12>(b, h, so, stage); break;
    }
    double *out = b.ak[stage];
    if (d.ps && e >= d.np) ps_volume_prepass(b.ytmp + so, rh[e - d.np], out + so, vout + vo);
    else if (d.ps) ps_prepass(b.ytmp + so, fr[e], out + so, vout + vo);
    else if (d.ap && e >= d.np) ap_volume_prepass(b.ytmp + so, rh[e - d.np], out + so, vout + vo);
    else if (d.ap) ap_prepass(b.ytmp + so, fr[e], out + so, vout + vo);
    else if (e < d.np) patch_prepass(b.ytmp + so, fr[e], out + so, vout + vo);
    else volume_prepass(b.ytmp + so, rh[e - d.np], out + so, vout + vo);
    if (b.v0) {
        const int nvk = elem_nv(d, e);
        for (int k = 0; k < nvk; k++) vout[vo + k] -= b.v0[vo + k];
    }
}

template <int MODE>
__global__ void __launch_bounds__(256) rhs_stage_kernel(PlainDims d, KOperand K,
                                                        const Friction *__restrict__ fr,
                                                        const Rheology *__restrict__ rh,
                                                        RkBuffers b, Control *ctl, int stage)
{
    if (ctl->done) return;
    const int lane = threadIdx.x & 63;
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= d.np + d.nv) return;
    const double *vin = (stage & 1) ? b.v : b.v2;
    double *vout = (stage & 1) ? b.v2 : b.v;
    if (stage == 1) {
        // a retried attempt keeps the step-start derivative (the reference's
        // RKQSm loop reuses dydt)
        if (ctl->need_rhs)
            elem_gemv_post<MODE>(d, K, fr, b.y, vin, b.dydt, nullptr, e, lane, &ctl->h, b.yscal,
                                 b.t0);
        if (lane == 0 && e == 0) ctl->errmax_bits = 0ull;
    } else {
        elem_gemv_post<MODE>(d, K, fr, b.ytmp, vin, b.ak[stage], nullptr, e, lane, nullptr,
                             nullptr, b.t0);
    }
    if (lane == 0) stage_elem(d, fr, rh, b, ctl->h, e, stage + 1, vout);
}

template <int MODE>
__global__ void __launch_bounds__(256) rhs_finish_kernel(PlainDims d, KOperand K,
                                                         const Friction *__restrict__ fr,
                                                         RkBuffers b, Control *ctl)
{
    if (ctl->done) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int e = blockIdx.x * 4 + w;
    const bool live = e < d.np + d.nv;
    if (live)
        elem_gemv_post<MODE>(d, K, fr, b.ytmp, b.v2, b.ak[6], nullptr, e, lane, nullptr, nullptr,
                             b.t0);
    double emax = 0.0;
    if (live && lane == 0) {
        const double h = ctl->h;
        const int so = elem_state_off(d, e), ns = elem_nstate(d, e);
        for (int k = 0; k < ns; k++) {
            const int i = so + k;
            const double k1 = b.dydt[i], k3 = b.ak[3][i], k4 = b.ak[4][i], k5 = b.ak[5][i],
                         k6 = b.ak[6][i];
            double yr = C1 * k1;
            yr = yr + C3 * k3;
            yr = yr + C4 * k4;
            yr = yr + C6 * k6;
            b.ycand[i] = b.y[i] + h * yr;
            double er = DC1 * k1;
            er = er + DC3 * k3;
            er = er + DC4 * k4;
            er = er + DC5 * k5;
            er = er + DC6 * k6;
            er = h * er;
            const double r = fabs(er / b.yscal[i]);
            // non-finite ratios propagate as NaN bits, which order above +inf
            emax = (r > emax || r != r) ? r : emax;
        }
    }
    __shared__ unsigned long long red[4];
    if (lane == 0) red[w] = dbits(emax);
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long m = red[0];
        for (int k = 1; k < 4; k++) m = red[k] > m ? red[k] : m;
        atomicMax(&ctl->errmax_bits, m);
    }
}

void launch_rhs_stage(hipStream_t st, const PlainDims &d, const KOperand &K, const Friction *fr,
                      const Rheology *rh, const RkBuffers &b, Control *ctl, int stage)
{
    const dim3 g((d.np + d.nv + 3) / 4), t(256);
    if (stage == 1 && K.prec == UCY_PREC_SPLIT_BF16)
        hipLaunchKernelGGL(rhs_stage_kernel<DOT_SPLIT_T0>, g, t, 0, st, d, K, fr, rh, b, ctl, stage);
    else if (stage == 1 && K.prec == UCY_PREC_MIXED)
        hipLaunchKernelGGL(rhs_stage_kernel<DOT_F64_T0>, g, t, 0, st, d, K, fr, rh, b, ctl, stage);
    else if (K.prec == UCY_PREC_F64)
        hipLaunchKernelGGL(rhs_stage_kernel<DOT_F64>, g, t, 0, st, d, K, fr, rh, b, ctl, stage);
    else
        hipLaunchKernelGGL(rhs_stage_kernel<DOT_SPLIT_INC>, g, t, 0, st, d, K, fr, rh, b, ctl, stage);
}

void launch_rhs_finish(hipStream_t st, const PlainDims &d, const KOperand &K, const Friction *fr,
                       const RkBuffers &b, Control *ctl)
{
    const dim3 g((d.np + d.nv + 3) / 4), t(256);
    if (K.prec == UCY_PREC_F64)
        hipLaunchKernelGGL(rhs_finish_kernel<DOT_F64>, g, t, 0, st, d, K, fr, b, ctl);
    else
        hipLaunchKernelGGL(rhs_finish_kernel<DOT_SPLIT_INC>, g, t, 0, st, d, K, fr, b, ctl);
}

__global__ void controller_kernel(RkBuffers b, Control *ctl)
{
    controller_step(b, ctl, true);
}

// the step-start state and derivative of the observed entries after an
// accepted step, at the step's log row (the controller has advanced
// log_count; y is committed at the next attempt's start)
__global__ void obs_log_kernel(RkBuffers b, Control *ctl)
{
    // only in the attempt that accepted the step: replays issued after the
    // run ended keep `accepted` but have committed y already
    if (!ctl->obs_pending) return;
    const int64_t row = ctl->log_count - 1;
    if (row < 0 || row >= ctl->log_cap) return;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < b.n_obs;
         j += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = b.obs_idx[j];
        b.obs_y[row * b.n_obs + j] = b.y[i];
        b.obs_dydt[row * b.n_obs + j] = b.dydt[i];
    }
}

// exportPoints (ratestate.f90:414-486, viscouscycles.f90:523-625): d = O u,
// the reference's DGEMV("T") on O(n, 3 npts), with u gathered from the state
// (strike and dip slip of each patch, e11..e33 of each volume).  One block per
// row of O, four waves across its columns.  df and dl split the same products
// as buildO splits O into Of and Ol (greens.f90:388-445): fault columns and
// the volumes' third component go to df, the volumes' first two to dl.
__global__ void __launch_bounds__(256)
disp_gemv_kernel(const double *__restrict__ O, int64_t rows, int64_t n, int np, int model,
                 const double *__restrict__ y, double *d, double *df, double *dl,
                 const Control *ctl)
{
    int64_t off = 0;
    if (ctl) {
        if (!ctl->obs_pending) return;
        const int64_t row = ctl->log_count - 1;
        if (row < 0 || row >= ctl->log_cap) return;
        off = row * rows;
    }
    const int64_t r = blockIdx.x;
    // model 0: the 3-D model (3 rows per point), 1: antiplane (1 row),
    // 2: plane strain (2 rows: east, down; one dip slip per patch)
    const bool ap = model == 1, ps = model == 2;
    const bool vertical = model == 0 && (r % 3) == 2;
    const double *Or = O + r * n;
    // the 2-D antiplane model: one slip per patch (state entry 0 of 4), then
    // e12, e13 per volume (entries 0, 1 of 4); one displacement component per point
    const int64_t nf = (ap || ps) ? np : 2 * (int64_t)np, vbase = 7 * (int64_t)np;
    double a = 0.0, af = 0.0, al = 0.0;
    for (int64_t j = threadIdx.x; j < n; j += blockDim.x) {
        double u;
        if (ps) {
            // plane strain: one dip slip per patch (entry 0 of 5), then e22,
            // e23, e33 per volume (entries 0..2 of 6); viscouscycles.f90
            // (2-D plane strain):546-566
            u = j < np ? y[5 * j] : y[5 * (int64_t)np + 6 * ((j - np) / 3) + (j - np) % 3];
        } else if (ap) {
            u = j < np ? y[4 * j] : y[4 * np + 4 * ((j - np) >> 1) + ((j - np) & 1)];
        } else if (j < nf) {
            u = y[7 * (j >> 1) + (j & 1)];
        } else {
            const int64_t q = (j - nf) / 6;
            u = y[vbase + 12 * q + (j - nf - 6 * q)];
        }
        const double p = Or[j] * u;
        a += p;
        if (j < nf || vertical) af += p;
        else al += p;
    }
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        af += __shfl_xor(af, o, 64);
        al += __shfl_xor(al, o, 64);
    }
    __shared__ double part[3][4];
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        part[0][w] = a;
        part[1][w] = af;
        part[2][w] = al;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nw = blockDim.x >> 6;
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        for (int k = 0; k < nw; k++) {
            s0 += part[0][k];
            s1 += part[1][k];
            s2 += part[2][k];
        }
        d[off + r] = s0;
        if (df) df[off + r] = s1;
        if (dl) dl[off + r] = s2;
    }
}

void launch_disp_gemv(hipStream_t st, const double *O, int64_t rows, int64_t n, int np, int model,
                      const double *y, double *d, double *df, double *dl, const Control *ctl)
{
    if (rows <= 0) return;
    hipLaunchKernelGGL(disp_gemv_kernel, dim3((unsigned)rows), dim3(256), 0, st, O, rows, n, np,
                       model, y, d, df, dl, ctl);
}

void launch_obs_log(hipStream_t st, const RkBuffers &b, Control *ctl)
{
    const int64_t blocks = b.n_obs < 256 * 64 ? (b.n_obs + 255) / 256 : 64;
    hipLaunchKernelGGL(obs_log_kernel, dim3((unsigned)blocks), dim3(256), 0, st, b, ctl);
}

// y <- ycand after an accepted attempt (ode45.f90:103)
__global__ void commit_kernel(int dim, RkBuffers b, Control *ctl)
{
    if (!ctl->accepted) return;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += gridDim.x * blockDim.x)
        b.y[i] = b.ycand[i];
}

void launch_controller(hipStream_t st, const RkBuffers &b, Control *ctl)
{
    hipLaunchKernelGGL(controller_kernel, dim3(1), dim3(1), 0, st, b, ctl);
}

void launch_commit(hipStream_t st, int dim, const RkBuffers &b, Control *ctl)
{
    int blocks = (dim + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(commit_kernel, dim3(blocks), dim3(256), 0, st, dim, b, ctl);
}

// ---------------------------------------------------------------------------
// One Cash-Karp evaluation for a host's own step loop (ucy_rkck, ucy_rkqs): the
// caller's h and k1, binary64 K whatever the context integrates with.  A launch
// per stage: as in the captured attempt a matvec's wave makes its element's next
// stage input, so that a step has 6 launches where combination, pre-pass and matvec
// apart made 16.  945 patches take 14.2 us per stage, 3 TB/s of their K of 43 MB from
// the last-level cache: 945 waves for 1024 SIMDs, each with an element's three rows
// and then its chain, do not have enough loads in flight for more.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(64)
rkck_begin_kernel(PlainDims d, const Friction *__restrict__ fr, const Rheology *__restrict__ rh,
                  RkBuffers b, double h)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < d.np + d.nv) stage_elem(d, fr, rh, b, h, e, 2, b.v2);
}

// N entries of the fifth-order solution and of the error (ode45.f90:190-200)
template <int N>
__device__ __forceinline__ void step_entries(const RkBuffers &b, double h, int so)
{
    double y[N], err[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int i = so + k;
        const double k1 = b.dydt[i], k3 = b.ak[3][i], k4 = b.ak[4][i], k5 = b.ak[5][i],
                     k6 = b.ak[6][i];
        double yr = C1 * k1;
        yr = yr + C3 * k3;
        yr = yr + C4 * k4;
        yr = yr + C6 * k6;
        y[k] = b.y[i] + h * yr;
        double er = DC1 * k1;
        er = er + DC3 * k3;
        er = er + DC4 * k4;
        er = er + DC5 * k5;
        er = er + DC6 * k6;
        err[k] = h * er;
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
        b.ycand[so + k] = y[k];
        b.yerr[so + k] = err[k];
    }
}

// stage 2..5: k_stage, then the input of the next stage; 6: k_6, then the
// fifth-order solution and the error
__global__ void __launch_bounds__(256)
rkck_stage_kernel(PlainDims d, KOperand K, const Friction *__restrict__ fr,
                  const Rheology *__restrict__ rh, RkBuffers b, double h, int stage)
{
    const int lane = threadIdx.x & 63;
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= d.np + d.nv) return;
    const double *vin = (stage & 1) ? b.v : b.v2;
    double *vout = (stage & 1) ? b.v2 : b.v;
    elem_gemv_post<DOT_F64>(d, K, fr, b.ytmp, vin, b.ak[stage], nullptr, e, lane, nullptr, nullptr,
                            nullptr);
    if (lane != 0) return;
    if (stage < 6) {
        stage_elem(d, fr, rh, b, h, e, stage + 1, vout);
        return;
    }
    const int so = elem_state_off(d, e);
    switch (elem_nstate(d, e)) {
    case 4: step_entries<4>(b, h, so); break;
    case 5: step_entries<5>(b, h, so); break;
    case 6: step_entries<6>(b, h, so); break;
    case 7: step_entries<7>(b, h, so); break;
    default: step_entries<12>(b, h, so); break;
    }
}

void launch_rkck(hipStream_t st, const PlainDims &d, const double *K, const Friction *fr,
                 const Rheology *rh, RkBuffers b, double h)
{
    const int ne = d.np + d.nv;
    b.v0 = nullptr;   // slip rates themselves, not their increments
    const KOperand k{K, nullptr, nullptr, 0};
    hipLaunchKernelGGL(rkck_begin_kernel, dim3((ne + 63) / 64), dim3(64), 0, st, d, fr, rh, b, h);
    for (int s = 2; s <= 6; s++)
        hipLaunchKernelGGL(rkck_stage_kernel, dim3((ne + 3) / 4), dim3(256), 0, st, d, k, fr, rh, b,
                           h, s);
}

}  // namespace ucy
