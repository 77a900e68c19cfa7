// k_resident.hip -- the single-instance integrator as one resident kernel.
//
// Reference: jdpmoore/unicycle fortran/3d/src/ratestate.f90:307-328 (main
// loop), 624-778 (odefun), ode45.f90:51-202 (RKQSm, RKCKm).
//
// The captured attempt (k_ode.hip) runs an RK45 attempt as 8 kernels.  For a
// small fault their launches are the whole cost: 40 us per attempt for one
// element, 70 us for 390 triangles whose K of 7 MB takes 6 us to read six
// times.  Here the blocks stay on the chip for many attempts.  Each block owns
// a range of elements and their rows of K, which live in its LDS; rows that do
// not fit are read through the caches or streamed.  Per stage a block forms its
// elements' slip rates, exchanges them with the other blocks and multiplies its
// rows.  Every block takes the step control's decision by itself, from the same
// exchanged maxima.
//
// us per attempt, captured and resident: 1 segment 40 -> 8.6; 241 segments
// 51 -> 18; 900 segments 58 -> 22; 20 patches 57 -> 16; 390 triangles 70 -> 24;
// 1024 patches 87 -> 37; 2048 patches (K of 201 MB) 228 -> 188; 4096 patches
// 770 -> 755, mixed 555 -> 484.  Small faults are bound by the chain exp, atan2,
// exchange, row sum, division of every stage; from about 1500 patches by the
// rows that are streamed (168 of 201 MB at 7 TB/s).
//
// Wave 0 holds the elements, one lane each, with their Cash-Karp sums in
// registers, and takes the step control; the other waves collect the exchanged
// slip rates and multiply rows.  The two parts are separate code between common
// barriers, so that the registers of one are free in the other.
//
// Exchange.  A block writes its slip rates with agent-scope relaxed atomic
// stores, which go through to the point that the 8 XCDs' L2s share; the others
// poll the entries themselves with agent-scope loads until they differ from
// kEmpty, a NaN that no arithmetic makes.  So a value is its own flag, and an
// exchange is one way out and one way in.  Buffers go round in fours: when a
// block publishes exchange k it has every block's k-1, so all have read k-2,
// whose buffer it empties for k+2; the emptying is complete (s_waitcnt) before
// it publishes k+1, and nobody polls k+2 without having that.  This needs every
// block to publish slip rates, so the plan has no block without an element
// (resident_plan.h): nobody would wait for one within an attempt, and its buffer
// would be emptied before it has read it.  No plain load or
// store touches exchanged data, so no cache has to be written back or
// invalidated: with agent-scope release and acquire fences an exchange took
// 59-64 us; with these accesses and a flag per block 1.8 us among 32 blocks
// and 3.8-5.1 us among 256.
//
// All blocks have to be resident before the first exchange.  They count
// themselves in; if they are not complete within 2 ms (another kernel holds
// the CUs), all of them leave before anything has changed, and the caller
// falls back on the captured attempt.  The later waits are bounded too, by 2 s: a
// block whose wait runs out raises a flag for the host and for the others' waits,
// and takes part until the attempt's end, where it leaves.  The launch's results
// are then void: the host puts back the state that the launch found, which every
// block has kept a copy of, and goes on with the captured attempt.
//
// The row sums keep wave_rows_dot's order and the element arithmetic is the
// captured attempt's (ode_dev.h): a run gives the same bits on either.
#include <hip/hip_runtime.h>
#include <type_traits>
#include "../../include/ucy.h"
#include "ode_dev.h"
#include "resident.h"

namespace ucy {

template <class T>
__device__ __forceinline__ T agent_load(const T *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void agent_store(T *p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

constexpr unsigned long long kEmpty = ~0ull;

// the bits of a value that is to be exchanged: never kEmpty
__device__ __forceinline__ unsigned long long exchange_bits(unsigned long long b)
{
    return b == kEmpty ? 0x7ff8000000000000ull : b;
}

// NR rows in LDS times v in LDS, in the order of wave_rows_dot (binary64) or
// wave_rows_dot_split (packed split-bf16 words)
template <int NR, class W>
__device__ __forceinline__ void lds_rows_dot(const W *K, int n, const double *v, int lane,
                                             double acc[NR])
{
#pragma unroll
    for (int r = 0; r < NR; r++) acc[r] = 0.0;
    const int n2 = n >> 1;
    const double2 *v2 = reinterpret_cast<const double2 *>(v);
#pragma unroll 4
    for (int j = lane; j < n2; j += 64) {
        const double2 vv = v2[j];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            if constexpr (sizeof(W) == 8) {
                const double2 kk = reinterpret_cast<const double2 *>(K + (size_t)r * n)[j];
                acc[r] = fma(kk.x, vv.x, acc[r]);
                acc[r] = fma(kk.y, vv.y, acc[r]);
            } else {
                const u32x2 kk = reinterpret_cast<const u32x2 *>(K + (size_t)r * n)[j];
                acc[r] = fma(split_entry(kk.x), vv.x, acc[r]);
                acc[r] = fma(split_entry(kk.y), vv.y, acc[r]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < NR; r++) acc[r] = wave_sum(acc[r]);
}

// the kernel is compiled per model, so that an element's few state entries stay
// in registers: 3-D patches, 3-D patches and volumes, the two 2-D models
enum { RES_PATCH = 0, RES_VOLUME = 1, RES_ANTIPLANE = 2, RES_PLANESTRAIN = 3 };

template <int M>
struct ResModel {
    // entries: state (largest), of them formed by the pre-pass, slip rates, rows
    static constexpr int ns = M == RES_PATCH ? 7 : M == RES_VOLUME ? 12 : M == RES_ANTIPLANE ? 4 : 6;
    static constexpr int nv = M == RES_PATCH ? 2 : M == RES_VOLUME ? 6 : M == RES_ANTIPLANE ? 2 : 3;
    static constexpr int nt = M == RES_PATCH ? 3 : M == RES_VOLUME ? 6 : M == RES_ANTIPLANE ? 2 : 3;
};

// what a lane keeps of its element between the pre-pass and the post-pass
struct ElemPre {
    PatchPre q;
    FrictionTerms g;
};

// the counts of an element: state entries, those that the pre-pass forms (as
// many as its slip rates), rows
template <int M>
__device__ __forceinline__ void elem_counts(bool vol, int &ns, int &nv, int &nt)
{
    if (M == RES_PATCH || (M == RES_VOLUME && !vol)) { ns = 7; nv = 2; nt = 3; }
    else if (M == RES_VOLUME) { ns = 12; nv = 6; nt = 6; }
    else if (M == RES_ANTIPLANE) { ns = 4; nv = nt = vol ? 2 : 1; }
    else { ns = vol ? 6 : 5; nv = vol ? 3 : 1; nt = vol ? 3 : 2; }
}

// the state entries that the right-hand side reads
template <int M>
__device__ __forceinline__ bool rhs_reads(bool vol, int k)
{
    if (M == RES_ANTIPLANE) return k >= 2;
    if (M == RES_PLANESTRAIN) return k >= 3;
    return vol ? k >= 6 : (k == 2 || k == 3 || k == 5 || k == 6);
}

// pre-pass of one element at the state p: dp's first entries, the slip-rate
// entries vp, the slip velocity (patch) in vel, the strain-rate norm (volume)
// in en
template <int M>
__device__ __forceinline__ void elem_pre(bool vol, const double *p, const Friction &f,
                                         const Rheology *rh, double *dp, double *vp, ElemPre &q,
                                         double &vel, double &en)
{
    vel = en = 0.0;
    if constexpr (M == RES_ANTIPLANE) {
        if (vol) en = ap_volume_prepass(p, *rh, dp, vp);
        else vel = q.q.velocity = ap_prepass(p, f, dp, vp);
    } else if constexpr (M == RES_PLANESTRAIN) {
        if (vol) en = ps_volume_prepass(p, *rh, dp, vp);
        else vel = q.q.velocity = ps_prepass(p, f, dp, vp);
    } else if (M == RES_PATCH || !vol) {
        patch_pre(p[2], p[3], p[6], q.q);
        const double vs = q.q.velocity * q.q.cr, vd = q.q.velocity * q.q.sr;
        dp[0] = vs;
        dp[1] = vd;
        vp[0] = vs - f.vplc;
        vp[1] = vd - f.vpls;
        vel = q.q.velocity;
    } else if constexpr (M == RES_VOLUME) {
        volume_prepass(p, *rh, dp, vp);
        en = sqrt((dp[0] * dp[0] + 2.0 * (dp[1] * dp[1]) + 2.0 * (dp[2] * dp[2]) +
                   dp[3] * dp[3] + 2.0 * (dp[4] * dp[4]) + dp[5] * dp[5]) / 2.0);
    }
}

// the part of the post-pass that needs no traction rate, taken while the slip
// rates travel
template <int M>
__device__ __forceinline__ void elem_early(bool vol, const double *p, const Friction &f, ElemPre &q)
{
    if (!vol)
        q.g = friction_terms(M == RES_ANTIPLANE ? p[2] : M == RES_PLANESTRAIN ? p[3] : p[5],
                             q.q.velocity, f);
}

// post-pass: the remaining entries of dp from the traction rates t
template <int M>
__device__ __forceinline__ void elem_post(bool vol, const double *t, const ElemPre &q, double *dp)
{
    if constexpr (M == RES_ANTIPLANE) {
        if (vol) {
            dp[2] = t[0];
            dp[3] = t[1];
        } else {
            ap_post(t[0], q.g, dp);
        }
    } else if constexpr (M == RES_PLANESTRAIN) {
        if (vol) {
            for (int k = 0; k < 3; k++) dp[3 + k] = t[k];
        } else {
            ps_post(t, q.g, dp);
        }
    } else if (M == RES_PATCH || !vol) {
        patch_post(t, q.q, q.g, dp);
    } else if constexpr (M == RES_VOLUME) {
        for (int k = 0; k < 6; k++) dp[6 + k] = t[k];
    }
}

// the Cash-Karp weights of k_j (j = 2..5) in the inputs of stages j+1, j+2, ..
__constant__ double kStageWeights[4][4] = {
    {B32, B42, B52, B62}, {B43, B53, B63, 0.0}, {B54, B64, 0.0, 0.0}, {B65, 0.0, 0.0, 0.0}};
// and of k_j (j = 2..6) in the solution and the error; 0: k_j is left out
__constant__ double kEndWeights[5][2] = {{0.0, 0.0}, {C3, DC3}, {C4, DC4}, {0.0, DC5}, {C6, DC6}};

template <int M, int PREC>
__global__ void __launch_bounds__(kResThreads)
resident_kernel(ResArgs a)
{
    typedef typename std::conditional<PREC == UCY_PREC_F64, double, uint32_t>::type Word;
    constexpr bool red_prec = PREC != UCY_PREC_F64;
    constexpr int NSM = ResModel<M>::ns, NVM = ResModel<M>::nv, NTM = ResModel<M>::nt;
    extern __shared__ __attribute__((aligned(16))) double lds[];
    __shared__ Control ctl;
    __shared__ int formed, stop, go, leave;
    const PlainDims &d = a.d;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, T = blockDim.x, nw = T >> 6;
    const int P = a.P, blk = blockIdx.x;

    // ---- every block counts itself in -------------------------------------
    if (t == 0) {
        formed = 1;
        if (P > 1) {
            if (atomicAdd(&a.head->arrived, 1u) == (unsigned)P - 1 && a.form_ticks)
                atomicCAS(&a.head->state, 0u, 1u);
            const unsigned long long t0 = wall_clock64();
            unsigned s;
            while ((s = agent_load(&a.head->state)) == 0) {
                if (wall_clock64() - t0 >= a.form_ticks) atomicCAS(&a.head->state, 0u, 2u);
                __builtin_amdgcn_s_sleep(1);
            }
            formed = s == 1;
        } else {
            a.head->state = 1;
        }
        ctl = *a.ctl;
        stop = leave = 0;
    }
    __syncthreads();
    if (!formed) return;

    // ---- this block's elements, rows and LDS ------------------------------
    const int e0 = a.bounds[blk], E = a.bounds[blk + 1] - e0;
    const int r0 = elem_row_off(d, e0), R = elem_row_off(d, e0 + E) - r0;
    const int n = d.n, nvt = elem_v_off(d, d.np + d.nv), EL = a.el_max;
    double *vL = lds;                          // [n]
    double *st = vL + n;                       // [2][NSM][EL]: yscal, dydt
    double *tL = st + (size_t)2 * NSM * EL;    // [rows_max] K v of the stage
    double *t0L = tL + a.rows_max;             // [rows_max] of the step start (reduced K)
    Word *KL = reinterpret_cast<Word *>(t0L + a.rows_max);
    const Word *Kg = red_prec ? reinterpret_cast<const Word *>(a.K.Kp)
                              : reinterpret_cast<const Word *>(a.K.K);
    auto scale = [&](int k) -> double & { return st[(size_t)k * EL + lane]; };
    auto dydt = [&](int k) -> double & { return st[(size_t)(NSM + k) * EL + lane]; };
    const int rl = R < a.rows_lds ? R : a.rows_lds;      // rows [0, rl) in LDS
    for (int i = t; i < n; i += T) vL[i] = 0.0;
    {
        // rl n is even: whole 8-byte (reduced) or 16-byte pairs
        typedef typename std::conditional<red_prec, u32x2, f64x2>::type Pair;
        const Pair *src = reinterpret_cast<const Pair *>(Kg + (int64_t)r0 * n);
        Pair *dst = reinterpret_cast<Pair *>(KL);
        const int c = (int)((int64_t)rl * n >> 1);
        for (int i = t; i < c; i += T) dst[i] = src[i];
    }
    // wave 0, one lane per element
    const bool mine = w == 0 && lane < E;
    const int e = e0 + (mine ? lane : 0);
    const bool vol = M != RES_PATCH && e >= d.np;
    const int so = elem_state_off(d, e), vo = elem_v_off(d, e), ro = elem_row_off(d, e) - r0;
    int ns, nv, nt;
    elem_counts<M>(vol, ns, nv, nt);
    const Rheology *rh = a.rh + (vol ? e - d.np : 0);
    Friction f{};
    ElemPre q{};
    // state, stage input (then the candidate), derivative, slip rates (the
    // step start's in v0); the sums over k_1..k_j so far of the solution, the
    // error and the inputs of the next four stages.  Each sum takes its terms
    // in stage_value's order, so that only the last is left when k_j arrives.
    double y[NSM], p[NSM], dp[NSM], vp[NVM], v0[NVM], ys[NSM], es[NSM], A[4][NSM];
    double vel = 0.0, en = 0.0;
#pragma unroll
    for (int k = 0; k < NSM; k++) y[k] = p[k] = dp[k] = ys[k] = es[k] = 0.0;
#pragma unroll
    for (int k = 0; k < NVM; k++) v0[k] = vp[k] = 0.0;
    if (mine) {
        double *const sy = a.saved, *const sd = sy + d.dim, *const ss = sd + d.dim;
        if (!vol) f = a.fr[e];
#pragma unroll
        for (int k = 0; k < NSM; k++)
            if (k < ns) {
                sy[so + k] = y[k] = p[k] = a.b.y[so + k];
                ss[so + k] = scale(k) = a.b.yscal[so + k];
                sd[so + k] = dydt(k) = a.b.dydt[so + k];
            }
        if (red_prec && !ctl.need_rhs) {
            double *const sv = ss + d.dim, *const st0 = sv + n;
#pragma unroll
            for (int k = 0; k < NVM; k++)
                if (k < nv) sv[vo + k] = v0[k] = a.b.v0[vo + k];
            for (int k = 0; k < nt; k++) st0[r0 + ro + k] = t0L[ro + k] = a.b.t0[r0 + ro + k];
        }
    }
    __syncthreads();

    unsigned sq = 0;      // exchanges so far

    // wave 0: the pre-pass at p and the slip rates out (less v0 if set); with
    // red set the block's maxima too
    auto publish = [&](bool red, bool less_v0, double err) {
        sq++;
        if (mine) elem_pre<M>(vol, p, f, rh, dp, vp, q, vel, en);
        if (P == 1) {
            if (mine) {
#pragma unroll
                for (int k = 0; k < NVM; k++)
                    if (k < nv) vL[vo + k] = less_v0 ? vp[k] - v0[k] : vp[k];
            }
        } else {
            __builtin_amdgcn_s_waitcnt(0);   // the emptied buffer of two exchanges ago
            asm volatile("" ::: "memory");
            unsigned long long *vb = a.v + (size_t)(sq & 3) * n;
            unsigned long long *ve = a.v + (size_t)((sq + 2) & 3) * n;
            if (mine) {
#pragma unroll
                for (int k = 0; k < NVM; k++)
                    if (k < nv) {
                        agent_store(vb + vo + k,
                                    exchange_bits(dbits(less_v0 ? vp[k] - v0[k] : vp[k])));
                        agent_store(ve + vo + k, kEmpty);
                    }
            }
            unsigned long long *re = a.red + (size_t)((sq + 2) & 3) * 3 * P + 3 * blk;
            if (red) {
                const unsigned long long be = wave_max_bits(dbits(err)),
                                         bv = wave_max_bits(dbits(vel)),
                                         bn = wave_max_bits(dbits(en));
                unsigned long long *rb = a.red + (size_t)(sq & 3) * 3 * P + 3 * blk;
                if (lane == 0) {
                    agent_store(rb, exchange_bits(be));
                    agent_store(rb + 1, exchange_bits(bv));
                    agent_store(rb + 2, exchange_bits(bn));
                }
            }
            if (lane < 3) agent_store(re + lane, kEmpty);
        }
        if (mine) elem_early<M>(vol, p, f, q);
    };
    // polls one entry; a wait that runs into its limit, or is behind one that has,
    // ends the block's part in the run
    auto poll = [&](const unsigned long long *x) {
        unsigned long long b, t0 = 0;
        for (int spin = 1; (b = agent_load(x)) == kEmpty; spin++)
            if ((spin & 1023) == 0 || a.wait_ticks == 0) {
                const unsigned long long now = wall_clock64();
                if (!t0) t0 = now;
                if (now - t0 >= a.wait_ticks || *(volatile int *)&stop ||
                    agent_load(&a.head->failed)) {
                    stop = 1;
                    agent_store(&a.head->failed, 1u);
                    return 0ull;
                }
            }
        return b;
    };
    // the workers: the slip rates of all blocks into LDS
    auto collect = [&]() {
        sq++;
        if (P == 1) return;
        const unsigned long long *vb = a.v + (size_t)(sq & 3) * n;
        for (int i = t - 64; i < nvt; i += T - 64)
            vL[i] = __longlong_as_double((long long)poll(vb + i));
    };
    // wave 0: the maxima of all blocks (P == 1: of this one), in every lane
    auto fold = [&](double err, unsigned long long &be, unsigned long long &bv,
                    unsigned long long &bn) {
        if (P == 1) {
            be = dbits(err);
            bv = dbits(vel);
            bn = dbits(en);
        } else {
            be = bv = bn = 0;
            const unsigned long long *rb = a.red + (size_t)(sq & 3) * 3 * P;
            for (int i = lane; i < P; i += 64) {
                const unsigned long long x = poll(rb + 3 * i), z = poll(rb + 3 * i + 1),
                                         u = poll(rb + 3 * i + 2);
                be = x > be ? x : be;
                bv = z > bv ? z : bv;
                bn = u > bn ? u : bn;
            }
        }
        be = wave_max_bits(be);
        bv = wave_max_bits(bv);
        bn = wave_max_bits(bn);
    };
    // the workers: rows [lo, hi) of this block from memory, in groups of nr
    auto stream_rows = [&](auto row_dot, int lo, int hi) {
        const int nr = min(4, (hi - lo + nw - 2) / (nw - 1));
        for (int r = lo + nr * (w - 1); r < hi; r += nr * (nw - 1)) {
            const int c = min(nr, hi - r);
            if (c == 4) row_dot(std::integral_constant<int, 4>(), r);
            else if (c == 3) row_dot(std::integral_constant<int, 3>(), r);
            else if (c == 2) row_dot(std::integral_constant<int, 2>(), r);
            else row_dot(std::integral_constant<int, 1>(), r);
        }
    };
    auto f64_rows = [&](auto count, int r) {
        constexpr int c = decltype(count)::value;
        double acc[c];
        if (r < a.rows_cached) wave_rows_dot<c, false>(a.K.K, r0 + r, n, vL, lane, acc);
        else wave_rows_dot<c, true>(a.K.K, r0 + r, n, vL, lane, acc);
        if (lane == 0)
            for (int k = 0; k < c; k++) tL[r + k] = acc[k];
    };
    auto split_rows = [&](auto count, int r) {
        constexpr int c = decltype(count)::value;
        double acc[c];
        wave_rows_dot_split<c>(a.K.Kp, a.K.rs, r0 + r, n, vL, lane, acc);
        if (lane == 0)
            for (int k = 0; k < c; k++) tL[r + k] = acc[k];
    };
    // K v of this block's rows with the stored K (the mixed form's step start
    // takes the binary64 K)
    auto dot = [&]() {
        // rows beyond LDS first: their latency is the longer one
        if constexpr (red_prec) stream_rows(split_rows, rl, R);
        else stream_rows(f64_rows, rl, R);
        // three rows per wave share the reads of v where there are enough; the
        // last workers, with the fewest rows from memory, begin
        const int wi = nw - 1 - w, wn = nw - 1, nr = rl >= 3 * wn ? 3 : 1;
        for (int r = nr * wi; r < rl; r += nr * wn) {
            if (nr == 3 && r + 3 <= rl) {
                double acc[3];
                lds_rows_dot<3>(KL + (size_t)r * n, n, vL, lane, acc);
                if (lane == 0)
                    for (int k = 0; k < 3; k++)
                        tL[r + k] = red_prec ? acc[k] * a.K.rs[r0 + r + k] : acc[k];
                continue;
            }
            for (int k = r; k < rl && k < r + nr; k++) {
                double acc[1];
                lds_rows_dot<1>(KL + (size_t)k * n, n, vL, lane, acc);
                if (lane == 0) tL[k] = red_prec ? acc[0] * a.K.rs[r0 + k] : acc[0];
            }
        }
    };
    // a lane's post-pass; start: of the step start, whose K v the stages add to
    auto post = [&](bool start) {
        double tr[NTM];
#pragma unroll
        for (int k = 0; k < NTM; k++) {
            tr[k] = 0.0;
            if (k < nt) {
                tr[k] = tL[ro + k];
                if (red_prec && start) t0L[ro + k] = tr[k];
                if (red_prec && !start) tr[k] += t0L[ro + k];
            }
        }
        elem_post<M>(vol, tr, q, dp);
    };

    // ---- the workers --------------------------------------------------------
    // They and wave 0 go through the same barriers: per exchange one when the
    // slip rates are in LDS, one when K v is.  Nobody polls between the two of a
    // step start, where wave 0 reads `stop` into `leave`: all waves leave alike.
    if (w != 0) {
        // 1: the call's first step start; 2..6: a stage; 7: an attempt's end,
        // with the next step's start if the step is accepted
        int phase = ctl.need_rhs && !ctl.done ? 1 : 2;
        for (int att = 0;;) {
            if (phase == 2 && !(att < a.max_attempts && !ctl.done && !leave)) break;
            collect();
            __syncthreads();
            const bool start = phase == 1 || phase == 7;
            if (phase != 7 || go) {
                if (PREC == UCY_PREC_MIXED && start) stream_rows(f64_rows, 0, R);
                else dot();
            }
            __syncthreads();
            att += phase == 7;
            phase = start ? 2 : phase + 1;
        }
        return;
    }

    // ---- wave 0: the elements and the step control --------------------------
    bool fresh = false;   // K v of a new step's start is in tL
    if (ctl.need_rhs && !ctl.done) {
        publish(true, false, 0.0);
        unsigned long long be, bv, bn;
        fold(0.0, be, bv, bn);
        __syncthreads();
        if (lane == 0) {
            ctl.vmax = __longlong_as_double((long long)bv);
            ctl.emax = __longlong_as_double((long long)bn);
            leave = stop;
        }
        __syncthreads();
        fresh = true;
    }

    for (int att = 0; att < a.max_attempts && !ctl.done && !leave; att++) {
        const double h = ctl.h;
        if (mine) {
            if (fresh) {   // a new step: dydt and yscal (ratestate.f90:309-315)
                post(true);
#pragma unroll
                for (int k = 0; k < NVM; k++) v0[k] = vp[k];
#pragma unroll
                for (int k = 0; k < NSM; k++)
                    if (k < ns) {
                        dydt(k) = dp[k];
                        scale(k) = fabs(y[k]) + fabs(h * dp[k]) + 1.0e-30;
                    }
            }
#pragma unroll
            for (int k = 0; k < NSM; k++) {
                if (k >= ns) continue;
                const double k1 = dydt(k);
                ys[k] = C1 * k1;
                es[k] = DC1 * k1;
                if (rhs_reads<M>(vol, k)) {
                    p[k] = y[k] + (h * B21) * k1;
                    A[0][k] = B31 * k1;
                    A[1][k] = B41 * k1;
                    A[2][k] = B51 * k1;
                    A[3][k] = B61 * k1;
                }
            }
        }
#pragma unroll 1
        for (int j = 2; j <= 6; j++) {
            publish(false, red_prec, 0.0);
            __syncthreads();
            __syncthreads();
            if (!mine) continue;
            post(false);
            const double c = kEndWeights[j - 2][0], dc = kEndWeights[j - 2][1];
            if (j < 6) {
                const double *b = kStageWeights[j - 2];
                const double b0 = b[0], b1 = b[1], b2 = b[2], b3 = b[3];
#pragma unroll
                for (int k = 0; k < NSM; k++) {
                    if (k >= ns) continue;
                    if (rhs_reads<M>(vol, k)) {
                        p[k] = y[k] + h * (A[0][k] + b0 * dp[k]);
                        A[0][k] = A[1][k] + b1 * dp[k];
                        A[1][k] = A[2][k] + b2 * dp[k];
                        A[2][k] = A[3][k] + b3 * dp[k];
                    }
                    if (c != 0.0) ys[k] = ys[k] + c * dp[k];
                    if (dc != 0.0) es[k] = es[k] + dc * dp[k];
                }
            }
        }
        // the candidate: the 5th-order solution and the largest error ratio
        // (ode45.f90:185-200, :75); the next step's pre-pass at it goes out with
        // the ratio
        double err = 0.0;
        if (mine) {
#pragma unroll
            for (int k = 0; k < NSM; k++) {
                if (k >= ns) continue;
                p[k] = y[k] + h * (ys[k] + C6 * dp[k]);
                const double er = h * (es[k] + DC6 * dp[k]);
                const double r = fabs(er / scale(k));
                // non-finite ratios propagate as NaN bits, which order above +inf
                err = (r > err || r != r) ? r : err;
            }
        }
        publish(true, false, err);
        unsigned long long be, bv, bn;
        fold(err, be, bv, bn);
        // as controller_step decides
        const double raw = __longlong_as_double((long long)be);
        fresh = raw <= 1.7976931348623157e308 && !(raw / ctl.epsilon > 1.0);
        if (lane == 0) go = fresh;
        __syncthreads();
        // the step control, two powers and a log row, while the workers
        // multiply the next step's start
        if (lane == 0) {
            ctl.errmax_bits = be;
            controller_step(a.b, &ctl, blk == 0);
            leave = stop;
            if (ctl.accepted) {
                ctl.vmax = __longlong_as_double((long long)bv);
                ctl.emax = __longlong_as_double((long long)bn);
            }
        }
        __syncthreads();
        if (fresh && mine) {
            // the export of the step-start entries (ratestate.f90:488-536)
            const int64_t row = ctl.log_count - 1;
            if (a.b.n_obs > 0 && row >= 0 && row < ctl.log_cap) {
                double *oy = a.b.obs_y + row * a.b.n_obs, *od = a.b.obs_dydt + row * a.b.n_obs;
                int col[NSM];
#pragma unroll
                for (int k = 0; k < NSM; k++) col[k] = k < ns ? a.obs_col[so + k] : -1;
#pragma unroll
                for (int k = 0; k < NSM; k++)
                    for (int v = col[k]; v >= 0;) {
                        const int j = v & ~kResMore;
                        oy[j] = y[k];
                        od[j] = dydt(k);
                        v = v & kResMore ? a.obs_next[j] : -1;
                    }
            }
#pragma unroll
            for (int k = 0; k < NSM; k++) y[k] = p[k];
        }
    }

    // ---- back to memory ---------------------------------------------------
    if (mine) {
#pragma unroll
        for (int k = 0; k < NSM; k++)
            if (k < ns) {
                a.b.y[so + k] = y[k];
                a.b.yscal[so + k] = scale(k);
                a.b.dydt[so + k] = dydt(k);
            }
        if (red_prec) {
#pragma unroll
            for (int k = 0; k < NVM; k++)
                if (k < nv) a.b.v0[vo + k] = v0[k];
            for (int k = 0; k < nt; k++) a.b.t0[r0 + ro + k] = t0L[ro + k];
        }
    }
    if (blk == 0 && t == 0) {
        ctl.accepted = 0;      // y is the accepted state already
        ctl.obs_pending = 0;
        if (ctl.need_rhs) {    // formed again by the next step start
            ctl.vmax = 0.0;
            ctl.emax = 0.0;
        }
        *a.ctl = ctl;
    }
}

typedef void (*ResKernel)(ResArgs);
template <int M>
static ResKernel resident_of(int prec)
{
    return prec == UCY_PREC_F64 ? resident_kernel<M, UCY_PREC_F64>
           : prec == UCY_PREC_MIXED ? resident_kernel<M, UCY_PREC_MIXED>
                                    : resident_kernel<M, UCY_PREC_SPLIT_BF16>;
}
static ResKernel resident_of(const PlainDims &d, int prec)
{
    if (d.ap) return resident_of<RES_ANTIPLANE>(prec);
    if (d.ps) return resident_of<RES_PLANESTRAIN>(prec);
    return d.nv ? resident_of<RES_VOLUME>(prec) : resident_of<RES_PATCH>(prec);
}

hipError_t launch_resident(hipStream_t st, const ResArgs &a, size_t lds)
{
    const ResKernel k = resident_of(a.d, a.K.prec);
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, dim3(a.P), dim3(a.threads), lds, st, a);
    return hipGetLastError();
}

}  // namespace ucy
