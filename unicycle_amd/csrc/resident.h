// resident.h -- the resident integrator (k_resident.hip): its arguments and plan
#pragma once
#include "resident_plan.h"
#include "ucy_internal.h"

namespace ucy {

constexpr int kResThreads = 512;      // at most, per block

struct ResHead {
    unsigned arrived, state;          // state 0: forming, 1: complete, 2: given up
    unsigned failed;                  // a wait of any block ran into its limit
    unsigned pad;
};

// The head lies behind the control block, so that the host reads both in one copy,
// and on a cache line of its own: the blocks poll it.
constexpr size_t kResHeadOffset = 256;
static_assert(sizeof(Control) <= kResHeadOffset, "the head would overlap the control block");
constexpr size_t kControlBytes = kResHeadOffset + sizeof(ResHead);
inline ResHead *resident_head(Control *ctl)
{
    return reinterpret_cast<ResHead *>(reinterpret_cast<char *>(ctl) + kResHeadOffset);
}

struct ResArgs {
    PlainDims d;
    KOperand K;
    const Friction *fr;
    const Rheology *rh;
    RkBuffers b;
    Control *ctl;
    ResHead *head;
    // the state, derivative and scale, and (reduced K) v0 and t0, as the launch found
    // them: [3 dim + n + m], in the order of the work buffers
    double *saved;
    // exchange buffers, all entries empty (all bits set) at launch
    unsigned long long *red;          // [4][P][3]: error norm, slip velocity, strain rate
    unsigned long long *v;            // [4][n] slip rates
    size_t xbytes;                    // of red and v together
    const int *bounds;                // [P + 1] first element of each block
    // columns of the log of observed entries (b.n_obs > 0): per state entry one, or
    // -1; with kResMore set another follows, in obs_next at the column
    const int *obs_col, *obs_next;
    int P, threads;
    int el_max, rows_max;             // largest share of a block, both even
    int rows_lds;                     // rows of a block kept in LDS
    int rows_cached;                  // rows up to this one are read through the caches,
                                      // later ones stream past them
    int max_attempts;
    // ticks of the 100 MHz clock: forming (0: the blocks find no room) and a wait
    // for other blocks' values
    unsigned long long form_ticks, wait_ticks;
};

hipError_t launch_resident(hipStream_t st, const ResArgs &a, size_t lds);

}  // namespace ucy
