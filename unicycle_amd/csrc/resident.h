// resident.h -- the resident integrator (k_resident.hip): its arguments and plan
#pragma once
#include "resident_plan.h"
#include "ucy_internal.h"

namespace ucy {

constexpr int kResThreads = 512;      // at most, per block

struct ResHead {
    unsigned arrived, state;          // state 0: forming, 1: complete, 2: given up
};

struct ResArgs {
    PlainDims d;
    KOperand K;
    const Friction *fr;
    const Rheology *rh;
    RkBuffers b;
    Control *ctl;
    ResHead *head;
    // exchange buffers, all entries empty (all bits set) at launch
    unsigned long long *red;          // [4][P][3]: error norm, slip velocity, strain rate
    unsigned long long *v;            // [4][n] slip rates
    size_t xbytes;                    // of red and v together
    const int *bounds;                // [P + 1] first element of each block
    int P, threads;
    int el_max, rows_max;             // largest share of a block, both even
    int rows_lds;                     // rows of a block kept in LDS
    int rows_cached;                  // rows up to this one are read through the caches,
                                      // later ones stream past them
    int max_attempts;
};

hipError_t launch_resident(hipStream_t st, const ResArgs &a, size_t lds);

}  // namespace ucy
