// resident_plan.h -- the resident integrator's blocks, their shares and LDS: host
// arithmetic alone, so that it can be checked without a GPU
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace ucy {

constexpr int kResMaxBlocks = 256;    // one per CU of a whole MI355X
constexpr int kResMaxElements = 64;   // of a block: one lane of wave 0 each

enum { RES_MODEL_3D = 0, RES_MODEL_ANTIPLANE = 1, RES_MODEL_PLANESTRAIN = 2 };

// state entries per element that the kernel holds in LDS, for its size
inline int resident_state_entries(int model, int nv)
{
    return model == RES_MODEL_ANTIPLANE ? 4 : model == RES_MODEL_PLANESTRAIN ? 6 : nv ? 12 : 7;
}

struct ResidentPlan {
    int P = 0;                 // blocks; 0: the model takes the captured attempt
    std::vector<int> bounds;   // [P + 1] first element of each block, strictly ascending
    int el_max = 0, rows_max = 0;   // largest share of a block, both even
    int rows_lds = 0;          // rows of a block kept in LDS
    int rows_cached = 0;       // rows up to this one are read through the caches
    size_t lds = 0;
};

// np patches, nv volumes, K of m rows and n columns (as stored, n even) with
// binary64 entries (f64) or packed words of 4 bytes, on a device of cus CUs.
//   - At most a block per CU, as all are resident at once and a block's LDS is most
//     of a CU's.  A device partition has fewer CUs than the whole: blocks beyond
//     them would find no room, and each call would wait 2 ms to learn it.
//   - Share of a block: 48 KB of K, so that a stage's products (0.2 us) take
//     less than the exchange among the blocks (1.5 us with 8, 3.8 us with 256).
//     8 to 72 KB measure within 10 % of each other; a reduced K has fewer bytes
//     per row and takes 16 KB (200 patches: 28 us per attempt, 35 us at 48 KB).
//   - One block where K fits it whole, as it needs no exchange.
//   - No block without an element: the exchange reuses its buffers on the strength
//     of every block's publishing slip rates (k_resident.hip).  Cut at equal numbers
//     of rows a range can be empty, as an element has up to 6; such ranges are
//     dropped.
//   - At most 1 GB of K in binary64 (4096 patches: 755 us per attempt, captured
//     770 us; 8192 patches: 2985 and 2910 us, the launches no longer show) and
//     2 GB reduced (8192 patches: 1775 and 1800 us).
//   - Rows beyond LDS up to 64 KB per CU are left to the L2 (1600 patches 103 us,
//     109 us if all stream; 2816 patches 368 and 353 us).
inline ResidentPlan resident_plan(int model, int np, int nv, int64_t m, int64_t n, bool f64,
                                  int cus)
{
    constexpr int64_t kLds = 158 * 1024, kOneBlock = 96 * 1024, kCachedBytes = 64 * 1024;
    const int64_t entry = f64 ? 8 : 4, share = (f64 ? 48 : 16) * 1024, kb = m * n * entry;
    const int ne = np + nv;
    ResidentPlan p;
    if (kb > (f64 ? 1ll << 30 : 2ll << 30)) return p;
    int64_t P = kb <= kOneBlock && ne <= kResMaxElements
                    ? 1 : std::max<int64_t>(2, (kb + share - 1) / share);
    P = std::max<int64_t>(P, (ne + 55) / 56);
    P = std::min<int64_t>(P, std::max(1, std::min(cus, kResMaxBlocks)));
    // element boundaries at equal numbers of rows
    const bool ap = model == RES_MODEL_ANTIPLANE, ps = model == RES_MODEL_PLANESTRAIN;
    const int64_t rp = ps ? 2 : ap ? 1 : 3, rv = ps ? 3 : ap ? 2 : 6;
    auto row = [&](int e) { return e <= np ? rp * e : rp * np + rv * (e - np); };
    p.bounds.push_back(0);
    for (int64_t b = 1; b <= P; b++) {
        const int64_t r = m * b / P;
        const int e = (int)(r <= rp * np ? (r + rp - 1) / rp : np + (r - rp * np + rv - 1) / rv);
        const int first = p.bounds.back();
        if (e == first) continue;
        p.bounds.push_back(e);
        p.el_max = std::max(p.el_max, e - first);
        p.rows_max = std::max(p.rows_max, (int)(row(e) - row(first)));
    }
    P = (int64_t)p.bounds.size() - 1;
    if (p.el_max > kResMaxElements) return p;
    p.el_max += p.el_max & 1;
    p.rows_max += p.rows_max & 1;
    const int64_t other =
        8 * (n + 2ll * resident_state_entries(model, nv) * p.el_max + 2ll * p.rows_max);
    if (other > kLds) return p;
    const int64_t lr = std::min<int64_t>(p.rows_max, (kLds - other) / (n * entry));
    p.lds = (size_t)(other + lr * n * entry);
    p.rows_lds = (int)lr;
    p.rows_cached = (int)(lr + kCachedBytes / (n * entry));
    p.P = (int)P;
    return p;
}

// The columns of each state entry in a log of observed entries idx[0, n_obs): the
// lane that holds an entry finds its columns without a look at the others' (700
// entries of 247 patches, each lane walking the list: 159 us per attempt, 27
// without).  An entry may be observed more than once.
constexpr int kResMore = 1 << 30;
inline void resident_observed(int dim, int64_t n_obs, const int64_t *idx, int *col, int *next)
{
    std::fill(col, col + dim, -1);
    for (int64_t j = 0; j < n_obs; j++) {
        int &head = col[idx[j]];
        next[j] = head;
        head = (int)j | (head == -1 ? 0 : kResMore);
    }
}

}  // namespace ucy
