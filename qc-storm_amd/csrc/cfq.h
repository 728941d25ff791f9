// cfq.h -- work-item records of the converged fitter's queue kernels (cfq.hip, cfs.hip).
#pragma once
#include "cfit_dev.h"

namespace qcs {

enum { CX_ROI = 0, CX_ST = 1, CX_T = 2, CX_ITERS = 3, CX_EVALS = 4, CX_SLOPE = 5, CX_ALPHA = 6, CX_DMAX = 7, CX_DU = 8 };

// record of one work item: theta, loss, gradient, "identity start" flag, packed D0, padding; a
// fit left by a one-lane wave adds the state of its line search and its counters at OX
template <int KK> struct CQ {
    static constexpr int P = CP<KK>::P, NS = CP<KK>::NS;
    static constexpr int OL = P, OG = P + 1, OF = 2 * P + 1, OD = 2 * P + 2;
    static constexpr int W = (2 * P + 2 + NS + 3) & ~3;   // floats, a multiple of 4
    static constexpr int OX = W, XW = (W + CX_DU + P + 3) & ~3;
};

enum { CQ_IDLE = 0, CQ_DIR = 1, CQ_LS = 2 };

// a wave's LDS accesses complete in order; this keeps the compiler from moving them
__device__ __forceinline__ void cf_wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// split launch over the sets of a (cfs.hip): fresh items, or where a.left[i].rec is set the left fits
int cfs_waves_per_cu(int KK, int RMAX);   // its resident waves per CU
int cfs_launch(const CfqArgs &a, int KK, int rmax, long long items, int cus, int max_waves_per_cu, hipStream_t s);

}  // namespace qcs
