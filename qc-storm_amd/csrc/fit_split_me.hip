// fit_split_me.hip -- multi-emitter kernels of fit_split.h by model, ROI size and lanes per ROI.
#include "fit_split.h"

namespace qcs {

template <int MODEL, bool FAST>
static int by_size(int R, int G, const SplitArgs &a, const FitConst &fc, hipStream_t s)
{
    if (R == 5 && G == 4) return launch_split<MODEL, 5, 4, FAST>(a, fc, s);
    if (R == 5 && G == 8) return launch_split<MODEL, 5, 8, FAST>(a, fc, s);
    if (R == 7 && G == 4) return launch_split<MODEL, 7, 4, FAST>(a, fc, s);
    if (R == 7 && G == 8) return launch_split<MODEL, 7, 8, FAST>(a, fc, s);
    if (R == 9 && G == 4) return launch_split<MODEL, 9, 4, FAST>(a, fc, s);
    if (R == 9 && G == 16) return launch_split<MODEL, 9, 16, FAST>(a, fc, s);
    if (R == 11 && G == 4) return launch_split<MODEL, 11, 4, FAST>(a, fc, s);
    if (R == 11 && G == 16) return launch_split<MODEL, 11, 16, FAST>(a, fc, s);
    if (R == 13 && G == 16) return launch_split<MODEL, 13, 16, FAST>(a, fc, s);
    return fail(QCS_ERR_ARG, "ROISize %d not supported by the multi-emitter fitter (odd, 5..13)", R);
}

int fit_split_me(int model, int R, int G, bool fast, const SplitArgs &a, const FitConst &fc, hipStream_t s)
{
    switch (model) {
    case MODEL_2E: return fast ? by_size<MODEL_2E, true>(R, G, a, fc, s) : by_size<MODEL_2E, false>(R, G, a, fc, s);
    case MODEL_3E: return fast ? by_size<MODEL_3E, true>(R, G, a, fc, s) : by_size<MODEL_3E, false>(R, G, a, fc, s);
    default: return fast ? by_size<MODEL_AS3D2E, true>(R, G, a, fc, s) : by_size<MODEL_AS3D2E, false>(R, G, a, fc, s);
    }
}

}  // namespace qcs
