// fit_split_1e.hip -- one-emitter kernels of fit_split.h by model, ROI size and lanes per ROI.
#include "fit_split.h"

namespace qcs {

template <int MODEL, bool FAST>
static int by_size(int R, int G, const SplitArgs &a, const FitConst &fc, hipStream_t s)
{
    if (R == 5 && G == 1) return launch_split<MODEL, 5, 1, FAST>(a, fc, s);
    if (R == 5 && G == 2) return launch_split<MODEL, 5, 2, FAST>(a, fc, s);
    if (R == 5 && G == 4) return launch_split<MODEL, 5, 4, FAST>(a, fc, s);
    if (R == 5 && G == 8) return launch_split<MODEL, 5, 8, FAST>(a, fc, s);
    if (R == 7 && G == 1) return launch_split<MODEL, 7, 1, FAST>(a, fc, s);
    if (R == 7 && G == 4) return launch_split<MODEL, 7, 4, FAST>(a, fc, s);
    if (R == 7 && G == 8) return launch_split<MODEL, 7, 8, FAST>(a, fc, s);
    if (R == 9 && G == 2) return launch_split<MODEL, 9, 2, FAST>(a, fc, s);
    if (R == 9 && G == 4) return launch_split<MODEL, 9, 4, FAST>(a, fc, s);
    if (R == 9 && G == 16) return launch_split<MODEL, 9, 16, FAST>(a, fc, s);
    if (R == 11 && G == 4) return launch_split<MODEL, 11, 4, FAST>(a, fc, s);
    if (R == 11 && G == 16) return launch_split<MODEL, 11, 16, FAST>(a, fc, s);
    if (R == 13 && G == 16) return launch_split<MODEL, 13, 16, FAST>(a, fc, s);
    if (R == 15 && G == 16) return launch_split<MODEL, 15, 16, FAST>(a, fc, s);
    if (R == 17 && G == 8) return launch_split<MODEL, 17, 8, FAST>(a, fc, s);
    if (R == 17 && G == 16) return launch_split<MODEL, 17, 16, FAST>(a, fc, s);
    if constexpr (FAST) {
        if (R == 9 && G == 1) return launch_split<MODEL, 9, 1, FAST>(a, fc, s);
        if constexpr (MODEL == MODEL_GS2D) {
            if (R == 13 && G == 2) return launch_split<MODEL, 13, 2, FAST>(a, fc, s);
        } else {
            if (R == 13 && G == 4) return launch_split<MODEL, 13, 4, FAST>(a, fc, s);
        }
    }
    return fail(QCS_ERR_ARG, "ROISize %d not supported by the fitter (odd, 5..17)", R);
}

int fit_split_1e(int model, int R, int G, bool fast, const SplitArgs &a, const FitConst &fc, hipStream_t s)
{
    if (model == MODEL_AS3D) return fast ? by_size<MODEL_AS3D, true>(R, G, a, fc, s) : by_size<MODEL_AS3D, false>(R, G, a, fc, s);
    return fast ? by_size<MODEL_GS2D, true>(R, G, a, fc, s) : by_size<MODEL_GS2D, false>(R, G, a, fc, s);
}

}  // namespace qcs
