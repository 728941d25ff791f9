// fit_dev.h -- models of the reference-schedule fitters: parameter layouts, start vectors, weights,
// acceptance rules and rows, used by the kernels of fit_split.h (instantiated in fit_split_1e.hip and
// fit_split_me.hip) and their host side (fit.hip).
//
// Reference kernels (DLL = MLEbfgs/bfgs_MLE_dll x64/bfgsMLE_dll/bfgsMLE_dll):
//   bfgsMLELoc_Gauss2D      DLL/bfgsMLE_Loc_LD/bfgsMLE_GS2D_core.h:56-310
//   bfgsMLELoc_AS3D         DLL/bfgsMLE_Loc_LD/bfgsMLE_AS3D_core.h:57-337
//   bfgsMLELoc_Gauss2D_2E   DLL/bfgsMLE_Loc_HD/bfgsMLE_GS2D_2Emitter_core.h:74-371, init :595-698
//   bfgsMLELoc_Gauss2D_3E   DLL/bfgsMLE_Loc_HD/bfgsMLE_GS2D_3Emitter_core.h:76-362, init :592-710
//   bfgsMLELoc_AS3D_2E      DLL/bfgsMLE_Loc_HD/bfgsMLE_AS3D_2Emitter_core.h:77-422, init :647-750
#pragma once
#include "qcs_internal.h"
#include "qcs_devmath.h"

namespace qcs {

// Arguments of the fits (fit_split.h): items i < n (or *n_dev) of list idx (or the ROIs themselves).  fa, by
// ROI: one-emitter fits that go to the two-emitter stage (finish_1e); fa and fb, by item: accepted second
// and rejected first emitters of the multi-emitter stages (finish_me), whose second rows go to second.
struct SplitArgs {
    const uint16_t *rois;
    const float *wle;
    const int *idx;
    int n;
    const int *n_dev;
    float *loc, *second;
    int *fa, *fb;
};
int fit_split_1e(int model, int R, int G, bool fast, const SplitArgs &a, const FitConst &fc, hipStream_t s);
int fit_split_me(int model, int R, int G, bool fast, const SplitArgs &a, const FitConst &fc, hipStream_t s);

enum { MODEL_GS2D = 0, MODEL_AS3D = 1, MODEL_2E = 2, MODEL_3E = 3, MODEL_AS3D2E = 4 };

// Parameter layout of each model: amplitude / x / y / sigma_x / sigma_y index of emitter k,
// background index, iteration count, loss clamp, WLE weighting.
template <int MODEL> struct Traits;
template <> struct Traits<MODEL_GS2D> {   // bfgsMLE_GS2D_core.h:25-37
    static constexpr int P = 5, ITERS = 8, K = 1, IB = 4;
    static constexpr bool WEIGHTED = true;
    static constexpr float CLAMP = 0.0f;
    __device__ static constexpr int ia(int) { return 0; }
    __device__ static constexpr int ix(int) { return 1; }
    __device__ static constexpr int iy(int) { return 2; }
    __device__ static constexpr int isx(int) { return 3; }
    __device__ static constexpr int isy(int) { return 3; }
};
template <> struct Traits<MODEL_AS3D> {   // bfgsMLE_AS3D_core.h:25-38, loss clamp :501-505
    static constexpr int P = 6, ITERS = 11, K = 1, IB = 5;
    static constexpr bool WEIGHTED = true;
    static constexpr float CLAMP = 0.01f;
    __device__ static constexpr int ia(int) { return 0; }
    __device__ static constexpr int ix(int) { return 1; }
    __device__ static constexpr int iy(int) { return 2; }
    __device__ static constexpr int isx(int) { return 3; }
    __device__ static constexpr int isy(int) { return 4; }
};
template <> struct Traits<MODEL_2E> {     // bfgsMLE_GS2D_2Emitter_core.h:24-51
    static constexpr int P = 8, ITERS = 13, K = 2, IB = 7;
    static constexpr bool WEIGHTED = true;
    static constexpr float CLAMP = 0.0f;
    __device__ static constexpr int ia(int k) { return 3 * k; }
    __device__ static constexpr int ix(int k) { return 3 * k + 1; }
    __device__ static constexpr int iy(int k) { return 3 * k + 2; }
    __device__ static constexpr int isx(int) { return 6; }
    __device__ static constexpr int isy(int) { return 6; }
};
template <> struct Traits<MODEL_3E> {     // bfgsMLE_GS2D_3Emitter_core.h:24-54 (unweighted)
    static constexpr int P = 11, ITERS = 16, K = 3, IB = 10;
    static constexpr bool WEIGHTED = false;
    static constexpr float CLAMP = 0.0f;
    __device__ static constexpr int ia(int k) { return 3 * k; }
    __device__ static constexpr int ix(int k) { return 3 * k + 1; }
    __device__ static constexpr int iy(int k) { return 3 * k + 2; }
    __device__ static constexpr int isx(int) { return 9; }
    __device__ static constexpr int isy(int) { return 9; }
};
template <> struct Traits<MODEL_AS3D2E> { // bfgsMLE_AS3D_2Emitter_core.h:24-54 (unweighted), clamp :590-594
    static constexpr int P = 11, ITERS = 16, K = 2, IB = 10;
    static constexpr bool WEIGHTED = false;
    static constexpr float CLAMP = 0.01f;
    __device__ static constexpr int ia(int k) { return 5 * k; }
    __device__ static constexpr int ix(int k) { return 5 * k + 1; }
    __device__ static constexpr int iy(int k) { return 5 * k + 2; }
    __device__ static constexpr int isx(int k) { return 5 * k + 3; }
    __device__ static constexpr int isy(int k) { return 5 * k + 4; }
};

template <int P>
__device__ __forceinline__ void normalize_dir(float (&d)[P])
{
    float tot = 0.0f;
#pragma unroll
    for (int k = 0; k < P; k++) tot = tot + __builtin_fabsf(d[k]);
    tot = (float)P / tot;
#pragma unroll
    for (int k = 0; k < P; k++) d[k] = d[k] * tot;
}

// WLEWeightsCalc (bfgsMLE_core.h:206-238), separable form: w(r, c) = wy[r] * wx[c]
template <int R>
__device__ __forceinline__ void wle_weights(float sgx, float sgy, bool mlefit, float (&wx)[R], float (&wy)[R])
{
    const float ctr = (float)R / 2.0f;
    const float sx1 = 1.0f / ((2.0f * sgx) * sgx);
    const float sy1 = 1.0f / ((2.0f * sgy) * sgy);
#pragma unroll
    for (int c = 0; c < R; c++) {
        const float d = ((float)c + 0.5f) - ctr;
        wx[c] = mlefit ? 1.0f : qexpf(-((d * d) * sx1));
        wy[c] = mlefit ? 1.0f : qexpf(-((d * d) * sy1));
    }
}

// Border sums of the ROI (PreEstimation_GS2D, bfgsMLE_GS2D_core.h:529-546).
template <int R, class Q>
__device__ __forceinline__ float border_bkg(Q q)
{
    float m1 = 0.0f, m2 = 0.0f, m3 = 0.0f, m4 = 0.0f;
#pragma unroll
    for (int k = 0; k < R; k++) {
        m1 = m1 + q(k * R + 0);
        m2 = m2 + q(k * R + R - 1);
        m3 = m3 + q(0 * R + k);
        m4 = m4 + q((R - 1) * R + k);
    }
    m1 = m1 < m2 ? m1 : m2;
    m3 = m3 < m4 ? m3 : m4;
    return ((m1 + m3) / 2.0f) / (float)R;
}

__device__ __forceinline__ float zpoly(const float (&pc)[5], float d, float corr)
{
    // bfgsMLE_AS3D_core.h:266-279 with d^k formed by multiplication
    const float d2 = d * d, d3 = d2 * d, d4 = d2 * d2;
    float z = pc[0] * d4;
    z = __builtin_fmaf(pc[1], d3, z);
    z = __builtin_fmaf(pc[2], d2, z);
    z = __builtin_fmaf(pc[3], d, z);
    z = z + pc[4];
    return z * corr;
}

// Start vector x and weights of the one-emitter fits; q(i) is pixel i, wp the ROI's WLE record.
template <int MODEL, int R, class Q>
__device__ __forceinline__ void start_1e(Q q, const float *__restrict__ wp, const FitConst &fc, float (&x)[Traits<MODEL>::P],
                                         float (&wx)[R], float (&wy)[R])
{
    constexpr int HALF = R / 2;
    const float sl = wp[1], sr = wp[2], su = wp[3], sd = wp[4];
    const int mt = (int)wp[5];
    const bool mlefit = (mt == QCS_MOLTYPE_MLEFIT);

    const float bkg = border_bkg<R>(q);
    const float amp = q(HALF * R + HALF) - bkg;
    if (MODEL == MODEL_GS2D) {
        // bfgsMLELoc_Gauss2D :188-228, PreEstimation_GS2D :548-574
        float ws = fminf(fminf(sl, sr), fminf(su, sd));
        ws = fminf(ws, ((float)R / 2.0f) / 2.35f);
        const float ps = 1.0f / ((2.0f * ws) * ws);
        x[0] = amp * 0.0078125f;
        x[1] = (float)HALF + 0.5f;
        x[2] = (float)HALF + 0.5f;
        x[3] = ps * 10.0f;
        x[4] = bkg * 0.015625f;
        if (!mlefit) {
            ws = ws / 1.2f;
            ws = fminf(ws, ((float)R / 2.0f) / 2.35f);
        }
        if (fc.WLEEn == 0 && mt != QCS_MOLTYPE_MULTIFIT) ws = (float)R;
        wle_weights<R>(ws, ws, mlefit, wx, wy);
    } else {
        // bfgsMLELoc_AS3D :188-228, PreEstimation_AS3D :578-606
        float wsx = fminf(sl, sr), wsy = fminf(su, sd);
        x[0] = amp * 0.0078125f;
        x[1] = (float)HALF + 0.5f;
        x[2] = (float)HALF + 0.5f;
        x[3] = 10.0f * (0.5f / (wsx * wsx));
        x[4] = 10.0f * (0.5f / (wsy * wsy));
        x[5] = bkg * 0.015625f;
        if (!mlefit) {
            const float cap = ((float)R / 1.6f) / 2.35f;
            wsx = fminf(wsx, cap);
            wsy = fminf(wsy, cap);
        }
        if (fc.WLEEn == 0 && mt != QCS_MOLTYPE_MULTIFIT) { wsx = (float)R; wsy = (float)R; }
        wle_weights<R>(wsx, wsy, mlefit, wx, wy);
    }
}

// Acceptance and 12-float row of a one-emitter fit; flag[roi] (if non-null) is set to 1 when a
// rejected fit qualifies for the two-emitter stage (valid background and SNR > 6,
// bfgsMLE_GS2D_core.h:279-297).
template <int MODEL, int R>
__device__ __forceinline__ void finish_1e(const float (&x)[Traits<MODEL>::P], const FitConst &fc, int xo, int yo, int fr, int roi,
                                          float *__restrict__ loc, int *__restrict__ flag)
{
    constexpr int HALF = R / 2;
    float row[QCS_REC_FLOATS];
    bool ok;
    float snr;
    bool valid;
    const float QE = fc.QE;
    if (MODEL == MODEL_GS2D) {
        // bfgsMLELoc_Gauss2D :236-308
        const float lb = (float)R / 2.0f - 1.5f, ub = (float)R / 2.0f + 1.5f;
        const float smax = fc.MultiEmitterFitEn ? ((float)R / 2.0f) / 2.35f : ((float)R / 1.5f) / 2.35f;
        const float pp = (x[0] * 128.0f) / QE;
        const float bg = (x[4] * 64.0f) / QE;
        float fx = x[1], fy = x[2];
        float sg = sqrtf(0.5f / (x[3] * 0.1f));
        fx = (fx != fx) ? -1.0f : fx;
        fy = (fy != fy) ? -1.0f : fy;
        sg = (sg != sg) ? -1.0f : sg;
        snr = (sqrtf(QE) * pp) / sqrtf(pp + bg);
        const float tp = (((pp * 2.0f) * 3.141593f) * sg) * sg;
        valid = !(bg != bg);
        ok = valid && snr > 4.0f && sg <= smax && sg >= 0.6f && fx > lb && fx < ub && fy > lb && fy < ub;
        row[0] = pp; row[1] = (fx - (float)HALF) + (float)xo; row[2] = (fy - (float)HALF) + (float)yo;
        row[3] = 0.0f; row[4] = sg; row[5] = sg; row[6] = tp; row[7] = bg; row[8] = snr;
        row[9] = 0.0f; row[10] = 0.0f; row[11] = (float)fr;
    } else {
        // bfgsMLELoc_AS3D :237-335
        const float lb = (float)R / 2.0f - 2.5f, ub = (float)R / 2.0f + 2.5f;
        const float smax = fc.MultiEmitterFitEn ? ((float)R / 2.0f) / 2.35f : ((float)R / 1.5f) / 2.35f;
        const float pe = x[0] * 128.0f, be = x[5] * 64.0f;
        float fx = x[1], fy = x[2];
        float sx = sqrtf(0.5f / (x[3] * 0.1f));
        float sy = sqrtf(0.5f / (x[4] * 0.1f));
        fx = (fx != fx) ? -1.0f : fx;
        fy = (fy != fy) ? -1.0f : fy;
        sx = (sx != sx) ? -1.0f : sx;
        sy = (sy != sy) ? -1.0f : sy;
        snr = pe / sqrtf(pe + be);
        const float pp = pe / QE, bg = be / QE;
        const float tp = (((pp * 2.0f) * 3.141593f) * sx) * sy;
        const float dif = (sx * sx) - (sy * sy);
        const float z = (dif >= 0.0f) ? zpoly(fc.pG, dif, fc.ZDepthCorrFactor) : zpoly(fc.pL, dif, fc.ZDepthCorrFactor);
        const float ms = (sx + sy) / 2.0f;
        valid = !(bg != bg);
        ok = valid && snr > 3.5f && ms > 0.8f && ms < smax && fx > lb && fx < ub && fy > lb && fy < ub;
        row[0] = pp; row[1] = (fx - (float)HALF) + (float)xo; row[2] = (fy - (float)HALF) + (float)yo;
        row[3] = z; row[4] = sx; row[5] = sy; row[6] = tp; row[7] = bg; row[8] = snr;
        row[9] = 0.0f; row[10] = 0.0f; row[11] = (float)fr;
    }
    if (!ok) {
#pragma unroll
        for (int k = 0; k < QCS_REC_FLOATS; k++) row[k] = 0.0f;
    }
    float4 *dst = reinterpret_cast<float4 *>(loc + (size_t)roi * QCS_REC_FLOATS);
    dst[0] = make_float4(row[0], row[1], row[2], row[3]);
    dst[1] = make_float4(row[4], row[5], row[6], row[7]);
    dst[2] = make_float4(row[8], row[9], row[10], row[11]);
    if (flag) flag[roi] = (!ok && valid && snr > 6.0f) ? 1 : 0;
}

// Block sums placing the extra emitters (PreEstimation_GS2D_2E :634-681; 3E takes two peaks).
template <int R, int NPK, class Q>
__device__ __forceinline__ void block_peaks(Q q, float (&px)[2], float (&py)[2])
{
    constexpr int HALF = R / 2, L = R / 3 + 1, LH = L / 2;
    const int start[3] = {0, HALF - LH, R - L};
    const float ctr = (float)R / 2.0f;
    const float rpos[3] = {ctr - (float)L / 2.0f, ctr, ctr + (float)L / 2.0f};
    float sum[9];
#pragma unroll
    for (int cnt = 0; cnt < 9; cnt++) {
        float s = 0.0f;
#pragma unroll
        for (int r = 0; r < L; r++)
#pragma unroll
            for (int c = 0; c < L; c++) s = s + q((r + start[cnt / 3]) * R + (c + start[cnt % 3]));
        sum[cnt] = s;
    }
    sum[4] = 0.0f;
#pragma unroll
    for (int k = 0; k < NPK; k++) {
        int mx = 0;
        float mv = sum[0];
#pragma unroll
        for (int cnt = 0; cnt < 9; cnt++)
            if (sum[cnt] > mv) { mx = cnt; mv = sum[cnt]; }
        // mx is per lane: select the block centre without dynamic register indexing
        float xs = rpos[0], ys = rpos[0];
#pragma unroll
        for (int cnt = 0; cnt < 9; cnt++)
            if (cnt == mx) { xs = rpos[cnt % 3]; ys = rpos[cnt / 3]; }
        px[k] = xs;
        py[k] = ys;
#pragma unroll
        for (int cnt = 0; cnt < 9; cnt++)
            if (cnt == mx) sum[cnt] = 0.0f;
    }
}

__device__ __forceinline__ float hypot_fma(float dx, float dy) { return sqrtf(__builtin_fmaf(dx, dx, dy * dy)); }

// Start vector x and weights of the multi-emitter fits; returns the nearest-neighbour distance
// (1000 for the models that do not read it).
template <int MODEL, int R, class Q>
__device__ __forceinline__ float start_me(Q q, const float *__restrict__ wp, const FitConst &fc, float (&x)[Traits<MODEL>::P],
                                          float (&wx)[R], float (&wy)[R])
{
    constexpr int HALF = R / 2;
    const float ctr = (float)R / 2.0f;
    // weights: 2E uses the fixed mask R/1.8/2.35 (R when WLE is off); 3E / AS3D-2E are unweighted
    float nn = 1000.0f;
    if (MODEL == MODEL_2E) {
        float ws = ((float)R / 1.8f) / 2.35f;
        if (fc.WLEEn == 0) ws = (float)R;
        wle_weights<R>(ws, ws, false, wx, wy);
        nn = wp[QCS_WLE_NEARDIST];
    } else {
#pragma unroll
        for (int c = 0; c < R; c++) { wx[c] = 1.0f; wy[c] = 1.0f; }
    }

    // pre-estimation
    float m1 = 0.0f, m2 = 0.0f, m3 = 0.0f, m4 = 0.0f;
#pragma unroll
    for (int k = 0; k < R; k++) {
        m1 = m1 + q(k * R + 0);
        m2 = m2 + q(k * R + R - 1);
        m3 = m3 + q(0 * R + k);
        m4 = m4 + q((R - 1) * R + k);
    }
    m1 = m1 < m2 ? m1 : m2;
    m3 = m3 < m4 ? m3 : m4;
    const float bkg = (MODEL == MODEL_2E) ? (m1 < m3 ? m1 : m3) / (float)R : ((m1 + m3) / 2.0f) / (float)R;
    const float amp = q(HALF * R + HALF) - bkg;
    const float s0 = ((float)R / 2.2f) / 2.35f;
    float px[2], py[2];
    block_peaks<R, (MODEL == MODEL_3E) ? 2 : 1>(q, px, py);
    if (MODEL == MODEL_2E) {
        const float s1 = 1.0f / ((2.0f * s0) * s0);
        x[0] = (0.8f * amp) * 0.0078125f; x[1] = ctr; x[2] = ctr;
        x[3] = (0.8f * amp) * 0.0078125f; x[4] = px[0]; x[5] = py[0];
        x[6] = s1 * 10.0f;
        x[7] = (0.8f * bkg) * 0.015625f;
    } else if (MODEL == MODEL_3E) {
        const float s1 = 1.0f / ((2.0f * s0) * s0);
        x[0] = (0.7f * amp) * 0.0078125f; x[1] = ctr; x[2] = ctr;
        x[3] = (0.7f * amp) * 0.0078125f; x[4] = px[0]; x[5] = py[0];
        x[6] = (0.3f * amp) * 0.0078125f; x[7] = px[1]; x[8] = py[1];
        x[9] = s1 * 10.0f;
        x[10] = (0.8f * bkg) * 0.015625f;
    } else {
        const float s1 = 10.0f * (0.5f / (s0 * s0));
        x[0] = (0.7f * amp) * 0.0078125f; x[1] = ctr; x[2] = ctr; x[3] = s1; x[4] = s1;
        x[5] = (0.7f * amp) * 0.0078125f; x[6] = px[0]; x[7] = py[0]; x[8] = s1; x[9] = s1;
        x[10] = (0.8f * bkg) * 0.015625f;
    }
    return nn;
}

// Emitter selection and acceptance of the multi-emitter fit of list entry j (ROI roi).  The first
// emitter is written to the ROI's row (zeroed when rejected); an accepted second emitter goes to
// second[j] with fs[j] = 1; a rejected first emitter sets ff[j] = 1 (re-route to 3E, or rejected).
template <int MODEL, int R>
__device__ __forceinline__ void finish_me(const float (&x)[Traits<MODEL>::P], const FitConst &fc, float nn, int xo, int yo, int fr,
                                          int roi, int j, float *__restrict__ loc, float *__restrict__ second,
                                          int *__restrict__ fs, int *__restrict__ ff)
{
    using T = Traits<MODEL>;
    constexpr int K = T::K, HALF = R / 2;
    constexpr bool ELLIP = (MODEL == MODEL_AS3D2E);
    const float ctr = (float)R / 2.0f;
    // emitter selection and acceptance
    const float QE = fc.QE;
    const float sqe = sqrtf(QE);
    float pk[K], ex[K], ey[K], sxv[K], syv[K], score[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        pk[k] = (x[T::ia(k)] * 128.0f) / QE;
        ex[k] = x[T::ix(k)];
        ey[k] = x[T::iy(k)];
        sxv[k] = sqrtf(0.5f / (x[T::isx(k)] * 0.1f));
        syv[k] = ELLIP ? sqrtf(0.5f / (x[T::isy(k)] * 0.1f)) : sxv[k];
    }
    const float bg = (x[T::IB] * 64.0f) / QE;
    const bool valid = !(bg != bg);
#pragma unroll
    for (int k = 0; k < K; k++) {
        float cx = ex[k], cy = ey[k];
        if (fabsf(cx - ctr) >= (float)HALF) cx = -100.0f;
        if (fabsf(cy - ctr) >= (float)HALF) cy = -100.0f;
        const float dist = hypot_fma(cx - ctr, cy - ctr);
        score[k] = pk[k] * ((float)R - dist);
    }
    int s0i = 0;
    float sb = score[0];
#pragma unroll
    for (int k = 0; k < K; k++)
        if (score[k] > sb) { s0i = k; sb = score[k]; }
    int s1i = 1 - s0i;
    if (K == 3) {
#pragma unroll
        for (int k = 0; k < K; k++)
            if (k == s0i) score[k] = -100.0f;
        s1i = 0;
        float b1 = score[0];
#pragma unroll
        for (int k = 0; k < K; k++)
            if (score[k] > b1) { s1i = k; b1 = score[k]; }
    }
    // pick the selected emitters' values without dynamic register indexing
    float pp0 = 0, x0 = 0, y0 = 0, sx0 = 0, sy0 = 0, pp1 = 0, x1 = 0, y1 = 0, sx1 = 0, sy1 = 0;
#pragma unroll
    for (int k = 0; k < K; k++) {
        if (k == s0i) { pp0 = pk[k]; x0 = ex[k]; y0 = ey[k]; sx0 = sxv[k]; sy0 = syv[k]; }
        if (k == s1i) { pp1 = pk[k]; x1 = ex[k]; y1 = ey[k]; sx1 = sxv[k]; sy1 = syv[k]; }
    }
    const float tp0 = (((pp0 * 2.0f) * 3.141593f) * sx0) * sy0;
    const float tp1 = (((pp1 * 2.0f) * 3.141593f) * sx1) * sy1;
    const float snr0 = (sqe * pp0) / sqrtf(pp0 + bg);
    const float snr1 = (sqe * pp1) / sqrtf(pp1 + bg);
    const float sep = hypot_fma(x0 - x1, y0 - y1);
    float z0 = 0.0f, z1 = 0.0f;
    bool ok0, ok1;
    if (ELLIP) {
        const float smax = ((float)R / 1.9f) / 2.35f;
        const float ms0 = (sx0 + sy0) / 2.0f, ms1 = (sx1 + sy1) / 2.0f;
        const float d0 = (sx0 * sx0) - (sy0 * sy0), d1 = (sx1 * sx1) - (sy1 * sy1);
        z0 = (d0 >= 0.0f) ? zpoly(fc.pG, d0, fc.ZDepthCorrFactor) : zpoly(fc.pL, d0, fc.ZDepthCorrFactor);
        z1 = (d1 >= 0.0f) ? zpoly(fc.pG, d1, fc.ZDepthCorrFactor) : zpoly(fc.pL, d1, fc.ZDepthCorrFactor);
        ok0 = valid && snr0 > 5.5f && ms0 > 0.6f && ms0 > 0.8f && ms0 <= smax;
        ok1 = sep > 1.5f && snr1 > 5.2f && nn > ctr && ms1 > 0.6f && ms1 > 0.8f && ms1 <= smax && pp1 > pp0 / 3.0f &&
              x1 > 1.0f && y1 > 1.0f && x1 < (float)(R - 1) && y1 < (float)(R - 1);
    } else {
        const float smax = ((float)R / 2.0f) / 2.35f;
        ok0 = valid && snr0 > 5.5f && sx0 > 0.6f && sx0 <= smax;
        const bool nn_ok = (MODEL == MODEL_2E) ? (nn >= ctr) : (nn > ctr);
        ok1 = sep > 1.5f && snr1 > 5.2f && nn_ok && pp1 > pp0 / 2.0f && x1 > 1.0f && y1 > 1.0f && x1 < (float)(R - 1) &&
              y1 < (float)(R - 1);
    }
    float4 *dst = reinterpret_cast<float4 *>(loc + (size_t)roi * QCS_REC_FLOATS);
    if (ok0) {
        dst[0] = make_float4(pp0, (x0 - (float)HALF) + (float)xo, (y0 - (float)HALF) + (float)yo, z0);
        dst[1] = make_float4(sx0, sy0, tp0, bg);
        dst[2] = make_float4(snr0, 0.0f, 0.0f, (float)fr);
    } else {
        dst[0] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        dst[1] = dst[0];
        dst[2] = dst[0];
    }
    const bool wr2 = ok0 && ok1;
    if (wr2) {
        float4 *d2 = reinterpret_cast<float4 *>(second + (size_t)j * QCS_REC_FLOATS);
        d2[0] = make_float4(pp1, (x1 - (float)HALF) + (float)xo, (y1 - (float)HALF) + (float)yo, z1);
        d2[1] = make_float4(sx1, sy1, tp1, bg);
        d2[2] = make_float4(snr1, 0.0f, 0.0f, (float)fr);
    }
    fs[j] = wr2 ? 1 : 0;
    ff[j] = ok0 ? 0 : 1;
}

}  // namespace qcs
