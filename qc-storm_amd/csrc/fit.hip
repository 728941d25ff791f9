// fit.hip -- host side of the reference-schedule fits (dispatch by ROI size and count, the
// multi-emitter cascade) and the CRLB kernel for gfx950.  The fitting kernels are in fit_split.h.
//
// Reference (DLL = MLEbfgs/bfgs_MLE_dll x64/bfgsMLE_dll/bfgsMLE_dll):
//   GaussianCRLB_Calc_top DLL/bfgsMLE_Loc_top/LocPrecCalc_GaussianCRLB.h:64-243
//   BFGS_MLELocalization  DLL/bfgsMLE_Loc_top/bfgs_top.cu:26-204
#include "fit_dev.h"

namespace qcs {

FitConst make_fit_const(const qcs_params &p)
{
    FitConst c;
    c.Offset = p.Offset; c.KAdc = p.KAdc; c.QE = p.QE; c.ReadNoise_e = p.ReadNoise_e; c.PixelSize = p.PixelSize;
    c.MultiEmitterFitEn = p.MultiEmitterFitEn; c.WLEEn = p.WLEEn; c.ZDepthCorrFactor = p.ZDepthCorrFactor;
    c.pG[0] = p.p4_XGY; c.pG[1] = p.p3_XGY; c.pG[2] = p.p2_XGY; c.pG[3] = p.p1_XGY; c.pG[4] = p.p0_XGY;
    c.pL[0] = p.p4_XLY; c.pL[1] = p.p3_XLY; c.pL[2] = p.p2_XLY; c.pL[3] = p.p1_XLY; c.pL[4] = p.p0_XLY;
    return c;
}

// ---------------------------------------------------------------------------------------------
// Diagonal-Fisher CRLB of x and y (GaussianCRLB_Calc_top, LocPrecCalc_GaussianCRLB.h:64-128):
// numeric second derivatives of the model and its log with dh = 0.02 on a G x G grid.
template <int G, bool NARROW>
__device__ __forceinline__ float crlb_psf(int r, int c, float peak, float ix, float iy, float x0, float y0, float B)
{
    const float cy = (float)(r - G / 2), cx = (float)(c - G / 2);
    const float dx = cx - x0, dy = cy - y0;
    const float arg = -__builtin_fmaf(dx * dx, ix, (dy * dy) * iy);
    return __builtin_fmaf(peak, NARROW ? qexpf_nonpos(arg) : qexpf(arg), B);
}

// x / 0.02f.  NARROW: as y = x * 50 corrected by one fma residual, which equals the IEEE quotient
// for x = 0 and every |x| in [1e-30, 1e30] (checked over all floats); the Fisher sums' numerators
// stay there when every model value lies in [1, 1e20].
template <bool NARROW>
__device__ __forceinline__ float div_dh(float x)
{
    if (!NARROW) return x / 0.02f;
    const float y = x * 50.0f;
    return __builtin_fmaf(__builtin_fmaf(-y, 0.02f, x), 50.0f, y);
}

// One grid point's terms of the diagonal Fisher sums of x and y.  NARROW (every model value in
// [1, 1e20], the argument of each exponential <= 0): qexpf_nonpos, qlogf_normal and div_dh<true>
// give the same bits as the general forms there.
template <int G, bool NARROW>
__device__ __forceinline__ void crlb_term(int r, int c, float peak, float ix, float iy, float be, float &tx, float &ty)
{
    const float dh = 0.02f;
    const float xp = 0.0f + dh, xn = (0.0f + dh) - 2.0f * dh;
    auto lg = [](float m) { return NARROW ? qlogf_normal(m) : qlogf(m); };
    const float m0 = crlb_psf<G, NARROW>(r, c, peak, ix, iy, 0.0f, 0.0f, be);
    const float l0 = lg(m0);
    {
        const float mp = crlb_psf<G, NARROW>(r, c, peak, ix, iy, xp, 0.0f, be);
        const float mn = crlb_psf<G, NARROW>(r, c, peak, ix, iy, xn, 0.0f, be);
        const float d2 = div_dh<NARROW>(div_dh<NARROW>(__builtin_fmaf(-2.0f, m0, mp) + mn));
        const float d2l = div_dh<NARROW>(div_dh<NARROW>(__builtin_fmaf(-2.0f, l0, lg(mp)) + lg(mn)));
        tx = __builtin_fmaf(-m0, d2l, d2);
    }
    {
        const float mp = crlb_psf<G, NARROW>(r, c, peak, ix, iy, 0.0f, xp, be);
        const float mn = crlb_psf<G, NARROW>(r, c, peak, ix, iy, 0.0f, xn, be);
        const float d2 = div_dh<NARROW>(div_dh<NARROW>(__builtin_fmaf(-2.0f, m0, mp) + mn));
        const float d2l = div_dh<NARROW>(div_dh<NARROW>(__builtin_fmaf(-2.0f, l0, lg(mp)) + lg(mn)));
        ty = __builtin_fmaf(-m0, d2l, d2);
    }
}

// sum += v of lane K of the 16, K = 0 .. 15 in turn (row_newbcast)
template <int K>
__device__ __forceinline__ void crlb_add16(float v, float &sum)
{
    sum = sum + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + K, 0xf, 0xf, true));
    if constexpr (K < 15) crlb_add16<K + 1>(v, sum);
}

// The sums over the G x G grid in raster order.  L = 1: a lane takes every point.  L = 16: lane l of the 16
// takes points 16 t + l, and all add the 16 terms of a round in the same order (points past the grid
// add 0 to a sum that is never -0).
template <int G, int L, bool NARROW>
__device__ __forceinline__ void crlb_fisher(float peak, float ix, float iy, float be, float &fx, float &fy)
{
    fx = 0.0f;
    fy = 0.0f;
    float tx, ty;
    if constexpr (L == 1) {
        for (int r = 0; r < G; r++) {
#pragma unroll
            for (int c = 0; c < G; c++) {
                crlb_term<G, NARROW>(r, c, peak, ix, iy, be, tx, ty);
                fx = fx + tx;
                fy = fy + ty;
            }
        }
    } else {
        static_assert(L == 16, "a DPP row");
        for (int p = threadIdx.x & 15; (p & ~15) < G * G; p += 16) {
            const int q = min(p, G * G - 1), r = q / G;
            crlb_term<G, NARROW>(r, q - r * G, peak, ix, iy, be, tx, ty);
            crlb_add16<0>(p < G * G ? tx : 0.0f, fx);
            crlb_add16<0>(p < G * G ? ty : 0.0f, fy);
        }
    }
}

// What bounds a small call is the chain of G^2 points of some 200 instructions, the same for one row as
// for a lane's worth of rows on every SIMD; with 16 lanes a row it is a sixteenth, and the ordered
// sums are 15% more instructions (crlb_launch has both sides).
template <int G, int L>
__global__ void __launch_bounds__(64) crlb_kernel(float *__restrict__ loc, int n, const int *__restrict__ n_dev, float QE,
                                                  float RN, float PS)
{
    const int i = blockIdx.x * (64 / L) + (int)threadIdx.x / L;
    if (n_dev) n = *n_dev;
    if (i >= n) return;
    float *row = loc + (size_t)i * QCS_REC_FLOATS;
    float te = row[6] * QE, be = row[7] * QE;
    const float sx = row[4], sy = row[5];
    float stdx = 100.0f, stdy = 100.0f;
    if (te > 1.0f && be > 1.0f && (double)sx > 0.1 && (double)sy > 0.1 && sx < 10.0f && sy < 10.0f) {
        be = __builtin_fmaf(be, QE, RN * RN) / QE;
        const float pi = 3.141592654f;
        const float peak = (1.0f / (((2.0f * pi) * sx) * sy)) * te;
        const float ix = 1.0f / ((2.0f * sx) * sx);
        const float iy = 1.0f / ((2.0f * sy) * sy);
        float fx, fy;
        // model values lie in [be, peak + be] with be > 1
        if (peak + be < 1e20f) crlb_fisher<G, L, true>(peak, ix, iy, be, fx, fy);
        else crlb_fisher<G, L, false>(peak, ix, iy, be, fx, fy);
        fx = (fx == 0.0f) ? 1.0f : fx;
        fy = (fy == 0.0f) ? 1.0f : fy;
        stdx = sqrtf(1.0f / fx) * PS;
        stdy = sqrtf(1.0f / fy) * PS;
    }
    if (threadIdx.x % L != 0) return;
    row[9] = stdx;
    row[10] = stdy;
}

// ---------------------------------------------------------------------------------------------
// Lanes per ROI of a one-emitter call of n ROIs (fit_split.h).  A group of G lanes shortens the
// serial chain of loss evaluations and puts G times as many waves on the chip, but repeats the
// parameter arithmetic in every lane; so small calls take the widest group that pays, and each
// line below lies where the narrower one measured faster (us per call with its CRLB, wide / narrow):
//   5x5   8 lanes to 24,000 ROIs (143 / 151 at 20,000, 214 / 203 at 40,000), 4 to 64,000 (203 / 214,
//         296 / 273 at 80,000), 2 to 240,000 (430 / 501 at 160,000; elliptical 1240 / 1068 at 320,000), then 1
//   7x7   8 to 24,000 (177 / 183, 270 / 258), 4 to 400,000 (1274 / 1343 at 320,000, 3829 / 3614 at
//         1,000,000; elliptical to 200,000: 987 / 1115 at 160,000, 1870 / 1726 at 320,000), then 1
//   9x9   16 to 28,000 (270 / 321, 471 / 446), 4 to 110,000 (688 / 744, 1247 / 1151), then 2
//   11x11 16 to 28,000 (311 / 333, 545 / 539), then 4 (two rows' worth of pixels per lane and more
//         hold the other sizes back: 2991 against 4082 with 2 lanes at 320,000)
//   13, 15  16 at every size (13: 1150 against 1364 and 1799 with 8 and 4 at 80,000)
//   17x17 16 to 20,000 (1082 / 1346, 1842 / 1840 at 40,000), then 8
//
// With the hardware exp and log (fast) an evaluation is half as long, the lines lie lower, and while a launch
// is less than one wave per SIMD (65,536 lanes) the group can be as wide as that allows (wide / narrow):
//   5x5   8 to 8,192 (65 / 73 at 5,000), 4 to 16,384 (76 / 89 at 10,000), 2 to 32,768 (103 / 126 at 30,000),
//         then 1 (147 against 171 at 60,000, 398 against 488 at 240,000)
//   7x7   8 to 8,192 (72 / 81 at 5,000), 4 to 36,000 (145 / 184 at 30,000, 193 / 191 at 40,000), then 1
//         (205 against 251 at 60,000, 759 against 1002 at 320,000) but for the start of its second round
//         (80,000: 311 / 344)
//   9x9   16 to 6,000 (102 / 114 at 5,000, 140 / 115 at 10,000), 4 to 16,384 (115 / 161 at 10,000,
//         202 / 168 at 20,000), 2 to 36,000 (181 / 277 at 30,000, 306 / 284 at 40,000) and from 65,536 to
//         100,000 (452 / 498 at 80,000), else 1 (1114 against 1345 at 320,000); elliptical 2 to 200,000
//         (960 / 1072 at 160,000, 1446 / 1372 at 240,000)
//   13x13 16 to 26,000 (285 / 314 at 20,000, 424 / 333 at 30,000), then 2 (559 against 624 and 755 with 4 and
//         16 at 60,000, 1233 against 1383 and 1709 at 160,000); elliptical 4 (486 against 605 with 2 at
//         30,000, 1956 against 2006 at 160,000)
static int lanes_1e(int model, int R, int n, bool fast)
{
    const bool el = model == MODEL_AS3D;
    if (fast) {
        switch (R) {
        case 5: return n <= 8192 ? 8 : n <= 16384 ? 4 : n <= 32768 ? 2 : 1;
        case 7: return n <= 8192 ? 8 : n <= 36000 || (n > 65536 && n <= 100000) ? 4 : 1;
        case 9: return n <= 6000 ? 16 : n <= 16384 ? 4 : (el ? n <= 200000 : n <= 36000 || (n > 65536 && n <= 100000)) ? 2 : 1;
        case 13: return n <= 26000 ? 16 : el ? 4 : 2;
        default: break;
        }
    }
    switch (R) {
    case 5: return n <= 24000 ? 8 : n <= 64000 ? 4 : n <= 240000 ? 2 : 1;
    case 7: return n <= 24000 ? 8 : n <= (el ? 200000 : 400000) ? 4 : 1;
    case 9: return n <= 28000 ? 16 : n <= 110000 ? 4 : 2;
    case 11: return n <= 28000 ? 16 : 4;
    case 17: return n <= 20000 ? 16 : 8;
    default: return 16;
    }
}

// The same for the multi-emitter stages, by the cascade's ROI count (a stage fits a part of them;
// us per cascade, wide / narrow): 8 lanes to 50,000 at 5x5 and 7x7 (7x7: 1519 / 1770 at 60,000, 3631 /
// 3099 at 200,000; elliptical 833 / 909 at 20,000, 1806 / 1570 at 60,000), 16 to 100,000 at 9x9 and 11x11
// (9x9: 2318 / 3282 at 60,000, 6284 / 5864 at 200,000; elliptical to 30,000: 1121 / 1345 at 20,000,
// 2408 / 1839 at 60,000), then 4; 16 at 13x13 (3792 against 8780 at 60,000).
static int lanes_me(int model, int R, int n)
{
    if (R <= 7) return n <= 50000 ? 8 : 4;
    if (R <= 11) return n <= (model == MODEL_AS3D2E ? 30000 : 100000) ? 16 : 4;
    return 16;
}

int fit_launch_1e(const qcs_params &p, const uint16_t *d_rois, const float *d_wle, const int *d_idx, int n,
                  const int *d_n, float *d_loc, int *d_flag, hipStream_t s)
{
    if (n <= 0) return QCS_OK;
    const int R = p.ROISize, model = (p.LocType == QCS_LOCTYPE_AS3D) ? MODEL_AS3D : MODEL_GS2D;
    const SplitArgs a{d_rois, d_wle, d_idx, n, d_n, d_loc, nullptr, d_flag, nullptr};
    const bool fast = p.FitMath == QCS_MATH_FAST;
    return fit_split_1e(model, R, lanes_1e(model, R, n, fast), fast, a, make_fit_const(p), s);
}

// multi-emitter stage over list[j], j < *n_dev (grid sized for n_max)
int fit_launch_me(const qcs_params &p, int model, const uint16_t *d_rois, const float *d_wle, const int *d_list, int n_max,
                  const int *d_n, float *d_loc, float *d_second, int *d_fs, int *d_ff, hipStream_t s)
{
    if (n_max <= 0) return QCS_OK;
    const SplitArgs a{d_rois, d_wle, d_list, n_max, d_n, d_loc, d_second, d_fs, d_ff};
    return fit_split_me(model, p.ROISize, lanes_me(model, p.ROISize, n_max), p.FitMath == QCS_MATH_FAST, a, make_fit_const(p), s);
}

int crlb_launch(const qcs_params &p, float *d_loc, int n, const int *d_n, hipStream_t s)
{
    if (n <= 0) return QCS_OK;
    const bool el = p.LocType == QCS_LOCTYPE_AS3D;
    // us per call, 16 lanes / one lane: 9 x 9 11 / 55 at 4,000 rows, 17 / 56 at 20,480, 39 / 55 at 64,000,
    // 58 / 58 at 100,000, 91 / 59 at 160,000; 15 x 15 24 / 145, 37 / 145, 87 / 140, 127 / 150, 196 / 151
    const bool split = n <= (el ? 110000 : 90000);
    const dim3 grid(split ? (n + 3) / 4 : (n + 63) / 64), block(64);
    const float q = p.QE, rn = p.ReadNoise_e, ps = p.PixelSize;
    if (el && split) hipLaunchKernelGGL((crlb_kernel<15, 16>), grid, block, 0, s, d_loc, n, d_n, q, rn, ps);
    else if (el) hipLaunchKernelGGL((crlb_kernel<15, 1>), grid, block, 0, s, d_loc, n, d_n, q, rn, ps);
    else if (split) hipLaunchKernelGGL((crlb_kernel<9, 16>), grid, block, 0, s, d_loc, n, d_n, q, rn, ps);
    else hipLaunchKernelGGL((crlb_kernel<9, 1>), grid, block, 0, s, d_loc, n, d_n, q, rn, ps);
    QCS_HIP(hipGetLastError());
    return QCS_OK;
}

// ---------------------------------------------------------------------------------------------
// Multi-emitter cascade (LDLocData_TypeDef::BFGS_MLELocalization, bfgs_top.cu:26-204, with
// gpuMoleculeFitClasify, bfgs_top_MoleculeClasify.cu:26-92).  The reference builds its lists
// with atomic counters (arbitrary order); here every list is a stable compaction (exclusive
// scan of flags), so list order and the rows appended for second emitters are deterministic:
//   1E list  = ROIs with WLE type <= WLEFit, in index order
//   2E list  = ROIs with WLE type MultiFit, in index order, then rejected 1E fits with SNR > 6
//   3E list  = rejected first emitters of the 2E stage, in 2E-list order (2D only)
//   appended = accepted second emitters of the 2E stage, then of the 3E stage, in list order
// All counts stay on the device; one read-back at the end.  The list building is launches, not
// work: 19 of them beside the fits (13 up to 16,384 ROIs), where a clear, a scan, a count and a tail
// clear per flag array were 48 (20,480 ROIs: 1056 -> 959 us).

// cnt layout: [0] n1, [1] n2 classified, [2] n2 total, [3] n3, [4] seconds from 2E, [5] seconds
// from 3E, [6] rejected, [7] rows, [8] loc_cap
__global__ void cascade_classify_kernel(const float *__restrict__ wle, int n, int *__restrict__ f1, int *__restrict__ rr,
                                        int *__restrict__ cnt, int loc_cap)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x < 16) cnt[threadIdx.x] = threadIdx.x == 8 ? loc_cap : 0;
    if (i >= n) return;
    const int mt = (int)wle[(size_t)i * QCS_WLE_FLOATS + QCS_WLE_FLUOTYPE];
    f1[i] = (mt <= QCS_MOLTYPE_WLEFIT) ? 1 : 0;
    rr[i] = 0;
}

// the 1E list and the classified part of the 2E list (the others), both in index order, with their counts
__global__ void __launch_bounds__(256) cascade_lists_kernel(const int *__restrict__ f1, const int *__restrict__ offs, int n,
                                                            int *__restrict__ list1, int *__restrict__ list2, int *__restrict__ cnt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) cnt[1] = cnt[2] = n - cnt[0];
    if (i >= n) return;
    const int o = offs[i];
    if (f1[i]) list1[o] = i;
    else list2[i - o] = i;
}

__global__ void cascade_rows_kernel(int n, int *__restrict__ cnt)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    int extra = cnt[4] + cnt[5];
    const int room = cnt[8] - n;
    extra = extra < room ? extra : room;
    cnt[7] = n + extra;
}

// append second-emitter rows: row = n + base + offs[j] for flagged j (bounded by the capacity)
__global__ void __launch_bounds__(256) append_kernel(const int *__restrict__ flags, const int *__restrict__ offs,
                                                     const int *__restrict__ n_list, const float *__restrict__ second,
                                                     const int *__restrict__ cnt, int base_slot, int n, int loc_cap,
                                                     float *__restrict__ loc)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= *n_list || !flags[j]) return;
    const int base = base_slot >= 0 ? cnt[base_slot] : 0;
    const int row = n + base + offs[j];
    if (row >= loc_cap) return;
    const float4 *src = reinterpret_cast<const float4 *>(second + (size_t)j * QCS_REC_FLOATS);
    float4 *dst = reinterpret_cast<float4 *>(loc + (size_t)row * QCS_REC_FLOATS);
    dst[0] = src[0];
    dst[1] = src[1];
    dst[2] = src[2];
}

size_t cascade_scratch_bytes(int n)
{
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t ni = (size_t)(n > 0 ? n : 1);
    return up(64) + 3 * up(sizeof(int) * ni) + up(sizeof(int) * (6 * ni + scan_tile_count(ni) + 1)) +
           up(sizeof(float) * QCS_REC_FLOATS * 2 * ni);
}

void cascade_carve(void *base, int n, CascadeBufs &b)
{
    auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t ni = (size_t)(n > 0 ? n : 1);
    char *p = static_cast<char *>(base);
    b.cnt = reinterpret_cast<int *>(p);
    p += up(64);
    b.list1 = reinterpret_cast<int *>(p);
    p += up(sizeof(int) * ni);
    b.list2 = reinterpret_cast<int *>(p);
    p += up(sizeof(int) * ni);
    b.list3 = reinterpret_cast<int *>(p);
    p += up(sizeof(int) * ni);
    b.flag = reinterpret_cast<int *>(p);
    p += up(sizeof(int) * (6 * ni + scan_tile_count(ni) + 1));
    b.rows = reinterpret_cast<float *>(p);
}

int fit_cascade_launch(const qcs_params &p, Timer *tm, const uint16_t *d_rois, const float *d_wle, int n, float *d_loc,
                       int loc_cap, const CascadeBufs &b, hipStream_t s)
{
    const bool as3d = (p.LocType == QCS_LOCTYPE_AS3D);
    int rc;
    int *list1 = b.list1, *list2 = b.list2, *list3 = b.list3;
    int *f1 = b.flag, *rr = f1 + n, *fs2 = rr + n, *ff2 = fs2 + n, *fs3 = ff2 + n;
    int *offs = fs3 + n, *tsum = offs + n;
    int *ff3 = f1;   // f1 is free again once the 1E list is built
    float *sec2 = b.rows, *sec3 = sec2 + (size_t)QCS_REC_FLOATS * n;
    int *cnt = b.cnt;
    const dim3 g((n + 255) / 256);
    // stage timers are recorded only when a timer is given and enabled
    auto tb = [&](hipEvent_t *ev) { *ev = nullptr; return tm ? timer_begin(*tm, s, ev) : QCS_OK; };
    auto te = [&](int cat, hipEvent_t ev) { return tm ? timer_end(*tm, cat, s, ev, n) : QCS_OK; };

    hipLaunchKernelGGL(cascade_classify_kernel, g, dim3(256), 0, s, d_wle, n, f1, rr, cnt, loc_cap);
    if ((rc = scan_exclusive(f1, n, offs, tsum, s, nullptr, cnt + 0))) return rc;
    hipLaunchKernelGGL(cascade_lists_kernel, g, dim3(256), 0, s, f1, offs, n, list1, list2, cnt);
    // one-emitter stage; rejected fits with SNR > 6 flag themselves in rr
    hipEvent_t ev;
    if ((rc = tb(&ev))) return rc;
    if ((rc = fit_launch_1e(p, d_rois, d_wle, list1, n, cnt + 0, d_loc, rr, s))) return rc;
    if ((rc = te(TM_FIT1E, ev))) return rc;
    // re-routed ROIs join the 2E list after the classified ones, in index order
    if ((rc = scan_exclusive(rr, n, offs, tsum, s, nullptr, cnt + 2, true)) ||
        (rc = compact_scatter(rr, offs, n, nullptr, cnt + 1, 0, list2, s)))
        return rc;
    // two-emitter stage (every entry of its list writes fs2 and ff2)
    if ((rc = tb(&ev))) return rc;
    if ((rc = fit_launch_me(p, as3d ? MODEL_AS3D2E : MODEL_2E, d_rois, d_wle, list2, n, cnt + 2, d_loc, sec2, fs2, ff2, s)))
        return rc;
    if ((rc = te(TM_FITME, ev))) return rc;
    if ((rc = scan_exclusive(fs2, n, offs, tsum, s, cnt + 2, cnt + 4))) return rc;
    hipLaunchKernelGGL(append_kernel, g, dim3(256), 0, s, fs2, offs, cnt + 2, sec2, cnt, -1, n, loc_cap, d_loc);
    if ((rc = scan_exclusive(ff2, n, offs, tsum, s, cnt + 2, cnt + (as3d ? 6 : 3)))) return rc;
    if (!as3d) {
        if ((rc = compact_scatter(ff2, offs, n, list2, nullptr, 0, list3, s, cnt + 2))) return rc;
        if ((rc = tb(&ev))) return rc;
        if ((rc = fit_launch_me(p, MODEL_3E, d_rois, d_wle, list3, n, cnt + 3, d_loc, sec3, fs3, ff3, s))) return rc;
        if ((rc = te(TM_FITME, ev))) return rc;
        if ((rc = scan_exclusive(fs3, n, offs, tsum, s, cnt + 3, cnt + 5))) return rc;
        hipLaunchKernelGGL(append_kernel, g, dim3(256), 0, s, fs3, offs, cnt + 3, sec3, cnt, 4, n, loc_cap, d_loc);
        if ((rc = scan_exclusive(ff3, n, offs, tsum, s, cnt + 3, cnt + 6))) return rc;
    }
    hipLaunchKernelGGL(cascade_rows_kernel, dim3(1), dim3(1), 0, s, n, cnt);
    QCS_HIP(hipGetLastError());
    if ((rc = tb(&ev))) return rc;
    if ((rc = crlb_launch(p, d_loc, loc_cap, cnt + 7, s))) return rc;
    return te(TM_CRLB, ev);
}

int fit_cascade(qcs_ctx *c, const uint16_t *d_rois, const float *d_wle, int n, float *d_loc, int loc_cap, int *n_rows,
                hipStream_t s)
{
    const qcs_params &p = c->p;
    const bool as3d = (p.LocType == QCS_LOCTYPE_AS3D);
    int rc;
    if ((rc = c->fit_flag.ensure(cascade_scratch_bytes(n))) || (rc = c->pin_cnt.ensure(64))) return rc;
    CascadeBufs b;
    cascade_carve(c->fit_flag.ptr, n, b);
    if ((rc = fit_cascade_launch(p, &c->timer, d_rois, d_wle, n, d_loc, loc_cap, b, s))) return rc;
    int *cnt = b.cnt;
    int *h = c->pin_cnt.as<int>();
    QCS_HIP(hipMemcpyAsync(h, cnt, 16 * sizeof(int), hipMemcpyDeviceToHost, s));
    QCS_HIP(hipStreamSynchronize(s));
    qcs_fit_stats &st = c->stats;
    st.n_in = n;
    st.n_single = h[0];
    st.n_2e = h[2];
    st.n_3e = h[3];
    st.n_rejected = h[6];
    st.n_rows = h[7];
    // FitRatio_* as bfgs_top.cu:64-173
    const float nd = (float)(n < 1 ? 1 : n);
    st.FitRatio_1E = (float)h[0] / nd;
    st.FitRatio_2E = (float)h[2] / nd;
    st.FitRatio_3E = (float)h[3] / nd;
    st.FitRatio_Final_1E = (float)(h[0] - (h[2] - h[1])) / nd;
    if (!as3d) {
        st.FitRatio_Final_2E = (float)(h[2] - h[3]) / nd;
        st.FitRatio_Final_3E = (float)(h[3] - h[6]) / nd;
    } else {
        st.FitRatio_Final_2E = (float)(h[2] - h[6]) / nd;
        st.FitRatio_Final_3E = 0.0f;
    }
    st.FitRatio_Final_4E = (float)h[6] / nd;
    if (n_rows) *n_rows = h[7];
    return QCS_OK;
}

}  // namespace qcs
