// fit_split.h -- reference-schedule BFGS Poisson-MLE fits for gfx950, one ROI split over a group of
// G = 1, 2, 4, 8 or 16 lanes.
//
// The schedule (gradient, 2 + 10 line-search evaluations, step, gradient, BFGS update;
// DLL/bfgsMLE_Loc_LD/bfgsMLE_GS2D_core.h:313-426) does not depend on the data: 176 loss
// evaluations for the 2D one-emitter model, up to 544 for three emitters, each waiting for the one
// before it but within a gradient.  A call that cannot fill the chip with one ROI per lane is
// bound by that chain, and a model whose pixels and matrix do not fit a lane's registers by
// occupancy.  So a group of G lanes holds an ROI, RL = ceil(R / G) rows per lane: q, the loss's
// data term and the row factors of its own rows, and RL of the column exponentials; column
// exponentials and row sums go round the group by DPP.  Parameters, gradient and direction are
// held by every lane of the group; row r of the inverse Hessian is on lane r % G.  With G = 1 it is
// one ROI per lane, for calls that fill the chip.  Every operation, and the order of every sum
// (rows in column order, then rows in ascending order), is the same for every G, so the rows are
// the same bit for bit.
//
// The loss: Poisson deviance of I = sum_k A_k exp(-(sx_k dx^2 + sy_k dy^2)) + B evaluated separably
// (one exp per emitter and ROI row / column).  The pixel term w (I - q - q (log I - log q)) is
// formed as fma(-q, log I + c, I) with c = 1 - log q and the log fused with c (logtabb_u,
// logtab_u); the weighted sum runs as sum_r wy[r] sum_c wx[c] t(r, c).  The loss clamps its
// argument in place, as the reference's does.
//
// Range check: with positions below 2^60 in magnitude and finite widths each exp term lies in
// [0, 1], so I lies in [B, sum of the amplitudes + B].  Multi-emitter models need B in
// [2^-126, 2^124] and amplitudes at most 2^124 (I a positive normal float); the one-emitter models
// use the binade table log and need B and A within [2^-10.5, 2^18.5] so that I stays inside the
// table.  A group that fails it (a line-search probe gone far out, a background at zero) takes the
// _any form of the log, whose range and special-value handling gives the value the CPU oracle
// computes.
//
// What bounds it: many ROIs, VALU issue (7x7 2D at G = 1: 163,800 VALU instructions per fit, 19 per pixel
// of an evaluation with everything; 210,200 at G = 4); few, the latency of the chain.  Measured, us per call
// with CRLB, against one ROI per lane with a uniform loop over the evaluations:
//   7x7 2D     20,480 ROIs 498 -> 173 (G = 8), 1,000,003 ROIs 4030 -> 3670 (G = 1)
//   9x9 3D     5,377 ROIs 1445 -> 191 (G = 16);  11x11 2D 100,001 ROIs 3090 -> 1090 (G = 4)
//   cascade    20,480 ROIs of dense frames, 7x7: 4850 -> 950 (G = 8)
#pragma once
#include <type_traits>
#include "fit_dev.h"

namespace qcs {

// f(integral_constant<int, i>) for i = B .. E - 1
template <int B, int E, class F>
__device__ __forceinline__ void fs_for(F &&f)
{
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        fs_for<B + 1, E>(f);
    }
}

// Value of lane J of each group of G lanes, in every lane of the group.
template <int G, int J>
__device__ __forceinline__ float group_bcast(float v)
{
    static_assert(G == 1 || G == 2 || G == 4 || G == 8 || G == 16, "group of 2, 4, 8 or 16 lanes");
    static_assert(J >= 0 && J < G, "lane of the group");
    const int i = __float_as_int(v);
    if constexpr (G == 1) {
        return v;
    } else if constexpr (G == 2) {
        return __int_as_float(__builtin_amdgcn_mov_dpp(i, J * 0x55 + 0xa0, 0xf, 0xf, true));   // quad_perm J,J,2+J,2+J
    } else if constexpr (G == 4) {
        return __int_as_float(__builtin_amdgcn_mov_dpp(i, J * 0x55, 0xf, 0xf, true));          // quad_perm J,J,J,J
    } else if constexpr (G == 16) {
        return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0x150 + J, 0xf, 0xf, true));         // row_newbcast:J
    } else {
        // lanes 0-7 of a DPP row take lane J, lanes 8-15 (banks 2 and 3) lane 8 + J
        const int lo = __builtin_amdgcn_mov_dpp(i, 0x150 + J, 0xf, 0xf, true);
        return __int_as_float(__builtin_amdgcn_update_dpp(lo, i, 0x150 + 8 + J, 0xf, 0xc, false));
    }
}

template <int MODEL, int R, int G> struct SplitShape {
    static constexpr int RL = (R + G - 1) / G;   // rows (and column exponentials) per lane
};

// Row sums of the lane's rows.
template <int MODEL, int R, int G, bool FAST, bool SAFE>
__device__ __forceinline__ void split_rows(const float (&q)[SplitShape<MODEL, R, G>::RL][R], const float (&c1)[SplitShape<MODEL, R, G>::RL][R],
                                           const float (&wx)[R], const float (&ex)[Traits<MODEL>::K][R],
                                           const float (&ay)[Traits<MODEL>::K][SplitShape<MODEL, R, G>::RL], float b, const float2 *lt,
                                           float (&acc)[SplitShape<MODEL, R, G>::RL])
{
    using T = Traits<MODEL>;
    constexpr int K = T::K;
#pragma unroll
    for (int m = 0; m < SplitShape<MODEL, R, G>::RL; m++) {
        float s = 0.0f;
#pragma unroll
        for (int c = 0; c < R; c++) {
            float I;
            if (K == 1) {
                I = __builtin_fmaf(ay[0][m], ex[0][c], b);
            } else {
                I = ay[0][m] * ex[0][c];
#pragma unroll
                for (int k = 1; k < K; k++) I = __builtin_fmaf(ay[k][m], ex[k][c], I);
                I = I + b;
            }
            const float cc = c1[m][c];
            float u;
            if (FAST) u = flogf(I) + cc;
            else if (K == 1) u = SAFE ? logtabb_u_any(I, cc, lt) : logtabb_u(I, cc, lt);
            else u = SAFE ? logtab_u_any(I, cc, lt) : logtab_u(I, cc, lt);
            const float t = __builtin_fmaf(-q[m][c], u, I);
            s = T::WEIGHTED ? __builtin_fmaf(wx[c], t, s) : s + t;
        }
        acc[m] = s;
    }
}

// Amplitudes, column exponentials and row factors of the model at p, over the group's lanes; returns
// whether the fast log holds for every model value (the range check above).
template <int MODEL, int R, int G, bool FAST>
__device__ __forceinline__ bool split_model(const float (&pos)[SplitShape<MODEL, R, G>::RL], const float (&p)[Traits<MODEL>::P],
                                            float (&ex)[Traits<MODEL>::K][R], float (&ay)[Traits<MODEL>::K][SplitShape<MODEL, R, G>::RL],
                                            float &b)
{
    using T = Traits<MODEL>;
    constexpr int K = T::K, RL = SplitShape<MODEL, R, G>::RL;
    b = p[T::IB] * 64.0f;
    constexpr float BLO = (K == 1) ? kLogTabBLo : 1.17549435082228751e-38f;
    constexpr float AHI = (K == 1) ? kLogTabBHi * 0.125f : 0x1p124f;
    bool inrange = (b >= BLO) && (b <= AHI);
#pragma unroll
    for (int k = 0; k < K; k++) {
        const float a = p[T::ia(k)] * 128.0f;
        const float sx = p[T::isx(k)] * 0.1f;
        const float sy = p[T::isy(k)] * 0.1f;
        inrange = inrange && (a <= AHI) && (sx <= 0x1p124f) && (sy <= 0x1p124f) &&
                  (__builtin_fabsf(p[T::ix(k)]) <= 0x1p60f) && (__builtin_fabsf(p[T::iy(k)]) <= 0x1p60f);
        float own[RL];
#pragma unroll
        for (int m = 0; m < RL; m++) {
            const float dx = pos[m] - p[T::ix(k)];
            own[m] = vexp_nonpos<FAST>((-(dx * dx)) * sx);
            const float dy = pos[m] - p[T::iy(k)];
            ay[k][m] = a * vexp_nonpos<FAST>((-(dy * dy)) * sy);
        }
        fs_for<0, R>([&](auto C) {
            constexpr int c = decltype(C)::value;
            ex[k][c] = group_bcast<G, c / RL>(own[c % RL]);
        });
    }
    return inrange;
}

// total of the group's row sums, rows in ascending order
template <int MODEL, int R, int G>
__device__ __forceinline__ float split_total(const float (&wy)[R], const float (&acc)[SplitShape<MODEL, R, G>::RL])
{
    using T = Traits<MODEL>;
    constexpr int RL = SplitShape<MODEL, R, G>::RL;
    float total = 0.0f;
    fs_for<0, R>([&](auto Rc) {
        constexpr int r = decltype(Rc)::value;
        const float a = group_bcast<G, r / RL>(acc[r % RL]);
        total = T::WEIGHTED ? __builtin_fmaf(wy[r], a, total) : total + a;
    });
    return total;
}

// The loss at p, which it clamps in place.  pos: the lane's row and column centres.
template <int MODEL, int R, int G, bool FAST>
__device__ __forceinline__ float split_loss(const float (&q)[SplitShape<MODEL, R, G>::RL][R], const float (&c1)[SplitShape<MODEL, R, G>::RL][R],
                                            const float (&wx)[R], const float (&wy)[R], const float (&pos)[SplitShape<MODEL, R, G>::RL],
                                            float (&p)[Traits<MODEL>::P], const float2 *lt)
{
    using T = Traits<MODEL>;
#pragma unroll
    for (int i = 0; i < T::P; i++) p[i] = (p[i] < T::CLAMP) ? T::CLAMP : p[i];
    float ex[T::K][R], ay[T::K][SplitShape<MODEL, R, G>::RL], acc[SplitShape<MODEL, R, G>::RL], b;
    const bool inrange = split_model<MODEL, R, G, FAST>(pos, p, ex, ay, b);
    if (FAST || inrange) split_rows<MODEL, R, G, FAST, false>(q, c1, wx, ex, ay, b, lt, acc);
    else split_rows<MODEL, R, G, FAST, true>(q, c1, wx, ex, ay, b, lt, acc);
    return split_total<MODEL, R, G>(wy, acc);
}

// Central differences at x (NumericalGradient: x_k - 0.002, then + 0.004, then - 0.002, the loss
// clamping its argument in place).  Probe k changes one parameter, so in straight-line code the
// factors of the others are computed once: 13 sets of exponentials instead of 20 for the 2D
// model.  That code has no range check per probe; it runs when every probe of every lane of
// the wave is inside the fast log's range, else the loop with the check per probe does.
template <int MODEL, int R, int G, bool FAST>
__device__ __forceinline__ void split_gradient(const float (&q)[SplitShape<MODEL, R, G>::RL][R], const float (&c1)[SplitShape<MODEL, R, G>::RL][R],
                                               const float (&wx)[R], const float (&wy)[R], const float (&pos)[SplitShape<MODEL, R, G>::RL],
                                               const float (&x)[Traits<MODEL>::P], float (&g)[Traits<MODEL>::P], const float2 *lt)
{
    using T = Traits<MODEL>;
    constexpr int P = T::P, K = T::K;
    float t[P];
#pragma unroll
    for (int k = 0; k < P; k++) t[k] = x[k];
    bool flat = true;
    if constexpr (!FAST) {
        constexpr float AHI = ((K == 1) ? kLogTabBHi * 0.125f : 0x1p124f) * 0.0009765625f;
        bool ok = t[T::IB] >= 0.004f && t[T::IB] <= AHI;
#pragma unroll
        for (int k = 0; k < K; k++)
            ok = ok && t[T::ia(k)] <= AHI && t[T::isx(k)] <= 0x1p120f && t[T::isy(k)] <= 0x1p120f && __builtin_fabsf(t[T::ix(k)]) <= 0x1p59f &&
                 __builtin_fabsf(t[T::iy(k)]) <= 0x1p59f;
        flat = __all(ok);
    }
    if (flat) {
        auto clamp = [&](int k) { t[k] = (t[k] < T::CLAMP) ? T::CLAMP : t[k]; };
#pragma unroll
        for (int k = 1; k < P; k++) clamp(k);
        fs_for<0, P>([&](auto Gi) {
            constexpr int gi = decltype(Gi)::value;
            float L[2];
            fs_for<0, 2>([&](auto Hc) {
                constexpr int h = decltype(Hc)::value;
                t[gi] = t[gi] + (h ? 0.004f : -0.002f);
                clamp(gi);
                float ex[K][R], ay[K][SplitShape<MODEL, R, G>::RL], acc[SplitShape<MODEL, R, G>::RL], b;
                (void)split_model<MODEL, R, G, FAST>(pos, t, ex, ay, b);
                split_rows<MODEL, R, G, FAST, false>(q, c1, wx, ex, ay, b, lt, acc);
                L[h] = split_total<MODEL, R, G>(wy, acc);
            });
            g[gi] = (L[1] - L[0]) * 250.0f;
            t[gi] = t[gi] - 0.002f;
            clamp(gi);
        });
        return;
    }
#pragma unroll 1
    for (int gi = 0; gi < P; gi++) {
        float ln = 0.0f;
#pragma unroll 1
        for (int h = 0; h < 2; h++) {
            const float delta = h ? 0.004f : -0.002f;
#pragma unroll
            for (int k = 0; k < P; k++) t[k] = (k == gi) ? t[k] + delta : t[k];
            const float L = split_loss<MODEL, R, G, FAST>(q, c1, wx, wy, pos, t, lt);
            if (h == 0) ln = L;
            else
#pragma unroll
                for (int k = 0; k < P; k++) {
                    g[k] = (k == gi) ? (L - ln) * 250.0f : g[k];
                    t[k] = (k == gi) ? t[k] - 0.002f : t[k];
                }
        }
    }
}

// ConstructD0 (bfgsMLE_core.h:87-182) and the new direction d = -D g.  Row r of D is on lane r % G of the group (D[r / G]).
template <int P, int G>
__device__ __forceinline__ void split_update(float (&D)[(P + G - 1) / G][P], int gl, const float (&s)[P], const float (&y)[P],
                                             const float (&g)[P], float (&d)[P])
{
    constexpr int MR = (P + G - 1) / G;
    float sy = 0.0f;
#pragma unroll
    for (int k = 0; k < P; k++) sy = __builtin_fmaf(s[k], y[k], sy);
    sy = 1.0f / sy;
    float ty[P], ts[P];
#pragma unroll
    for (int k = 0; k < P; k++) { ty[k] = y[k] * sy; ts[k] = s[k] * sy; }
    float T[MR][P], sr[MR], dr[MR];
#pragma unroll
    for (int m = 0; m < MR; m++) {
        const int r = gl + G * m;
        sr[m] = dr[m] = 0.0f;
#pragma unroll
        for (int k = 0; k < P; k++) sr[m] = (k == r) ? s[k] : sr[m];
#pragma unroll
        for (int c = 0; c < P; c++) T[m][c] = 0.0f;
    }
    fs_for<0, P>([&](auto Kc) {
        constexpr int k = decltype(Kc)::value;
        float a[MR];
#pragma unroll
        for (int m = 0; m < MR; m++) a[m] = __builtin_fmaf(-sr[m], ty[k], (gl + G * m == k) ? 1.0f : 0.0f);   // A[r][k]
#pragma unroll
        for (int c = 0; c < P; c++) {
            const float dk = group_bcast<G, k % G>(D[k / G][c]);
#pragma unroll
            for (int m = 0; m < MR; m++) T[m][c] = __builtin_fmaf(a[m], dk, T[m][c]);
        }
    });
#pragma unroll
    for (int c = 0; c < P; c++) {
        float acc[MR];
#pragma unroll
        for (int m = 0; m < MR; m++) acc[m] = 0.0f;
#pragma unroll
        for (int k = 0; k < P; k++) {
            const float a = __builtin_fmaf(-s[c], ty[k], (c == k) ? 1.0f : 0.0f);   // A[c][k]
#pragma unroll
            for (int m = 0; m < MR; m++) acc[m] = __builtin_fmaf(T[m][k], a, acc[m]);
        }
#pragma unroll
        for (int m = 0; m < MR; m++) {
            D[m][c] = acc[m] + sr[m] * ts[c];
            dr[m] = __builtin_fmaf(-D[m][c], g[c], dr[m]);   // MatMulVector (bfgsMLE_core.h:184-204)
        }
    }
    fs_for<0, P>([&](auto Rc) {
        constexpr int r = decltype(Rc)::value;
        d[r] = group_bcast<G, r % G>(dr[r / G]);
    });
}

// The fixed schedule (MLELocalization_GS2D, bfgsMLE_GS2D_core.h:313-426): gradient, then per iteration probes at 1e-4 and 1, ten bisection
// evaluations (eleven halvings of [1e-5, 1]), step, clamp >= 0.01, and -- except after the last
// iteration -- gradient, update and new direction.
template <int MODEL, int R, int G, bool FAST>
__device__ __forceinline__ void split_fit(const float (&q)[SplitShape<MODEL, R, G>::RL][R], const float (&c1)[SplitShape<MODEL, R, G>::RL][R],
                                          const float (&wx)[R], const float (&wy)[R], const float (&pos)[SplitShape<MODEL, R, G>::RL],
                                          float (&x)[Traits<MODEL>::P], int gl, const float2 *lt)
{
    constexpr int P = Traits<MODEL>::P, IT = Traits<MODEL>::ITERS, MR = (P + G - 1) / G;
    float D[MR][P];
#pragma unroll
    for (int m = 0; m < MR; m++)
#pragma unroll
        for (int c = 0; c < P; c++) D[m][c] = (gl + G * m == c) ? 1.0f : 0.0f;
    float g[P], gp[P], d[P], s[P];
#pragma unroll
    for (int k = 0; k < P; k++) g[k] = gp[k] = d[k] = s[k] = 0.0f;
#pragma unroll 1
    for (int it = 0; it < IT; it++) {
        split_gradient<MODEL, R, G, FAST>(q, c1, wx, wy, pos, x, g, lt);
        if (it == 0) {
#pragma unroll
            for (int k = 0; k < P; k++) d[k] = -g[k];
        } else {
            float y[P];
#pragma unroll
            for (int k = 0; k < P; k++) y[k] = g[k] - gp[k];
            split_update<P, G>(D, gl, s, y, g, d);
        }
        normalize_dir<P>(d);
        float lo = 0.00001f, hi = 1.0f, L0 = 0.0f, L1 = 0.0f;
        bool sel = false;
#pragma unroll 1
        for (int j = 0; j < 12; j++) {
            const float step = j == 0 ? 0.0001f : (j == 1 ? 1.0f : (sel ? hi : lo));
            float pr[P];
#pragma unroll
            for (int k = 0; k < P; k++) pr[k] = __builtin_fmaf(d[k], step, x[k]);
            const float L = split_loss<MODEL, R, G, FAST>(q, c1, wx, wy, pos, pr, lt);
            if (j == 0) {
                L0 = L;
                continue;
            }
            if (j == 1 || sel) L1 = L;
            else L0 = L;
            sel = (L0 < L1);
            const float mid = (lo + hi) * 0.5f;
            if (sel) hi = mid;
            else lo = mid;
        }
        const float scale = (lo + hi) * 0.5f;
#pragma unroll
        for (int k = 0; k < P; k++) {
            s[k] = d[k] * scale;
            x[k] = x[k] + s[k];
            x[k] = (x[k] < 0.01f) ? 0.01f : x[k];   // IninfConstrain (bfgsMLE_core.h:76-85)
            gp[k] = g[k];
        }
    }
}

// work-group: its four waves share the log table (32 KB for the one-emitter models).  G = 1, and the
// fast 13x13 pair of lanes (91 pixels a lane), are held to two waves per SIMD: the 7x7 2D kernel then
// takes 225 VGPRs without spills, and the 13x13 one spills 58 but runs 60,000 fits in one round (638 -> 559 us).
constexpr int FS_BLOCK = 256;
template <int R, int G> constexpr bool kTwoWaves = G == 1 || ((R + G - 1) / G) * R > 80;

// Items i < n (or *n_dev) of list idx (or the ROIs themselves).  One-emitter models write the ROI's
// row and flag a[roi]; multi-emitter models write as finish_me does (second rows, a = fs, b = ff).
template <int MODEL, int R, int G, bool FAST>
__global__ void __launch_bounds__(FS_BLOCK) __attribute__((amdgpu_waves_per_eu(kTwoWaves<R, G> ? 2 : 1, kTwoWaves<R, G> ? 2 : 10))) fit_split_kernel(const uint16_t *__restrict__ rois, const float *__restrict__ wle,
                                                             const int *__restrict__ idx, int n, const int *__restrict__ n_dev,
                                                             float *__restrict__ loc, float *__restrict__ second, int *__restrict__ fa,
                                                             int *__restrict__ fb, FitConst fc)
{
    using T = Traits<MODEL>;
    constexpr int P = T::P, K = T::K, RL = SplitShape<MODEL, R, G>::RL, NG = FS_BLOCK / G;
    __shared__ float2 ltab[K == 1 ? kLogTabBN : 32];
    if (n_dev) n = *n_dev;
    const int i0 = blockIdx.x * NG;
    if (i0 >= n) return;   // uniform over the work-group
    if constexpr (K == 1) log_tabb_load(ltab);
    else log_tab_load(ltab);
    const int gl = threadIdx.x % G, item = i0 + threadIdx.x / G;
    // groups past the end repeat the last item, so every lane takes part in the exchanges
    const int i = min(item, n - 1);
    const int roi = idx ? idx[i] : i;
    const uint16_t *rec = rois + (size_t)roi * (R * (R + 1));
    auto pixel = [&](int k) {
        const float e = ((float)rec[k] - fc.Offset) * fc.KAdc;   // bfgsMLE_GS2D_core.h:144
        return (e > 1.0f) ? e : 1.0f;
    };
    float x[P], wx[R], wy[R];
    float nn = 0.0f;
    const float *wp = wle + (size_t)roi * QCS_WLE_FLOATS;
    if constexpr (K == 1) start_1e<MODEL, R>(pixel, wp, fc, x, wx, wy);
    else nn = start_me<MODEL, R>(pixel, wp, fc, x, wx, wy);
    float q[RL][R], c1[RL][R], pos[RL];
#pragma unroll
    for (int m = 0; m < RL; m++) {
        const int r = gl * RL + m;
        pos[m] = (float)r + 0.5f;
#pragma unroll
        for (int c = 0; c < R; c++) {
            q[m][c] = (r < R) ? pixel(r * R + c) : 1.0f;   // rows past the ROI enter no sum
            c1[m][c] = 1.0f - qlogf_normal(q[m][c]);       // q >= 1
        }
    }
    split_fit<MODEL, R, G, FAST>(q, c1, wx, wy, pos, x, gl, ltab);
    if (gl != 0 || item >= n) return;
    const int xo = rec[R * R], yo = rec[R * R + 1], fr = (int)rec[R * R + 2] + 65536 * (int)rec[R * R + 3];
    if constexpr (K == 1) finish_1e<MODEL, R>(x, fc, xo, yo, fr, roi, loc, fa);
    else finish_me<MODEL, R>(x, fc, nn, xo, yo, fr, roi, i, loc, second, fa, fb);
}

template <int MODEL, int R, int G, bool FAST>
static int launch_split(const SplitArgs &a, const FitConst &fc, hipStream_t s)
{
    constexpr int NG = FS_BLOCK / G;
    hipLaunchKernelGGL((fit_split_kernel<MODEL, R, G, FAST>), dim3((unsigned)((a.n + NG - 1) / NG)), dim3(FS_BLOCK), 0, s, a.rois, a.wle,
                       a.idx, a.n, a.n_dev, a.loc, a.second, a.fa, a.fb, fc);
    QCS_HIP(hipGetLastError());
    return QCS_OK;
}

}  // namespace qcs
