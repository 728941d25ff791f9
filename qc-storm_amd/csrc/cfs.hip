// cfs.hip -- converged fits split over 16 lanes each (gfx950): short launches and the tails of long ones.
//
// One fit per lane (cfq.hip) is the better use of the chip while there are many fits, but a single
// long fit then takes as long as its evaluations take one lane: a three-emitter elliptical fit runs
// up to a thousand evaluations of 81 pixels x 3 emitters and 16 x 16 matrix products, and the launch
// waits for the slowest.  Here a DPP row of 16 lanes holds a fit:
//   lane r < R     the pixels of ROI row r (loss terms, weights, row sums) and the exponentials of
//                  column r, which go round the row by row_newbcast;
//   lane i < P     parameter i: its value, gradient, step and row i of the inverse Hessian;
//   sums           the sums over all pixels are serial in pixel order, as in the one-lane kernels: the
//                  rows leave each pixel's terms in LDS, and the lanes of the x, width and background
//                  parameters (and lane 0 for the loss) each run one of those sums.
// Every operation and the order of every sum are those of cfq_run (cfit_dev.h), so parameters,
// iteration counts and flags are the same bit for bit; sums over parameters are repeated in every lane.
//
// The launch takes either fresh work items (the prep pass's records) or the fits that the waves of a
// one-lane launch left when their queue ran dry (CqLeft records), each resumed where it stood.
//
// Backtracking: the long fits reject most of their trials (a three-emitter elliptical fit accepts 41%),
// and a rejected trial's successors are known: alpha 0.3, 0.09, ...  Once a wave has no more fits to
// take, its idle groups join one that runs (pairs for two fits, all four groups for one), and the
// groups try consecutive step lengths at once; the first that passes counts, so the path and the
// evaluation count are those of the serial search.  Launches of at most one fit per resident wave
// start that way.
//
// What bounds it: a lone fit, the latency of a round (2.5 us elliptical K = 3: 81 chained FMAs over LDS, the
// 16-parameter products); many, VALU issue (0.76 of the cycles on 2^18 elliptical ROIs at K = 3), 312
// instructions per loss evaluation or 1,250 per round of four fits, of which the pixel terms use 9 of 16 lanes
// at 9x9.  Measured against one fit per lane to the end, three launches and selection: elliptical 9x9,
// 500 ROIs 21.1 -> 1.6 ms, 16,461 ROIs 35.3 -> 6.1 ms; 2D 7x7, 2,000 ROIs 2.6 -> 0.56 ms.
#include <string.h>
#include "cfq.h"

namespace qcs {

// Value of lane J of the 16-lane row, in all its lanes.
template <int J>
__device__ __forceinline__ float row_bcast(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + J, 0xf, 0xf, true));
}
template <int N>
__device__ __forceinline__ float row_ror(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x120 + N, 0xf, 0xf, true));
}
// largest magnitude over the row, at least 0 (NaN entries are passed over, as fmaxf does)
__device__ __forceinline__ float row_absmax(float v)
{
    v = fmaxf(0.0f, fabsf(v));
    v = fmaxf(v, row_ror<8>(v));
    v = fmaxf(v, row_ror<4>(v));
    v = fmaxf(v, row_ror<2>(v));
    return fmaxf(v, row_ror<1>(v));
}

// per-fit LDS: the pixel terms (loss, weight, weighted emitter values) by row, then the row sums
template <int KK, int R> struct CsLds {
    static constexpr int K = CM<KK>::K, NA = 2 + K;
    static constexpr int PITCH = (R + 3) & ~3;
    static constexpr int ARR = R * PITCH;              // one pixel array
    static constexpr int ROWS = NA * ARR;              // sw[k][16], then (2D) sx2[k][16]
    static constexpr int SIZE = ROWS + (CM<KK>::AS ? K : 2 * K) * 16;
};

enum { ROLE_N = 0, ROLE_X = 1, ROLE_Y = 2, ROLE_SX = 3, ROLE_SY = 4, ROLE_B = 5, ROLE_NONE = 6 };

template <int KK, int R>
__device__ __forceinline__ void cfs_run(const CfqSet &S, int *head, const CqLeft *left, const CFitConst &c, int ways, float *lds)
{
    using M = CM<KK>;
    using Q = CQ<KK>;
    using LD = CsLds<KK, R>;
    constexpr int P = Q::P, K = M::K;
    const int lane = threadIdx.x & 63, gl = lane & 15, gi = lane >> 4;
    const int wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int nfits = gridDim.x * (blockDim.x >> 6) * 4 / ways;   // fits in flight
    lds += ((threadIdx.x >> 6) * 4 + gi) * LD::SIZE;
    const int n = left ? min(*left->cnt, left->cap) : (S.n_dev ? min(*S.n_dev, S.n) : S.n);

    // the lane's parameter: emitter, role, units
    int role = ROLE_NONE, ke = 0;
    float sc = 1.0f;
    if (gl == P - 1) role = ROLE_B;
    else if (gl < P - 1) {
        if constexpr (M::AS) { ke = gl / 5; role = gl % 5; }
        else if (gl == P - 2) role = ROLE_SX;   // the shared width
        else { ke = gl / 3; role = gl % 3; }
    }
    if (role == ROLE_N) sc = 1000.0f;
    if (role == ROLE_B) sc = 100.0f;
    // box bounds of cf_project
    float blo = -__builtin_inff(), bhi = __builtin_inff();
    if (role == ROLE_N) blo = 1.0f;
    if (role == ROLE_X || role == ROLE_Y) { blo = -0.5f; bhi = (float)R + 0.5f; }
    if (role == ROLE_SX || role == ROLE_SY) { blo = 0.4f; bhi = 0.5f * (float)R; }
    if (role == ROLE_B) blo = 0.01f;
    const int src = role == ROLE_B ? 1 : ((role == ROLE_X || (M::AS && role == ROLE_SX)) ? 2 + ke : 0);
    const float pos = (float)gl + 0.5f;   // the lane's row and column centre

    int st = CQ_IDLE, roi = 0, iters = 0, evals = 0, t = 0, pin_run = 0, next = (wave * 4 + gi) / ways;
    bool first = false;
    float th = 0.0f, g = 0.0f, du = 0.0f, D[P], q[R], rq[R];
    float L = 0.0f, slope = 0.0f, alpha = 1.0f, dmax = 0.0f;
#pragma unroll
    for (int j = 0; j < P; j++) D[j] = 0.0f;
#pragma unroll
    for (int cc = 0; cc < R; cc++) q[cc] = rq[cc] = 1.0f;

    auto finish = [&](int flags) {
        st = CQ_IDLE;
        if (gi & (ways - 1)) return;   // one of the groups that share the fit writes it
        if (gl < P) S.theta[(size_t)roi * S.ostride + gl] = th;
        if (S.info && gl == 0) {
            int *inf = S.info + (size_t)roi * 4;
            inf[0] = iters;
            inf[1] = flags;
            inf[2] = evals;
            inf[3] = 0;
        }
    };
    auto from = [&](float &v, int l) { v = __shfl(v, l, 64); };
    auto from_i = [&](int &v, int l) { v = __shfl(v, l, 64); };

    while (true) {
        if (st == CQ_IDLE && next < n) {   // uniform over the group
            // the first items are dealt out by position (one atomic per group would queue up at the L2)
            const int j = next;
            {
                const float *rec;
                if (left) {
                    rec = left->rec + (size_t)j * Q::XW;
                    const int *h = reinterpret_cast<const int *>(rec + Q::OX);
                    roi = h[CX_ROI];
                    st = h[CX_ST];
                    t = h[CX_T];
                    iters = h[CX_ITERS];
                    evals = h[CX_EVALS];
                    pin_run = 0;   // only the models without it have left fits
                    slope = rec[Q::OX + CX_SLOPE];
                    alpha = rec[Q::OX + CX_ALPHA];
                    dmax = rec[Q::OX + CX_DMAX];
                    du = gl < P ? rec[Q::OX + CX_DU + gl] : 0.0f;
                } else {
                    rec = S.rec + (size_t)j * Q::W;
                    roi = S.idx ? S.idx[j] : j;
                    st = CQ_DIR;
                    iters = pin_run = 0;
                    evals = 1;
                }
                L = rec[Q::OL];
                first = rec[Q::OF] != 0.0f;
                th = gl < P ? rec[gl] : 0.0f;
                g = gl < P ? rec[Q::OG + gl] : 0.0f;
#pragma unroll
                for (int jj = 0; jj < P; jj++) {
                    const int a = min(gl, jj), b2 = max(gl, jj);
                    D[jj] = gl < P ? rec[Q::OD + tri(a, b2, P)] : 0.0f;
                }
                if (gl < R) {
                    const uint16_t *px = S.rois + (size_t)roi * (R * (R + 1)) + gl * R;
#pragma unroll
                    for (int cc = 0; cc < R; cc++) {
                        q[cc] = fmaxf(((float)px[cc] - c.offset) * c.kadc, 1.0f) * c.inv_qe;
                        rq[cc] = __builtin_amdgcn_rcpf(q[cc]);
                    }
                }
                if (ways == 1) {
                    int nx = 0;
                    if (gl == 0) nx = atomicAdd(head, 1);
                    next = nfits + __builtin_amdgcn_mov_dpp(nx, 0x150, 0xf, 0xf, true);
                } else {
                    next = n;   // a shared start deals every fit out by position
                }
            }
        }
        const unsigned long long act = __ballot(st != CQ_IDLE);
        if (act == 0ull) {
            if (__all(next >= n)) break;
            continue;
        }
        if (ways < 4 && __all(next >= n)) {
            // Nothing more to take: groups without a fit join one that still runs.  With one fit left
            // the wave's four groups share it, with two, pairs do; each then tries the step lengths
            // that a rejected trial would lead to next, so a backtracking search takes a quarter of
            // the rounds.
            int owner[4], nf = 0;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (k % ways == 0 && ((act >> (16 * k)) & 1ull)) {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (e == nf) owner[e] = k;
                    nf++;
                }
            const int nw = nf == 1 ? 4 : (nf == 2 ? 2 : 1);
            if (nw > ways) {
                const int l = (nw == 4 || gi < 2 ? owner[0] : owner[1]) * 16 + gl;
                from(th, l); from(g, l); from(du, l); from(L, l); from(slope, l); from(alpha, l); from(dmax, l);
#pragma unroll
                for (int jj = 0; jj < P; jj++) from(D[jj], l);
#pragma unroll
                for (int cc = 0; cc < R; cc++) { from(q[cc], l); from(rq[cc], l); }
                from_i(st, l); from_i(roi, l); from_i(iters, l); from_i(evals, l); from_i(t, l); from_i(pin_run, l);
                int f = first ? 1 : 0;
                from_i(f, l);
                first = f != 0;
                ways = nw;
            }
        }
        if (st == CQ_DIR) {   // quasi-Newton direction (cf_direction)
            const float gu = g * sc;
            bool pin = false;
            if (c.active_set) {
                if (role == ROLE_N || role == ROLE_B) pin = th <= blo && gu > 0.0f;
                else if (role != ROLE_NONE) pin = (th <= blo && gu > 0.0f) || (th >= bhi && gu < 0.0f);
            }
            const unsigned pm = (unsigned)(__ballot(pin) >> (lane & 48));
            float GU[P];
            cf_sfor<0, P>([&](auto J) { GU[decltype(J)::value] = row_bcast<decltype(J)::value>(gu); });
            float a = 0.0f;
            if (__any(pin)) {
#pragma unroll
                for (int jj = 0; jj < P; jj++) {
                    const float v = fmaf(D[jj], GU[jj], a);
                    a = ((pm >> jj) & 1u) ? a : v;
                }
            } else {
#pragma unroll
                for (int jj = 0; jj < P; jj++) a = fmaf(D[jj], GU[jj], a);
            }
            du = (pin || gl >= P) ? 0.0f : -a;
            auto dot = [&]() {
                slope = 0.0f;
                cf_sfor<0, P>([&](auto J) { slope = fmaf(row_bcast<decltype(J)::value>(du), GU[decltype(J)::value], slope); });
            };
            dot();
            if (row_absmax(du) < c.tol && slope <= 0.0f) {
                finish(CF_CONVERGED);
            } else {
                if (!(slope < 0.0f)) {   // not a descent direction: restart from the gradient
                    du = (pin || gl >= P) ? 0.0f : -gu;
                    dot();
#pragma unroll
                    for (int jj = 0; jj < P; jj++) D[jj] = (gl == jj) ? 1.0f : 0.0f;
                    first = true;
                }
                if (first) {   // identity inverse Hessian: limit the first step to 0.1 scaled units
                    const float m = row_absmax(du);
                    if (m > 0.1f) {
                        du *= 0.1f / m;
                        dot();
                    }
                }
                dmax = row_absmax(du);
                alpha = 1.0f;
                t = 0;
                st = CQ_LS;
            }
        }
        if (st != CQ_LS) continue;

        // Loss (cf_lossgrad_q) at the trial point: group h of the fit's groups takes the step length
        // that h rejections from here lead to.
        const int h = gi & (ways - 1);
        float al[5];
        al[0] = alpha;
#pragma unroll
        for (int e = 1; e < 5; e++) al[e] = al[e - 1] * 0.3f;
        const float ah = h == 0 ? al[0] : (h == 1 ? al[1] : (h == 2 ? al[2] : al[3]));
        float tn = fmaf(ah, du * sc, th);
        if (role != ROLE_NONE) tn = fminf(fmaxf(tn, blo), bhi);
        float T[P];
        cf_sfor<0, P>([&](auto J) { T[decltype(J)::value] = row_bcast<decltype(J)::value>(tn); });
        const float b = T[M::IB];
        float isx2[K], isy2[K], ex[K][R], ay[K], dy[K];
        // the emitters' divisions: each lane those of its own emitter, the photon lanes' go round
        {
            float sx = T[M::isx(0)], sy = T[M::isy(0)], nN = T[M::iN(0)];
#pragma unroll
            for (int k = 1; k < K; k++) {
                if constexpr (M::AS) {
                    sx = ke == k ? T[M::isx(k)] : sx;
                    sy = ke == k ? T[M::isy(k)] : sy;
                }
                nN = ke == k ? T[M::iN(k)] : nN;
            }
            const float ix2 = 1.0f / (sx * sx);
            const float iy2 = M::AS ? 1.0f / (sy * sy) : ix2;
            const float nl = nN * (M::AS ? 0.15915494309189535f / (sx * sy) : 0.15915494309189535f * ix2);
            cf_sfor<0, K>([&](auto Kc) {
                constexpr int k = decltype(Kc)::value;
                isx2[k] = M::AS ? row_bcast<M::iN(k)>(ix2) : ix2;
                isy2[k] = M::AS ? row_bcast<M::iN(k)>(iy2) : ix2;
                const float nk = row_bcast<M::iN(k)>(nl);
                const float hx = -0.5f * isx2[k], hy = -0.5f * isy2[k];
                const float dxl = pos - T[M::ix(k)];
                const float exl = __expf(hx * dxl * dxl);
                cf_sfor<0, R>([&](auto Cc) { ex[k][decltype(Cc)::value] = row_bcast<decltype(Cc)::value>(exl); });
                dy[k] = pos - T[M::iy(k)];
                ay[k] = nk * __expf(hy * dy[k] * dy[k]);
            });
        }
        cf_wave_fence();   // the terms of the evaluation before have been read
        {
            float sw[K], sx2[K];
#pragma unroll
            for (int k = 0; k < K; k++) sw[k] = sx2[k] = 0.0f;
            float *o = lds + gl * LD::PITCH;
            // four pixels at a time, and no further: the terms of a whole row would cost registers
#pragma unroll
            for (int v = 0; v < LD::PITCH; v += 4) {
                float tv[4], wv[4], gv[K][4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int cc = v + e;
                    tv[e] = wv[e] = 0.0f;
#pragma unroll
                    for (int k = 0; k < K; k++) gv[k][e] = 0.0f;
                    if (cc >= R) continue;
                    float gk[K], mu = b;
#pragma unroll
                    for (int k = 0; k < K; k++) {
                        gk[k] = ay[k] * ex[k][cc];
                        mu += gk[k];
                    }
                    mu = fmaxf(mu, 1e-6f);
                    tv[e] = (mu - q[cc]) - q[cc] * cf_logf(mu * rq[cc]);
                    wv[e] = 1.0f - q[cc] * __builtin_amdgcn_rcpf(mu);
#pragma unroll
                    for (int k = 0; k < K; k++) {
                        gv[k][e] = wv[e] * gk[k];
                        sw[k] += gv[k][e];
                        if constexpr (!M::AS) {
                            const float dx = ((float)cc + 0.5f) - T[M::ix(k)];
                            sx2[k] = fmaf(gv[k][e], dx * dx, sx2[k]);
                        }
                    }
                }
                if (gl < R) {
                    *reinterpret_cast<float4 *>(o + v) = make_float4(tv[0], tv[1], tv[2], tv[3]);
                    *reinterpret_cast<float4 *>(o + LD::ARR + v) = make_float4(wv[0], wv[1], wv[2], wv[3]);
#pragma unroll
                    for (int k = 0; k < K; k++)
                        *reinterpret_cast<float4 *>(o + (2 + k) * LD::ARR + v) = make_float4(gv[k][0], gv[k][1], gv[k][2], gv[k][3]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (gl < R) {
#pragma unroll
                for (int k = 0; k < K; k++) {
                    lds[LD::ROWS + k * 16 + gl] = sw[k];
                    if constexpr (!M::AS) lds[LD::ROWS + (K + k) * 16 + gl] = sx2[k];
                }
            }
        }
        cf_wave_fence();
        // the lane's sum over the pixels, in pixel order
        float xk = T[M::ix(0)], yk = T[M::iy(0)];
#pragma unroll
        for (int k = 1; k < K; k++) {
            xk = ke == k ? T[M::ix(k)] : xk;
            yk = ke == k ? T[M::iy(k)] : yk;
        }
        float pixsum = 0.0f;
        {
            float mul[LD::PITCH];
#pragma unroll
            for (int cc = 0; cc < R; cc++) {
                const float dx = ((float)cc + 0.5f) - xk;
                mul[cc] = role == ROLE_X ? dx : 1.0f;
                if constexpr (M::AS) mul[cc] = role == ROLE_SX ? dx * dx : mul[cc];
            }
            const float *p = lds + src * LD::ARR;
#pragma unroll
            for (int r = 0; r < R; r++) {
                float v[LD::PITCH];
#pragma unroll
                for (int e = 0; e < LD::PITCH; e += 4) {
                    const float4 x = *reinterpret_cast<const float4 *>(p + r * LD::PITCH + e);
                    v[e] = x.x; v[e + 1] = x.y; v[e + 2] = x.z; v[e + 3] = x.w;
                }
#pragma unroll
                for (int cc = 0; cc < R; cc++) pixsum = fmaf(v[cc], mul[cc], pixsum);
            }
        }
        float Lt = row_bcast<0>(pixsum);
        // the first trial, in the order of the step lengths, that ends the search
        const bool good = t + h < 16 && Lt == Lt && Lt < L && Lt <= fmaf(1e-4f * ah, slope, L);
        const bool tiny = t == 0 && h == 0 && !(Lt < L) && dmax < 20.0f * c.tol;
        const unsigned long long bg = __ballot(good), bt = __ballot(tiny);
        int w = ways;   // groups before the accepted one; ways: none
        const int g0 = gi - h;
#pragma unroll
        for (int e = 3; e >= 0; e--)
            if (e < ways && ((bg >> (16 * (g0 + e))) & 1ull)) w = e;
        if ((bt >> (16 * g0)) & 1ull) {
            // the full step is tiny and the FP32 loss cannot resolve it: take it and stop
            evals++;
            iters++;
            if (ways > 1) from(tn, g0 * 16 + gl);
            th = tn;
            finish(CF_CONVERGED);
            continue;
        }
        if (w == ways) {
            const int tries = min(ways, 16 - t);
            evals += tries;
            t += tries;
            alpha = ways == 4 ? al[4] : (ways == 2 ? al[2] : al[1]);
            if (t >= 16) {   // no decrease in 16 backtracks
                iters++;
                finish(CF_STALLED);
            }
            continue;
        }
        evals += w + 1;
        // gradient at the accepted point
        // sums over the rows: the lane's own (photons, y, y width), and (2D) the shared width's
        float rowsum = 0.0f, gd2 = 0.0f, gw = 0.0f;
        {
            const float *p = lds + LD::ROWS + ke * 16;
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float d = ((float)r + 0.5f) - yk;
                float m = role == ROLE_Y ? d : 1.0f;
                if constexpr (M::AS) m = role == ROLE_SY ? d * d : m;
                rowsum = fmaf(p[r], m, rowsum);
            }
            if constexpr (!M::AS) {
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int k = 0; k < K; k++) {
                        const float sw = lds[LD::ROWS + k * 16 + r], d = ((float)r + 0.5f) - T[M::iy(k)];
                        gw += sw;
                        gd2 = fmaf(sw, d * d, gd2 + lds[LD::ROWS + (K + k) * 16 + r]);
                    }
            }
        }
        float gt = 0.0f;
        if constexpr (M::AS) {
            float gNk = row_bcast<M::iN(0)>(rowsum), sxk = T[M::isx(0)], syk = T[M::isy(0)], ix2 = isx2[0], iy2 = isy2[0];
            cf_sfor<1, K>([&](auto Kc) {
                constexpr int k = decltype(Kc)::value;
                const float gN = row_bcast<M::iN(k)>(rowsum);
                gNk = ke == k ? gN : gNk;
                sxk = ke == k ? T[M::isx(k)] : sxk;
                syk = ke == k ? T[M::isy(k)] : syk;
                ix2 = ke == k ? isx2[k] : ix2;
                iy2 = ke == k ? isy2[k] : iy2;
            });
            const float sum = role == ROLE_SX ? fmaf(pixsum, ix2, -gNk) : fmaf(rowsum, iy2, -gNk);
            const float num = role == ROLE_N ? rowsum : sum;
            const float den = role == ROLE_N ? fmaxf(tn, 1e-3f) : (role == ROLE_SX ? sxk : syk);
            const float quo = num / den;
            gt = role == ROLE_X ? pixsum * ix2 : (role == ROLE_Y ? rowsum * iy2 : (role == ROLE_B ? pixsum : quo));
        } else {
            const float is2 = isx2[0];
            const float num = role == ROLE_N ? rowsum : (gd2 * is2 - 2.0f * gw);
            const float den = role == ROLE_N ? fmaxf(tn, 1e-3f) : T[M::isx(0)];
            const float quo = num / den;
            gt = role == ROLE_X ? pixsum * is2 : (role == ROLE_Y ? rowsum * is2 : (role == ROLE_B ? pixsum : quo));
        }
        if (role == ROLE_NONE) gt = 0.0f;
        if (ways > 1) {   // the accepted group's point to the others
            const int l = (g0 + w) * 16 + gl;
            from(tn, l);
            from(gt, l);
            from(Lt, l);
        }
        {
            // accepted: BFGS update of the inverse Hessian (cf_bfgs_update)
            iters++;
            const float s = (tn - th) / sc, y = (gt - g) * sc;
            float Sv[P], Y[P], sy = 0.0f, yy = 0.0f;
            cf_sfor<0, P>([&](auto J) {
                constexpr int j = decltype(J)::value;
                Sv[j] = row_bcast<j>(s);
                Y[j] = row_bcast<j>(y);
                sy = fmaf(Sv[j], Y[j], sy);
                yy = fmaf(Y[j], Y[j], yy);
            });
            if (sy > 1e-12f) {
                if (first) {
                    const float d0 = sy / yy;
#pragma unroll
                    for (int jj = 0; jj < P; jj++) D[jj] = (gl == jj) ? d0 : 0.0f;
                    first = false;
                }
                const float rho = 1.0f / sy;
                float u = 0.0f, U[P], yu = 0.0f;
#pragma unroll
                for (int jj = 0; jj < P; jj++) u = fmaf(D[jj], Y[jj], u);
                cf_sfor<0, P>([&](auto J) {
                    constexpr int j = decltype(J)::value;
                    U[j] = row_bcast<j>(u);
                    yu = fmaf(Y[j], U[j], yu);
                });
                const float cs = fmaf(rho * rho, yu, rho);
                // entry (i, j), i <= j, by the formula of its upper-triangular place
#pragma unroll
                for (int jj = 0; jj < P; jj++) {
                    const bool up = gl <= jj;
                    const float si = up ? s : Sv[jj], sj = up ? Sv[jj] : s, ui = up ? u : U[jj], uj = up ? U[jj] : u;
                    D[jj] = fmaf(cs * si, sj, fmaf(-rho, fmaf(si, uj, ui * sj), D[jj]));
                }
            }
            th = tn;
            g = gt;
            const float Lold = L;
            L = Lt;
            if constexpr (M::AS && K == 3)
                if (c.pin_stop) {
                    const bool at = role != ROLE_NONE && role != ROLE_B && (th <= blo || th >= bhi);
                    pin_run = ((unsigned)(__ballot(at) >> (lane & 48)) & 0xffffu) ? pin_run + 1 : 0;
                }
            if (Lold - L < c.ftol) finish(CF_CONVERGED | CF_FLAT);   // the likelihood has stopped moving
            else if (pin_run >= CF_PIN_RUN) finish(CF_PINNED);
            else if (iters >= c.max_iter) finish(CF_MAXITER);
            else st = CQ_DIR;
        }
    }
}

constexpr int CS_BLOCK = 64;

template <int KK, int RMAX>
__global__ void __launch_bounds__(CS_BLOCK) cfs_kernel(CfqArgs a, int ways)
{
    __shared__ __align__(16) float lds[(CS_BLOCK / 16) * CsLds<KK, RMAX>::SIZE];
    for (int si = 0; si < a.nsets; si++) {
        const int R = a.set[si].R;
        const CqLeft *left = a.left[si].rec ? &a.left[si] : nullptr;
        if constexpr (RMAX >= 11) {
            if (R == 11) cfs_run<KK, 11>(a.set[si], a.heads + si, left, a.c, ways, lds);
        }
        if constexpr (RMAX >= 9) {
            if (R == 9) cfs_run<KK, 9>(a.set[si], a.heads + si, left, a.c, ways, lds);
        }
        if (R == 7) cfs_run<KK, 7>(a.set[si], a.heads + si, left, a.c, ways, lds);
    }
}

// resident single-wave work-groups per CU (cached)
int cfs_waves_per_cu(int KK, int RMAX)
{
    static int cache[2][3][3] = {{{0}}};
    const int ri = RMAX == 7 ? 0 : (RMAX == 9 ? 1 : 2);
    const int as = KK > CF_ELLIPTIC ? 1 : 0, K = as ? KK - CF_ELLIPTIC : KK;
    int &v = cache[as][K - 1][ri];
    if (v == 0) {
        const void *f = nullptr;
        switch (KK) {
        case 1: case 2: case 3: case 11: case 12: case 13: break;
        default: return 1;
        }
        auto pick = [&]() -> int {
            CF_DISPATCH_KK(KK, CF_DISPATCH_R(RMAX, f = reinterpret_cast<const void *>(&cfs_kernel<KT, RT>)))
            return QCS_OK;
        };
        if (pick() != QCS_OK) return 1;
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, CS_BLOCK, 0) != hipSuccess || nb < 1) nb = 1;
        v = nb;
    }
    return v;
}

int cfs_launch(const CfqArgs &a, int KK, int rmax, long long items, int cus, int max_waves_per_cu, hipStream_t s)
{
    int wpc = cfs_waves_per_cu(KK, rmax);
    if (max_waves_per_cu > 0 && max_waves_per_cu < wpc) wpc = max_waves_per_cu;
    const long long most = (long long)cus * wpc;
    // one fit per wave, its four groups sharing it, while every fit gets a wave at once
    const int ways = !a.left[0].rec && items <= most ? 4 : 1;
    long long waves = ways == 4 ? items : (items + 3) / 4;
    if (waves > most) waves = most;
    const dim3 grid((unsigned)waves), block(CS_BLOCK);
    CF_DISPATCH_KK(KK, CF_DISPATCH_R(rmax, hipLaunchKernelGGL((cfs_kernel<KT, RT>), grid, block, 0, s, a, ways)))
    QCS_HIP(hipGetLastError());
    return QCS_OK;
}

}  // namespace qcs
