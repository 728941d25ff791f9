// stats.hip -- statistics of a batch of localization rows on gfx950.
//
// Reference (DLL = MLEbfgs/bfgs_MLE_dll x64/bfgsMLE_dll/bfgsMLE_dll):
//   CalcLocResultStatInf       DLL/StatisticsInfo/statisticsInfo.cu:19-91
//   GetStatisticalInf          DLL/StatisticsInfo/statisticsInfo_top.cu:61-128
//   CalcLocalizationDensity2D  DLL/StatisticsInfo/statisticsInfo_top.cu:130-205
//   UpdateStatDat              DLL/StatisticsInfo/statisticsInfo_top.cu:208-225
//   FillerMoleculesInCurFrame, CalcOverlapFluoNum  DLL/StatisticsInfo/statisticsInfo_densityCalc.cu:17-107
//   GetActivationDensity, GetHistogramMeanData     DLL/StatisticsInfo/statisticsInfo_rc.cu:17-74
//   GetFirstFrame, GetLastFrame                    DLL/bfgsMLE_Loc_top/bfgs_top.cu:345-381
//
// The row pass builds the four histograms in LDS per work-group (one global add per non-empty
// bin) and the sums in FP64, one add per work-group.  The reference counts neighbours by an
// all-pairs scan of every frame's molecules, one frame per launch with a host synchronisation
// each; here the molecules of all frames go into a hash table of (frame, cell of the neighbour
// radius) buckets (count, scan, scatter) and each scans the buckets of the 3x3 cells around its own,
// which visits every pair closer than the radius: the counts are the same integers.
// The batch is small (an output call has some ten thousand rows), so launches and waits are what
// it costs: the frame range stays on the device and everything is read back once, eight launches
// and one wait.  Sorting the molecules by (frame, cell) and searching the sorted keys took 19
// launches and five waits, and each search is a chain of fifteen dependent loads (20,480 rows:
// neighbours 28.8 -> 10 us, row pass 28.6 -> 6 us; with compaction and rendering 417 -> 215 us; 2,200,000 rows
// in 200 frames 1,890 -> 660 us, 8,000,000 in 100,000 frames 4,390 -> 2,670 us).
#include <limits.h>
#include <stddef.h>
#include <algorithm>
#include <math.h>
#include <string.h>
#include "qcs_internal.h"

namespace qcs {

namespace {

constexpr int SB = QCS_STAT_BINS, SL = 400;

// device accumulator: histograms, FP64 sums, counters
struct StatAcc {
    int hist[4][SB];
    double sum[4];   // loc prec, peak SNR, PSF width, background
    // first and last rows with a frame: row index above, frame (int) below; none: ~0 and 0
    unsigned long long first, last;
    int valid, kept, n0, n1;
};

// frames the density looks at: both ends are dropped when more than 3 (GetFirstFrame, GetLastFrame)
struct FrameRange {
    int fs, fe;
};
__host__ __device__ inline FrameRange frame_range(const StatAcc &a)
{
    FrameRange r;
    r.fs = a.first == ~0ull ? 0 : (int)(unsigned)a.first;
    r.fe = a.last == 0ull ? 0 : (int)(unsigned)a.last;
    if ((long long)r.fe - r.fs + 1 > 3) {
        r.fs++;
        r.fe--;
    }
    return r;
}

// bin of a quotient value / width, clamped to [0, SB - 1] (the reference converts to int with
// saturation and clamps; clamping the float first gives the same bin without an out-of-range
// conversion)
__device__ __forceinline__ int sbin(float q) { return q >= (float)SB ? SB - 1 : (q > 0.0f ? (int)q : 0); }

constexpr int RT = 512;   // threads of a row pass work-group

__global__ void __launch_bounds__(RT) stat_rows_kernel(const float *__restrict__ loc, int n, StatAcc *__restrict__ acc)
{
    __shared__ int h[4][SB];
    __shared__ double ws[4][RT / 64];
    __shared__ int wi[3][RT / 64];
    for (int k = threadIdx.x; k < 4 * SB; k += RT) (&h[0][0])[k] = 0;
    __syncthreads();
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    int valid = 0, first = INT_MAX, last = -1;
    for (int i = blockIdx.x * RT + threadIdx.x; i < n; i += gridDim.x * RT) {
        const float *r = loc + (size_t)i * QCS_REC_FLOATS;
        const int fr = (int)r[QCS_POS_FRME];
        if (fr != 0) {
            first = min(first, i);
            if (i > 0) last = max(last, i);
        }
        const float tp = r[QCS_POS_TPHO], bg = r[QCS_POS_BAKG];
        const float sg = (r[QCS_POS_SIGX] + r[QCS_POS_SIGY]) / 2;
        const float snr = r[QCS_POS_PSNR];
        const float cx = r[QCS_POS_CRBX], cy = r[QCS_POS_CRBY];
        const float lp = sqrtf(cx * cx + cy * cy);
        if (!((tp > 30.0f) && (bg > 2.0f) && (snr >= 3.0f) && (sg >= 0.01f) && (lp > 0.01f) && (lp < 55.0f))) continue;
        atomicAdd(&h[0][sbin(tp / (10000.0f / SL))], 1);
        atomicAdd(&h[1][sbin(lp / (60.0f / SL))], 1);
        atomicAdd(&h[2][sbin(snr / (50.0f / SL))], 1);
        atomicAdd(&h[3][sbin(sg / (5.0f / SL))], 1);
        valid++;
        s[0] += lp;
        s[1] += snr;
        s[2] += sg;
        s[3] += bg;
    }
    for (int off = 32; off > 0; off >>= 1) {
        for (int k = 0; k < 4; k++) s[k] += __shfl_down(s[k], off, 64);
        valid += __shfl_down(valid, off, 64);
        first = min(first, __shfl_down(first, off, 64));
        last = max(last, __shfl_down(last, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        const int w = threadIdx.x >> 6;
        for (int k = 0; k < 4; k++) ws[k][w] = s[k];
        wi[0][w] = valid;
        wi[1][w] = first;
        wi[2][w] = last;
    }
    __syncthreads();
    if (threadIdx.x < 7) {
        const int k = threadIdx.x;
        if (k < 4) {
            double t = 0.0;
            for (int w = 0; w < RT / 64; w++) t += ws[k][w];
            if (t != 0.0) atomicAdd(&acc->sum[k], t);
        } else if (k == 4) {
            int t = 0;
            for (int w = 0; w < RT / 64; w++) t += wi[0][w];
            if (t) atomicAdd(&acc->valid, t);
        } else if (k == 5) {
            int t = INT_MAX;
            for (int w = 0; w < RT / 64; w++) t = min(t, wi[1][w]);
            if (t != INT_MAX)
                atomicMin(&acc->first, ((unsigned long long)(unsigned)t << 32) |
                                           (unsigned)(int)loc[(size_t)t * QCS_REC_FLOATS + QCS_POS_FRME]);
        } else {
            int t = -1;
            for (int w = 0; w < RT / 64; w++) t = max(t, wi[2][w]);
            if (t >= 0)
                atomicMax(&acc->last, ((unsigned long long)(unsigned)t << 32) |
                                          (unsigned)(int)loc[(size_t)t * QCS_REC_FLOATS + QCS_POS_FRME]);
        }
    }
    for (int k = threadIdx.x; k < 4 * SB; k += RT) {
        const int v = (&h[0][0])[k];
        if (v) atomicAdd(&(&acc->hist[0][0])[k], v);
    }
}

// The neighbour grid.  Cells are `cell` = radius * (1 + 2^-10) wide: two molecules whose float
// distance test passes are then at most one cell apart in x and in y even after the rounding of the
// quotients.  A molecule's bucket is a hash of its frame and cell; the cells around one molecule may
// share a bucket, so an entry carries its frame and cell and counts for its own cell only.
// The hash: the cell times Knuth's multiplicative constant (2^32 / golden ratio), plus the frame times
// xxHash32's second prime, then a shift and the multiplier 0x2c1b3c6d of the 32-bit mixers in common use; its
// upper bits are the bucket.
struct Grid {
    int W, H, ncx, lb;   // 2^lb buckets
    float cell, r2;
};
__device__ __forceinline__ int bucket(const Grid &g, int frame, unsigned c)
{
    unsigned u = c * 2654435769u + (unsigned)frame * 2246822519u;
    u ^= u >> 15;
    u *= 739982445u;
    return (int)(u >> (32 - g.lb));
}
__device__ __forceinline__ unsigned cell_id(const Grid &g, int cx, int cy) { return (unsigned)cy * (unsigned)g.ncx + (unsigned)cx; }

// Molecules of frames fs..fe at least 5 px inside the image (FillerMoleculesInCurFrame).  Pass 1
// (ent == null): molecules per bucket; pass 2: the entries {x, y, frame, cell}, counting cnt down.
__global__ void __launch_bounds__(256) stat_bins_kernel(const float *__restrict__ loc, int n, Grid g, const StatAcc *__restrict__ acc,
                                                        int *__restrict__ cnt, const int *__restrict__ offs, float4 *__restrict__ ent)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const FrameRange fr = frame_range(*acc);
    const float *r = loc + (size_t)i * QCS_REC_FLOATS;
    const float X = r[QCS_POS_XPOS], Y = r[QCS_POS_YPOS];
    const int x = (int)X, y = (int)Y, cf = (int)r[QCS_POS_FRME];
    if (!(x >= 5 && x < g.W - 5 && y >= 5 && y < g.H - 5 && cf >= fr.fs && cf <= fr.fe)) return;
    const unsigned c = cell_id(g, (int)(X / g.cell), (int)(Y / g.cell));
    const int b = bucket(g, cf, c);
    if (!ent) atomicAdd(&cnt[b], 1);
    else ent[offs[b] + atomicSub(&cnt[b], 1) - 1] = make_float4(X, Y, __int_as_float(cf), __int_as_float((int)c));
}

// Neighbours within the radius in the same frame (CalcOverlapFluoNum): molecules with 0 and with 1.
// 16 lanes per molecule, one per cell of the 3x3 block: the nine bucket walks are one round of
// loads instead of nine.  A molecule finds itself once, at distance 0.  NEIGH_BLOCKS work-groups at the
// most take all molecules in turn: each ends with two additions to the same words, one at a time for the
// whole chip at 11 ns (8,000,000 rows: 5,650 us with a work-group per 16 molecules).
// Where a bucket of the wave's is longer than NEIGH_LONG, the 16 lanes walk the nine buckets one after the
// other, an entry each: 2,000,000 molecules in one elliptical frame of 2048 x 2048, 200 a cell, 8,750 -> 4,180 us
// per call (7,500 with a thread a molecule), 20,000 in 256 x 256 124 -> 93 us, short buckets unchanged.
constexpr int NEIGH_BLOCKS = 2048, NEIGH_LONG = 24;
__global__ void __launch_bounds__(256) stat_neigh_kernel(const float4 *__restrict__ ent, const int *__restrict__ offs, Grid g,
                                                         int nb, StatAcc *__restrict__ acc)
{
    __shared__ int wc[2][4];
    const int m = offs[nb];
    if (blockIdx.x == 0 && threadIdx.x == 0) acc->kept = m;
    const int l = threadIdx.x & 15;
    int c0 = 0, c1 = 0;
    for (int p0 = blockIdx.x * 16; p0 < m; p0 += gridDim.x * 16) {   // uniform over the work-group
        const int p = p0 + (int)(threadIdx.x >> 4);
        int cnt = 0;
        float4 e = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        unsigned c = 0;
        int q0 = 0, q1 = 0;   // the bucket of the lane's cell
        if (p < m) {
            e = ent[p];
            const int cx = (int)(e.x / g.cell) + l % 3 - 1, cy = (int)(e.y / g.cell) + l / 3 - 1;
            if (l < 9 && cx >= 0 && cy >= 0) {
                c = cell_id(g, cx, cy);
                const int b = bucket(g, __float_as_int(e.z), c);
                q0 = offs[b];
                q1 = offs[b + 1];
            }
        }
        auto near = [&](int q, unsigned cell) {
            const float4 o = ent[q];
            const float ox = o.x - e.x, oy = o.y - e.y;
            return (ox * ox + oy * oy) <= g.r2 && __float_as_int(o.z) == __float_as_int(e.z) && (unsigned)__float_as_int(o.w) == cell;
        };
        if (__any(q1 - q0 > NEIGH_LONG)) {   // uniform over the wave
            for (int k = 0; k < 9; k++) {
                const unsigned ck = (unsigned)__shfl((int)c, k, 16);
                const int e1 = __shfl(q1, k, 16);
                for (int q = __shfl(q0, k, 16) + l; q < e1; q += 16) cnt += near(q, ck);
            }
        } else {
            for (int q = q0; q < q1; q++) cnt += near(q, c);
        }
        for (int off = 8; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 16);
        const bool lead = p < m && l == 0;
        c0 += __popcll(__ballot(lead && cnt == 1));
        c1 += __popcll(__ballot(lead && cnt == 2));
    }
    if ((threadIdx.x & 63) == 0) {
        wc[0][threadIdx.x >> 6] = c0;
        wc[1][threadIdx.x >> 6] = c1;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const int t = wc[threadIdx.x][0] + wc[threadIdx.x][1] + wc[threadIdx.x][2] + wc[threadIdx.x][3];
        if (t) atomicAdd(threadIdx.x ? &acc->n1 : &acc->n0, t);
    }
}

// accumulator and bucket counts; one writer per word
__global__ void stat_init_kernel(StatAcc *acc, int *cnt, int nb)
{
    int *p = reinterpret_cast<int *>(acc);
    const int nw = (int)(sizeof(StatAcc) / sizeof(int)), wf = (int)(offsetof(StatAcc, first) / sizeof(int));
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nw + nb; k += gridDim.x * blockDim.x) {
        if (k < nw) p[k] = (k == wf || k == wf + 1) ? -1 : 0;
        else cnt[k - nw] = 0;
    }
}

// GetHistogramMeanData (statisticsInfo_rc.cu:44-74), float arithmetic in bin order
float hist_mean(const int *h, int len, float pct)
{
    int mx = h[0];
    for (int i = 0; i < len; i++) mx = h[i] > mx ? h[i] : mx;
    pct = pct * (float)mx;
    float ws = 0.0f, os = 0.0f;
    for (int i = 0; i < len; i++) {
        const float v = (float)h[i];
        if (v >= pct) {
            ws += v * ((float)i + 0.5f);
            os += v;
        }
    }
    if (os == 0) os = 1;
    return ws / os;
}

// GetActivationDensity (statisticsInfo_rc.cu:17-41)
float activation_density(float r0, float r1, float radius_um)
{
    const float PI = 3.14159f;
    if (r0 <= 0.001f) r0 = 0.001f;
    if (r1 <= 0.001f) r1 = 0.001f;
    if (r0 > 1) r0 = 1;
    if (r1 > 1) r1 = 1;
    const float l0 = logf(r0);
    const float l1 = logf(r1 / PI / radius_um / radius_um);
    const float d0 = -l0 / PI / radius_um / radius_um;
    const float d1 = -l1 / PI / radius_um / radius_um;
    return r0 * d0 + (1.0f - r0) * d1;
}

}  // namespace

}  // namespace qcs

using namespace qcs;

extern "C" int qcs_loc_stats_dev(qcs_ctx *ctx, const float *d_loc, int n, qcs_loc_stats *out, void *stream)
{
    if (!ctx || !out || n < 0 || (n > 0 && !d_loc)) return fail(QCS_ERR_ARG, "invalid argument");
    memset(out, 0, sizeof(*out));
    if (n == 0) return QCS_OK;
    hipStream_t s = (hipStream_t)stream;
    const qcs_params &p = ctx->p;
    if (n > 1 << 27) return fail(QCS_ERR_ARG, "statistics of %d rows exceed the supported size", n);
    const float rad = (p.LocType == QCS_LOCTYPE_GS2D) ? 10.0f : 20.0f;
    Grid g;
    g.W = p.ImageWidth;
    g.H = p.ImageHigh;
    g.cell = rad * 1.0009765625f;
    g.ncx = (int)((float)p.ImageWidth / g.cell) + 2;
    g.r2 = rad * rad;
    for (g.lb = 8; g.lb < 24 && (1 << g.lb) < n; g.lb++) {}   // a bucket per molecule, as far as one scan goes
    const int nb = 1 << g.lb;
    // scratch: accumulator, entries, bucket counts, offsets (one more than buckets), scan sums
    const size_t acc_b = (sizeof(StatAcc) + 255) & ~(size_t)255, ent_b = (size_t)n * sizeof(float4);
    int rc;
    if ((rc = ctx->st_buf.ensure(acc_b + ent_b + sizeof(int) * (2 * (size_t)nb + 1 + scan_tile_count((size_t)nb) + 1))) ||
        (rc = ctx->pin_cnt.ensure(sizeof(StatAcc))))
        return rc;
    char *buf = ctx->st_buf.as<char>();
    StatAcc *acc = reinterpret_cast<StatAcc *>(buf), *h = ctx->pin_cnt.as<StatAcc>();
    float4 *ent = reinterpret_cast<float4 *>(buf + acc_b);
    int *cnt = reinterpret_cast<int *>(buf + acc_b + ent_b), *offs = cnt + nb, *tsum = offs + nb + 1;
    const dim3 gr((n + 255) / 256), blk(256);
    hipLaunchKernelGGL(stat_init_kernel, dim3(std::min((nb + 2047) / 2048 + 1, 1024)), blk, 0, s, acc, cnt, nb);
    hipLaunchKernelGGL(stat_rows_kernel, dim3(std::min((n + RT - 1) / RT, 512)), dim3(RT), 0, s, d_loc, n, acc);
    hipLaunchKernelGGL(stat_bins_kernel, gr, blk, 0, s, d_loc, n, g, acc, cnt, nullptr, nullptr);
    QCS_HIP(hipGetLastError());
    if ((rc = scan_exclusive(cnt, nb, offs, tsum, s, nullptr, offs + nb))) return rc;
    hipLaunchKernelGGL(stat_bins_kernel, gr, blk, 0, s, d_loc, n, g, acc, cnt, offs, ent);
    hipLaunchKernelGGL(stat_neigh_kernel, dim3(std::min((n + 15) / 16, NEIGH_BLOCKS)), blk, 0, s, ent, offs, g, nb, acc);
    QCS_HIP(hipGetLastError());
    QCS_HIP(hipMemcpyAsync(h, acc, sizeof(StatAcc), hipMemcpyDeviceToHost, s));
    QCS_HIP(hipStreamSynchronize(s));
    memcpy(out->hist_total_photon, h->hist[0], sizeof(out->hist_total_photon));
    memcpy(out->hist_loc_prec, h->hist[1], sizeof(out->hist_loc_prec));
    memcpy(out->hist_peak_snr, h->hist[2], sizeof(out->hist_peak_snr));
    memcpy(out->hist_psf_width, h->hist[3], sizeof(out->hist_psf_width));
    out->valid = h->valid;
    out->sum_loc_prec = h->sum[0];
    out->sum_peak_snr = h->sum[1];
    out->sum_psf_width = h->sum[2];
    out->sum_background = h->sum[3];
    const double vn = h->valid > 0 ? (double)h->valid : 1.0;
    out->mean_total_photon = (10000.0f / SL) * hist_mean(out->hist_total_photon, SB, 0.1f);
    out->mean_loc_prec = (float)(out->sum_loc_prec / vn);
    out->mean_peak_snr = (float)(out->sum_peak_snr / vn);
    out->mean_background = (float)(out->sum_background / vn);
    out->mean_psf_width = (float)(out->sum_psf_width / vn);
    out->mean_psf_width_ctl = out->mean_psf_width * (-out->mean_peak_snr);

    const FrameRange fr = frame_range(*h);
    out->density_first_frame = fr.fs;
    out->density_last_frame = fr.fe;
    if (fr.fe < fr.fs) return QCS_OK;
    const int kept = h->kept;
    out->density_total = kept;
    out->density_n0 = h->n0;
    out->density_n1 = h->n1;
    if (kept > 50) {
        const float r0 = (float)h->n0 / (float)kept, r1 = (float)h->n1 / (float)kept;
        float d = activation_density(r0, r1, rad * p.PixelSize / 1000);
        d = p.MultiEmitterFitEn ? d * d * 0.5098f + d * 0.6364f : d * d * 0.8082f + d * 0.519f;
        out->loc_density_2d = d;
    }
    return QCS_OK;
}
