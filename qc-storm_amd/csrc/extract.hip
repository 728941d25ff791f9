// extract.hip -- ROI extraction from uint16 sCMOS frames on gfx950.
//
// Reference (SE = MLEbfgs/bfgs_MLE_dll x64/bfgsMLE_dll/bfgsMLE_dll/SubregionExtraction):
//   FilterInit                    SE/LDROIExtraction_ImageFiltering.cu:22-81
//   ImageFiltering pass order     SE/LDROIExtraction_ImageFiltering.cu:85-121
//   gpuRemoveBackgroundIntensity  SE/LDROIExtraction_ImageFiltering.cu:125-282
//   gpuImageConv_Seperable_H / V  SE/LDROIExtraction_ImageFiltering.cu:286-470
//   ImageVarianceCalc             SE/LDROIExtraction.cu:140-177, ..._ImageFiltering.cu:503-544
//   gpuROIFindingLD               SE/LDROIExtraction_ROIExtraction.cu:25-177
//   gpuDetectedROIClasify         SE/LDROIExtraction_ROIExtraction.cu:181-253
//   gpuSubregionExtractionLD      SE/LDROIExtraction_ROIExtraction.cu:257-316
//   ExtractMolecules / ROIExtraction SE/LDROIExtraction.cu:30-138
//
// Pipeline for one call (any number of frames, batches of BatchedImageNum frames; no host
// synchronisation until the final count read):
//   1. walk_kernel<0>     background-removed values over each batch's variance region
//   2. var_reduce_kernel  exact integer sums of the variance samples per batch
//   3. walk_kernel<1>     one wave per 56-column strip walks down the rows: raw rows enter a
//                         16-row LDS ring, background removal, 5-tap H and V smoothing (uint16
//                         truncation after each pass, as the reference stores them), 3x3
//                         local-maximum test against the batch's thresholds.  Candidates and
//                         marks leave as one 56-bit ballot mask per row and strip; per-row
//                         candidate counts via integer atomics.
//   4. scan               exclusive prefix sum of the row counts -> raster-order offsets
//   5. batch_kernel       per-batch found / kept (capacity) / output offsets
//   6. emit_kernel        candidate (x, y) list in raster order
//   7. cut_kernel         detector classification (multi mode), raw R x R cut, header
//   8. WLE                PSF width, nearest neighbour (sorted sweep over the list), type
#include <string.h>
#include <algorithm>
#include <type_traits>
#include "qcs_internal.h"

namespace qcs {

int wle_launch_extract(const qcs_params &p, const uint16_t *d_rois, const int3 *d_xyb, int B, int H, const int *d_n, int cap,
                       float *d_wle, hipStream_t s);
void filter_taps_host(int R, int loc_type, int multi, float taps[5]);

// FilterInit (SE/LDROIExtraction_ImageFiltering.cu:22-81): host FP32 without contraction; the
// exponential is evaluated in double and rounded once.
void filter_taps_host(int R, int loc_type, int multi, float taps[5])
{
    volatile float s7 = 0.5f, s11 = 1.0f;
    float ss = s7 + ((float)(R - 7) * (s11 - s7)) / (float)(11 - 7);
    if (ss < 0.5f) ss = 0.5f;
    if (loc_type == QCS_LOCTYPE_AS3D) ss = ss * 1.5f;
    else if (multi == 0 && loc_type == QCS_LOCTYPE_GS2D) ss = ss * 1.2f;
    ss = -1.0f / ((2.0f * ss) * ss);
    const float ctr = 2.0f;
    for (int c = 0; c < 5; c++) {
        volatile float d = ((float)c - ctr) * ((float)c - ctr);
        volatile float arg = d * ss;
        taps[c] = (float)exp((double)arg);
    }
    float sum = 0.0f;
    for (int i = 0; i < 5; i++)
        for (int j = 0; j < 5; j++) {
            volatile float pr = taps[i] * taps[j];
            sum = sum + pr;
        }
    sum = sqrtf(1.0f / sum);
    for (int c = 0; c < 5; c++) taps[c] = taps[c] * sum;
}

struct ExtractConst {
    int W, H;              // frame size
    int B;                 // frames per batch
    int nframes;           // frames in this call
    int nbatch;
    int R;
    int loc_type, multi;
    int smooth;            // 0: detection on the background-removed image (2D multi mode)
    int batch_cap;         // candidates kept per batch
    int cap;               // output capacity
    int start_frame;
    int nseg;              // SEGW-column segments per row (one walking wave each)
    int walk_rows;         // image rows per walking wave of the full pass
    int var_rows;          // ... of the variance region's
    float taps[5];
    const int *start_dev;  // when set: the call's first frame number is read here at run time (graph replays)
};

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// rows of batch b and its first frame
__device__ __forceinline__ int batch_rows(const ExtractConst &c, int b)
{
    const int f0 = b * c.B;
    const int nb = (c.nframes - f0) < c.B ? (c.nframes - f0) : c.B;
    return nb * c.H;
}

// variance region of batch b: S x S samples at (cx + i, cy + j), each the minimum of the
// background-removed image at (X, Y), (X - S, Y), (X, Y - S), (X - S, Y - S)
// (ImageVarianceCalc, SE/LDROIExtraction.cu:140-177; gpuImageVarianceCalcOnSelectRegion,
// SE/LDROIExtraction_ImageFiltering.cu:503-533)
__device__ __forceinline__ int var_side(const ExtractConst &c, int BH)
{
    int sw = c.W / 2 - 5, sh = BH / 2 - 5;
    sw = sw > 256 ? 256 : sw;
    sh = sh > 256 ? 256 : sh;
    sw = sw < 1 ? 1 : sw;
    sh = sh < 1 ? 1 : sh;
    return sw < sh ? sw : sh;
}

__device__ __forceinline__ void batch_thresholds(const ExtractConst &c, const unsigned long long *sums, int b, int BH,
                                                 float &th, float &th1)
{
    const int S = var_side(c, BH);
    const double n = (double)S * (double)S;
    const double m1 = (double)sums[2 * b] / n, m2 = (double)sums[2 * b + 1] / n;
    float var = (float)(m2 - m1 * m1);
    var = (var < 100.0f) ? 100.0f : var;
    const float sd = sqrtf(var);
    if (c.loc_type == QCS_LOCTYPE_AS3D || (c.multi == 0 && c.loc_type == QCS_LOCTYPE_GS2D)) {
        th = 8.5f * sd;
        th1 = 3.5f * sd;
    } else {
        th = 9.5f * sd;
        th1 = 3.8f * sd;
    }
}

// ---- 1+2. row-walking filter wave ----------------------------------------------------------
// One wave (64 lanes, one column each) walks down a strip of the batched image.  Lane l owns
// column xc = x0 - 4 + l; the background sum needs raw columns xc-4..xc+4, so the raw rows in
// LDS are 72 wide (8 halo columns loaded by lanes 0..7).  Each stage narrows the valid lanes by
// its stencil reach: background sums on lanes 0..63, background-removed values on 1..62,
// H-smoothed values on 3..60, detection on 4..59 -- SEGW = 56 output columns per wave.
//
// A step handles 4 image rows r..r+3: the raw rows r+4..r+7 (loaded from HBM during the previous
// step) enter a 16-row LDS ring, then for each row r:
//   bk(r, x) = sum_{i<8} min(R(r-4, x-4+i), R(r-4+i, x+4), R(r+4, x+4-i), R(r+4-i, x-4))
//              with R the raw image, row/column indices clamped to the batch
//              (gpuRemoveBackgroundIntensity, SE/LDROIExtraction_ImageFiltering.cu:125-267);
//   tv(r, x) = uint16 trunc(max(raw - ((bk[xl] / 8 + bk[x] / 8) + bk[xr] / 8) / 3, 0)), xl/xr the
//              neighbours clamped to x's 32-column group.  The float expression equals the
//              integer max(raw - ceil((bk[xl] + bk[x] + bk[xr]) / 24), 0) exactly: the three
//              eighths sum exactly, s/3 rounds to within 2^-9 of S/24, and S/24 is either an
//              integer or at least 1/24 from one, so the truncation never changes;
//   hc(r, x) = uint16(min(fma-chain of tv(r, clamp(x-2+t)) * tap[t], 65535))      (H pass)
//   sv(y, x) = uint16(min(fma-chain of hc(clamp(y-2+t), x) * tap[t], 65535))      (V pass,
//              gpuImageConv_Seperable_H/V, SE/LDROIExtraction_ImageFiltering.cu:286-470);
//   detection of rows r-3..r once sv(r+1) exists (gpuROIFindingLD,
//   SE/LDROIExtraction_ROIExtraction.cu:25-164).
// Only the raw rows go through LDS (one barrier per step, after they are staged), as the 16-bit
// pairs (R(x), R(x+1)) of every column: the sums take two neighbouring terms per instruction from
// pairs that start at any column, and a pair read whole is an aligned word with one bank a lane.
// (Reading eight 16-bit columns at the lane's odd address as one 16-byte word kept the LDS busy 92% of
// the pass, 83% of it in stalls for the alignment.)  Everything else moves between lanes by DPP wave
// shifts, mostly inside the instruction that uses it -- the neighbours' background sums, tv of
// lanes l-2..l+2 for the H pass, sv of lanes l-1, l+1 for detection -- and between rows in registers;
// the lanes whose results are used never reach past the wave, and a strip at the image border takes
// its clamped columns by readlane.  Rows with no pixel at the threshold, most of them, stop there.
// What bounds the full pass is instruction issue: 32 frames of 2048 x 2048, 720 -> 410 us.
// MODE 0 computes tv only, over the variance region, into tvbuf; MODE 1 is the full pass.
// Wave shifts by one lane (DPP wave_shr:1 / wave_shl:1).  Bound control writes 0 where the
// source lane is outside the wave (lane 0 for prev, lane 63 for next), so no old value is needed.
__device__ __forceinline__ int lane_prev(int v) { return __builtin_amdgcn_mov_dpp(v, 0x138, 0xf, 0xf, true); }
__device__ __forceinline__ int lane_next(int v) { return __builtin_amdgcn_mov_dpp(v, 0x130, 0xf, 0xf, true); }
__device__ __forceinline__ float lane_prev(float v) { return __int_as_float(lane_prev(__float_as_int(v))); }
__device__ __forceinline__ float lane_next(float v) { return __int_as_float(lane_next(__float_as_int(v))); }

// acc[k] += x[k] of lane l - 1 (PREV) or l + 1, times w, for four rows: the shift is part of the
// instruction (the compiler makes it a move of its own before a multiply-add).  A DPP operand needs two
// wait states after the instruction that wrote it, once for the four.  acc[0] is written before x[1] is
// read, so no sum may share a register with an input of the same value ("+&v").
template <bool PREV>
__device__ __forceinline__ void fma_shifted(float (&acc)[4], const float (&x)[4], float w)
{
    if constexpr (PREV)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %0, %4, %8 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
            "v_fmac_f32_dpp %1, %5, %8 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
            "v_fmac_f32_dpp %2, %6, %8 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
            "v_fmac_f32_dpp %3, %7, %8 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1"
            : "+&v"(acc[0]), "+&v"(acc[1]), "+&v"(acc[2]), "+&v"(acc[3]) : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(w));
    else
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %0, %4, %8 wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
            "v_fmac_f32_dpp %1, %5, %8 wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
            "v_fmac_f32_dpp %2, %6, %8 wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
            "v_fmac_f32_dpp %3, %7, %8 wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1"
            : "+&v"(acc[0]), "+&v"(acc[1]), "+&v"(acc[2]), "+&v"(acc[3]) : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(w));
}

// two 16-bit lanes of a 32-bit register
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2 as_u16x2(uint32_t w) { return __builtin_bit_cast(u16x2, w); }
__device__ __forceinline__ u16x2 swap16(u16x2 v) { return __builtin_shufflevector(v, v, 1, 0); }
__device__ __forceinline__ u16x2 pmin16(u16x2 a, u16x2 b) { return __builtin_elementwise_min(a, b); }
constexpr u16x2 kOnes16 = {1, 1};
typedef uint32_t __attribute__((may_alias)) u32_alias;

constexpr int SEGW = 56;             // output columns per wave
constexpr int RAWW = 72;             // raw columns per row in LDS
constexpr int ROWW = 2 * RAWW + 2;   // 16-bit words per row of pairs: column x is words 2x + 2 and 2x + 1
constexpr int VAR_MAX = 512;         // region side bound (2 * 256)

constexpr int WALK_RS = 4;   // image rows per step
constexpr int WALK_NR = 16;  // raw ring rows (a step needs rows r-4 .. r+RS+3); power of two

// The walk of one strip.  BORDER: a lane of 1..62 has an H-pass column clamped to the image
// (the strips at the left and right image edges); only those carry the clamping code.
template <int MODE, bool SMOOTH, bool BORDER>
__device__ __forceinline__ void walk_body(const uint16_t *__restrict__ frames, const ExtractConst &c,
                                          const unsigned long long *__restrict__ var_sums,
                                          uint16_t *__restrict__ tvbuf,
                                          unsigned long long *__restrict__ cand_mask,
                                          unsigned long long *__restrict__ mark_mask,
                                          int *__restrict__ row_count, uint16_t (*raw)[ROWW])
{
    constexpr int RS = WALK_RS;
    constexpr int NR = WALK_NR;

    const int b = blockIdx.z;
    const int BH = batch_rows(c, b);
    const int seg = blockIdx.x;
    const int W = c.W;
    const uint16_t *img = frames + (size_t)b * c.B * c.H * W;
    const int l = threadIdx.x;

    int x0, ys, ye, rb, rlast;
    int S = 0, rx0 = 0, ry0 = 0;
    if (MODE == 0) {
        S = var_side(c, BH);
        rx0 = W / 2 - S;
        ry0 = BH / 2 - S;
        x0 = rx0 + blockIdx.x * SEGW;
        if (x0 >= rx0 + 2 * S) return;
        ys = ry0 + blockIdx.y * c.var_rows;
        if (ys >= ry0 + 2 * S) return;
        ye = min(ys + c.var_rows, ry0 + 2 * S);
        rb = ys;          // steps compute tv rows r .. r+3
        rlast = ye - 1;
    } else {
        x0 = seg * SEGW;
        ys = blockIdx.y * c.walk_rows;
        if (ys >= BH) return;
        ye = min(ys + c.walk_rows, BH);
        rb = ys - 4;      // step r: hc rows r..r+3, sv rows r-2..r+1, detection rows r-3..r
        rlast = ye + 2;
    }
    // ring slots are relative to rb; a step starts at rb + 4 * (4n + PH), so in interior steps the
    // slots are compile-time functions of the phase PH
    auto slot = [&](int v) { return (v - rb + 2 * NR) & (NR - 1); };
    const int xc = x0 - 4 + l;
    const int xcl = clampi(xc, 0, W - 1);
    // halo columns: lanes 0..3 -> x0-8+l (slot l), lanes 4..7 -> x0+60+(l-4) (slot 68+l-4)
    const int hx = (l < 4) ? clampi(x0 - 8 + l, 0, W - 1) : clampi(x0 + 56 + l, 0, W - 1);
    const int hslot = (l < 4) ? l : 64 + l;
    auto ldp = [&](const uint16_t *src, uint16_t &main, uint16_t &halo) {
        main = src[xcl];
        halo = (l < 8) ? src[hx] : (uint16_t)0;
    };
    auto ld = [&](int v, uint16_t &main, uint16_t &halo) { ldp(img + (unsigned)(clampi(v, 0, BH - 1) * W), main, halo); };

    // Column x of a row: the first half of pair x and the second half of pair x - 1.  The latter's place
    // is kept from the compiler, which else joins the two into one store at an odd word: any LDS access
    // that is not aligned to its size takes 64 cycles, one a lane, an aligned one 3 to 5.
    int m2 = 2 * (l + 4) + 1, h2 = 2 * hslot + 1;
    asm("" : "+v"(m2), "+v"(h2));
    auto put = [&](int rs, uint16_t m, uint16_t h) {
        raw[rs][2 * (l + 4) + 2] = m;
        raw[rs][m2] = m;
        if (l < 8) {
            raw[rs][2 * hslot + 2] = h;
            raw[rs][h2] = h;
        }
    };
    auto col = [&](int rs, int x) { return (uint32_t)raw[rs][2 * x + 2]; };
    auto pair = [&](int rs, int x) { return *reinterpret_cast<const u32_alias *>(&raw[rs][2 * x + 2]); };
    for (int v = rb - 4; v < rb + 4; v++) {
        uint16_t m, h;
        ld(v, m, h);
        put(slot(v), m, h);
    }
    uint16_t pf[RS], pfh[RS];
#pragma unroll
    for (int k = 0; k < RS; k++) ld(rb + 4 + k, pf[k], pfh[k]);

    float th = 0.0f, th1 = 0.0f;
    float tap[5] = {0, 0, 0, 0, 0};
    if (MODE == 1) {
        batch_thresholds(c, var_sums, b, BH, th, th1);
#pragma unroll
        for (int t = 0; t < 5; t++) tap[t] = c.taps[t];
    }
    const int g0 = xc & ~31;
    const int li = max(min(((xc - 1 < g0) ? g0 : xc - 1) - (x0 - 4), 63), 0);
    const int ri = max(min(((xc + 1 > g0 + 31) ? g0 + 31 : xc + 1) - (x0 - 4), 63), 0);
    // weights of the three sums in the background, -1/24 each
    const float wc = -(float)(1 + (li == l ? 1 : 0) + (ri == l ? 1 : 0)) / 24.0f, wl = li == l ? 0.0f : -1.0f / 24.0f,
                wr = ri == l ? 0.0f : -1.0f / 24.0f;
    int hci[5];   // H-pass source lanes (columns clamped to the image)
#pragma unroll
    for (int t = 0; t < 5; t++) hci[t] = max(min(clampi(xc - 2 + t, 0, W - 1) - (x0 - 4), 63), 0);
    // lanes of image columns 0 and W-1 when the strip reaches a border (the H pass clamps to them)
    const int lane_lo = max(min(0 - (x0 - 4), 63), 0), lane_hi = max(min(W - 1 - (x0 - 4), 63), 0);
    const int half = c.R / 2;
    const bool out_lane = (l >= 4 && l < 4 + SEGW);
    const bool det_col = out_lane && xc < W && xc >= half && xc < W - half;
    const float thc = det_col ? th : 3.0e38f;   // no value reaches it outside the detection columns
    const int ylo = max(ys - 1, 0), yhi = min(ye, BH - 1);   // sv rows this wave needs
    unsigned long long *cmask = cand_mask + (size_t)b * c.B * c.H * c.nseg + seg;
    unsigned long long *mmask = mark_mask + (size_t)b * c.B * c.H * c.nseg + seg;
    int *rcount = row_count + (size_t)b * c.B * c.H;
    const int nseg = c.nseg, H = c.H;
    int ryd = ((rb - 3) % H + H) % H;   // frame row of detection row r-3 for the current step
    // 16-bit pairs (col[m], col[m+1]) of raw column xc+4 from row r-4 and of column xc-4 from row r-3.  A
    // step keeps the previous step's six newest; of the new ones, column xc+4 is in the pairs that
    // the sums read (rows r+4 .. r+6 in this step's, r+3 in the last step's), and so is the centre
    // of the rows (in the last step's).
    uint32_t CR[RS + 6], CL[RS + 6], b3, cen[RS];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 6; m++) {   // as a step before the first would leave them
        CR[RS + m] = col(slot(rb + m - 4), l + 8) | col(slot(rb + m - 3), l + 8) << 16;
        CL[RS + m] = col(slot(rb + m - 3), l) | col(slot(rb + m - 2), l) << 16;
    }
    b3 = col(slot(rb + 3), l + 8) << 16;
#pragma unroll
    for (int k = 0; k < RS; k++) cen[k] = col(slot(rb + k), l + 4) << 16;
    // the lane's H-smoothed rows r-4 .. r+RS-1 and V-smoothed rows r-4 .. r+RS-3: the last RS rows are
    // this step's; detection takes lanes l-1 and l+1 of the latter by DPP wave shifts
    float hcr[RS + 4], svr[RS + 2];
#pragma unroll
    for (int i = 0; i < RS + 4; i++) hcr[i] = 0.0f;
#pragma unroll
    for (int i = 0; i < RS + 2; i++) svr[i] = 0.0f;
    const unsigned moff = (unsigned)l * (unsigned)c.nseg;   // lanes 0 .. RS-1: their row of a step's masks

    // One step of 4 rows.  EDGE: rows near the batch or walk ends (bounds checks, clamped rows,
    // dynamic ring slots); otherwise every row is in range and PH fixes the ring slots.
    auto step = [&](int r, auto edge_tag, auto ph_tag) {
        constexpr bool EDGE = decltype(edge_tag)::value;
        constexpr int PH = decltype(ph_tag)::value;
        auto rs = [&](int off) { if constexpr (EDGE) return slot(r + off); else return (4 * PH + off + 2 * NR) & (NR - 1); };
        // stage rows r+4 .. r+7 (loaded one step ago), then prefetch rows r+8 .. r+11
#pragma unroll
        for (int k = 0; k < RS; k++) put(rs(4 + k), pf[k], pfh[k]);
        if constexpr (EDGE) {
#pragma unroll
            for (int k = 0; k < RS; k++) ld(r + 8 + k, pf[k], pfh[k]);
        } else {
            const uint16_t *p8 = img + (unsigned)((r + 8) * W);
#pragma unroll
            for (int k = 0; k < RS; k++) ldp(p8 + k * W, pf[k], pfh[k]);
        }
        __syncthreads();
        // background sums of rows r .. r+3
#pragma unroll
        for (int m = 0; m < 6; m++) {
            CR[m] = CR[m + RS];
            CL[m] = CL[m + RS];
        }
        // Two terms per instruction: term i takes rA[l+i], colR[k+i], rB[l+8-i] and colL[k+7-i],
        // so terms 2j and 2j+1 read the 16-bit pairs (rA[l+2j], rA[l+2j+1]) and
        // (colR[k+2j], colR[k+2j+1]) in order and (rB[l+7-2j], rB[l+8-2j]) and
        // (colL[k+6-2j], colL[k+7-2j]) with their halves swapped.  Packed 16-bit minima, then a
        // dot product with (1, 1) adds both halves into the 32-bit sum.
        float bkv[RS];
        uint32_t cn[RS], cl = CL[5] >> 16;
#pragma unroll
        for (int k = 0; k < RS; k++) {
            CR[6 + k] = __builtin_amdgcn_perm(b3, CR[5 + k], 0x07060302);   // the upper halves of both
            const uint32_t c = col(rs(k + 4), l);
            CL[6 + k] = cl | c << 16;
            cl = c;
            uint32_t bk = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t bp = pair(rs(k + 4), l + 7 - 2 * j);
                if (j == 0) b3 = bp;
                if (j == 2) cn[k] = bp;
                const u16x2 m1 = pmin16(as_u16x2(pair(rs(k - 4), l + 2 * j)), as_u16x2(CR[k + 2 * j]));
                const u16x2 m2 = pmin16(swap16(as_u16x2(bp)), swap16(as_u16x2(CL[k + 6 - 2 * j])));
                bk = __builtin_amdgcn_udot2(pmin16(m1, m2), kOnes16, bk, false);
            }
            bkv[k] = (float)bk;
        }
        // tv = max(raw - ceil(S / 24), 0), S the three sums' total, as trunc(max(raw - S / 24 + 1/48, 0)) in
        // float: raw - S / 24 is a multiple of 1/24, so with the 1/48 it is that far from every integer,
        // and the four roundings (2^-9 each, no value reaches 2^16) and those of the weights
        // (65535 * 2^-24) add up to less than 0.012.
        float tvk[RS];
#pragma unroll
        for (int k = 0; k < RS; k++) {
            tvk[k] = __builtin_fmaf(bkv[k], wc, (float)(cen[k] >> 16) + 1.0f / 48.0f);
            cen[k] = cn[k];
        }
        fma_shifted<true>(tvk, bkv, wl);
        fma_shifted<false>(tvk, bkv, wr);
#pragma unroll
        for (int k = 0; k < RS; k++) tvk[k] = __builtin_truncf(fmaxf(tvk[k], 0.0f));
        if constexpr (MODE == 0) {
#pragma unroll
            for (int k = 0; k < RS; k++) {
                const int v = r + k;
                if (out_lane && v < ye && xc < rx0 + 2 * S)
                    tvbuf[(size_t)b * VAR_MAX * VAR_MAX + (size_t)(v - ry0) * VAR_MAX + (xc - rx0)] = (uint16_t)tvk[k];
            }
            return;
        }
        // H pass.  The values of lanes l-2 .. l+2 come by DPP wave shifts; a strip at the image border
        // takes its clamped columns from the border lane (readlane).  Lanes 3 .. 60, the ones whose
        // results are used, never read a lane outside the wave.  Rows outside the batch repeat its
        // first and last row.
        float h0 = hcr[RS], h1 = hcr[RS + 1], h2 = hcr[RS + 2], h3 = hcr[RS + 3], hn[RS];
        float hv[RS];
        if constexpr (!SMOOTH) {
#pragma unroll
            for (int k = 0; k < RS; k++) hv[k] = tvk[k];
        } else {
            // no value is negative: the first tap's product has the bits of fma(src, tap, 0)
            float m1[RS], p1[RS];   // lanes l-1, l+1
#pragma unroll
            for (int k = 0; k < RS; k++) {
                m1[k] = lane_prev(tvk[k]);
                p1[k] = lane_next(tvk[k]);
            }
            if constexpr (BORDER) {
#pragma unroll
                for (int k = 0; k < RS; k++) {
                    const float v0 = tvk[k];
                    float src[5] = {lane_prev(m1[k]), m1[k], v0, p1[k], lane_next(p1[k])};
                    const float vl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v0), lane_lo));
                    const float vr = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v0), lane_hi));
#pragma unroll
                    for (int t = 0; t < 5; t++) src[t] = hci[t] == lane_lo ? vl : (hci[t] == lane_hi ? vr : src[t]);
                    float acc = src[0] * tap[0];
#pragma unroll
                    for (int t = 1; t < 5; t++) acc = __builtin_fmaf(src[t], tap[t], acc);
                    hv[k] = acc;
                }
            } else {
#pragma unroll
                for (int k = 0; k < RS; k++) hv[k] = 0.0f;
                fma_shifted<true>(hv, m1, tap[0]);
#pragma unroll
                for (int k = 0; k < RS; k++)
                    hv[k] = __builtin_fmaf(p1[k], tap[3], __builtin_fmaf(tvk[k], tap[2], __builtin_fmaf(m1[k], tap[1], hv[k])));
                fma_shifted<false>(hv, p1, tap[4]);
            }
#pragma unroll
            for (int k = 0; k < RS; k++) hv[k] = __builtin_truncf(fminf(hv[k], 65535.0f));   // >= 0: the uint16 store's truncation
        }
#pragma unroll
        for (int k = 0; k < RS; k++) {
            if (EDGE && r + k >= BH) {   // uniform
                hn[k] = k > 0 ? hn[k - 1] : h3;
                continue;
            }
            hn[k] = hv[k];
            if (EDGE && r + k <= 0) {   // uniform
                h0 = h1 = h2 = h3 = hv[k];
#pragma unroll
                for (int i = 0; i < k; i++) hn[i] = hv[k];
            }
        }
        hcr[0] = h0;
        hcr[1] = h1;
        hcr[2] = h2;
        hcr[3] = h3;
#pragma unroll
        for (int k = 0; k < RS; k++) hcr[RS + k] = hn[k];
        // V pass: sv rows r-2 .. r+1, held as integral floats
#pragma unroll
        for (int k = 0; k < RS; k++) {
            float sv = hcr[k + 2];
            if constexpr (SMOOTH) {
                float acc = hcr[k] * tap[0];
#pragma unroll
                for (int t = 1; t < 5; t++) acc = __builtin_fmaf(hcr[k + t], tap[t], acc);
                sv = __builtin_truncf(fminf(acc, 65535.0f));
            }
            if (EDGE && (r - 2 + k < ylo || r - 2 + k > yhi)) sv = 0.0f;   // uniform
            svr[2 + k] = sv;
        }
        // detection rows r-3 .. r (sv rows r-4 .. r+1) that have a pixel at the threshold; the shifts
        // run on the whole wave, ahead of the per-lane tests.  The eight-neighbour count s8 >= 7 of the
        // reference is "at most one neighbour <= th1": with cv >= th > th1 the centre is not one of them, so
        // it is the 3 x 3 count of the low flags (column sums, then lanes l-1, l, l+1) being at most one.
        unsigned long long hit[RS];
        bool any = false;
#pragma unroll
        for (int k = 0; k < RS; k++) {
            int ry = ryd + k;
            ry = ry >= H ? ry - H : ry;
            const unsigned long long m = __ballot(svr[k + 1] >= thc);
            hit[k] = ry >= half && ry < H - half ? m : 0ull;
            any |= hit[k] != 0;
        }
        if (!EDGE && !any) {   // uniform
            if (l < RS) {
                cmask[(size_t)(r - 3) * nseg + moff] = 0;
                mmask[(size_t)(r - 3) * nseg + moff] = 0;
            }
        } else {
#pragma unroll
            for (int k = 0; k < RS; k++) {
                const int d = r - 3 + k;
                if (EDGE && (d < ys || d >= ye)) continue;   // uniform
                unsigned long long cm = 0, mm = 0;
                const float p01 = svr[k], cv = svr[k + 1], p21 = svr[k + 2];
                if (hit[k] && __ballot((cv >= thc) & (cv > p01) & (cv >= p21))) {   // uniform
                    const float p00 = lane_prev(p01), p02 = lane_next(p01);
                    const float p10 = lane_prev(cv), p12 = lane_next(cv);
                    const float p20 = lane_prev(p21), p22 = lane_next(p21);
                    const int lc = (p01 > th1 ? 0 : 1) + (cv > th1 ? 0 : 1) + (p21 > th1 ? 0 : 1);
                    const int low9 = lane_prev(lc) + lc + lane_next(lc);
                    const bool sin4 = (cv > p01) & (cv >= p12) & (cv >= p21) & (cv > p10);
                    const bool a = cv > p00, bb = cv > p02, cc = cv > p20, dd = cv > p22;
                    const bool sout3 = (a & bb & (cc | dd)) | (cc & dd & (a | bb));
                    const bool mark = (cv >= thc) & (low9 <= 1) & sin4 & sout3;
                    cm = (__ballot(mark & a & bb & cc & dd) >> 4) & ((1ULL << SEGW) - 1);
                    mm = (__ballot(mark) >> 4) & ((1ULL << SEGW) - 1);
                }
                if (l == 0) {
                    cmask[(size_t)d * nseg] = cm;
                    mmask[(size_t)d * nseg] = mm;
                    if (cm) atomicAdd(&rcount[d], __popcll(cm));
                }
            }
        }
        svr[0] = svr[RS];
        svr[1] = svr[RS + 1];
    };

    using E = std::true_type;
    using I = std::false_type;
    for (int r = rb; r <= rlast; r += RS) {
        bool edge;
        if (MODE == 0) edge = (r - 4 < 0) || (r + 11 > BH - 1) || (r + RS - 1 >= ye);
        else edge = (r - 4 < 0) || (r + 11 > BH - 1) || (r - 2 < ylo) || (r + 1 > yhi) || (r - 3 < ys) || (r >= ye);
        if (edge) {
            step(r, E{}, std::integral_constant<int, 0>{});
        } else {
            switch (((r - rb) >> 2) & 3) {
            case 0: step(r, I{}, std::integral_constant<int, 0>{}); break;
            case 1: step(r, I{}, std::integral_constant<int, 1>{}); break;
            case 2: step(r, I{}, std::integral_constant<int, 2>{}); break;
            default: step(r, I{}, std::integral_constant<int, 3>{}); break;
            }
        }
        ryd += RS;
        ryd = ryd >= H ? ryd - H : ryd;
    }
}

// The full pass is held to five waves per SIMD (at most 96 VGPRs, no spills; six spill): issue slots are
// 85% taken.
template <int MODE, bool SMOOTH>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(MODE == 1 ? 5 : 1))) walk_kernel(const uint16_t *__restrict__ frames, ExtractConst c,
                                                  const unsigned long long *__restrict__ var_sums,
                                                  uint16_t *__restrict__ tvbuf,
                                                  unsigned long long *__restrict__ cand_mask,
                                                  unsigned long long *__restrict__ mark_mask,
                                                  int *__restrict__ row_count)
{
    __shared__ __align__(4) uint16_t raw[WALK_NR][ROWW];
    const int xs = (int)blockIdx.x * SEGW;
    if (MODE == 1 && (xs - 4 + 1 < 2 || xs - 4 + 62 > c.W - 3))   // uniform
        walk_body<MODE, SMOOTH, true>(frames, c, var_sums, tvbuf, cand_mask, mark_mask, row_count, raw);
    else
        walk_body<MODE, SMOOTH, false>(frames, c, var_sums, tvbuf, cand_mask, mark_mask, row_count, raw);
}

// integer sums of the variance samples of each batch from the region's background-removed values: a
// work-group takes every VAR_BLOCKS-th row of samples (S <= 256: one a thread), four rows at the most,
// whose loads are all in flight together (32 regions: 18 -> 11 us)
constexpr int VAR_BLOCKS = 64;
__global__ void __launch_bounds__(256) var_reduce_kernel(ExtractConst c, const uint16_t *__restrict__ tvbuf,
                                                         unsigned long long *__restrict__ sums)
{
    __shared__ unsigned long long sh[2][4];
    const int b = blockIdx.y;
    const int BH = batch_rows(c, b);
    const int S = var_side(c, BH);
    const uint16_t *t = tvbuf + (size_t)b * VAR_MAX * VAR_MAX;
    const int i = threadIdx.x;
    unsigned long long s1 = 0, s2 = 0;
    if (i < S) {
        // sample (X, Y) = (cx + i, cy + j), region origin (cx - S, cy - S)
        int v[256 / VAR_BLOCKS];
#pragma unroll
        for (int q = 0; q < 256 / VAR_BLOCKS; q++) {
            const int j = blockIdx.x + q * VAR_BLOCKS;
            v[q] = 0;
            if (j < S) {
                const int d1 = t[(size_t)(S + j) * VAR_MAX + S + i], d2 = t[(size_t)(S + j) * VAR_MAX + i];
                const int d3 = t[(size_t)j * VAR_MAX + S + i], d4 = t[(size_t)j * VAR_MAX + i];
                v[q] = min(min(d1, d2), min(d3, d4));
            }
        }
#pragma unroll
        for (int q = 0; q < 256 / VAR_BLOCKS; q++) {
            s1 += (unsigned long long)v[q];
            s2 += (unsigned long long)v[q] * (unsigned long long)v[q];
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        s1 += __shfl_down(s1, off, 64);
        s2 += __shfl_down(s2, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = s1;
        sh[1][threadIdx.x >> 6] = s2;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const unsigned long long *p = sh[threadIdx.x];
        const unsigned long long s = (p[0] + p[1]) + (p[2] + p[3]);
        if (s) atomicAdd(&sums[2 * b + threadIdx.x], s);
    }
}

// ---- 3. exclusive scan of int counts ----------------------------------------------------------
// Items at and past *n_dev count as zero.  Up to SCAN_ONE items, one tile of 16 waves, are one launch
// (4,096 items 3.7 us); more items take two, tile totals and then the tiles, each of which adds up the
// totals before it: 20,480 items 9.3 us and 65,536 items 9.6 us, where one work-group walking the
// tiles takes 13 and 35 us, and tile totals, their scan and an addition were three launches of 4 us.
constexpr int SCAN_BLOCK = 256, SCAN_ITEMS = 16, SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;
constexpr int SCAN_ONE_T = 1024, SCAN_ONE = SCAN_ONE_T * SCAN_ITEMS;

__device__ __forceinline__ int wave_inclusive_sum(int v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

// One tile of 16 items a thread over W waves: chunk c of the tile is 4 consecutive items a thread, so a
// wave's loads cover whole lines.  v becomes each item's prefix within the tile; returns the tile's
// sum.  sh: 4 W + 1 ints.
template <int W>
__device__ __forceinline__ int tile_exclusive_sum(int (&v)[4][4], int *sh)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int pre[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const int s = (v[c][0] + v[c][1]) + (v[c][2] + v[c][3]);
        const int incl = wave_inclusive_sum(s);
        if (lane == 63) sh[c * W + w] = incl;
        pre[c] = incl - s;
    }
    __syncthreads();
    if (w == 0) {
        const int t = lane < 4 * W ? sh[lane] : 0;
        const int incl = wave_inclusive_sum(t);
        if (lane < 4 * W) sh[lane] = incl - t;
        if (lane == 63) sh[4 * W] = incl;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; c++) {
        int p = pre[c] + sh[c * W + w];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int x = v[c][k];
            v[c][k] = p;
            p += x;
        }
    }
    return sh[4 * W];
}

template <int W>
__device__ __forceinline__ void tile_load(int (&v)[4][4], const int *__restrict__ in, int base, int m)
{
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = base + (c * W * 64 + (int)threadIdx.x) * 4 + k;
            v[c][k] = i < m ? in[i] : 0;
        }
}

template <int W>
__device__ __forceinline__ void tile_store(const int (&v)[4][4], int *__restrict__ out, int base, int n, int add)
{
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = base + (c * W * 64 + (int)threadIdx.x) * 4 + k;
            if (i < n) out[i] = v[c][k] + add;
        }
}

// where the grand total goes besides tile_sums[ntiles]: *out = (add: *out +) total
struct ScanTotal {
    int *out;
    int add;
};
__device__ __forceinline__ void scan_put_total(const ScanTotal &t, int total)
{
    if (t.out) *t.out = t.add ? *t.out + total : total;
}

__global__ void __launch_bounds__(SCAN_ONE_T) scan_one_kernel(const int *__restrict__ in, int n, const int *__restrict__ n_dev,
                                                              int *__restrict__ out, int *__restrict__ total, ScanTotal tot)
{
    constexpr int W = SCAN_ONE_T / 64;
    __shared__ int sh[4 * W + 1];
    int v[4][4];
    tile_load<W>(v, in, 0, n_dev ? min(*n_dev, n) : n);
    const int all = tile_exclusive_sum<W>(v, sh);
    tile_store<W>(v, out, 0, n, 0);
    if (threadIdx.x == 0) {
        *total = all;
        scan_put_total(tot, all);
    }
}

// sum of v over a work-group of SCAN_BLOCK threads; sh: one int a wave
__device__ __forceinline__ int block_sum(int v, int *sh)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    v = 0;
#pragma unroll
    for (int w = 0; w < SCAN_BLOCK / 64; w++) v += sh[w];
    return v;
}

__global__ void __launch_bounds__(SCAN_BLOCK) scan_tiles_kernel(const int *__restrict__ in, int n, const int *__restrict__ n_dev,
                                                                int *__restrict__ tile_sums)
{
    __shared__ int sh[SCAN_BLOCK / 64];
    const int m = n_dev ? min(*n_dev, n) : n;
    int v[4][4], s = 0;
    tile_load<SCAN_BLOCK / 64>(v, in, blockIdx.x * SCAN_TILE, m);
#pragma unroll
    for (int c = 0; c < 4; c++) s += (v[c][0] + v[c][1]) + (v[c][2] + v[c][3]);
    s = block_sum(s, sh);
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = s;
}

// total at tile_sums[ntiles]
__global__ void __launch_bounds__(SCAN_BLOCK) scan_apply_kernel(const int *__restrict__ in, int n, const int *__restrict__ n_dev,
                                                                int *__restrict__ out, int *__restrict__ tile_sums, int ntiles,
                                                                ScanTotal tot)
{
    constexpr int W = SCAN_BLOCK / 64;
    __shared__ int sh[4 * W + 1], shb[W];
    const int m = n_dev ? min(*n_dev, n) : n;
    int v[4][4], s = 0;
    tile_load<W>(v, in, blockIdx.x * SCAN_TILE, m);
    for (int t = threadIdx.x; t < (int)blockIdx.x; t += SCAN_BLOCK) s += tile_sums[t];
    const int before = block_sum(s, shb);
    const int all = tile_exclusive_sum<W>(v, sh);
    tile_store<W>(v, out, blockIdx.x * SCAN_TILE, n, before);
    if (threadIdx.x == 0 && (int)blockIdx.x == ntiles - 1) {
        tile_sums[ntiles] = before + all;
        scan_put_total(tot, before + all);
    }
}

// ---- 4. per-batch bookkeeping ----------------------------------------------------------------
// info layout: [0] kept total, [1] found total, then per batch b: found, kept, out offset
// One wave, a batch a lane: a batch's candidates are cut off at its own capacity, and all batches' at the
// call's, which is the prefix sum of the former cut off.
__global__ void __launch_bounds__(64) batch_kernel(ExtractConst c, const int *__restrict__ row_off, const int *__restrict__ tile_sums,
                                                   int nrows, int ntiles, int *__restrict__ info)
{
    const int lane = threadIdx.x, total = tile_sums[ntiles];
    int out = 0;   // candidates of the chunks before, not cut off
    for (int b0 = 0; b0 < c.nbatch; b0 += 64) {
        const int b = b0 + lane;
        int found = 0, want = 0;
        if (b < c.nbatch) {
            const int r0 = b * c.B * c.H, r1 = r0 + batch_rows(c, b);
            found = (r1 < nrows ? row_off[r1] : total) - row_off[r0];
            want = min(found, c.batch_cap);
        }
        const int incl = wave_inclusive_sum(want), before = out + incl - want;
        if (b < c.nbatch) {
            info[2 + 3 * b + 0] = found;
            info[2 + 3 * b + 1] = max(min(want, c.cap - before), 0);
            info[2 + 3 * b + 2] = min(before, c.cap);
        }
        out += __shfl(incl, 63, 64);
    }
    if (lane == 0) {
        info[0] = min(out, c.cap);
        info[1] = total;
    }
}

// ---- 5. candidate list in raster order -------------------------------------------------------
// One wave per EMIT_U stacked rows, whose loads are in flight together: lane s takes segment s's
// candidate mask (coalesced loads), and a wave prefix sum of the masks' popcounts gives each segment
// its first slot, so a row's candidates come out in raster order (65,536 rows with some six candidates each: 19 -> 15 us).
constexpr int EMIT_WAVES = 4, EMIT_U = 4;
__global__ void __launch_bounds__(64 * EMIT_WAVES) emit_kernel(ExtractConst c, const unsigned long long *__restrict__ cand_mask,
                                                               const int *__restrict__ row_off, int nrows,
                                                               const int *__restrict__ info, int3 *__restrict__ xyb)
{
    const int row0 = (blockIdx.x * EMIT_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * EMIT_U, lane = threadIdx.x & 63;
    unsigned long long m0[EMIT_U];
    int off[EMIT_U];
#pragma unroll
    for (int u = 0; u < EMIT_U; u++) {
        const int row = row0 + u;
        const bool in = row < nrows;
        m0[u] = in && lane < c.nseg ? cand_mask[(size_t)row * c.nseg + lane] : 0ull;
        off[u] = in ? row_off[row] : 0;
    }
#pragma unroll
    for (int u = 0; u < EMIT_U; u++) {
        const int row = row0 + u;
        if (row >= nrows || (c.nseg <= 64 && __ballot(m0[u] != 0) == 0)) continue;   // uniform
        const int b = row / (c.B * c.H);
        const int r0 = b * c.B * c.H;
        const int kept = info[2 + 3 * b + 1], out0 = info[2 + 3 * b + 2];
        int base = off[u] - row_off[r0];
        const int y = row - r0;   // batch-relative row
        for (int s0 = 0; s0 < c.nseg; s0 += 64) {
            const int sgi = s0 + lane;
            unsigned long long m = s0 == 0 ? m0[u] : ((sgi < c.nseg) ? cand_mask[(size_t)row * c.nseg + sgi] : 0ull);
            const int cnt = __popcll(m);
            const int incl = wave_inclusive_sum(cnt);
            int local = base + incl - cnt;
            while (m) {
                const int bit = __ffsll((long long)m) - 1;
                m &= m - 1;
                if (local < kept) xyb[out0 + local] = make_int3(sgi * SEGW + bit, y, b);
                local++;
            }
            base += __shfl(incl, 63, 64);
        }
    }
}

// ---- 6. classification + cut -----------------------------------------------------------------
__device__ __forceinline__ int mark_count(const unsigned long long *mark, int nseg, size_t row, int xa, int xb)
{
    // number of marks in [xa, xb] of one stacked row (segments of SEGW columns)
    int cnt = 0;
    for (int sgi = xa / SEGW; sgi <= xb / SEGW; sgi++) {
        unsigned long long m = mark[row * nseg + sgi];
        const int lo = sgi * SEGW;
        if (xa > lo) m &= ~0ULL << (xa - lo);
        if (xb < lo + SEGW - 1) m &= ~0ULL >> (63 - (xb - lo));
        cnt += __popcll(m);
    }
    return cnt;
}

// a mark in columns x - half .. x + half of one row's segment masks (two at the most: 2 half + 1 < SEGW),
// x - 1 .. x + 1 left out with `centre`
__device__ __forceinline__ bool other_marks(const unsigned long long *__restrict__ mark, int x, int half, bool centre)
{
    const int s0 = (x - half) / SEGW, s1 = (x + half) / SEGW;
    unsigned long long m0 = mark[s0], m1 = mark[s1];   // the same word when one segment holds them all
    // bits of the window in either segment, from its column 0
    auto window = [](int lo, int hi) {
        lo = max(lo, 0);
        hi = min(hi, SEGW - 1);
        return lo > hi ? 0ull : (~0ull << lo) & (~0ull >> (63 - hi));
    };
    const int c0 = x - s0 * SEGW, c1 = x - s1 * SEGW;
    unsigned long long w0 = window(c0 - half, c0 + half), w1 = window(c1 - half, c1 + half);
    if (centre) {
        w0 &= ~window(c0 - 1, c0 + 1);
        w1 &= ~window(c1 - 1, c1 + 1);
    }
    return ((m0 & w0) | (m1 & w1)) != 0;
}

// one wave per group of CUT_U consecutive ROI records (grid-stride over the kept count): lanes
// write consecutive uint16 words of each record, so the stores are contiguous; the CUT_U records'
// pixels are loaded before any is stored, so a wave keeps CUT_U independent memory round trips in
// flight instead of one.  The marks of all CUT_U windows are one round of loads too, eight lanes a
// record, and a record's header is one lane's work.  32 frames of 2048 x 2048 with 0.003 molecules per
// pixel, 7 x 7: 65 -> 60 us, most of it the 64-byte sectors of seven rows a record; CUT_BLOCKS
// waves fill the chip, and a call of 180 records pays for no more (6.6 -> 4.4 us).
constexpr int CUT_U = 8, CUT_BLOCKS = 4096;

// R is the cut size; with sel set, record j is candidate sel[j] for j < *sel_n (a set of the
// mixed-size extraction), else record i is candidate i for i < info[0]
__global__ void __launch_bounds__(64) cut_kernel(const uint16_t *__restrict__ frames, ExtractConst c, int R,
                                                 const unsigned long long *__restrict__ mark_mask,
                                                 const int *__restrict__ info, const int3 *__restrict__ xyb,
                                                 const int *__restrict__ sel, const int *__restrict__ sel_n,
                                                 uint16_t *__restrict__ rois)
{
    // the CUT_U records are assembled in LDS and leave as one contiguous block (16-byte stores
    // when the block is 16-byte aligned)
    __shared__ __align__(16) uint16_t stage[CUT_U * 17 * 18];
    const int n = sel ? *sel_n : info[0];
    const int half = R / 2, WR = R * (R + 1), RR = R * R;
    const int l = threadIdx.x;
    const int start = c.start_dev ? *c.start_dev : c.start_frame;
    const int BH = c.B * c.H;
    for (int i0 = blockIdx.x * CUT_U; i0 < n; i0 += gridDim.x * CUT_U) {
        // lane j holds record j's list entry and works out its header
        int3 e = make_int3(half, half, 0);
        if (l < CUT_U && i0 + l < n) e = xyb[sel ? sel[i0 + l] : i0 + l];
        const int valid = min(CUT_U, n - i0);   // uniform
        int x[CUT_U], y[CUT_U], z[CUT_U];       // uniform
#pragma unroll
        for (int j = 0; j < CUT_U; j++) {
            x[j] = __builtin_amdgcn_readlane(e.x, j);
            y[j] = __builtin_amdgcn_readlane(e.y, j);
            z[j] = __builtin_amdgcn_readlane(e.z, j);
        }
        int ft = QCS_ROITYPE_SINGLE;
        if (c.multi) {
            // eight lanes a record, a window row each: marks outside the centre's 3 x 3
            const int q = l & 7, ex = __shfl(e.x, l >> 3, 64), ey = __shfl(e.y, l >> 3, 64), ez = __shfl(e.z, l >> 3, 64);
            bool other = false;
            for (int r = q; r < R && (l >> 3) < valid; r += 8)
                other |= other_marks(mark_mask + ((size_t)ez * BH + ey - half + r) * c.nseg, ex, half, r >= half - 1 && r <= half + 1);
            const unsigned long long m = __ballot(other);
            if (l < CUT_U && ((m >> (8 * l)) & 0xff)) ft = QCS_ROITYPE_MULTI;
        }
        for (int k = l; k < RR; k += 64) {
            uint16_t v[CUT_U];
            const int r = k / R;
            const size_t off = (size_t)r * c.W + (k - r * R);
#pragma unroll
            for (int j = 0; j < CUT_U; j++)
                v[j] = j < valid ? (frames + (((size_t)z[j] * BH + y[j] - half) * c.W + x[j] - half))[off] : (uint16_t)0;
#pragma unroll
            for (int j = 0; j < CUT_U; j++) stage[j * WR + k] = v[j];
        }
        if (l < CUT_U) {
            uint16_t *h = stage + l * WR + RR;
            const int f = e.y / c.H, fr = start + e.z * c.B + f;
            h[0] = (uint16_t)e.x;
            h[1] = (uint16_t)(e.y - f * c.H);
            h[2] = (uint16_t)(fr % 65536);
            h[3] = (uint16_t)(fr / 65536);
            h[4] = (uint16_t)ft;
            for (int k = 5; k < R; k++) h[k] = 0;
        }
        __syncthreads();
        const int nv = min(CUT_U, n - i0);
        uint16_t *dst = rois + (size_t)i0 * WR;
        const uintptr_t al = reinterpret_cast<uintptr_t>(dst);
        if (nv == CUT_U && (al & 15) == 0) {   // uniform; CUT_U records are 16 R (R + 1) bytes
            for (int t = l; t < CUT_U * WR / 8; t += 64)
                reinterpret_cast<uint4 *>(dst)[t] = reinterpret_cast<const uint4 *>(stage)[t];
        } else if ((al & 3) == 0) {   // records are a whole number of 4-byte words (R (R + 1) even)
            for (int t = l; t < nv * WR / 2; t += 64)
                reinterpret_cast<uint32_t *>(dst)[t] = reinterpret_cast<const uint32_t *>(stage)[t];
        } else {
            for (int t = l; t < nv * WR; t += 64) dst[t] = stage[t];
        }
        __syncthreads();   // the next group reuses stage
    }
}

__global__ void fill_kernel(int *__restrict__ p, size_t n, int v)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

void fill_async(int *p, size_t n, int v, hipStream_t s)
{
    if (n == 0) return;
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
}

int scan_tile_count(size_t n) { return (int)((n + SCAN_TILE - 1) / SCAN_TILE); }

int scan_exclusive(const int *in, int n, int *out, int *tile_sums, hipStream_t s, const int *n_dev, int *total, bool add)
{
    if (n <= 0) return QCS_OK;
    const int ntiles = scan_tile_count((size_t)n);
    if (ntiles > SCAN_TILE) return fail(QCS_ERR_ARG, "scan of %d items exceeds the supported size", n);
    const ScanTotal t{total, add ? 1 : 0};
    if (n <= SCAN_ONE) {
        hipLaunchKernelGGL(scan_one_kernel, dim3(1), dim3(SCAN_ONE_T), 0, s, in, n, n_dev, out, tile_sums + ntiles, t);
    } else {
        hipLaunchKernelGGL(scan_tiles_kernel, dim3(ntiles), dim3(SCAN_BLOCK), 0, s, in, n, n_dev, tile_sums);
        hipLaunchKernelGGL(scan_apply_kernel, dim3(ntiles), dim3(SCAN_BLOCK), 0, s, in, n, n_dev, out, tile_sums, ntiles, t);
    }
    QCS_HIP(hipGetLastError());
    return QCS_OK;
}

__global__ void __launch_bounds__(256) scatter_kernel(const int *__restrict__ flags, const int *__restrict__ offs, int n,
                                                      const int *__restrict__ src, const int *__restrict__ base_dev,
                                                      int base_const, int *__restrict__ out, const int *__restrict__ n_dev)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n || (n_dev && j >= *n_dev) || !flags[j]) return;
    const int base = base_dev ? *base_dev : base_const;
    out[base + offs[j]] = src ? src[j] : j;
}

int compact_scatter(const int *flags, const int *offs, int n, const int *src, const int *base_dev, int base_const, int *out,
                    hipStream_t s, const int *n_dev)
{
    if (n <= 0) return QCS_OK;
    hipLaunchKernelGGL(scatter_kernel, dim3((n + 255) / 256), dim3(256), 0, s, flags, offs, n, src, base_dev, base_const, out, n_dev);
    QCS_HIP(hipGetLastError());
    return QCS_OK;
}

}  // namespace qcs

namespace qcs {

// Everything of one extraction call up to the candidate list (no host synchronisation):
// variance, walking filter + detection, row scan, per-batch bookkeeping, raster-order (x, y,
// batch) list.  info[0] receives the kept count (at most cap), info[1] the found count.
struct ExtractRun {
    ExtractConst c;
    int *info;
    int3 *xyb;
    const unsigned long long *mark;
};

static int extract_candidates(qcs_ctx *ctx, const qcs_params &p, const uint16_t *d_frames, int nframes, int start_frame,
                              const int *d_start, int cap, hipStream_t s, ExtractRun &run)
{
    const int R = p.ROISize;
    ExtractConst &c = run.c;
    memset(&c, 0, sizeof(c));
    c.W = p.ImageWidth;
    c.H = p.ImageHigh;
    c.B = p.BatchedImageNum > 0 ? p.BatchedImageNum : 1;
    c.nframes = nframes;
    c.nbatch = (nframes + c.B - 1) / c.B;
    c.R = R;
    c.loc_type = p.LocType;
    c.multi = p.MultiEmitterFitEn;
    c.smooth = !(p.LocType == QCS_LOCTYPE_GS2D && p.MultiEmitterFitEn > 0);
    c.batch_cap = p.MaxROIPerBatch > 0 ? p.MaxROIPerBatch : QCS_MAX_POINT_NUM;
    c.cap = cap;
    c.start_frame = start_frame;
    c.start_dev = d_start;
    c.nseg = (c.W + SEGW - 1) / SEGW;
    filter_taps_host(R, p.LocType, p.MultiEmitterFitEn, c.taps);
    // Rows per walking wave: long walks amortise the 14-row pipeline fill (32 frames of 2048 x 2048 at 96,
    // 128, 256 and 512 rows: 413, 410, 426 and 445 us); shorter ones keep small calls spread over the
    // chip, the shortest while there is not a wave for every SIMD (one frame of 256 x 256 at 8, 16 and 32
    // rows: 13, 16 and 23 us).
    const int rows_per_batch = c.B * c.H;
    auto waves = [&](int strips, int rows, int per) { return (long long)strips * ((rows + per - 1) / per) * c.nbatch; };
    c.walk_rows = 128;
    while (c.walk_rows > 8 && waves(c.nseg, rows_per_batch, c.walk_rows) < (c.walk_rows > 16 ? 8192 : 1024)) c.walk_rows /= 2;
    // variance region extent (largest over the batches: the first batch is a full one) and its walks
    // (8 rows of fill; 32 regions of 512 x 512 at 16, 32, 64 and 128 rows: 35, 32, 39 and 58 us; one of
    // 246 x 246 at 8, 16 and 32 rows: 9, 13 and 17 us)
    int Smax;
    {
        int sw = c.W / 2 - 5, sh = rows_per_batch / 2 - 5;
        sw = sw > 256 ? 256 : (sw < 1 ? 1 : sw);
        sh = sh > 256 ? 256 : (sh < 1 ? 1 : sh);
        Smax = sw < sh ? sw : sh;
    }
    const int var_strips = (2 * Smax + SEGW - 1) / SEGW;
    c.var_rows = 32;
    while (c.var_rows > 8 && waves(var_strips, 2 * Smax, c.var_rows) < 4096) c.var_rows /= 2;

    const size_t nrows = (size_t)nframes * c.H;
    if (nrows > (size_t)SCAN_TILE * SCAN_TILE) return fail(QCS_ERR_ARG, "too many rows in one extraction call");
    if ((size_t)rows_per_batch * c.W >= ((size_t)1 << 31)) return fail(QCS_ERR_ARG, "batched image larger than 2^31 pixels");
    const int ntiles = (int)((nrows + SCAN_TILE - 1) / SCAN_TILE);
    int rc;
    const size_t nvs = 4 * (size_t)c.nbatch;   // ints of the variance sums, ahead of the row counts: one fill clears both
    if ((rc = ctx->ex_det.ensure(sizeof(uint16_t) * VAR_MAX * VAR_MAX * (size_t)c.nbatch)) ||
        (rc = ctx->ex_mark.ensure(sizeof(unsigned long long) * nrows * c.nseg * 2)) ||
        (rc = ctx->ex_cnt.ensure(sizeof(int) * (nvs + nrows * 2 + ntiles + 1))) ||
        (rc = ctx->ex_xy.ensure(sizeof(int3) * (size_t)(cap > 0 ? cap : 1))) ||
        (rc = ctx->ex_tmp.ensure(sizeof(int) * (2 + 3 * (size_t)c.nbatch))))
        return rc;
    unsigned long long *var_sums = ctx->ex_cnt.as<unsigned long long>();
    uint16_t *tvbuf = ctx->ex_det.as<uint16_t>();
    unsigned long long *cand = ctx->ex_mark.as<unsigned long long>();
    unsigned long long *mark = cand + nrows * c.nseg;
    int *row_count = ctx->ex_cnt.as<int>() + nvs;
    int *row_off = row_count + nrows;
    int *tile_sums = row_off + nrows;
    int *info = ctx->ex_tmp.as<int>();
    int3 *xyb = ctx->ex_xy.as<int3>();

    fill_async(ctx->ex_cnt.as<int>(), nvs + nrows, 0, s);
    hipLaunchKernelGGL((walk_kernel<0, false>), dim3(var_strips, (2 * Smax + c.var_rows - 1) / c.var_rows, c.nbatch),
                       dim3(64), 0, s, d_frames, c, var_sums, tvbuf, cand, mark, row_count);
    QCS_HIP(hipGetLastError());
    hipLaunchKernelGGL(var_reduce_kernel, dim3(VAR_BLOCKS, c.nbatch), dim3(256), 0, s, c, tvbuf, var_sums);
    QCS_HIP(hipGetLastError());
    const dim3 wgrid(c.nseg, (rows_per_batch + c.walk_rows - 1) / c.walk_rows, c.nbatch);
    if (c.smooth)
        hipLaunchKernelGGL((walk_kernel<1, true>), wgrid, dim3(64), 0, s, d_frames, c, var_sums, tvbuf, cand, mark, row_count);
    else
        hipLaunchKernelGGL((walk_kernel<1, false>), wgrid, dim3(64), 0, s, d_frames, c, var_sums, tvbuf, cand, mark, row_count);
    QCS_HIP(hipGetLastError());
    if ((rc = scan_exclusive(row_count, (int)nrows, row_off, tile_sums, s))) return rc;
    hipLaunchKernelGGL(batch_kernel, dim3(1), dim3(64), 0, s, c, row_off, tile_sums, (int)nrows, ntiles, info);
    hipLaunchKernelGGL(emit_kernel, dim3((unsigned)((nrows + EMIT_WAVES * EMIT_U - 1) / (EMIT_WAVES * EMIT_U))), dim3(64 * EMIT_WAVES), 0,
                       s, c, cand, row_off, (int)nrows, info, xyb);
    QCS_HIP(hipGetLastError());
    run.info = info;
    run.xyb = xyb;
    run.mark = mark;
    return QCS_OK;
}

static int check_extract_args(const qcs_params &p, int R)
{
    if (p.ImageWidth <= 0 || p.ImageHigh <= 0) return fail(QCS_ERR_ARG, "ImageWidth/ImageHigh not set");
    if (p.ImageWidth < R || p.ImageHigh < R) return fail(QCS_ERR_ARG, "image smaller than the ROI");
    return QCS_OK;
}

// ---- mixed ROI sizes (no reference counterpart) ----------------------------------------------
// Each candidate of the base-size-7 extraction gets an ROI size in {7, 9, 11}:
//   s    = min(SigmaL, SigmaR, SigmaU, SigmaD) of its 7 x 7 WLE record;
//   Rpsf = 7 if s <= 1.4, 9 if s <= 1.9, else 11 (about +-2.5 s);
//   c(d) = detector marks in the (2d + 1)^2 window, rows of the candidate's own frame only;
//   dmin = smallest d in 1..5 with c(d) > 1 (6 if none);
//   Rnb  = 2 dmin + 3 for dmin 3 or 4 (a neighbour on the edge of the 7 x 7 window is taken in
//          whole, with a pixel of margin), else 7;
//   R    = max(Rpsf, Rnb), reduced by 2 while R > 7 and the window holds more than 2 other marks
//          (a fit models at most 3 emitters), then while R > 7 and the window leaves the frame.
// flags[s * ncap + i] = 1 when candidate i gets size 7 + 2 s; entries i >= *n are cleared.
__global__ void __launch_bounds__(256) mixed_size_kernel(ExtractConst c, const unsigned long long *__restrict__ mark_mask,
                                                         const int *__restrict__ info, const int3 *__restrict__ xyb,
                                                         const float *__restrict__ wle7, int ncap, int *__restrict__ flags)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ncap) return;
    int R = 0;
    if (i < info[0]) {
        const int3 e = xyb[i];
        const int x = e.x, y = e.y;                 // y: row of the stacked batch
        const int fy0 = (y / c.H) * c.H, ry = y - fy0;
        const size_t rbase = (size_t)e.z * c.B * c.H;
        const float *w = wle7 + (size_t)i * QCS_WLE_FLOATS;
        float sg = w[QCS_WLE_SIGMAL];
        sg = w[QCS_WLE_SIGMAR] < sg ? w[QCS_WLE_SIGMAR] : sg;
        sg = w[QCS_WLE_SIGMAU] < sg ? w[QCS_WLE_SIGMAU] : sg;
        sg = w[QCS_WLE_SIGMAD] < sg ? w[QCS_WLE_SIGMAD] : sg;
        const int rpsf = (sg <= 1.4f) ? 7 : ((sg <= 1.9f) ? 9 : 11);
        int cnt[6];
        cnt[0] = 1;
        for (int d = 1; d <= 5; d++) {
            const int xa = x - d < 0 ? 0 : x - d, xb = x + d > c.W - 1 ? c.W - 1 : x + d;
            int ya = y - d, yb = y + d;
            ya = ya < fy0 ? fy0 : ya;
            yb = yb > fy0 + c.H - 1 ? fy0 + c.H - 1 : yb;
            int n = 0;
            for (int yy = ya; yy <= yb; yy++) n += mark_count(mark_mask, c.nseg, rbase + yy, xa, xb);
            cnt[d] = n;
        }
        int dmin = 6;
        for (int d = 5; d >= 1; d--)
            if (cnt[d] > 1) dmin = d;
        const int rnb = (dmin == 3 || dmin == 4) ? 2 * dmin + 3 : 7;
        R = rpsf > rnb ? rpsf : rnb;
        while (R > 7 && cnt[R / 2] - 1 > 2) R -= 2;
        while (R > 7 && !(x - R / 2 >= 0 && x + R / 2 < c.W && ry - R / 2 >= 0 && ry + R / 2 < c.H)) R -= 2;
    }
    flags[i] = R == 7;
    flags[(size_t)ncap + i] = R == 9;
    flags[2 * (size_t)ncap + i] = R == 11;
}

// set lists: sel[off[i]] = i for flagged i with off[i] < cap; *n_out = min(total, cap)
__global__ void __launch_bounds__(256) mixed_scatter_kernel(const int *__restrict__ flags, const int *__restrict__ offs, int ncap,
                                                            int cap, int *__restrict__ sel)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ncap || !flags[i]) return;
    const int o = offs[i];
    if (o < cap) sel[o] = i;
}

__global__ void mixed_count_kernel(const int *__restrict__ tile_sums, int ntiles, int cap, int *__restrict__ n_out)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const int t = tile_sums[ntiles];
    *n_out = t < cap ? t : cap;
}

// Mixed-size extraction (launches only): candidates of the base-size-7 extraction (at most cap),
// their 7 x 7 cuts and WLE records in ctx scratch, the size rule, and per set s (sizes 7, 9, 11)
// the candidate list cand_s (ctx scratch, returned), the count sets[s].d_n and the records
// sets[s].d_rois (at most sets[s].n).
int extract_mixed_launch(qcs_ctx *ctx, const uint16_t *d_frames, int nframes, int start_frame, const int *d_start, int cap,
                         const qcs_roi_set *sets, int *cand_lists[3], int **cand_info, hipStream_t s)
{
    qcs_params p = ctx->p;
    p.ROISize = 7;
    int rc;
    if ((rc = check_extract_args(p, 11))) return rc;
    for (int k = 0; k < 3; k++)
        if (sets[k].roi_size != 7 + 2 * k || sets[k].n < 0 || (sets[k].n > 0 && !sets[k].d_rois) || !sets[k].d_n)
            return fail(QCS_ERR_ARG, "set %d: sizes 7, 9, 11 in order, a record buffer and a device count are required", k);
    ExtractRun run;
    if ((rc = extract_candidates(ctx, p, d_frames, nframes, start_frame, d_start, cap, s, run))) return rc;
    const int ncap = cap > 0 ? cap : 1;
    const int ntiles = scan_tile_count((size_t)ncap);
    // scratch: 7 x 7 cuts, WLE records, flags (3 ncap), offsets (3 ncap), tile sums (3 (ntiles + 1)), lists (3 ncap)
    const size_t r7w = (size_t)QCS_ROI_WORDS(7) * ncap;
    if ((rc = ctx->mx_rois.ensure(sizeof(uint16_t) * r7w + sizeof(float) * QCS_WLE_FLOATS * (size_t)ncap)) ||
        (rc = ctx->mx_list.ensure(sizeof(int) * (9 * (size_t)ncap + 3 * ((size_t)ntiles + 1)))))
        return rc;
    uint16_t *r7 = ctx->mx_rois.as<uint16_t>();
    float *w7 = reinterpret_cast<float *>(r7 + r7w);
    int *flags = ctx->mx_list.as<int>();
    int *offs = flags + 3 * (size_t)ncap;
    int *lists = offs + 3 * (size_t)ncap;
    int *tsum = lists + 3 * (size_t)ncap;
    if (cap > 0) {
        const int cut_blocks = (int)std::min<long long>(((long long)cap + CUT_U - 1) / CUT_U, CUT_BLOCKS);
        hipLaunchKernelGGL(cut_kernel, dim3(cut_blocks), dim3(64), 0, s, d_frames, run.c, 7, run.mark, run.info, run.xyb, nullptr, nullptr,
                           r7);
        QCS_HIP(hipGetLastError());
        if ((rc = wle_launch_extract(p, r7, run.xyb, run.c.B, run.c.H, run.info, cap, w7, s))) return rc;
    }
    hipLaunchKernelGGL(mixed_size_kernel, dim3((ncap + 255) / 256), dim3(256), 0, s, run.c, run.mark, run.info, run.xyb, w7, ncap, flags);
    QCS_HIP(hipGetLastError());
    for (int k = 0; k < 3; k++) {
        int *f = flags + (size_t)k * ncap, *o = offs + (size_t)k * ncap, *l = lists + (size_t)k * ncap;
        int *ts = tsum + (size_t)k * (ntiles + 1);
        if ((rc = scan_exclusive(f, ncap, o, ts, s))) return rc;
        hipLaunchKernelGGL(mixed_scatter_kernel, dim3((ncap + 255) / 256), dim3(256), 0, s, f, o, ncap, sets[k].n, l);
        hipLaunchKernelGGL(mixed_count_kernel, dim3(1), dim3(1), 0, s, ts, ntiles, sets[k].n, sets[k].d_n);
        QCS_HIP(hipGetLastError());
        if (sets[k].n > 0) {
            const int blocks = (int)std::min<long long>(((long long)sets[k].n + CUT_U - 1) / CUT_U, CUT_BLOCKS);
            hipLaunchKernelGGL(cut_kernel, dim3(blocks), dim3(64), 0, s, d_frames, run.c, 7 + 2 * k, run.mark, run.info, run.xyb, l,
                               sets[k].d_n, sets[k].d_rois);
            QCS_HIP(hipGetLastError());
        }
        cand_lists[k] = l;
    }
    if (cand_info) *cand_info = run.info;
    return QCS_OK;
}

}  // namespace qcs

using namespace qcs;

extern "C" int qcs_extract_dev(qcs_ctx *ctx, const uint16_t *d_frames, int nframes, int start_frame, uint16_t *d_rois,
                               float *d_wle, int cap, int *n_out, int *n_found, void *stream)
{
    if (n_out) *n_out = 0;
    if (n_found) *n_found = 0;
    if (!ctx || nframes < 0 || cap < 0 || (nframes > 0 && !d_frames) || (cap > 0 && (!d_rois || !d_wle)))
        return fail(QCS_ERR_ARG, "invalid argument");
    const qcs_params &p = ctx->p;
    int rc;
    if ((rc = check_extract_args(p, p.ROISize))) return rc;
    if (nframes == 0) return QCS_OK;
    hipStream_t s = (hipStream_t)stream;
    if ((rc = ctx->pin_cnt.ensure(64))) return rc;
    hipEvent_t ev;
    if ((rc = timer_begin(ctx->timer, s, &ev))) return rc;
    ExtractRun run;
    if ((rc = extract_candidates(ctx, p, d_frames, nframes, start_frame, nullptr, cap, s, run))) return rc;
    if (cap > 0) {
        const int cut_blocks = (int)std::min<long long>(((long long)cap + CUT_U - 1) / CUT_U, CUT_BLOCKS);
        hipLaunchKernelGGL(cut_kernel, dim3(cut_blocks), dim3(64), 0, s, d_frames, run.c, run.c.R, run.mark, run.info, run.xyb, nullptr,
                           nullptr, d_rois);
        QCS_HIP(hipGetLastError());
        rc = wle_launch_extract(p, d_rois, run.xyb, run.c.B, run.c.H, run.info, cap, d_wle, s);
        if (rc) return rc;
    }
    if ((rc = timer_end(ctx->timer, TM_EXTRACT, s, ev, nframes))) return rc;
    int *h = ctx->pin_cnt.as<int>();
    QCS_HIP(hipMemcpyAsync(h, run.info, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
    QCS_HIP(hipStreamSynchronize(s));
    if (n_out) *n_out = h[0];
    if (n_found) *n_found = h[1];
    if (h[1] > h[0]) return fail(QCS_ERR_CAPACITY, "%d candidates found, %d kept (capacity)", h[1], h[0]);
    return QCS_OK;
}

extern "C" int qcs_extract_mixed_dev(qcs_ctx *ctx, const uint16_t *d_frames, int nframes, int start_frame, int cap,
                                     const qcs_roi_set *sets, int *n_counts, void *stream)
{
    if (!ctx || !sets || nframes < 0 || cap < 0 || (nframes > 0 && !d_frames)) return fail(QCS_ERR_ARG, "invalid argument");
    hipStream_t s = (hipStream_t)stream;
    int rc;
    if (nframes == 0) {
        for (int k = 0; k < 3; k++) {
            if (!sets[k].d_n) return fail(QCS_ERR_ARG, "set %d: a device count is required", k);
            fill_async(sets[k].d_n, 1, 0, s);
        }
        QCS_HIP(hipGetLastError());
    } else {
        hipEvent_t ev;
        if ((rc = timer_begin(ctx->timer, s, &ev))) return rc;
        int *lists[3], *info = nullptr;
        if ((rc = extract_mixed_launch(ctx, d_frames, nframes, start_frame, nullptr, cap, sets, lists, &info, s))) return rc;
        if ((rc = timer_end(ctx->timer, TM_EXTRACT, s, ev, nframes))) return rc;
    }
    if (!n_counts) return QCS_OK;
    int h[3];
    for (int k = 0; k < 3; k++) QCS_HIP(hipMemcpyAsync(&h[k], sets[k].d_n, sizeof(int), hipMemcpyDeviceToHost, s));
    QCS_HIP(hipStreamSynchronize(s));
    for (int k = 0; k < 3; k++) n_counts[k] = h[k];
    return QCS_OK;
}

extern "C" int qcs_extract(qcs_ctx *ctx, const uint16_t *frames, int nframes, int start_frame, uint16_t *rois, float *wle,
                           int cap, int *n_out, int *n_found)
{
    if (n_out) *n_out = 0;
    if (n_found) *n_found = 0;
    if (!ctx || nframes < 0 || cap < 0 || (nframes > 0 && !frames) || (cap > 0 && (!rois || !wle)))
        return fail(QCS_ERR_ARG, "invalid argument");
    if (nframes == 0) return QCS_OK;
    const qcs_params &p = ctx->p;
    const size_t fb = (size_t)nframes * p.ImageWidth * p.ImageHigh * sizeof(uint16_t);
    const int R = p.ROISize;
    int rc;
    if ((rc = ctx->ex_frames.ensure(fb)) || (rc = ctx->h_rois_dev.ensure((size_t)(cap > 0 ? cap : 1) * QCS_ROI_WORDS(R) * 2)) ||
        (rc = ctx->h_wle_dev.ensure((size_t)(cap > 0 ? cap : 1) * QCS_WLE_FLOATS * 4)))
        return rc;
    QCS_HIP(hipMemcpy(ctx->ex_frames.ptr, frames, fb, hipMemcpyHostToDevice));
    int no = 0, nf = 0;
    rc = qcs_extract_dev(ctx, ctx->ex_frames.as<uint16_t>(), nframes, start_frame, ctx->h_rois_dev.as<uint16_t>(),
                         ctx->h_wle_dev.as<float>(), cap, &no, &nf, nullptr);
    if (rc && rc != QCS_ERR_CAPACITY) return rc;
    QCS_HIP(hipMemcpy(rois, ctx->h_rois_dev.ptr, (size_t)no * QCS_ROI_WORDS(R) * 2, hipMemcpyDeviceToHost));
    QCS_HIP(hipMemcpy(wle, ctx->h_wle_dev.ptr, (size_t)no * QCS_WLE_FLOATS * 4, hipMemcpyDeviceToHost));
    if (n_out) *n_out = no;
    if (n_found) *n_found = nf;
    return rc;
}
