// sort.hip -- stable LSD radix sort of (key, index) pairs, of localization rows by frame, and an
// inclusive max-scan (gfx950).
//
// The localization path sorts rows by frame (frame-sorted compaction) and by (frame, cell) keys
// (link search of consecutive-frame merging).  Each pass sorts by one 8-bit digit:
//   radix_hist_kernel     one work-group per tile of 2048 items: LDS digit histogram, written
//                         digit-major (counts[d * ntiles + tile]);
//   scan                  exclusive scan of the 256 x ntiles counts (digit-major), so a tile's
//                         slice of digit d starts after every earlier digit and every earlier
//                         tile's keys of digit d;
//   radix_scatter_kernel  the tile again, 256 items per round in index order: each wave finds the
//                         lanes holding its digit by 8 ballots (one per digit bit), ranks itself
//                         among the lower lanes, adds the counts of the lower waves (LDS) and the
//                         tile's running base of the digit.
// Equal digits keep their input order (stable), so the passes from the lowest digit up sort the
// keys stably; there are no atomics on the data path, so the result is deterministic.
//
// A pass reads its items from a source and writes them to a destination.  The row sort's first pass
// reads the rows themselves, where rows that are not kept count nowhere, and its last pass writes
// rows (in calls of up to SORT_COPY_ROWS): up to 256 frames are one pass of three launches with no flags, no list and no key arrays,
// and the number of kept rows stays on the device until the end.
#include <limits.h>
#include "qcs_internal.h"

namespace qcs {

namespace {

constexpr int SB = 256;                  // threads per work-group (4 waves)
constexpr int SI = 8;                    // keys per thread per tile
constexpr int STILE = SB * SI;           // keys per tile
constexpr int RADIX = 256;

// sources: get() gives the item's key and value, false if there is none
template <typename K>
struct PairSrc {
    const K *k;
    const int *v;
    int n;
    const int *n_dev;   // items on the device, or null
    __device__ __forceinline__ int count() const { return n_dev ? min(*n_dev, n) : n; }
    __device__ __forceinline__ bool key(int i, int m, K &key) const
    {
        if (i >= m) return false;
        key = k[i];
        return true;
    }
    __device__ __forceinline__ int val(int i) const { return v[i]; }
};

// float -> int truncation with NaN -> 0 and saturation (the CUDA conversion the reference relies on)
__device__ __forceinline__ int f2i_sat(float v)
{
    if (v != v) return 0;
    if (v >= 2147483647.0f) return 2147483647;
    if (v <= -2147483648.0f) return (-2147483647 - 1);
    return (int)v;
}

// the rows with photons of frames first..end (RemoveZero_SortFrame), key = frame - first
struct RowSrc {
    const float *loc;
    int n, first, end;
    __device__ __forceinline__ int count() const { return n; }
    __device__ __forceinline__ bool key(int i, int m, unsigned &key) const
    {
        if (i >= m) return false;
        const float *r = loc + (size_t)i * QCS_REC_FLOATS;
        const int pp = f2i_sat(r[QCS_POS_PPHO]), fr = f2i_sat(r[QCS_POS_FRME]);
        key = (unsigned)fr - (unsigned)first;
        return ((float)pp > 1.0f) && fr >= first && fr <= end;
    }
    __device__ __forceinline__ int val(int i) const { return i; }
};

template <typename K>
struct PairDst {
    K *k;
    int *v;
    __device__ __forceinline__ void put(int pos, K key, int val) const
    {
        k[pos] = key;
        v[pos] = val;
    }
};

struct RowDst {
    const float *loc;
    float *out;
    __device__ __forceinline__ void put(int pos, unsigned, int val) const
    {
        const float4 *src = reinterpret_cast<const float4 *>(loc + (size_t)val * QCS_REC_FLOATS);
        float4 *dst = reinterpret_cast<float4 *>(out + (size_t)pos * QCS_REC_FLOATS);
        dst[0] = src[0];
        dst[1] = src[1];
        dst[2] = src[2];
    }
};

template <typename K, class Src>
__global__ void __launch_bounds__(SB) radix_hist_kernel(Src src, int shift, int ntiles, int *__restrict__ counts)
{
    __shared__ int h[RADIX];
    const int tid = threadIdx.x;
    h[tid] = 0;
    __syncthreads();
    const int t0 = blockIdx.x * STILE, m = src.count();
#pragma unroll
    for (int k = 0; k < SI; k++) {
        K key;
        if (src.key(t0 + k * SB + tid, m, key)) atomicAdd(&h[(int)((key >> shift) & (K)(RADIX - 1))], 1);
    }
    __syncthreads();
    counts[(size_t)tid * ntiles + blockIdx.x] = h[tid];
}

template <typename K, class Src, class Dst>
__global__ void __launch_bounds__(SB) radix_scatter_kernel(Src src, Dst dst, int shift, int ntiles, const int *__restrict__ offs)
{
    __shared__ int base[RADIX];
    __shared__ int wcnt[SB / 64][RADIX];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    base[tid] = offs[(size_t)tid * ntiles + blockIdx.x];
    const int t0 = blockIdx.x * STILE, n = src.count();
    for (int k = 0; k < SI; k++) {
#pragma unroll
        for (int w = 0; w < SB / 64; w++) wcnt[w][tid] = 0;
        __syncthreads();
        const int i = t0 + k * SB + tid;
        K key = 0;
        const bool valid = src.key(i, n, key);
        const int val = valid ? src.val(i) : 0;   // in flight while the ranks are worked out
        const int d = (int)((key >> shift) & (K)(RADIX - 1));
        unsigned long long m = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const unsigned long long bb = __ballot((d >> b) & 1);
            m &= ((d >> b) & 1) ? bb : ~bb;
        }
        const int rank = __popcll(m & ((1ull << lane) - 1ull));
        if (valid && rank == 0) wcnt[wv][d] = __popcll(m);   // one lane per digit present in the wave
        __syncthreads();
        if (valid) {
            int pos = base[d] + rank;
            for (int w = 0; w < wv; w++) pos += wcnt[w][d];
            dst.put(pos, key, val);
        }
        __syncthreads();
        int add = 0;
#pragma unroll
        for (int w = 0; w < SB / 64; w++) add += wcnt[w][tid];
        base[tid] += add;
    }
}

// rows idx[0 .. *m_dev) of loc, 16 bytes a lane
__global__ void __launch_bounds__(SB) copy_rows_kernel(const float4 *__restrict__ loc, const int *__restrict__ idx, int n,
                                                       const int *__restrict__ m_dev, float4 *__restrict__ out)
{
    const size_t t = (size_t)blockIdx.x * SB + threadIdx.x, j = t / 3;
    if (j >= (size_t)min(*m_dev, n)) return;
    out[t] = loc[(size_t)idx[j] * 3 + (t - j * 3)];
}

// inclusive max-scan: per-tile scan, scan of the tile maxima, then the carry-in
constexpr int MB = 256, MI = 16, MTILE = MB * MI;

__device__ __forceinline__ int block_inclusive_max(int v, int *sh)
{
    const int tid = threadIdx.x;
    sh[tid] = v;
    __syncthreads();
    for (int off = 1; off < MB; off <<= 1) {
        const int t = (tid >= off) ? sh[tid - off] : INT_MIN;
        __syncthreads();
        sh[tid] = sh[tid] > t ? sh[tid] : t;
        __syncthreads();
    }
    const int r = sh[tid];
    __syncthreads();
    return r;
}

__global__ void __launch_bounds__(MB) max_scan_tiles_kernel(const int *__restrict__ in, int n, int *__restrict__ out,
                                                           int *__restrict__ tile_max)
{
    __shared__ int sh[MB];
    const int base = blockIdx.x * MTILE + threadIdx.x * MI;
    int v[MI], run = INT_MIN;
#pragma unroll
    for (int k = 0; k < MI; k++) {
        v[k] = (base + k < n) ? in[base + k] : INT_MIN;
        run = run > v[k] ? run : v[k];
    }
    const int incl = block_inclusive_max(run, sh);   // sh keeps every thread's inclusive maximum
    int carry = (threadIdx.x > 0) ? sh[threadIdx.x - 1] : INT_MIN;
#pragma unroll
    for (int k = 0; k < MI; k++) {
        carry = carry > v[k] ? carry : v[k];
        if (base + k < n) out[base + k] = carry;
    }
    if (threadIdx.x == MB - 1) tile_max[blockIdx.x] = incl;
}

__global__ void __launch_bounds__(MB) max_scan_sums_kernel(int *__restrict__ tile_max, int ntiles)
{
    __shared__ int sh[MB];
    const int base = threadIdx.x * MI;
    int v[MI], run = INT_MIN;
#pragma unroll
    for (int k = 0; k < MI; k++) {
        v[k] = (base + k < ntiles) ? tile_max[base + k] : INT_MIN;
        run = run > v[k] ? run : v[k];
    }
    (void)block_inclusive_max(run, sh);   // sh keeps every thread's inclusive maximum
    int carry = (threadIdx.x > 0) ? sh[threadIdx.x - 1] : INT_MIN;
    // exclusive carry per tile: the maximum of the tiles before it
#pragma unroll
    for (int k = 0; k < MI; k++) {
        const int x = v[k];
        if (base + k < ntiles) tile_max[base + k] = carry;
        carry = carry > x ? carry : x;
    }
}

__global__ void __launch_bounds__(256) max_scan_add_kernel(int *__restrict__ out, int n, const int *__restrict__ tile_max)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int c = tile_max[i / MTILE];
    out[i] = out[i] > c ? out[i] : c;
}

// one pass over up to n items; counts -> offs -> tsum are the ints of radix_sort_tmp_ints(n);
// *total (may be null) receives the number of items
template <typename K, class Src, class Dst>
int radix_pass(const Src &src, const Dst &dst, int n, int shift, int *tmp, int *total, hipStream_t s)
{
    const int ntiles = (n + STILE - 1) / STILE;
    const long long ncount = (long long)RADIX * ntiles;
    if (ncount > 16LL * 1024 * 1024) return fail(QCS_ERR_ARG, "sort of %d keys exceeds the supported size", n);
    int *counts = tmp, *offs = tmp + ncount, *tsum = offs + ncount;
    hipLaunchKernelGGL((radix_hist_kernel<K, Src>), dim3(ntiles), dim3(SB), 0, s, src, shift, ntiles, counts);
    QCS_HIP(hipGetLastError());
    const int rc = scan_exclusive(counts, (int)ncount, offs, tsum, s, nullptr, total);
    if (rc) return rc;
    hipLaunchKernelGGL((radix_scatter_kernel<K, Src, Dst>), dim3(ntiles), dim3(SB), 0, s, src, dst, shift, ntiles, offs);
    QCS_HIP(hipGetLastError());
    return QCS_OK;
}

}  // namespace

size_t radix_sort_tmp_ints(int n)
{
    const size_t ntiles = ((size_t)(n > 0 ? n : 1) + STILE - 1) / STILE;
    const size_t ncount = (size_t)RADIX * ntiles;
    return 2 * ncount + (size_t)scan_tile_count(ncount) + 1;
}

int radix_sort_pairs_u64(unsigned long long *k0, int *v0, unsigned long long *k1, int *v1, int n, int bits, int *tmp,
                         hipStream_t s, unsigned long long **kres, int **vres)
{
    using K = unsigned long long;
    K *ki = k0, *ko = k1;
    int *vi = v0, *vo = v1;
    for (int shift = 0; n > 0 && shift < bits && shift < 64; shift += 8) {
        const int rc = radix_pass<K>(PairSrc<K>{ki, vi, n, nullptr}, PairDst<K>{ko, vo}, n, shift, tmp, nullptr, s);
        if (rc) return rc;
        K *tk = ki; ki = ko; ko = tk;
        int *tv = vi; vi = vo; vo = tv;
    }
    *kres = ki;
    *vres = vi;
    return QCS_OK;
}

size_t sort_rows_tmp_ints(int n, int first, int end)
{
    return radix_sort_tmp_ints(n) + (((unsigned)end - (unsigned)first) > 255u ? (size_t)n * 4 : 0);
}

// Of several passes the last writes the rows itself up to SORT_COPY_ROWS; beyond, where the rows are far from
// the caches, it leaves the order and a launch of its own copies the rows, all in flight at once (us per call,
// rows in the last pass / copied; frames in order and shuffled, 5,000 frames: 1,000,000 rows 82 / 91 and
// 111 / 112; 2,200,000 145 / 134 and 255 / 191; 8,000,000 521 / 427 and 881 / 651).  A single pass reads
// its rows in order and writes them: 96 / 98 and 99 / 125 at 2,200,000 rows of 10 frames, 394 / 341 and
// 415 / 452 at 8,000,000.
constexpr int SORT_COPY_ROWS = 1500000;

int sort_rows_by_frame(const float *d_loc, int n, int first, int end, float *d_out, int *d_m, int *tmp, hipStream_t s)
{
    const unsigned span = ((unsigned)end - (unsigned)first);
    const RowSrc rows{d_loc, n, first, end};
    const RowDst out{d_loc, d_out};
    int rc;
    if (span <= 255u) return radix_pass<unsigned>(rows, out, n, 0, tmp, d_m, s);
    unsigned *k0 = reinterpret_cast<unsigned *>(tmp + radix_sort_tmp_ints(n)), *k1 = k0 + n;
    int *v0 = reinterpret_cast<int *>(k1 + n), *v1 = v0 + n;
    if ((rc = radix_pass<unsigned>(rows, PairDst<unsigned>{k0, v0}, n, 0, tmp, d_m, s))) return rc;
    for (int shift = 8; shift < 32 && (span >> shift) != 0; shift += 8) {
        const PairSrc<unsigned> src{k0, v0, n, d_m};
        const bool last = shift + 8 >= 32 || (span >> (shift + 8)) == 0;
        if (last && n <= SORT_COPY_ROWS) return radix_pass<unsigned>(src, out, n, shift, tmp, nullptr, s);
        if ((rc = radix_pass<unsigned>(src, PairDst<unsigned>{k1, v1}, n, shift, tmp, nullptr, s))) return rc;
        unsigned *tk = k0; k0 = k1; k1 = tk;
        int *tv = v0; v0 = v1; v1 = tv;
    }
    static_assert(QCS_REC_FLOATS == 12, "a row is three 16-byte words");
    hipLaunchKernelGGL(copy_rows_kernel, dim3((unsigned)(((size_t)n * 3 + SB - 1) / SB)), dim3(SB), 0, s,
                       reinterpret_cast<const float4 *>(d_loc), v0, n, d_m, reinterpret_cast<float4 *>(d_out));
    QCS_HIP(hipGetLastError());
    return QCS_OK;
}

size_t max_scan_tmp_ints(int n) { return (size_t)(((size_t)(n > 0 ? n : 1) + MTILE - 1) / MTILE) + 1; }

int scan_inclusive_max(const int *in, int n, int *out, int *tmp, hipStream_t s)
{
    if (n <= 0) return QCS_OK;
    const int ntiles = (n + MTILE - 1) / MTILE;
    if (ntiles > MTILE) return fail(QCS_ERR_ARG, "max-scan of %d items exceeds the supported size", n);
    hipLaunchKernelGGL(max_scan_tiles_kernel, dim3(ntiles), dim3(MB), 0, s, in, n, out, tmp);
    hipLaunchKernelGGL(max_scan_sums_kernel, dim3(1), dim3(MB), 0, s, tmp, ntiles);
    hipLaunchKernelGGL(max_scan_add_kernel, dim3((n + 255) / 256), dim3(256), 0, s, out, n, tmp);
    QCS_HIP(hipGetLastError());
    return QCS_OK;
}

}  // namespace qcs
