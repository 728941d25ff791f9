// nn_gemm.h -- BF16 MFMA building blocks of the warm-start network (gfx950).
//
// C[M][N] (fp32) = A[M][K] * B[N][K]^T with A and B bf16, both K-contiguous ("NT"), K a multiple
// of 16, lda/ldb multiples of 4.  One work-group of 4 waves computes a 64 x 64 or 32 x 32 tile, each wave
// a quarter of it in v_mfma_f32_16x16x16_bf16 tiles.  MFMA operand layout (16 x 16 x 16): lane
// l supplies A[l % 16][4 (l / 16) + 0..3] and B^T[l % 16][4 (l / 16) + 0..3] (that is
// B[k][n] with n = l % 16); the result D[4 (l / 16) + i][l % 16] sits in accumulator i of lane l.
// Both operands are read with one 8-byte load per lane per tile straight from global memory:
// the matrices here are at most a few MB and stay L2-resident.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace qcs {

typedef short bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// round-to-nearest-even float -> bf16 (NaN stays NaN)
__device__ __forceinline__ uint16_t f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// What a product's tile leaves: fp32 values; bias and ReLU in bf16 (a layer's output); bias in fp32
// (the last layer); or, going back, the values where the layer input m was positive (its ReLU), in
// fp32 (c) and bf16 (o).
enum { EPI_F32 = 0, EPI_RELU = 1, EPI_BIAS = 2, EPI_MASK = 3 };
struct GemmEpi {
    const float *bias = nullptr;
    uint16_t *o = nullptr;
    const uint16_t *m = nullptr;
    int ldo = 0, ldm = 0;
};

// The operands of eight k-steps are loaded before their MFMAs, so a wave waits for memory once per 128
// of K instead of once per 16: with few tiles (n = 2,048: 32 work-groups for the 576-wide layer) that
// latency is the kernel's time.
//
// T x T MFMA tiles per wave, 2 x 2 waves per work-group: T = 2 (64 x 64 outputs) reads each operand half
// as often, T = 1 (32 x 32) puts four times as many waves on the chip.
template <int EPI, int T>
__global__ void __launch_bounds__(256) gemm_nt_kernel(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                                                      float *__restrict__ C, int M, int N, int K, int lda, int ldb, int ldc, GemmEpi ep)
{
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int m0 = (blockIdx.y * 2 + (w >> 1)) * 16 * T, n0 = (blockIdx.x * 2 + (w & 1)) * 16 * T;
    const int lr = lane & 15, lk = (lane >> 4) * 4;
    f32x4_t acc[T][T];
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
        for (int j = 0; j < T; j++) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const bf16x4_t zero = {0, 0, 0, 0};
    // rows past the end read row 0 and count as zero
    const uint16_t *a[T], *b[T];
    bool ra[T], rb[T];
#pragma unroll
    for (int i = 0; i < T; i++) {
        ra[i] = m0 + 16 * i + lr < M;
        rb[i] = n0 + 16 * i + lr < N;
        a[i] = A + (size_t)(ra[i] ? m0 + 16 * i + lr : 0) * lda + lk;
        b[i] = B + (size_t)(rb[i] ? n0 + 16 * i + lr : 0) * ldb + lk;
    }
    auto steps = [&](int k0, auto U) {
        constexpr int u = decltype(U)::value;
        bf16x4_t va[T][u], vb[T][u];
#pragma unroll
        for (int e = 0; e < u; e++)
#pragma unroll
            for (int i = 0; i < T; i++) {
                va[i][e] = *reinterpret_cast<const bf16x4_t *>(a[i] + k0 + 16 * e);
                vb[i][e] = *reinterpret_cast<const bf16x4_t *>(b[i] + k0 + 16 * e);
            }
#pragma unroll
        for (int e = 0; e < u; e++) {
#pragma unroll
            for (int i = 0; i < T; i++) {
                if (!ra[i]) va[i][e] = zero;
                if (!rb[i]) vb[i][e] = zero;
            }
#pragma unroll
            for (int i = 0; i < T; i++)
#pragma unroll
                for (int j = 0; j < T; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(va[i][e], vb[j][e], acc[i][j], 0, 0, 0);
        }
    };
    int k0 = 0;
    for (; k0 + 128 <= K; k0 += 128) steps(k0, std::integral_constant<int, 8>{});
    for (; k0 + 64 <= K; k0 += 64) steps(k0, std::integral_constant<int, 4>{});
    for (; k0 < K; k0 += 16) steps(k0, std::integral_constant<int, 1>{});
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
        for (int j = 0; j < T; j++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int row = m0 + i * 16 + lk + t, col = n0 + j * 16 + lr;
                if (row >= M || col >= N) continue;
                float v = acc[i][j][t];
                if (EPI == EPI_RELU || EPI == EPI_BIAS) v += ep.bias[col];
                if (EPI == EPI_RELU) {
                    ep.o[(size_t)row * ep.ldo + col] = f2bf(fmaxf(v, 0.0f));
                } else if (EPI == EPI_MASK) {
                    v = bf2f(ep.m[(size_t)row * ep.ldm + col]) > 0.0f ? v : 0.0f;
                    C[(size_t)row * ldc + col] = v;
                    ep.o[(size_t)row * ep.ldo + col] = f2bf(v);
                } else {
                    C[(size_t)row * ldc + col] = v;
                }
            }
}

// Weight and bias gradients, dW[m][n] = sum_r dY[r][m] X[r][n] (bf16, rows contiguous) and
// db[m] = sum_r dY[r][m] (fp32), of up to WG_MAX layers in one launch.  The sums run over the batch's
// rows (up to 25 per ROI) and the results are small (16 x 64 to 64 x 576), so the rows are split: a
// work-group takes one slice of the rows and 64 columns of X, stages 64 rows at a time transposed in
// LDS (the MFMA operands need consecutive rows of one column), and leaves its partial sums; a second
// launch adds the slices in order.  A slice is at least 64 rows; at most WG_PARTS slices per layer.
// n = 2,048, all five layers: 2,150 us as transposes, one work-group per output tile and one
// column sum per layer; 25 us and 6 us for adding the slices here (the whole pass 2,400 -> 180 us).
constexpr int WG_MAX = 5, WG_PARTS = 128;
struct WgLayer {
    const uint16_t *dy, *x;
    const float *dyf;
    int rows, M, N, ldx;
    int parts, slice;    // row slices, rows of one
    int b0;              // first work-group of the layer
    int woff, boff;      // gradients in the parameter block
    size_t poff;         // partial sums: parts x (M N + M) floats
};
struct WgArgs {
    WgLayer l[WG_MAX];
    int nl, blocks;
    float *partial;
};

constexpr int WG_PITCH = 72;   // u16 per LDS row (64 batch rows, 8-byte aligned)

__global__ void __launch_bounds__(256) wgrad_kernel(WgArgs a)
{
    __shared__ __align__(16) uint16_t sy[64][WG_PITCH], sx[64][WG_PITCH];
    int li = 0;
    while (li + 1 < a.nl && (int)blockIdx.x >= a.l[li + 1].b0) li++;
    const WgLayer L = a.l[li];
    const int tiles = (L.N + 63) / 64, t0 = blockIdx.x - L.b0, tile = t0 % tiles, part = t0 / tiles;
    const int n0 = tile * 64, r0 = part * L.slice, r1 = min(r0 + L.slice, L.rows);
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, lr = lane & 15, lk = (lane >> 4) * 4;
    float *out = a.partial + L.poff + (size_t)part * (L.M * L.N + L.M);
    f32x4_t acc[4];   // the wave's 16 columns of X against up to 64 rows of dW
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int r = r0; r < r1; r += 64) {
        // 64 rows x 64 columns of each operand, four columns per load
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int q = tid + e * 256, rr = q >> 4, cc = (q & 15) * 4;
            uint2 vy = make_uint2(0, 0), vx = make_uint2(0, 0);
            if (r + rr < r1) {
                if (cc < L.M) vy = *reinterpret_cast<const uint2 *>(L.dy + (size_t)(r + rr) * L.M + cc);
                if (n0 + cc < L.N) vx = *reinterpret_cast<const uint2 *>(L.x + (size_t)(r + rr) * L.ldx + n0 + cc);
            }
            sy[cc][rr] = (uint16_t)vy.x;
            sy[cc + 1][rr] = (uint16_t)(vy.x >> 16);
            sy[cc + 2][rr] = (uint16_t)vy.y;
            sy[cc + 3][rr] = (uint16_t)(vy.y >> 16);
            sx[cc][rr] = (uint16_t)vx.x;
            sx[cc + 1][rr] = (uint16_t)(vx.x >> 16);
            sx[cc + 2][rr] = (uint16_t)vx.y;
            sx[cc + 3][rr] = (uint16_t)(vx.y >> 16);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 64; k += 16) {
            const bf16x4_t vb = *reinterpret_cast<const bf16x4_t *>(&sx[w * 16 + lr][k + lk]);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const bf16x4_t va = *reinterpret_cast<const bf16x4_t *>(&sy[i * 16 + lr][k + lk]);
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(va, vb, acc[i], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    const int col = n0 + w * 16 + lr;
    if (col < L.N) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int row = i * 16 + lk + t;
                if (row < L.M) out[row * L.N + col] = acc[i][t];
            }
    }
    if (tile == 0) {   // the slice's column sums of dY: M (16, 32 or 64) columns, 256 / M rows at a time
        float *red = reinterpret_cast<float *>(&sy[0][0]);
        const int c = tid % L.M, g = tid / L.M, ng = 256 / L.M;
        float s = 0.0f;
#pragma unroll 8
        for (int r = r0 + g; r < r1; r += ng) s += L.dyf[(size_t)r * L.M + c];
        red[tid] = s;
        __syncthreads();
        if (g == 0) {
            for (int k = 1; k < ng; k++) s += red[k * L.M + c];
            out[L.M * L.N + c] = s;
        }
    }
}

// g = (or +=, for the later chunks of a batch) the slices' sums, in slice order
__global__ void __launch_bounds__(256) wgrad_reduce_kernel(WgArgs a, float *__restrict__ g, int add)
{
    const WgLayer &L = a.l[blockIdx.y];
    const int i = blockIdx.x * 256 + threadIdx.x, sz = L.M * L.N + L.M;
    if (i >= sz) return;
    const float *p = a.partial + L.poff + i;
    float s = 0.0f;
#pragma unroll 16
    for (int k = 0; k < L.parts; k++) s += p[(size_t)k * sz];
    float *o = g + (i < L.M * L.N ? L.woff + i : L.boff + i - L.M * L.N);
    *o = add ? *o + s : s;
}

}  // namespace qcs
