// fh3_short.hip -- the product of short F16 rows (the video patch projection) on gfx950.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fh3_kernels.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Short F16 rows (K <= 128, K % 8 == 0: the video patch projection) in one
// launch: what such a product cannot do without is storing Y, and the general
// route spent as long on its two preparations and on the padding of K to 256.
// A workgroup takes 128 tokens x 128 columns, 32 columns to a wavefront, which
// holds its weight fragments, read in place, in registers; the tokens' fp16
// fragments are made here (k_xprep_any's scale rule and rounding) and shared
// through LDS.  The same products in the same k order as k_gemm16, so the same
// bits.  2880 x 96 -> 5376 with its bias: 43.5 -> 17.3 us per call (3.7 TB/s),
// 16384 tokens 191 -> 82, 100 tokens 29.9 -> 5.8, one token 10.2 -> 5.1 (K = 96).
// y must not lie over x.
constexpr int SHORT_K = 128, SHORT_M = 128, SHORT_N = 128;
__global__ __launch_bounds__(256) void k_short16(const _Float16 *__restrict__ W16, int N, int K,
                                                 const float *__restrict__ X, const float *__restrict__ bias,
                                                 float *__restrict__ Y, int M, int n_tiles) {
    constexpr int KS = SHORT_K / 16, ROW = SHORT_K + 8;  // LDS rows padded: consecutive tokens on different banks
    __shared__ __align__(16) _Float16 sx[SHORT_M][ROW];
    __shared__ __align__(16) float sinv[SHORT_M];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hf = lane >> 5;
    const int mt = blockIdx.x / n_tiles, nt = blockIdx.x - mt * n_tiles;
    const int m0 = mt * SHORT_M, o = nt * SHORT_N + 32 * wave + l32;
    const int kc = K / 8, ks = (kc + 1) / 2;  // chunks of 8 k, MFMA steps
    half8 w[KS];
    const half8 *wr = reinterpret_cast<const half8 *>(W16 + (size_t)(o < N ? o : N - 1) * K);
#pragma unroll
    for (int i = 0; i < KS; i++) w[i] = 2 * i + hf < kc ? wr[2 * i + hf] : half8{};
    {  // two threads to a token, its chunks in turn
        const int r = tid >> 1, c0 = tid & 1;
        const bool real = m0 + r < M;
        const f32x4 *xr = reinterpret_cast<const f32x4 *>(X + (size_t)(m0 + r) * K);
        f32x4 v[KS][2];
        float mx = 0.f;
#pragma unroll
        for (int i = 0; i < KS; i++) {
            const int c = 2 * i + c0;
#pragma unroll
            for (int p = 0; p < 2; p++) {
                v[i][p] = real && c < kc ? xr[2 * c + p] : f32x4{0.f, 0.f, 0.f, 0.f};
                mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[i][p].x), fabsf(v[i][p].y)),
                                     fmaxf(fabsf(v[i][p].z), fabsf(v[i][p].w))));
            }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 1));
        int e = 0;
        if (mx > 0.f && mx <= 3.4028234663852886e38f) {
            int E;
            (void)frexpf(mx, &E);
            e = 15 - E;
            e = e > 126 ? 126 : (e < -126 ? -126 : e);
        }
        const float s = ldexpf(1.0f, e);
        if (c0 == 0) sinv[r] = ldexpf(1.0f, -e);
#pragma unroll
        for (int i = 0; i < KS; i++)
            if (i < ks) {
                const f32x4 a = v[i][0], b = v[i][1];
                *reinterpret_cast<half8 *>(&sx[r][8 * (2 * i + c0)]) =
                    half8{(_Float16)(a.x * s), (_Float16)(a.y * s), (_Float16)(a.z * s), (_Float16)(a.w * s),
                          (_Float16)(b.x * s), (_Float16)(b.y * s), (_Float16)(b.z * s), (_Float16)(b.w * s)};
            }
    }
    const float bo = bias && o < N ? bias[o] : 0.f;
    __syncthreads();
    f32x16 acc[4];
#pragma unroll
    for (int tb = 0; tb < 4; tb++) acc[tb] = f32x16{};
#pragma unroll
    for (int i = 0; i < KS; i++)
        if (i < ks) {
#pragma unroll
            for (int tb = 0; tb < 4; tb++) {
                const half8 a = *reinterpret_cast<const half8 *>(&sx[32 * tb + l32][16 * i + 8 * hf]);
                acc[tb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, w[i], acc[tb], 0, 0, 0);
            }
        }
    if (N % 4 || ((uintptr_t)Y & 15)) {
        if (o >= N) return;
#pragma unroll
        for (int tb = 0; tb < 4; tb++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int tl = 32 * tb + 8 * g + 4 * hf;
                const f32x4 xs = *reinterpret_cast<const f32x4 *>(&sinv[tl]);
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (m0 + tl + v < M) Y[(size_t)(m0 + tl + v) * N + o] = acc[tb][4 * g + v] * xs[v] + bo;
            }
        return;
    }
    // 32 tokens at a time through LDS, so that a store takes 512 bytes of each of two
    // tokens (4 bytes a lane: 28.2 us at 2880 x 96 -> 5376, this 18.6, past the caches 17.3)
    float *so = reinterpret_cast<float *>(sx);
    const int c4 = nt * SHORT_N + 4 * (tid & 31);
#pragma unroll
    for (int tb = 0; tb < 4; tb++) {
        float *b = so + (tb & 1) * 32 * SHORT_N;
        if (tb == 0) __syncthreads();  // sx is read
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const f32x4 xs = *reinterpret_cast<const f32x4 *>(&sinv[32 * tb + 8 * g + 4 * hf]);
#pragma unroll
            for (int v = 0; v < 4; v++)
                b[(8 * g + 4 * hf + v) * SHORT_N + 32 * wave + l32] = acc[tb][4 * g + v] * xs[v] + bo;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = (tid >> 5) + 8 * i, t = m0 + 32 * tb + r;
            if (t < M && c4 < N)
                __builtin_nontemporal_store(*reinterpret_cast<const f32x4 *>(b + r * SHORT_N + 4 * (tid & 31)),
                                            reinterpret_cast<f32x4 *>(Y + (size_t)t * N + c4));
        }
    }
}

// Workgroups of M x N outputs, token tiles first; in 64 bits: M + 127 does not fit an int at the largest M.
constexpr int64_t short_tiles(int64_t M, int64_t N) {
    return (M + SHORT_M - 1) / SHORT_M * ((N + SHORT_N - 1) / SHORT_N);
}
static_assert(short_tiles(0x7FFFFFFF, 1) == 0x1000000 && short_tiles(0x7FFFFFFF, 0x7FFFFFFF) > 0x7FFFFFFF, "");

}  // namespace

extern "C" int fh3k_short16_fits(int K, int N, int M) {
    return K >= 8 && K <= SHORT_K && K % 8 == 0 && N <= 0x7FFFFFFF - SHORT_N &&
           short_tiles(M, N) <= 0xFFFFFF;  // a launch holds fewer than 2^32 threads
}

extern "C" hipError_t fh3k_short16(const void *W16, int N, int K, const float *x, const float *bias, float *y, int M,
                                   hipStream_t st) {
    if (!fh3k_short16_fits(K, N, M)) return hipErrorInvalidValue;
    const int n_tiles = (N + SHORT_N - 1) / SHORT_N;
    hipLaunchKernelGGL(k_short16, dim3((unsigned)short_tiles(M, N)), dim3(256), 0, st,
                       (const _Float16 *)W16, N, K, x, bias, y, M, n_tiles);
    return hipGetLastError();
}
