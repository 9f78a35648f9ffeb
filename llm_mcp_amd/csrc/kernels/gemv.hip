// K25: projection of one or two rows:  C[M, N] = epi(A[M, K] . W[N, K]^T)
// bf16 in, fp32 accumulate.
//
// A step of one stream does nothing but stream weights, and every kernel built on MFMA operands
// reads them as 16 rows x 64 B (or through an LDS ring with its barriers). Here a wave takes whole
// rows of W, 1 KB of one row an instruction, non-temporal, and multiplies by fp32 FMAs: at one row
// 40 vector instructions for 2 KB, well under the stream. Two rows a wave (a gate row and
// its up row under the pair epilogues), two instructions of each in flight, 8 waves a SIMD;
// no LDS, no barrier. The activations (8 KB a row at K = 4096) come from the vector L1.
// Measured, cold weights, one row (before: the fastest of K11 and K23): 16384 x 2048 with the
// SwiGLU 12.3 us (18.0), 6144 x 4096 10.4 (13.7), 3072 x 2048 4.5 (5.5), 4096 x 4096 7.8 (9.2), 2048 x
// 8192 in two slices 7.9 (9.3), 28672 x 4096 37.8 (39.2), 128256 x 4096 151 (160): 2.8 TB/s for 13 MB, 4.2
// to 4.8 for 34 to 50, 5.5 for 67, 6.2 to 7 from 235 on. Two rows 0.4 to 2 us more up to 150 MB, beyond 2
// to 10 % (17 % at K = 25600, where the rows pass the vector L1), four no better than before. A read of the
// same bytes that does nothing else takes 11.5, 9.3, 3.4 and 6.8 for the first four. Where a measured
// kernel of the table is faster the product stays there (ops.table_keeps). Blocks in plain order (not a range of rows per XCD)
// cost 10 % at K = 4096.
#include "common.h"

namespace lmx {
namespace {

enum { GV_PLAIN = 0, GV_PARTIAL = 2, GV_SWIGLU = 3, GV_RELUGLU = 4, GV_BIAS = 5 };
constexpr int GV_STEP = 1024;      // elements of K a pass

typedef uint32_t gv_u4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void gv_unpack(const gv_u4_t& v, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(v[i] << 16);
    f[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
  }
}

// grid (N / 8, splits), 4 waves: passes of slice blockIdx.y
template <int M, int EPI>
__global__ void __launch_bounds__(256) gemv_kernel(void* __restrict__ C, const bf16_t* __restrict__ A,
                                                   const bf16_t* __restrict__ W, int N, int K, long lda,
                                                   long ldw, long ldc, const bf16_t* __restrict__ bias) {
  constexpr bool PAIR = EPI == GV_SWIGLU || EPI == GV_RELUGLU;
  const int lane = threadIdx.x & 63;
  const int g = xcd_remap(blockIdx.x, gridDim.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the wave's two rows of W
  const int n0 = PAIR ? 32 * (g >> 4) + (g & 15) : 2 * g, n1 = PAIR ? n0 + 16 : n0 + 1;
  const int per = K / GV_STEP / (int)gridDim.y * GV_STEP;
  const long k0 = (long)blockIdx.y * per + 8 * lane;
  const bf16_t* w[2] = {W + n0 * ldw + k0, W + n1 * ldw + k0};
  const bf16_t* a = A + k0;
  float s[M][2];
#pragma unroll
  for (int m = 0; m < M; ++m) s[m][0] = s[m][1] = 0.f;
  for (int k = 0; k < per; k += GV_STEP) {
    gv_u4_t wv[2][2], av[2][M];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 2; ++r)
        wv[u][r] = __builtin_nontemporal_load(reinterpret_cast<const gv_u4_t*>(w[r] + k + 512 * u));
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int m = 0; m < M; ++m)
        av[u][m] = *reinterpret_cast<const gv_u4_t*>(a + m * lda + k + 512 * u);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float x[2][8];
      gv_unpack(wv[u][0], x[0]);
      gv_unpack(wv[u][1], x[1]);
#pragma unroll
      for (int m = 0; m < M; ++m) {
        float y[8];
        gv_unpack(av[u][m], y);
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int i = 0; i < 8; ++i) s[m][r] = fmaf(x[r][i], y[i], s[m][r]);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int r = 0; r < 2; ++r) s[m][r] = wave_sum(s[m][r]);
  // lane m writes row m
#pragma unroll
  for (int m = 0; m < M; ++m) {
    if (lane != m) continue;
    const float x = s[m][0], y = s[m][1];
    if constexpr (EPI == GV_PARTIAL) {
      *reinterpret_cast<float2*>((float*)C + ((long)blockIdx.y * M + m) * N + n0) = make_float2(x, y);
    } else if constexpr (PAIR) {
      const float act = EPI == GV_SWIGLU ? x / (1.f + __expf(-x)) : fmaxf(x, 0.f);
      ((bf16_t*)C)[m * ldc + 16 * (g >> 4) + (g & 15)] = f2bf(act * y);
    } else {
      const float b0 = EPI == GV_BIAS ? bf2f(bias[n0]) : 0.f, b1 = EPI == GV_BIAS ? bf2f(bias[n1]) : 0.f;
      *reinterpret_cast<uint32_t*>((bf16_t*)C + m * ldc + n0) = pack_bf16x2(x + b0, y + b1);
    }
  }
}

template <int M>
int gv_launch(void* C, const bf16_t* A, const bf16_t* W, int N, int K, long lda, long ldw, long ldc, int epi,
              int splits, const bf16_t* bias, hipStream_t stream) {
  const dim3 grid(N / 8, splits), block(256);
#define LMX_GV(E) gemv_kernel<M, E><<<grid, block, 0, stream>>>(C, A, W, N, K, lda, ldw, ldc, bias)
  switch (epi) {
    case GV_PLAIN: LMX_GV(GV_PLAIN); break;
    case GV_PARTIAL: LMX_GV(GV_PARTIAL); break;
    case GV_SWIGLU: LMX_GV(GV_SWIGLU); break;
    case GV_RELUGLU: LMX_GV(GV_RELUGLU); break;
    case GV_BIAS: LMX_GV(GV_BIAS); break;
    default: return -1;
  }
#undef LMX_GV
  return (int)hipGetLastError();
}

}  // namespace

// epi as dgemm's: 0 plain, 2 fp32 slabs [splits][M][N] in C, 3 SwiGLU and 4 ReLU-GLU over 16-row pairs,
// 5 + bias. splits > 1 only with the slabs.
int gemv(void* C, const void* A, const void* W, int M, int N, int K, long lda, long ldw, long ldc, int epi,
         int splits, const void* bias, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 2 || N % 32 || K % GV_STEP || splits < 1 || (splits > 1 && epi != 2) || K / GV_STEP % splits)
    return -1;
  if (lda % 8 || ldw % 8 || ldc % 2 || (((uintptr_t)A | (uintptr_t)W) & 15) || ((uintptr_t)C & 3) ||
      (epi == 2 && ((uintptr_t)C & 7)) || (epi == 5) != (bias != nullptr) || ((uintptr_t)bias & 1))
    return -1;
  auto A_ = (const bf16_t*)A;
  auto W_ = (const bf16_t*)W;
  auto b_ = (const bf16_t*)bias;
  return M == 1 ? gv_launch<1>(C, A_, W_, N, K, lda, ldw, ldc, epi, splits, b_, stream)
                : gv_launch<2>(C, A_, W_, N, K, lda, ldw, ldc, epi, splits, b_, stream);
}

}  // namespace lmx
