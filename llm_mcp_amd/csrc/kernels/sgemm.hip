// K23: projection of a few rows (1 to 64; ops.sgemm_splits and the encoders take it to 32, and one and
// two rows of K in whole thousands go to gemv.hip) with small weights:
//     C[M, N] = epi(A[M, K] . W[N, K]^T)      bf16 in, fp32 accumulate
//
// Such a product is bound by latencies, not by its weight stream: the decode GEMM
// (dgemm.hip) stages both operands through an LDS ring whose every step waits for
// a barrier, and reaches a small weight with few workgroups or with K slices that
// another kernel has to sum. Here a workgroup owns 16 NT columns over all of K (or
// a slice) and its 8 waves share K: a wave loads its fragments straight to registers,
// U K32 steps (16 B a lane) at a time and the next U behind them, so the whole
// workgroup has 64 KB of weights in flight without a barrier (128 with one row tile and two column
// tiles, 32 with four row tiles and one column tile); one exchange through LDS
// adds the 8 partial tiles. Every weight is read once, the activations once per
// workgroup from L2.
//
// Operands swapped as in dgemm.hip: D = W_tile . A_tile^T, so a lane holds 4
// consecutive columns of one row.
//
// Measured (cold weights, one row / 16 rows; before: K11 with its slices): 3072 x 2048 5.4 / 6.7 us
// (11.2 / 11.4), 2048 x 2048 as two slabs 4.1 / 4.7 (7.1 / 7.3), 2304 x 768 4.0 / 4.5 (- / 5.7),
// 4096 x 4096 9.1 / 12.8 (10.9 / 11.6): above 32 rows and some 20 MB the ring kernels are the better
// ones, since every workgroup reads all activations (28672 x 4096 50.9 / 62.2 against 38.8). Long K
// needs slices: a workgroup walks all of its K alone (the lines, measured: ops.sgemm_splits).
#include "common.h"

namespace lmx {
namespace {

constexpr int SG_WAVES = 8;

enum { SG_PLAIN = 0, SG_PARTIAL = 2, SG_SWIGLU = 3, SG_RELUGLU = 4, SG_BIAS = 5, SG_GELU = 6 };

// rows [0, 16 MT), columns 16 NT blockIdx.x .., K32 steps of slice blockIdx.y
template <int MT, int NT, int EPI>
__global__ void __launch_bounds__(64 * SG_WAVES) sgemm_kernel(
    void* __restrict__ C, const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int M, int N,
    int K, long lda, long ldw, long ldc, const bf16_t* __restrict__ bias) {
  constexpr int U = MT * NT >= 4 ? 2 : 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 15, fg = lane >> 4;
  const int n0 = xcd_remap(blockIdx.x, gridDim.x) * 16 * NT;
  // this wave's steps of this slice
  const int steps = K / 32, per = steps / (int)gridDim.y;
  const int s0 = blockIdx.y * per + per * wave / SG_WAVES;
  const int s1 = blockIdx.y * per + per * (wave + 1) / SG_WAVES;
  const bf16_t* wp[NT];
  const bf16_t* ap[MT];
#pragma unroll
  for (int j = 0; j < NT; ++j) wp[j] = W + (long)(n0 + 16 * j + fr) * ldw + 8 * fg;
#pragma unroll
  for (int i = 0; i < MT; ++i) ap[i] = A + (long)min(16 * i + fr, M - 1) * lda + 8 * fg;
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  struct Batch { bf16x8_t w[U][NT], a[U][MT]; };
  // steps past the end re-read the last one (never multiplied)
  auto load = [&](Batch& b, int s) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long k = 32L * min(s + u, s1 - 1);
#pragma unroll
      for (int j = 0; j < NT; ++j) b.w[u][j] = load_frag16B(wp[j] + k);
#pragma unroll
      for (int i = 0; i < MT; ++i) b.a[u][i] = load_frag16B(ap[i] + k);
    }
  };
  auto mma = [&](const Batch& b, int s) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u >= s1) break;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = mfma16(b.w[u][j], b.a[u][i], acc[i][j]);
    }
  };
  if (s0 < s1) {
    Batch x, y;
    load(x, s0);
    for (int s = s0; s < s1; s += 2 * U) {
      if (s + U < s1) load(y, s + U);
      mma(x, s);
      if (s + 2 * U < s1) load(x, s + 2 * U);
      if (s + U < s1) mma(y, s + U);
    }
  }

  // the waves' partial tiles, summed in wave order
  __shared__ f32x4_t part[SG_WAVES][MT * NT][64];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) part[wave][i * NT + j][lane] = acc[i][j];
  __syncthreads();
  constexpr bool PAIR = EPI == SG_SWIGLU || EPI == SG_RELUGLU;
  constexpr int OT = PAIR ? MT : MT * NT;                  // 16 x 16 output tiles
  static_assert(!PAIR || NT == 2, "gate and up columns side by side");
  for (int o = wave; o < OT; o += SG_WAVES) {
    const int i = PAIR ? o : o / NT, j = PAIR ? 0 : o % NT, m = 16 * i + fr;
    f32x4_t s = part[0][i * NT + j][lane];
#pragma unroll
    for (int v = 1; v < SG_WAVES; ++v) s += part[v][i * NT + j][lane];
    if constexpr (PAIR) {
      f32x4_t up = part[0][i * NT + 1][lane];
#pragma unroll
      for (int v = 1; v < SG_WAVES; ++v) up += part[v][i * NT + 1][lane];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        s[r] = (EPI == SG_SWIGLU ? s[r] / (1.f + __expf(-s[r])) : fmaxf(s[r], 0.f)) * up[r];
    }
    if (m >= M) continue;
    const int n = (PAIR ? n0 / 2 : n0 + 16 * j) + 4 * fg;
    if constexpr (EPI == SG_PARTIAL) {
      *reinterpret_cast<f32x4_t*>((float*)C + ((long)blockIdx.y * M + m) * N + n) = s;
    } else {
      bf16x4_t v;
      if constexpr (EPI == SG_BIAS || EPI == SG_GELU) {
        const bf16x4_t b = *reinterpret_cast<const bf16x4_t*>(bias + n);
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] += bf2f((uint16_t)b[r]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = (short)f2bf(EPI == SG_GELU ? gelu_erf(s[r]) : s[r]);
      *reinterpret_cast<bf16x4_t*>((bf16_t*)C + (long)m * ldc + n) = v;
    }
  }
}

template <int MT, int NT>
int sg_launch(void* C, const bf16_t* A, const bf16_t* W, int M, int N, int K, long lda, long ldw,
              long ldc, int epi, int splits, const bf16_t* bias, hipStream_t stream) {
  const dim3 grid(N / (16 * NT), splits), block(64 * SG_WAVES);
#define LMX_SG(E) sgemm_kernel<MT, NT, E><<<grid, block, 0, stream>>>(C, A, W, M, N, K, lda, ldw, ldc, bias)
  switch (epi) {
    case SG_PLAIN: LMX_SG(SG_PLAIN); break;
    case SG_PARTIAL: LMX_SG(SG_PARTIAL); break;
    case SG_BIAS: LMX_SG(SG_BIAS); break;
    case SG_GELU: LMX_SG(SG_GELU); break;
    case SG_SWIGLU:
      if constexpr (NT == 2) { LMX_SG(SG_SWIGLU); break; } else return -1;
    case SG_RELUGLU:
      if constexpr (NT == 2) { LMX_SG(SG_RELUGLU); break; } else return -1;
    default: return -1;
  }
#undef LMX_SG
  return (int)hipGetLastError();
}

}  // namespace

// epi as dgemm's: 0 plain, 2 fp32 slabs [splits][M][N] in C, 3 SwiGLU and 4 ReLU-GLU over
// 16-row pairs, 5 + bias, 6 gelu(+ bias). splits > 1 only with the slabs.
int sgemm(void* C, const void* A, const void* W, int M, int N, int K, long lda, long ldw, long ldc,
          int epi, int splits, const void* bias, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 64 || N % 32 || K % 32 || splits < 1 || (splits > 1 && epi != 2) || K / 32 % splits) return -1;
  if (lda % 8 || ldw % 8 || ldc % 4 || (((uintptr_t)A | (uintptr_t)W) & 15) || ((uintptr_t)C & 7) ||
      (epi == 2 && ((uintptr_t)C & 15)) || (epi >= 5) != (bias != nullptr) || ((uintptr_t)bias & 7))
    return -1;
  auto A_ = (const bf16_t*)A;
  auto W_ = (const bf16_t*)W;
  auto b_ = (const bf16_t*)bias;
  const int mt = (M + 15) / 16;
  const bool two = epi == SG_SWIGLU || epi == SG_RELUGLU || (N / 16 * splits > 512);
#define LMX_SGM(MTV)                                                                              \
  return two ? sg_launch<MTV, 2>(C, A_, W_, M, N, K, lda, ldw, ldc, epi, splits, b_, stream)      \
             : sg_launch<MTV, 1>(C, A_, W_, M, N, K, lda, ldw, ldc, epi, splits, b_, stream);
  if (mt == 1) { LMX_SGM(1) }
  if (mt == 2) { LMX_SGM(2) }
  LMX_SGM(4)
#undef LMX_SGM
}

}  // namespace lmx
