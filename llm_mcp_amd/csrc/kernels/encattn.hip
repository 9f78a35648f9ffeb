// K24: bidirectional attention of the embedding encoders (head dim 64) on the rows of the
// fused projection, packed sequences; no cache pages and no pass that writes them.
//
//   qkv [T][ld]: q | k | v, H heads each; sequence s holds rows cu[s] .. cu[s + 1] - 1
//   tiles[t] = {sequence, first query}, EA_Q queries each, longest sequences first
//   cos_sin (or null): [positions][64] cos | sin; q and k are rotated by their place
//   in the sequence, in fp32, and rounded to bf16 as rope_cache.hip does
//
// A workgroup of 4 waves serves 128 queries of a head, 32 a wave (the columns of 32 x 32 x 16
// MFMAs): S^T = K Q^T leaves a lane with half of a query's 64 scores of a tile, so that maxima
// and sums take one lane swap, and the weights are the PV product's B operand as they
// are (keys in the order of the accumulators; V^T is read in that order by the transposing
// LDS read, from the same row-major image that the rows arrive in).  K / V rows go through
// registers (they are rotated there) into a double buffer: the next tile's loads are in flight
// while a tile is computed, one barrier a tile.
// The grid has the heads innermost: the workgroups of a head run on 8 / gcd(H, 8) XCDs (one for 16 heads,
// two for 12), which read its K / V through their L2, and the longest sequences start first.
// Bound by vector instructions (150 a wave and tile, 32 of them exponentials, 56 more for the
// rotation): 16 heads, 48 sequences of 512: 70 us, 739 TF/s; 12 heads, 16 of 735, rotated: 58 us.
// Cache pages written by one kernel and read by the prompt attention took 85 + 40 us for 19153
// tokens of 16 heads (now 55) and 72 + 23 us for 11760 of 12 (58).  Operands of whole products
// loaded ahead (155 registers, 3 waves a SIMD) and the angles kept in registers for a tile measured
// the same.
#include "attention.h"

namespace lmx {

namespace {

constexpr int EA_Q = 128, EA_K = 64, EA_D = 64, EA_THREADS = 256;
constexpr int EA_IMG = EA_K * EA_D;       // elements of a tile's K or V image

typedef short ea_s4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) ea_s4_t ea_lds4_t;

// cos and sin of 8 consecutive pairs (elements d and d + 32)
struct EaAngles { float4 c[2], s[2]; };
__device__ __forceinline__ EaAngles ea_angles(const float* __restrict__ cs) {
  const float4* p = reinterpret_cast<const float4*>(cs);
  return {{p[0], p[1]}, {p[8], p[9]}};
}

__device__ __forceinline__ void ea_rotate(bf16x8_t& lo, bf16x8_t& hi, const EaAngles& r) {
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  u32x4_t x = __builtin_bit_cast(u32x4_t, lo), y = __builtin_bit_cast(u32x4_t, hi);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float4 &c4 = r.c[j >> 1], &s4 = r.s[j >> 1];
    const float c0 = j & 1 ? c4.z : c4.x, c1 = j & 1 ? c4.w : c4.y;
    const float s0 = j & 1 ? s4.z : s4.x, s1 = j & 1 ? s4.w : s4.y;
    const float a0 = __uint_as_float(x[j] << 16), a1 = __uint_as_float(x[j] & 0xffff0000u);
    const float b0 = __uint_as_float(y[j] << 16), b1 = __uint_as_float(y[j] & 0xffff0000u);
    x[j] = cvt_pk(a0 * c0 - b0 * s0, a1 * c1 - b1 * s1);
    y[j] = cvt_pk(b0 * c0 + a0 * s0, b1 * c1 + a1 * s1);
  }
  lo = __builtin_bit_cast(bf16x8_t, x);
  hi = __builtin_bit_cast(bf16x8_t, y);
}

// orders LDS accesses only: __syncthreads would also wait for the loads in flight
__device__ __forceinline__ void ea_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <bool ROPE>
__global__ void __launch_bounds__(EA_THREADS, 4) enc_attention_kernel(
    const bf16_t* __restrict__ qkv, long ld, int H, const int* __restrict__ cu,
    const int* __restrict__ tiles, const float* __restrict__ cos_sin, bf16_t* __restrict__ out,
    long ldo, float scale_log2, float rescale_thr) {
  __shared__ __attribute__((aligned(16))) bf16_t lds[2][2][EA_IMG];    // [buffer][K, V][key][d]
  const int t = blockIdx.x / H, head = blockIdx.x - t * H;
  const int seq = tiles[2 * t], q0 = tiles[2 * t + 1];
  const int beg = cu[seq], len = cu[seq + 1] - beg;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 31, h = lane >> 5;
  const int ntiles = (len + EA_K - 1) / EA_K;
  const bf16_t* const rows = qkv + (long)beg * ld + head * EA_D;
  const bf16_t* const krows = rows + (long)H * EA_D;
  const bf16_t* const vrows = krows + (long)H * EA_D;

  // staging: a thread moves elements 8 p .. and 32 + 8 p .. of key row sr (a rotation's pairs)
  const int sr = threadIdx.x >> 2, sp = threadIdx.x & 3;
  bf16x8_t kl, kh, vl, vh;
  auto load = [&](int tile) {
    const int key = min(tile * EA_K + sr, len - 1);
    const long off = (long)key * ld + 8 * sp;
    kl = load_frag16B(krows + off);
    kh = load_frag16B(krows + off + 32);
    vl = load_frag16B(vrows + off);
    vh = load_frag16B(vrows + off + 32);
  };
  // K image: 16-byte pieces at piece ^ (row / 2 % 8); V image: halves of a row swapped by row / 2
  // % 2: no bank is read twice by the 16 lanes of a K read or the 32 of a V read
  const int kswz = (sr >> 1) & 7, vswz = (sr >> 1) & 1;
  const int kat = sr * EA_D + 8 * (sp ^ kswz), kat2 = sr * EA_D + 8 * ((sp + 4) ^ kswz);
  const int vat = sr * EA_D + 32 * vswz + 8 * sp, vat2 = vat ^ 32;
  auto store = [&](int tile) {
    const int key = tile * EA_K + sr;
    bf16_t* const ki = lds[tile & 1][0];
    bf16_t* const vi = lds[tile & 1][1];
    if constexpr (ROPE) ea_rotate(kl, kh, ea_angles(cos_sin + (long)min(key, len - 1) * EA_D + 8 * sp));
    if (key >= len) vl = vh = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};      // weighs 0: must be finite
    *reinterpret_cast<bf16x8_t*>(ki + kat) = kl;
    *reinterpret_cast<bf16x8_t*>(ki + kat2) = kh;
    *reinterpret_cast<bf16x8_t*>(vi + vat) = vl;
    *reinterpret_cast<bf16x8_t*>(vi + vat2) = vh;
  };

  load(0);
  const int q = q0 + wave * 32 + c;                     // this lane's query
  const bool idle = q0 + wave * 32 >= len;              // the wave's: none
  bf16x8_t qf[4];
#pragma unroll
  for (int s = 0; s < 4; ++s)
    qf[s] = load_frag16B(rows + (long)min(q, len - 1) * ld + 16 * s + 8 * h);
  if constexpr (ROPE) {
    const float* cs = cos_sin + (long)min(q, len - 1) * EA_D + 8 * h;
    ea_rotate(qf[0], qf[2], ea_angles(cs));
    ea_rotate(qf[1], qf[3], ea_angles(cs + 16));
  }
  // used up here: a wait for them inside the loop would be one for the tiles in flight too
#pragma unroll
  for (int s = 0; s < 4; ++s) asm volatile("" : "+v"(qf[s]));
  store(0);
  if (ntiles > 1) load(1);
  ea_barrier();

  int kr[4];                                            // K operand: row c, elements 16 s + 8 h ..
#pragma unroll
  for (int s = 0; s < 4; ++s) kr[s] = c * EA_D + 8 * ((2 * s + h) ^ ((c >> 1) & 7));
  // V^T operand (rows d, keys 4 h .. and 8 + 4 h .. of 16): a group of 16 lanes turns 4 rows x 16
  const int vi16 = lane & 15, vrow = 4 * h + (vi16 >> 2);
  const int vr = vrow * EA_D + 32 * ((vrow >> 1) & 1) + 16 * ((lane >> 4) & 1) + 4 * (vi16 & 3);

  float m = -INFINITY, l = 0.f;
  f32x16_t acc[2];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.f;
  for (int tile = 0; tile < ntiles; ++tile) {
    if (tile + 1 < ntiles) {
      store(tile + 1);           // its buffer was read last before the barrier of tile - 1
      if (tile + 2 < ntiles) load(tile + 2);
    }
    if (!idle) {
      const bf16_t* const ki = lds[tile & 1][0];
      bf16_t* const vi = lds[tile & 1][1];
      f32x16_t s[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[b][i] = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          s[b] = mfma32(load_frag16B(ki + kr[k] + b * 32 * EA_D), qf[k], s[b]);
      }
      if (tile == ntiles - 1) {
        const int left = len - tile * EA_K - 4 * h;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            s[b][i] = 32 * b + 8 * (i >> 2) + (i & 3) < left ? s[b][i] : -INFINITY;
      }
      float mx4[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) mx4[i] = max2f(s[0][i], s[1][i]);
#pragma unroll
      for (int i = 4; i < 16; ++i) mx4[i & 3] = max3f(mx4[i & 3], s[0][i], s[1][i]);
      float mx = max3f(max2f(mx4[0], mx4[1]), mx4[2], mx4[3]);
      {
        const unsigned u = __float_as_uint(mx);
        const auto w = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        mx = max2f(__uint_as_float(w[0]), __uint_as_float(w[1])) * scale_log2;
      }
      // the running maximum is raised for the whole wave, and only where a query's
      // weights would pass 2^rescale_thr (attention.hip's rule)
      if (__ballot(!(mx <= m + rescale_thr))) {
        const float mn = max2f(m, mx), al = mn == -INFINITY ? 1.f : fast_exp2(m - mn);
        l *= al;
        m = mn;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          acc[0][i] *= al;
          acc[1][i] *= al;
        }
      }
      const float mu = m == -INFINITY ? 0.f : m;
      float sum[2] = {0.f, 0.f};
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[b][i] = fast_exp2(fmaf(s[b][i], scale_log2, -mu));
          sum[i & 1] += s[b][i];
        }
      l += sum[0] + sum[1];                             // of this lane's keys
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        union { uint32_t u[4]; bf16x8_t v; } p;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          p.u[j] = cvt_pk(s[k >> 1][8 * (k & 1) + 2 * j], s[k >> 1][8 * (k & 1) + 2 * j + 1]);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          bf16_t* const at = vi + (vr ^ (32 * b)) + k * 16 * EA_D;
          const ea_s4_t x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ea_lds4_t*)at);
          const ea_s4_t y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ea_lds4_t*)(at + 8 * EA_D));
          const bf16x8_t vf = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
          acc[b] = mfma32(vf, p.v, acc[b]);
        }
      }
    }
    ea_barrier();
  }
  {
    const unsigned u = __float_as_uint(l);
    const auto w = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    l = __uint_as_float(w[0]) + __uint_as_float(w[1]);
  }
  if (q >= len) return;
  // a lane holds elements 8 i + 4 h .. of its query; the swap leaves it with whole 16-byte
  // pieces 2 i + h
  const float inv = l == 0.f ? 0.f : 1.f / l;
  bf16_t* const o = out + (long)(beg + q) * ldo + head * EA_D + 8 * h;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f32x16_t& a = acc[b];
      const int e = 8 * i;
      const uint32_t x0 = cvt_pk(a[e] * inv, a[e + 1] * inv);
      const uint32_t x1 = cvt_pk(a[e + 2] * inv, a[e + 3] * inv);
      const uint32_t y0 = cvt_pk(a[e + 4] * inv, a[e + 5] * inv);
      const uint32_t y1 = cvt_pk(a[e + 6] * inv, a[e + 7] * inv);
      const auto w0 = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
      const auto w1 = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
      *reinterpret_cast<uint4*>(o + 32 * b + 16 * i) = make_uint4(w0[0], w1[0], w0[1], w1[1]);
    }
}

}  // namespace

int enc_attention(const void* qkv, long ld, int H, int D, const int* cu, const int* tiles, int ntiles,
                  const float* cos_sin, void* out, long ldo, float scale, float rescale_thr,
                  hipStream_t stream) {
  if (ntiles <= 0) return 0;
  if (D != EA_D || ld % 8 || ldo % 8 || ((uintptr_t)qkv & 15) || ((uintptr_t)out & 15) ||
      ((uintptr_t)cos_sin & 15))
    return -1;
  if ((long)ntiles * H > 0x7fffffffL) return -2;
  const dim3 grid(ntiles * H), block(EA_THREADS);
  const float sl = scale * LOG2E;
  if (cos_sin)
    enc_attention_kernel<true><<<grid, block, 0, stream>>>((const bf16_t*)qkv, ld, H, cu, tiles, cos_sin,
                                                           (bf16_t*)out, ldo, sl, rescale_thr);
  else
    enc_attention_kernel<false><<<grid, block, 0, stream>>>((const bf16_t*)qkv, ld, H, cu, tiles, cos_sin,
                                                            (bf16_t*)out, ldo, sl, rescale_thr);
  return (int)hipGetLastError();
}

}  // namespace lmx
