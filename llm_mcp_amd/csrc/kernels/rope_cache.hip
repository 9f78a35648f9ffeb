// K2 + K5: rotary embedding (neox / rotate-half form, as Llama-3 and
// nomic-bert use) applied in place to the q and k heads of the fused QKV
// projection output, fused with the scatter of k and v into the paged KV cache.
//
// KV-cache layout (MI355X-first, chosen for the MFMA operand maps of the
// attention kernels, see decode_attn.hip):
//   k_cache [num_blocks][Hkv][BS][D]   token-major: a K row is the 16-B A/B
//                                      fragment source of S = K.Q^T
//   v_cache [num_blocks][Hkv][BS/4][D][4]   key-quad: the 4 consecutive
//                                      tokens of one d are the contiguous 8-B
//                                      fragment run of O^T = V^T.P^T, and one
//                                      token's D values share D/16 128-B lines
//                                      (a d-major page [D][BS] spread a token
//                                      over D/2 lines: 17-20 us per decode
//                                      call of partial-line writes)
// cos/sin come from a host-precomputed fp32 table [max_pos][D] (cos | sin),
// so no transcendental runs on the device (guide App. B, element-wise).
#include "common.h"

namespace lmx {

// Optional per-head RMSNorm of q and k before the rotation (Qwen3's q_norm /
// k_norm).  The 16 lanes that own one head (tph = D/8 lanes x 8 elements)
// are consecutive and 16-aligned in every loop below, so the head's sum of
// squares is a 16-wide xor-shuffle reduction; normalisation stays in fp32
// through the rotation (one bf16 rounding).
__device__ __forceinline__ void qk_norm(float (&a)[4], float (&b)[4], const bf16_t* w, int i,
                                        int half, int D, float eps) {
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) ss += a[j] * a[j] + b[j] * b[j];
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 16);
  const float r = rsqrtf(ss / (float)D + eps);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    a[j] *= r * bf2f(w[i + j]);
    b[j] *= r * bf2f(w[half + i + j]);
  }
}

// Decode rows: one workgroup per token.  A thread owns up to IT rotation
// items (4 pairs of one head each); all of its q/k and cos/sin loads are
// issued before the first use (IT is a template parameter: a runtime-bounded
// loop re-serialised them into IT dependent memory latencies), then the V row
// goes to the transposed page 4 elements (one 8-B load) per thread.
template <int IT>
__global__ void __launch_bounds__(256) rope_cache_kernel(
    bf16_t* __restrict__ qkv, long qkv_stride, const int* __restrict__ positions,
    const float* __restrict__ cos_sin, int Hq, int Hkv, int D,
    const int* __restrict__ slot_mapping, bf16_t* __restrict__ k_cache,
    bf16_t* __restrict__ v_cache, int BS, int rotate_k_inplace,
    const bf16_t* __restrict__ q_norm, const bf16_t* __restrict__ k_norm, float eps) {
  const int t = blockIdx.x;
  const int half = D >> 1;
  const int tph = half >> 2;  // threads per head, each owns 4 rotation pairs
  bf16_t* row = qkv + (long)t * qkv_stride;
  const int pos = positions[t];
  const float* cs = cos_sin + (long)pos * D;
  const int slot = slot_mapping ? slot_mapping[t] : -1;
  const int blk = slot >= 0 ? slot / BS : 0, off = slot >= 0 ? slot % BS : 0;
  const int nrot = (Hq + Hkv) * tph;

  bf16x4_t x1[IT], x2[IT];
  float4 c[IT], sn[IT];
#pragma unroll
  for (int k = 0; k < IT; ++k) {
    const int it = threadIdx.x + k * 256;
    if (it < nrot) {
      const int h = it / tph, i = (it % tph) * 4;
      const bf16_t* hp = row + (long)h * D;
      x1[k] = *reinterpret_cast<const bf16x4_t*>(hp + i);
      x2[k] = *reinterpret_cast<const bf16x4_t*>(hp + half + i);
      c[k] = *reinterpret_cast<const float4*>(cs + i);
      sn[k] = *reinterpret_cast<const float4*>(cs + half + i);
    }
  }
  // V row loads issued with the rest (4 elements per thread per pass)
  const bf16_t* vrow = row + (long)(Hq + Hkv) * D;
  const int nv = Hkv * D;
  constexpr int VP = 2;                       // V passes held in registers (nv <= 2048)
  bf16x4_t vv[VP];
#pragma unroll
  for (int k = 0; k < VP; ++k) {
    const int e = (threadIdx.x + k * 256) * 4;
    if (slot >= 0 && v_cache && e < nv) vv[k] = *reinterpret_cast<const bf16x4_t*>(vrow + e);
  }
#pragma unroll
  for (int k = 0; k < IT; ++k) {
    const int it = threadIdx.x + k * 256;
    if (it >= nrot) continue;
    const int h = it / tph, i = (it % tph) * 4;
    bf16_t* hp = row + (long)h * D;
    const float cc[4] = {c[k].x, c[k].y, c[k].z, c[k].w};
    const float ss[4] = {sn[k].x, sn[k].y, sn[k].z, sn[k].w};
    const bool is_k = h >= Hq;
    float a[4], b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j] = bf2f((uint16_t)x1[k][j]), b[j] = bf2f((uint16_t)x2[k][j]);
    if (q_norm) qk_norm(a, b, is_k ? k_norm : q_norm, i, half, D, eps);
    bf16x4_t o1, o2;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o1[j] = (short)f2bf(a[j] * cc[j] - b[j] * ss[j]);
      o2[j] = (short)f2bf(b[j] * cc[j] + a[j] * ss[j]);
    }
    if (!is_k || rotate_k_inplace || slot < 0) {
      *reinterpret_cast<bf16x4_t*>(hp + i) = o1;
      *reinterpret_cast<bf16x4_t*>(hp + half + i) = o2;
    }
    if (is_k && slot >= 0 && k_cache) {
      bf16_t* kp = k_cache + (((long)blk * Hkv + (h - Hq)) * BS + off) * D;
      *reinterpret_cast<bf16x4_t*>(kp + i) = o1;
      *reinterpret_cast<bf16x4_t*>(kp + half + i) = o2;
    }
  }
  if (slot < 0 || !v_cache) return;
  // v -> key-quad cache page (2-B stores 8 B apart: one token's D values
  // share D/16 lines of its page)
#pragma unroll
  for (int k = 0; k < VP; ++k) {
    const int e = (threadIdx.x + k * 256) * 4;
    if (e >= nv) continue;
    const int h = e / D, d = e % D;
    bf16_t* vp = v_cache + ((long)blk * Hkv + h) * BS * D + vq_off(d, off, D);
#pragma unroll
    for (int j = 0; j < 4; ++j) vp[4 * j] = (bf16_t)vv[k][j];
  }
}

// Prefill rows: a workgroup of grid.x takes 32 consecutive tokens, one of grid.y
// a group of their heads: rotation of q / k heads (with the K write) or a group
// of V heads.  V goes through an LDS tile so that the key-quad cache page
// ([BS/4][D][4]) is written in 16-B pieces -- a thread stores 4 consecutive
// tokens of 2 d whenever their slots are consecutive and 4-aligned (always
// true inside a prefill chunk), and a wave covers 8 whole 128-B lines.
// The per-token kernel's 2-B stores remain for decode rows (one token per
// page per step, nothing to coalesce).
//
// The work is copying: memory bound when it fills the chip, otherwise bound by
// one chain of dependent latencies (slot, row, store) per workgroup.  A workgroup
// that walked all heads of its tokens ran 6 (Llama-3) to 9 (nomic) such chains one after
// the other on T / 32 workgroups; a head group is ONE chain.
// Measured, all heads in a workgroup -> groups of heads: 16 nomic tokens 17.0 -> 4.5 us, 160 Llama-3
// tokens (k and v only) 19.0 -> 5.0, 6,464 of them 30 -> 17, 11,760 nomic tokens 37.7 -> 24.4 (108 MB).
constexpr int RT = 32;
constexpr int RT_VCOLS = 256;    // V columns of a workgroup (at least a head)

// q / k heads that one workgroup rotates: up to 4 per thread, whose threads
// cover (token, 8-pair chunk) pairs of one head, or of several where D is small
__host__ __device__ constexpr int rope_head_step(int D) {
  return RT * (D / 16) >= 256 ? 1 : 256 / (RT * (D / 16));
}
__host__ __device__ constexpr int rope_v_heads(int D) { return D >= RT_VCOLS ? 1 : RT_VCOLS / D; }

// V heads h0 .. h0 + hg of tokens t0 .. t0 + nt (v: the first token's V row) to
// their pages; vt: RT rows of LD elements
__device__ __forceinline__ void v_to_pages(const bf16_t* __restrict__ v, long stride, int nt, int h0,
                                           int hg, int Hkv, int D, const int* sslot, bf16_t* vt,
                                           int LD, bf16_t* __restrict__ v_cache, int BS) {
  const int chunks = hg * D / 8;
#pragma unroll 4
  for (int it = threadIdx.x; it < nt * chunks; it += 256) {
    const int tt = it / chunks, c = it - tt * chunks;
    *reinterpret_cast<u16x8*>(&vt[tt * LD + 8 * c]) =
        *reinterpret_cast<const u16x8*>(v + (long)tt * stride + (long)h0 * D + 8 * c);
  }
  __syncthreads();
  // one 16-B store per (head, key quad, d pair): 4 tokens x 2 d of the
  // key-quad page, whenever the quad's 4 slots are consecutive and
  // 4-aligned (always, inside a prefill chunk's whole pages)
  const int per_h = (D / 2) * (RT / 4);
  for (int it = threadIdx.x; it < hg * per_h; it += 256) {
    const int hl = it / per_h, r = it - hl * per_h;
    const int d = 2 * (r % (D / 2)), tt0 = (r / (D / 2)) * 4, h = h0 + hl;
    if (tt0 >= nt) continue;
    const int col = hl * D + d;
    const int s0 = sslot[tt0];
    bool vec = tt0 + 4 <= nt && s0 >= 0 && (s0 % 4) == 0;
#pragma unroll
    for (int j = 1; j < 4; ++j) vec = vec && sslot[tt0 + j] == s0 + j;
    if (vec) {
      u16x8 w;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        w.v[j] = vt[(tt0 + j) * LD + col];
        w.v[4 + j] = vt[(tt0 + j) * LD + col + 1];
      }
      *reinterpret_cast<u16x8*>(v_cache + ((long)(s0 / BS) * Hkv + h) * BS * D +
                                vq_off(d, s0 % BS, D)) = w;
    } else {
      for (int j = 0; j < 4 && tt0 + j < nt; ++j) {
        const int sl = sslot[tt0 + j];
        if (sl < 0) continue;
        bf16_t* vp = v_cache + ((long)(sl / BS) * Hkv + h) * BS * D + vq_off(d, sl % BS, D);
        vp[0] = vt[(tt0 + j) * LD + col];
        vp[4] = vt[(tt0 + j) * LD + col + 1];
      }
    }
  }
}

// grid (32-token tiles, rotation groups + V groups)
__global__ void __launch_bounds__(256) rope_cache_tiled_kernel(
    bf16_t* __restrict__ qkv, long qkv_stride, const int* __restrict__ positions,
    const float* __restrict__ cos_sin, int row0, int T, int Hq, int Hkv, int D,
    const int* __restrict__ slot_mapping, bf16_t* __restrict__ k_cache,
    bf16_t* __restrict__ v_cache, int BS, int rotate_k_inplace,
    const bf16_t* __restrict__ q_norm, const bf16_t* __restrict__ k_norm, float eps, int skip_q,
    int rot_groups) {
  extern __shared__ __attribute__((aligned(16))) bf16_t vt[];   // [RT][rope_v_heads * D + 8]
  __shared__ int sslot[RT];
  const int t0 = row0 + blockIdx.x * RT;
  const int nt = min(RT, T - t0);
  if (threadIdx.x < RT)
    sslot[threadIdx.x] = (threadIdx.x < nt && slot_mapping) ? slot_mapping[t0 + threadIdx.x] : -1;
  __syncthreads();
  const int H = Hq + Hkv;
  if ((int)blockIdx.y >= rot_groups) {
    const int hv = rope_v_heads(D), h0 = ((int)blockIdx.y - rot_groups) * hv;
    v_to_pages(qkv + (long)t0 * qkv_stride + (long)H * D, qkv_stride, nt, h0, min(hv, Hkv - h0), Hkv,
               D, sslot, vt, hv * D + 8, v_cache, BS);
    return;
  }
  // a thread owns one (token, 8-pair chunk) of up to HU heads, whose loads are
  // issued before their arithmetic; the cos/sin chunk is loaded once for them
  // (heads of more than 128 channels take two turns)
  constexpr int HU = 4;
  const int half = D >> 1, tph = half >> 3;   // 8-pair chunks per head
  const int hs = rope_head_step(D), lanes = RT * tph;
  const int h0 = (skip_q ? Hq : 0) + blockIdx.y * HU * hs + (lanes < 256 ? threadIdx.x / lanes : 0);
  if (lanes < 256 && (int)threadIdx.x >= lanes * hs) return;
  for (int it = lanes < 256 ? threadIdx.x % lanes : threadIdx.x; it < nt * tph; it += 256) {
    const int tt = it / tph, i = (it % tph) * 8;
    bf16_t* row = qkv + (long)(t0 + tt) * qkv_stride;
    const float* cs = cos_sin + (long)positions[t0 + tt] * D;
    const int slot = sslot[tt];
    u16x8 x1[HU], x2[HU];
#pragma unroll
    for (int u = 0; u < HU; ++u) {
      if (h0 + u * hs < H) {
        const bf16_t* hp = row + (long)(h0 + u * hs) * D;
        x1[u] = *reinterpret_cast<const u16x8*>(hp + i);
        x2[u] = *reinterpret_cast<const u16x8*>(hp + half + i);
      }
    }
    float cc[8], ss[8];
#pragma unroll
    for (int q4 = 0; q4 < 2; ++q4) {
      const float4 c = *reinterpret_cast<const float4*>(cs + i + 4 * q4);
      const float4 sn = *reinterpret_cast<const float4*>(cs + half + i + 4 * q4);
      cc[4 * q4] = c.x; cc[4 * q4 + 1] = c.y; cc[4 * q4 + 2] = c.z; cc[4 * q4 + 3] = c.w;
      ss[4 * q4] = sn.x; ss[4 * q4 + 1] = sn.y; ss[4 * q4 + 2] = sn.z; ss[4 * q4 + 3] = sn.w;
    }
#pragma unroll
    for (int u = 0; u < HU; ++u) {
      const int h = h0 + u * hs;
      if (h >= H) break;
      bf16_t* hp = row + (long)h * D;
      const bool is_k = h >= Hq;
      float a[8], b[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = bf2f(x1[u].v[j]), b[j] = bf2f(x2[u].v[j]);
      if (q_norm) {
        // per-head RMSNorm of q / k (Qwen3): the head's D values are spread
        // over the 8 consecutive lanes of this (token, head)
        float sq = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) sq += a[j] * a[j] + b[j] * b[j];
#pragma unroll
        for (int o = 4; o > 0; o >>= 1) sq += __shfl_xor(sq, o, 8);
        const float r = rsqrtf(sq / (float)D + eps);
        const bf16_t* w = is_k ? k_norm : q_norm;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          a[j] *= r * bf2f(w[i + j]);
          b[j] *= r * bf2f(w[half + i + j]);
        }
      }
      u16x8 o1, o2;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        o1.v[j] = f2bf(a[j] * cc[j] - b[j] * ss[j]);
        o2.v[j] = f2bf(b[j] * cc[j] + a[j] * ss[j]);
      }
      if (!is_k || rotate_k_inplace || slot < 0) {
        *reinterpret_cast<u16x8*>(hp + i) = o1;
        *reinterpret_cast<u16x8*>(hp + half + i) = o2;
      }
      if (is_k && slot >= 0 && k_cache) {
        bf16_t* kp = k_cache + (((long)(slot / BS) * Hkv + (h - Hq)) * BS + slot % BS) * D;
        *reinterpret_cast<u16x8*>(kp + i) = o1;
        *reinterpret_cast<u16x8*>(kp + half + i) = o2;
      }
    }
  }
}

int rope_cache(void* qkv, long qkv_stride, const int* positions, const float* cos_sin, int T,
               int Hq, int Hkv, int D, const int* slot_mapping, void* k_cache, void* v_cache,
               int BS, int rotate_k_inplace, int tile_from, const void* q_norm,
               const void* k_norm, float eps, int skip_q, hipStream_t stream) {
  if (T <= 0) return 0;
  // skip_q only for the tiled (prefill) rows and without q/k norms
  if (skip_q && (tile_from > 0 || q_norm != nullptr)) return -1;
  if (D % 16 != 0 || D > 256) return -1;       // 8-pair rotation chunks
  if ((q_norm == nullptr) != (k_norm == nullptr) || (q_norm && D != 128)) return -1;
  const int n1 = tile_from < 0 ? 0 : (tile_from > T ? T : tile_from);
  if (n1 > 0) {
    const int nrot = (Hq + Hkv) * (D / 8);
    if (Hkv * D > 2048 || nrot > 6 * 256) return -1;
#define LMX_RC(IT)                                                                            \
    rope_cache_kernel<IT><<<dim3(n1), dim3(256), 0, stream>>>(                                 \
        (bf16_t*)qkv, qkv_stride, positions, cos_sin, Hq, Hkv, D, slot_mapping,               \
        (bf16_t*)k_cache, (bf16_t*)v_cache, BS, rotate_k_inplace, (const bf16_t*)q_norm,      \
        (const bf16_t*)k_norm, eps)
    if (nrot <= 256) LMX_RC(1);
    else if (nrot <= 512) LMX_RC(2);
    else if (nrot <= 768) LMX_RC(3);
    else if (nrot <= 1024) LMX_RC(4);
    else LMX_RC(6);
#undef LMX_RC
  }
  if (T > n1) {
    const bool v = v_cache && slot_mapping;
    const int hv = rope_v_heads(D), per = 4 * rope_head_step(D);
    const int rot = ((skip_q ? Hkv : Hq + Hkv) + per - 1) / per, vg = v ? (Hkv + hv - 1) / hv : 0;
    const size_t smem = v ? (size_t)RT * (hv * D + 8) * sizeof(bf16_t) : 0;
    rope_cache_tiled_kernel<<<dim3((T - n1 + RT - 1) / RT, rot + vg), dim3(256), smem, stream>>>(
        (bf16_t*)qkv, qkv_stride, positions, cos_sin, n1, T, Hq, Hkv, D, slot_mapping,
        (bf16_t*)k_cache, (bf16_t*)v_cache, BS, rotate_k_inplace, (const bf16_t*)q_norm,
        (const bf16_t*)k_norm, eps, skip_q, rot);
  }
  return (int)hipGetLastError();
}

// Attention heads padded to D channels (true size dk): q and k RMS-normed over
// the head (gains fp32 [D], zero in the padding), the first n channels turned by
// the row's angles (ang [T][n]: cos | sin, neighbouring channels a pair), k and v
// into their cache pages, q to rows.  A thread owns 8 channels of one head in up
// to 4 rows that share a key quad (quads: row starts, then the end; null: one
// row each), so values leave as whole quads.  D / 8 lanes reduce a head's norm.
// grid (row groups, ceil(heads D / 2048)), block 256
template <typename T>
__global__ void __launch_bounds__(256) norm_rope_cache_kernel(
    const T* __restrict__ p, long p_ld, const float* __restrict__ q_norm,
    const float* __restrict__ k_norm, const float* __restrict__ ang, int n,
    const int* __restrict__ slots, const int* __restrict__ quads, T* __restrict__ q,
    T* __restrict__ kc, T* __restrict__ vc, int Hq, int Hkv, int D, int dk, int BS, float eps) {
  const int c0 = (blockIdx.y * 256 + threadIdx.x) * 8;
  const int head = c0 / D, d = c0 - head * D;
  if (head >= Hq + 2 * Hkv) return;            // whole heads leave together
  const int r0 = quads ? quads[blockIdx.x] : blockIdx.x;
  const int cnt = quads ? min(4, quads[blockIdx.x + 1] - r0) : 1;
  float x[4][8];
  int slot[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    slot[t] = -1;
    if (t < cnt) {
      ldv<8>(x[t], p + (long)(r0 + t) * p_ld + c0);
      slot[t] = slots[r0 + t];
    }
  }
  if (head >= Hq + Hkv) {
    const long kvh = head - Hq - Hkv;
    bool quad = cnt == 4 && slot[0] >= 0 && slot[0] % 4 == 0;
#pragma unroll
    for (int t = 1; t < 4; ++t) quad = quad && slot[t] == slot[0] + t;
    if (quad) {
      T* vp = vc + ((long)(slot[0] / BS) * Hkv + kvh) * BS * D + vq_off(d, slot[0] % BS, D);
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float w[8] = {x[0][e], x[1][e], x[2][e], x[3][e],
                            x[0][e + 1], x[1][e + 1], x[2][e + 1], x[3][e + 1]};
        stv<8>(vp + 4 * e, w);
      }
      return;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t >= cnt || slot[t] < 0) continue;
      T* vp = vc + ((long)(slot[t] / BS) * Hkv + kvh) * BS * D + vq_off(d, slot[t] % BS, D);
#pragma unroll
      for (int e = 0; e < 8; ++e) st1(vp + 4 * e, x[t][e]);
    }
    return;
  }
  float w[8];
  ldv<8>(w, (head < Hq ? q_norm : k_norm) + d);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t >= cnt) continue;
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += x[t][e] * x[t][e];
    for (int o = D >> 4; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
    const float inv = rsqrtf(ss / (float)dk + eps);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[t][e] *= inv * w[e];
    if (d < n) {
      const float* a = ang + (long)(r0 + t) * n;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        if (d + e >= n) continue;
        const float c = a[(d + e) >> 1], s = a[(n + d + e) >> 1];
        const float u = x[t][e], v = x[t][e + 1];
        x[t][e] = u * c - v * s;
        x[t][e + 1] = v * c + u * s;
      }
    }
    if (head < Hq) {
      stv<8>(q + (long)(r0 + t) * Hq * D + c0, x[t]);
    } else if (slot[t] >= 0) {
      stv<8>(kc + (((long)(slot[t] / BS) * Hkv + head - Hq) * BS + slot[t] % BS) * D + d, x[t]);
    }
  }
}

int norm_rope_cache(const void* p, long p_ld, const float* q_norm, const float* k_norm,
                    const float* ang, int n, const int* slots, const int* quads, int groups,
                    void* q, void* kc, void* vc, int Hq, int Hkv, int D, int dk, int BS, float eps,
                    int is_bf16, hipStream_t stream) {
  if (groups <= 0) return 0;
  // a head's D / 8 lanes reduce inside one wave: D a power of two, 8..512
  if (D < 8 || D > 512 || (D & (D - 1)) || dk < 1 || dk > D || n < 0 || n % 2 || n > dk ||
      (n && !ang) || BS % 4 || p_ld % 8 || (((uintptr_t)p | (uintptr_t)q) & 15))
    return -1;
  const dim3 grid(groups, ((Hq + 2 * Hkv) * D / 8 + 255) / 256);
  if (is_bf16)
    norm_rope_cache_kernel<bf16_t><<<grid, dim3(256), 0, stream>>>(
        (const bf16_t*)p, p_ld, q_norm, k_norm, ang, n, slots, quads, (bf16_t*)q, (bf16_t*)kc,
        (bf16_t*)vc, Hq, Hkv, D, dk, BS, eps);
  else
    norm_rope_cache_kernel<float><<<grid, dim3(256), 0, stream>>>(
        (const float*)p, p_ld, q_norm, k_norm, ang, n, slots, quads, (float*)q, (float*)kc,
        (float*)vc, Hq, Hkv, D, dk, BS, eps);
  return (int)hipGetLastError();
}

// As above for q and k RMS-normed over the whole projection (all heads' true
// channels at once, gains fp32 [heads D]), after the projections' biases (fp32,
// all heads); v heads divided by their own root mean square over dv channels.
// One workgroup per row group; a thread owns IT pieces of 8 channels in its rows.
template <typename T, int IT>
__global__ void __launch_bounds__(1024) qkv_norm_rope_cache_kernel(
    const T* __restrict__ p, long p_ld, const float* __restrict__ bias,
    const float* __restrict__ q_norm, const float* __restrict__ k_norm,
    const float* __restrict__ ang, int n, const int* __restrict__ slots,
    const int* __restrict__ quads, T* __restrict__ q, T* __restrict__ kc, T* __restrict__ vc, int Hq,
    int Hkv, int D, int dk, int dv, int BS, float eps) {
  __shared__ float part[16][8];                // per wave: sums of squares of q and k, 4 rows
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int pieces = (Hq + 2 * Hkv) * D / 8;
  const int r0 = quads ? quads[blockIdx.x] : blockIdx.x;
  const int cnt = quads ? min(4, quads[blockIdx.x + 1] - r0) : 1;
  float x[IT][4][8], sq[4] = {0.f, 0.f, 0.f, 0.f}, sk[4] = {0.f, 0.f, 0.f, 0.f};
  int slot[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) slot[t] = t < cnt ? slots[r0 + t] : -1;
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int c = threadIdx.x + i * blockDim.x;
    if (c >= pieces) continue;
    const int head = 8 * c / D;
    float b[8];
    ldv<8>(b, bias + 8 * c);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t >= cnt) continue;
      ldv<8>(x[i][t], p + (long)(r0 + t) * p_ld + 8 * c);
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[i][t][e] += b[e];
        ss += x[i][t][e] * x[i][t][e];
      }
      if (head < Hq) sq[t] += ss; else if (head < Hq + Hkv) sk[t] += ss;
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t >= cnt) continue;
    const float a = wave_sum(sq[t]), b = wave_sum(sk[t]);
    if (lane == 0) { part[wave][t] = a; part[wave][4 + t] = b; }
  }
  __syncthreads();
  float iq[4], ik[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t >= cnt) continue;
    float a = 0.f, b = 0.f;
    for (int w = 0; w < nw; ++w) { a += part[w][t]; b += part[w][4 + t]; }
    iq[t] = rsqrtf(a / ((float)Hq * dk) + eps);
    ik[t] = rsqrtf(b / ((float)Hkv * dk) + eps);
  }
  bool quad = cnt == 4 && slot[0] >= 0 && slot[0] % 4 == 0;
#pragma unroll
  for (int t = 1; t < 4; ++t) quad = quad && slot[t] == slot[0] + t;
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int c = threadIdx.x + i * blockDim.x;
    if (c >= pieces) continue;                 // whole heads leave together
    const int head = 8 * c / D, d = 8 * c - head * D;
    if (head >= Hq + Hkv) {
      const long kvh = head - Hq - Hkv;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (t >= cnt) continue;
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += x[i][t][e] * x[i][t][e];
        for (int o = D >> 4; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
        const float inv = rsqrtf(ss / (float)dv + eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[i][t][e] *= inv;
      }
      if (quad) {
        T* vp = vc + ((long)(slot[0] / BS) * Hkv + kvh) * BS * D + vq_off(d, slot[0] % BS, D);
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const float w[8] = {x[i][0][e], x[i][1][e], x[i][2][e], x[i][3][e],
                              x[i][0][e + 1], x[i][1][e + 1], x[i][2][e + 1], x[i][3][e + 1]};
          stv<8>(vp + 4 * e, w);
        }
        continue;
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (t >= cnt || slot[t] < 0) continue;
        T* vp = vc + ((long)(slot[t] / BS) * Hkv + kvh) * BS * D + vq_off(d, slot[t] % BS, D);
#pragma unroll
        for (int e = 0; e < 8; ++e) st1(vp + 4 * e, x[i][t][e]);
      }
      continue;
    }
    const bool isq = head < Hq;
    float w[8];
    ldv<8>(w, isq ? q_norm + 8 * c : k_norm + 8 * c - Hq * D);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t >= cnt) continue;
      const float inv = isq ? iq[t] : ik[t];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[i][t][e] *= inv * w[e];
      if (d < n) {
        const float* a = ang + (long)(r0 + t) * n;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          if (d + e >= n) continue;
          const float cs = a[(d + e) >> 1], sn = a[(n + d + e) >> 1];
          const float u = x[i][t][e], v = x[i][t][e + 1];
          x[i][t][e] = u * cs - v * sn;
          x[i][t][e + 1] = v * cs + u * sn;
        }
      }
      if (isq) {
        stv<8>(q + (long)(r0 + t) * Hq * D + 8 * c, x[i][t]);
      } else if (slot[t] >= 0) {
        stv<8>(kc + (((long)(slot[t] / BS) * Hkv + head - Hq) * BS + slot[t] % BS) * D + d,
               x[i][t]);
      }
    }
  }
}

int qkv_norm_rope_cache(const void* p, long p_ld, const float* bias, const float* q_norm,
                        const float* k_norm, const float* ang, int n, const int* slots,
                        const int* quads, int groups, void* q, void* kc, void* vc, int Hq, int Hkv,
                        int D, int dk, int dv, int BS, float eps, int is_bf16, hipStream_t stream) {
  if (groups <= 0) return 0;
  // a head's D / 8 lanes reduce inside one wave: D a power of two, 64..512
  if (D < 64 || D > 512 || (D & (D - 1)) || dk < 1 || dk > D || dv < 1 || dv > D || n < 0 || n % 2 ||
      n > dk || (n && !ang) || BS % 4 || p_ld % 8 || (((uintptr_t)p | (uintptr_t)q) & 15) || Hq < 1 ||
      Hkv < 1)
    return -1;
  const int pieces = (Hq + 2 * Hkv) * D / 8;
  const int threads = pieces >= 1024 ? 1024 : (pieces + 63) / 64 * 64;
  const int it = (pieces + threads - 1) / threads;
  if (it > 4) return -2;
#define LMX_QN(T, I)                                                                            \
  qkv_norm_rope_cache_kernel<T, I><<<dim3(groups), dim3(threads), 0, stream>>>(                 \
      (const T*)p, p_ld, bias, q_norm, k_norm, ang, n, slots, quads, (T*)q, (T*)kc, (T*)vc, Hq, \
      Hkv, D, dk, dv, BS, eps)
#define LMX_QNT(T) if (it == 1) LMX_QN(T, 1); else if (it == 2) LMX_QN(T, 2); else LMX_QN(T, 4);
  if (is_bf16) { LMX_QNT(bf16_t) } else { LMX_QNT(float) }
#undef LMX_QNT
#undef LMX_QN
  return (int)hipGetLastError();
}

// Plain cache write (no rotation): models without rotary embeddings.  Any head
// size and alignment, one token per workgroup: few tokens are bound by latency, and this is one
// trip to memory and no barrier (a token of 8 heads of 128 3.4 us, 600 tokens 5.4).
__global__ void kv_write_kernel(const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
                                long kv_stride, const int* __restrict__ slot_mapping, int Hkv,
                                int D, bf16_t* __restrict__ k_cache, bf16_t* __restrict__ v_cache,
                                int BS) {
  const int t = blockIdx.x;
  const int slot = slot_mapping[t];
  if (slot < 0) return;
  const int blk = slot / BS, off = slot % BS;
  for (int it = threadIdx.x; it < Hkv * D; it += blockDim.x) {
    const int h = it / D, d = it % D;
    k_cache[(((long)blk * Hkv + h) * BS + off) * D + d] = k[(long)t * kv_stride + it];
    v_cache[((long)blk * Hkv + h) * BS * D + vq_off(d, off, D)] = v[(long)t * kv_stride + it];
  }
}

// The same for rows of whole 16-B pieces: grid (32-token tiles, K groups + V
// groups) as rope_cache_tiled_kernel, V in key quads through LDS instead of 2-B
// stores 8 B apart: many tokens, bound by the stores.  19,153 tokens of 16 heads of 64: 53 -> 39 us
// (157 MB); 600 of 8 heads of 128 6.0, longer than a workgroup a token.
__global__ void __launch_bounds__(256) kv_write_tiled_kernel(
    const bf16_t* __restrict__ k, const bf16_t* __restrict__ v, long kv_stride,
    const int* __restrict__ slot_mapping, int T, int Hkv, int D, bf16_t* __restrict__ k_cache,
    bf16_t* __restrict__ v_cache, int BS, int k_groups) {
  extern __shared__ __attribute__((aligned(16))) bf16_t vt[];
  __shared__ int sslot[RT];
  const int t0 = blockIdx.x * RT, nt = min(RT, T - t0);
  if (threadIdx.x < RT) sslot[threadIdx.x] = threadIdx.x < nt ? slot_mapping[t0 + threadIdx.x] : -1;
  __syncthreads();
  const int hv = rope_v_heads(D);
  const bool is_k = (int)blockIdx.y < k_groups;
  const int h0 = ((int)blockIdx.y - (is_k ? 0 : k_groups)) * hv, hg = min(hv, Hkv - h0);
  if (!is_k) {
    v_to_pages(v + (long)t0 * kv_stride, kv_stride, nt, h0, hg, Hkv, D, sslot, vt, hv * D + 8, v_cache,
               BS);
    return;
  }
  const int per = D / 8, chunks = hg * per;
#pragma unroll 4
  for (int it = threadIdx.x; it < nt * chunks; it += 256) {
    const int tt = it / chunks, c = it - tt * chunks, h = h0 + c / per;
    const int slot = sslot[tt];
    if (slot < 0) continue;
    *reinterpret_cast<u16x8*>(k_cache + (((long)(slot / BS) * Hkv + h) * BS + slot % BS) * D +
                              c % per * 8) =
        *reinterpret_cast<const u16x8*>(k + (long)(t0 + tt) * kv_stride + (long)h0 * D + 8 * c);
  }
}

int kv_write(const void* k, const void* v, long kv_stride, const int* slot_mapping, int T, int Hkv,
             int D, void* k_cache, void* v_cache, int BS, hipStream_t stream) {
  if (T <= 0) return 0;
  // whole 16-B pieces of rows and pages, whole key quads (BS % 4).  The line is where both take the same time:
  // 800,000 elements at 4 to 16 heads (1600 tokens of 4 heads of 128 5.9 / 6.0 us, 600 of 8 5.4 / 6.0, 1200
  // of 8 7.2 / 6.6), 4096 tokens at one or two (of one of 128 5.2 / 4.8, 3000 4.5 / 4.9)
  if ((T >= 4096 || (long)T * Hkv * D >= 800000) && D % 8 == 0 && D <= 256 && BS % 4 == 0 && kv_stride % 8 == 0 &&
      (((uintptr_t)k | (uintptr_t)v | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0) {
    const int hv = rope_v_heads(D), groups = (Hkv + hv - 1) / hv;
    kv_write_tiled_kernel<<<dim3((T + RT - 1) / RT, 2 * groups), dim3(256),
                            (size_t)RT * (hv * D + 8) * sizeof(bf16_t), stream>>>(
        (const bf16_t*)k, (const bf16_t*)v, kv_stride, slot_mapping, T, Hkv, D, (bf16_t*)k_cache,
        (bf16_t*)v_cache, BS, groups);
    return (int)hipGetLastError();
  }
  kv_write_kernel<<<dim3(T), dim3(256), 0, stream>>>((const bf16_t*)k, (const bf16_t*)v,
                                                     kv_stride, slot_mapping, Hkv, D,
                                                     (bf16_t*)k_cache, (bf16_t*)v_cache, BS);
  return (int)hipGetLastError();
}

}  // namespace lmx
