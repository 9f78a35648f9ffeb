// The layers of the embedding encoders (BERT, nomic-bert) as one host call: every
// launch of a forward from here, so that a short request is bound by its kernels
// and not by the interpreter (96 to 290 launches of 3 to 6 us each).
//
//   qkv = x Wqkv^T + b;  attention on its rows (K24), with the rotation (nomic)
//   h = LN(x + attn Wo^T + b);  g = act(h W1^T + b);  x = LN(h + g W2^T + b)
//
// Requests range from one query of ten tokens to 64 k tokens, so a projection has
// two kernels: K13's persistent 256 x 256 tiles for many rows, and the decode GEMM's
// smaller tiles (dgemm.hip) below, where K13 leaves compute units idle (its tile
// takes 16 us at K = 768 and 50 us at K = 3072 however few rows it holds). The two
// that end in a LayerNorm may also split K: their fp32 slabs are summed by the norm.
// enc_plan picks by estimated time.
#include "common.h"

#include <algorithm>

#include "encoder.h"

namespace lmx {

int layernorm(void*, const void*, const void*, const void*, const void*, int, int, float, hipStream_t);
int layernorm_slabs(void*, const float*, int, long, const void*, const void*, const void*, const void*,
                    int, int, float, hipStream_t);
int enc_attention(const void*, long, int, int, const int*, const int*, int, const float*, void*, long,
                  float, float, hipStream_t);
int dgemm(void*, const void*, const void*, float*, unsigned*, int, int, int, int, long, long, long,
          int, int, int, hipStream_t, const void*);
int pgemm(void*, const void*, const void*, const void*, int, int, int, long, long, long, int, int, int,
          int, float*, hipStream_t, float*, unsigned*);
long pgemm_tail_floats(int, int, int);
float pgemm_us(int, int, int, int);
int pgemm_cus();
int sgemm(void*, const void*, const void*, int, int, int, long, long, long, int, int, const void*,
          hipStream_t);

namespace {

// Time of a decode-GEMM tile configuration in us: base + rounds x (start + step x
// K / 64), rounds of a workgroup per CU; fill: the slabs' writes at a full
// round. Least squares over 12 shapes (N 384 to 6144, K 384 to 4096) x 16 row counts
// (16 to 12288) x slices, each within 5 to 8 % rms of the measured time.
struct EncTile { int cfg, bm, bn; float base, start, step, fill; };
constexpr EncTile kTiles[] = {
    {21, 64, 64, 1.13f, 1.48f, 0.281f, 0.58f},
    {31, 64, 128, 1.01f, 1.94f, 0.386f, 1.25f},
    {20, 128, 64, 0.45f, 2.20f, 0.423f, 1.42f},
    {22, 128, 128, 0.46f, 3.05f, 0.592f, 3.06f},
    {11, 128, 256, 2.02f, 3.80f, 0.945f, 3.96f},
};
constexpr int kSlices[] = {1, 2, 3, 4, 6, 8, 12, 16};      // layernorm_slabs' S
constexpr float kBytesUs = 4.5e6f;                         // memory traffic, bytes per us

}  // namespace

// act: 0 none, 3 SwiGLU over 16-row pairs, 4 gelu (exact). partials: the
// product's fp32 slabs go to a LayerNorm (no activation). cus: compute units (0: the device's).
EncPlan enc_plan(int M, int N, int K, int act, bool partials, int cus) {
  if (cus <= 0) cus = pgemm_cus();
  EncPlan best{-1, 0};
  // few rows: K23, except where K slices of the 64 x 64 tile fill the chip (at 16 rows:
  // qkv of nomic 4.5 us against 5.7, gate / up 5.8 against 7.3, but o 3.5 against 3.0 and down 4.6
  // against 4.0; qkv at 32 rows 5.5 against 5.9, at 64 7.5 against 6.1). K is d, 2048 at most. Weights
  // over 12 M elements, which no preset has, would do better on the 64 x 64 tile from 17 rows on (6144 x 2048 at
  // 16 / 32 rows 12.2 / 17.1 us against 12.2 / 12.4; K13 36.4)
  if (!partials && M <= 32 && N % 32 == 0 && K % 32 == 0) return {kEncSmall, 1};
  const bool k13 = N % 256 == 0 && K % 64 == 0 && K >= 192;
  float t = k13 ? pgemm_us(M, N, K, cus) : 1e30f;
  for (const EncTile& c : kTiles) {
    const int bk = c.cfg == 11 ? 64 : 128;
    if (N % c.bn || (act == 3 && c.cfg == 21)) continue;   // a wave holds whole 16-row pairs
    const long tiles = (long)((M + c.bm - 1) / c.bm) * (N / c.bn);
    if (tiles > 4096) continue;
    for (int s : kSlices) {
      if ((s > 1 && !partials) || K % (bk * s)) continue;
      const long wgs = tiles * s, rounds = (wgs + cus - 1) / cus;
      float u = c.base + rounds * (c.start + c.step * (K / 64.f / s));
      if (partials)      // the slabs' writes and reads against bf16 rows
        u += c.fill * wgs / cus + (4.f * s - 2.f) * M * N / kBytesUs;
      if (u < t) {
        t = u;
        best = {c.cfg, s};
      }
    }
  }
  return best;
}

// floats of slabs that the layers' partial products need
long enc_slab_floats(int T, int d, int I) {
  const EncPlan o = enc_plan(T, d, d, 0, true), m = enc_plan(T, d, I, 0, true);
  return (long)std::max(o.splits, m.splits) * T * d;
}

// floats that K13 takes for the last rounds of the products it runs
long enc_tail_floats(int T, int d, int I, bool gelu) {
  long n = 0;
  auto add = [&](int N, int K, int act, bool partials) {
    if (enc_plan(T, N, K, act, partials).cfg < 0) n = std::max(n, pgemm_tail_floats(T, N, K));
  };
  add(3 * d, d, 0, false);
  add(d, d, 0, true);
  add(gelu ? I : 2 * I, d, gelu ? 4 : 3, false);
  add(d, I, 0, true);
  return n;
}

int encoder_layers(const EncArgs& a, const uintptr_t* w, hipStream_t stream) {
  const int T = a.T, d = a.d, I = a.I;
  if (T <= 0) return 0;
  if (d != a.H * a.D || d % 256 || I % 256 || a.D != 64) return -1;
  for (int i = 0; i < a.layers * kEncPtrs; ++i)
    if (w[i] & 15) return -2;
  auto k13 = [&](void* out, const void* x, uintptr_t W, uintptr_t b, int N, int K, int ldc, int act) {
    const long n = pgemm_tail_floats(T, N, K);
    float* tail = n > 0 && n <= a.tail_floats ? a.tail : nullptr;
    return pgemm(out, x, (void*)W, (void*)b, T, N, K, K, K, ldc, act, 0, 0, 0, nullptr, stream, tail,
                 a.cnt);
  };
  auto full = [&](void* out, const void* x, uintptr_t W, uintptr_t b, int N, int K, int act) {
    const EncPlan p = enc_plan(T, N, K, act, false);
    const int ldc = act == 3 ? N / 2 : N;
    if (p.cfg < 0)
      return k13(out, x, W, b, N, K, ldc, act);
    const int epi = act == 3 ? 3 : act == 4 ? 6 : b ? 5 : 0;
    if (p.cfg == kEncSmall)
      return sgemm(out, x, (void*)W, T, N, K, K, K, ldc, epi, 1, (void*)b, stream);
    return dgemm(out, x, (void*)W, nullptr, nullptr, 0, T, N, K, K, K, ldc, p.cfg, 1, epi, stream,
                 (void*)b);
  };
  // out = LN(x W^T + b + residual)
  auto normed = [&](void* out, const void* x, uintptr_t W, uintptr_t b, const void* residual,
                    uintptr_t g, uintptr_t s, int K, void* tmp) {
    const EncPlan p = enc_plan(T, d, K, 0, true);
    if (p.cfg < 0) {
      const int e = k13(tmp, x, W, b, d, K, d, 0);
      return e ? e : layernorm(out, tmp, residual, (void*)g, (void*)s, T, d, a.eps, stream);
    }
    if ((long)p.splits * T * d > a.slab_floats) return -3;
    const int e = dgemm(nullptr, x, (void*)W, a.slabs, nullptr, 0, T, d, K, K, K, d, p.cfg, p.splits, 2,
                        stream, nullptr);
    return e ? e : layernorm_slabs(out, a.slabs, p.splits, (long)T * d, (void*)b, residual, (void*)g,
                                   (void*)s, T, d, a.eps, stream);
  };
  for (int l = 0; l < a.layers; ++l, w += kEncPtrs) {
    const bool gelu = a.gelu;
    int e = full(a.qkv, a.x, w[0], w[1], 3 * d, d, 0);
    if (!e)
      e = enc_attention(a.qkv, 3L * d, a.H, a.D, a.cu, a.tiles, a.ntiles, a.cos_sin, a.attn, d, a.scale,
                        8.f, stream);
    if (!e) e = normed(a.h, a.attn, w[2], w[3], a.x, w[4], w[5], d, a.qkv);
    if (!e) e = full(a.g, a.h, w[6], w[7], gelu ? I : 2 * I, d, gelu ? 4 : 3);
    if (!e) e = normed(a.x, a.g, w[8], w[9], a.h, w[10], w[11], I, a.qkv);
    if (e) return e;
  }
  return 0;
}

}  // namespace lmx
