// Arguments of encoder_layers (encoder.hip), filled by the bindings.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lmx {

// weights of a layer, in this order, 0 where there is none: Wqkv, its bias, Wo, bias, the
// first norm's gain and shift, W1 (gate / up interleaved by 16 rows, or the plain one), bias,
// W2, bias, the second norm's gain and shift
constexpr int kEncPtrs = 12;

struct EncArgs {
  int layers, T, d, I, H, D;
  bool gelu;                       // gelu(h W1 + b) instead of SwiGLU
  float eps, scale;
  // rows of T tokens, bf16: x [d] (in: the first norm's output, out: the last one's),
  // h [d], qkv [3 d], attn [d], g [I]
  void *x, *h, *qkv, *attn, *g;
  float* slabs;
  long slab_floats;
  const float* cos_sin;            // null: no rotation
  const int *cu, *tiles;           // enc_attention's
  int ntiles;
  float* tail;                     // K13's last round in pieces (pgemm): floats and counters
  long tail_floats;
  unsigned* cnt;
};

struct EncPlan { int cfg, splits; };   // cfg: dgemm's, -1: K13, kEncSmall: K23
constexpr int kEncSmall = 100;

EncPlan enc_plan(int M, int N, int K, int act, bool partials, int cus = 0);
long enc_slab_floats(int T, int d, int I);
long enc_tail_floats(int T, int d, int I, bool gelu);
int encoder_layers(const EncArgs& a, const uintptr_t* w, hipStream_t stream);

}  // namespace lmx
