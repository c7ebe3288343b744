// Launch interfaces of the float32 model's kernels (gemm_f32.hip, attn_f32.hip).
#pragma once

#include "common.h"

namespace mlcv {

// What a float32 linear does with its product y = x . W^T (each op rounds once, no contraction):
enum F32Epi : int {
  FE_STORE = 0,  // out = act(y + b), act: 0 none, 1 SiLU
  FE_QKV = 1,    // q and k roped (q then scaled), v plain, each to its own place
  FE_RES = 2,    // out = out + y, or out + y * gate
  FE_GEGLU = 3,  // out = gelu_tanh(y_gate) * y_up
  FE_EULER = 4,  // out = out + dt * (y + b)
};

// One of the equally shaped linears of a table launch.
struct F32Tab {
  const float* w;
  const float* b;
};

// y[m][n] over x [M][ldx] and weight rows of K floats.  Logical rows n come in slabs of 16: FE_GEGLU
// pairs 8 gate rows with their 8 up rows, q and k pair dims d .. d + 7 with their RoPE partners
// d + hd/2 .. (so a pair is 8 rows apart in one tile); the rest are in order.
// Needs K % 8 == 0, N % 8 == 0, ldx % 4 == 0 (checked) and 16-byte aligned pointers and output rows,
// which the caller sees to (F32Model::fast, f32_aligned).
struct F32Op {
  const float* x;
  int ldx, M, K, N;
  const float* w[3];       // FE_QKV: q, k, v; else w[0]
  const float* b;          // [N] or null
  const F32Tab* tab;       // (host) ntab linears over the same x: w, b from the table, out + z * tab_stride
  int ntab;
  size_t tab_stride;
  // x is normalised first: x / sqrt(mean(x^2) + eps), then * (1 + nw) (RMSNorm) or
  // * (1 + mod[k]) + mod[K + k] (adaRMS); in the kernel's pass over x, or by a launch into xn [M][K]
  const float* nw;
  const float* mod;
  float eps;
  float* xn;
  int epi, act;
  float* out;
  int ldo;
  const float* gate;       // [N] or null (FE_RES)
  int F;                   // FE_GEGLU: gate rows, then F up rows
  // FE_QKV: q [M][nq] from row n, k and v element (m, head, d) at m * kv_m + head * kv_h + d
  float *qo, *ko, *vo;
  int nq, nkv, hd, kv_m;
  size_t kv_h;
  const float *cos, *sin;  // [M][hd/2]
  float qscale, dt;
};
int f32_gemm_launch(const F32Op& a, hipStream_t st);

// softmax(q . k + mask) . v over the prefix keys kp / vp [KV][Sp][hd] (additive mask [Sp] or null) and
// the suffix rows ks / vs [Ts][s_ld] (kv head h at h hd): q [Tq][q_ld] -> out [Tq][o_ld], query head h
// at h hd reading kv head h / (H / KV).  hd one of 16, 32, 64, 128, 256; 16-byte aligned rows.
struct F32Attn {
  const float* q;
  int q_ld, Tq, H, KV, hd;
  const float *kp, *vp;
  const float* const* kv;  // or: kp = kv[0] + kv_off, vp = kv[1] + kv_off, read on the device (a
  size_t kv_off;           // captured launch then serves any cache)
  int Sp;
  const float* mask;
  const float *ks, *vs;
  int s_ld, Ts;
  float* out;
  int o_ld;
  float* ws;  // f32_attn_ws_floats of the plan
};
int f32_attn_launch(const F32Attn& a, hipStream_t st);

}  // namespace mlcv
