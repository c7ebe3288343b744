// The float32 model (Pi0Config(dtype="float32"), the reference's default dtype,
// pi0_config.py:97): prefill, denoise_step_kv, denoise_loop_kv and the chunk computed in float32
// from end to end, for the small shapes the reference runs in float32 (its CPU dummy model, the
// 2-layer test model).  With dtype = float32 every cast point of the reference is the identity:
// linears are fp32 products with fp32 sums (gemma_dual.py: nn.Linear at the model dtype), RMSNorm
// and adaRMS normalise in fp32 (:60-88), RoPE rotates in fp32 (:47-57), attention takes fp32
// logits, softmax and probabilities (:97-122), GeGLU (:125-135) and the gated residual (:91-94)
// round after each op, and the Euler update is x + dt * v in fp32 (pi0_model.py:165-194).
//
// The linears run on the fp32 matrix cores with the norms beside them and RoPE, cache writes, GeGLU and
// residuals in their epilogues (gemm_f32.hip), where widths, head dim and pointers allow
// (F32Model::fast); the general kernels here (one tiled FMA GEMM, one workgroup per row or per query
// row and head elsewhere) take everything else.  The elementwise steps round after each op as the
// reference does (floating-point contraction is off in these files; explicit fmaf in the general GEMM,
// the dot products and the sums of squares), but for one: a norm before a linear of few rows divides
// after the product, sum(x (1 + s) w) / sqrt(mean(x^2) + eps) + shift . w, where the reference divides
// x first.  Against 64 bits the models' errors are 0.36 to 1.01 times those of the general kernels.
#include <cmath>
#include <memory>
#include <vector>

#include "../../include/mlcvla.h"
#include "f32.h"
#include "kernels.h"

#pragma clang fp contract(off)

namespace mlcv {
namespace {

constexpr int F32_NT = 256;

// Y[m][n] = act(sum_k X[m][k] W[n][k] + b[n]) for row-major X (ldx) and W [N][K]: 64 x 64
// tiles of 256 threads (4 x 4 outputs each), k in steps of 16 through LDS, sums in k order.
// act: 0 none, 1 SiLU (x / (1 + exp(-x)))
__global__ __launch_bounds__(F32_NT) void f32_gemm_kernel(const float* __restrict__ X, int ldx,
                                                          const float* __restrict__ W, const float* __restrict__ b,
                                                          float* __restrict__ Y, int ldy, int M, int N, int K,
                                                          int act) {
  __shared__ float xs[16][64 + 4];
  __shared__ float ws[16][64 + 4];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
  for (int k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = threadIdx.x + F32_NT * i, r = e >> 4, kk = e & 15;
      const int gk = k0 + kk;
      xs[kk][r] = (m0 + r < M && gk < K) ? X[(size_t)(m0 + r) * ldx + gk] : 0.f;
      ws[kk][r] = (n0 + r < N && gk < K) ? W[(size_t)(n0 + r) * K + gk] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      float a[4], w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = xs[kk][ty * 4 + i];
        w[i] = ws[kk][tx * 4 + i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      float y = acc[i][j];
      if (b) y = y + b[n];
      if (act == 1) y = y / (1.0f + expf(-y));
      Y[(size_t)m * ldy + n] = y;
    }
  }
}

// sum over the workgroup (256 threads) of each thread's v
__device__ __forceinline__ float f32_block_sum(float v, float* red) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  if (lane == 0) red[w] = v;
  __syncthreads();
  const float s = ((red[0] + red[1]) + red[2]) + red[3];
  __syncthreads();
  return s;
}
__device__ __forceinline__ float f32_block_max(float v, float* red) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  if (lane == 0) red[w] = v;
  __syncthreads();
  const float s = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  return s;
}

// row r of x [rows][W]: xn = x / sqrt(mean(x^2) + eps), then xn * (1 + w) (Gemma RMSNorm,
// w non-null) or xn * (1 + scale) + shift (adaRMS, mod = [scale | shift | gate] of 3W)
__global__ __launch_bounds__(F32_NT) void f32_norm_kernel(const float* __restrict__ x, int W,
                                                          const float* __restrict__ w,
                                                          const float* __restrict__ mod, float eps,
                                                          float* __restrict__ out) {
  __shared__ float red[4];
  const float* xr = x + (size_t)blockIdx.x * W;
  float ss = 0.f;
  for (int i = threadIdx.x; i < W; i += F32_NT) ss += xr[i] * xr[i];
  const float var = f32_block_sum(ss, red) / (float)W;
  const float den = sqrtf(var + eps);
  float* o = out + (size_t)blockIdx.x * W;
  for (int i = threadIdx.x; i < W; i += F32_NT) {
    const float xn = xr[i] / den;
    o[i] = w ? xn * (1.0f + w[i]) : xn * (1.0f + mod[i]) + mod[W + i];
  }
}

// in place on columns [col0, col0 + heads * hd) of row t of buf (ld): the half-split rotation
// of each head by cos / sin [rows][hd / 2], then * scale
__global__ void f32_rope_kernel(float* buf, int ld, int col0, int heads, int hd, const float* __restrict__ cs,
                                const float* __restrict__ sn, float scale) {
  const int t = blockIdx.x, half = hd / 2;
  for (int e = threadIdx.x; e < heads * half; e += blockDim.x) {
    const int hh = e / half, i = e % half;
    float* p = buf + (size_t)t * ld + col0 + hh * hd;
    const float c = cs[(size_t)t * half + i], s = sn[(size_t)t * half + i];
    const float x1 = p[i], x2 = p[i + half];
    p[i] = (x1 * c - x2 * s) * scale;
    p[i + half] = (x2 * c + x1 * s) * scale;
  }
}

// the layer's cache slices keys / values [KV][P][hd] from k / v [P][KV * hd]
__global__ void f32_kv_write_kernel(const float* __restrict__ k, const float* __restrict__ v, int P, int KV, int hd,
                                    float* __restrict__ keys, float* __restrict__ values) {
  const size_t n = (size_t)P * KV * hd;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const int d = (int)(e % hd), p = (int)((e / hd) % P), kh = (int)(e / ((size_t)hd * P));
    keys[e] = k[(size_t)p * KV * hd + kh * hd + d];
    values[e] = v[(size_t)p * KV * hd + kh * hd + d];
  }
}

// out[t][h hd + d] = sum_j p_j val_j[d], p = softmax over the keys j of (q_t,h . key_j + mask_j):
// keys [0, Sp) from the prefix cache kp / vp [KV][Sp][hd] with the additive mask, then keys
// [Sp, Sp + Ts) from the suffix rows ks / vs [Ts][s_ld] (mask 0).  Query head h reads kv head
// h / (H / KV).  One workgroup per (query row, head); logits in LDS.
__global__ __launch_bounds__(F32_NT) void f32_attn_kernel(const float* __restrict__ q, int q_ld, int H, int KV,
                                                          int hd, const float* __restrict__ kp,
                                                          const float* __restrict__ vp, int Sp,
                                                          const float* __restrict__ mask,
                                                          const float* __restrict__ ks,
                                                          const float* __restrict__ vs, int s_ld, int Ts,
                                                          float* __restrict__ out, int o_ld) {
  extern __shared__ float sm[];
  float* qs = sm;       // [hd]
  float* lg = sm + hd;  // [Sp + Ts]
  __shared__ float red[4];
  const int t = blockIdx.x, h = blockIdx.y, kvh = h / (H / KV), nk = Sp + Ts;
  for (int d = threadIdx.x; d < hd; d += F32_NT) qs[d] = q[(size_t)t * q_ld + h * hd + d];
  __syncthreads();
  float mx = -INFINITY;
  for (int j = threadIdx.x; j < nk; j += F32_NT) {
    const float* kr = j < Sp ? kp + ((size_t)kvh * Sp + j) * hd : ks + (size_t)(j - Sp) * s_ld + kvh * hd;
    float s = 0.f;
    for (int d = 0; d < hd; ++d) s = fmaf(qs[d], kr[d], s);
    if (j < Sp && mask) s = s + mask[j];
    lg[j] = s;
    mx = fmaxf(mx, s);
  }
  mx = f32_block_max(mx, red);
  float sum = 0.f;
  for (int j = threadIdx.x; j < nk; j += F32_NT) {
    const float e = expf(lg[j] - mx);
    lg[j] = e;
    sum += e;
  }
  sum = f32_block_sum(sum, red);
  for (int j = threadIdx.x; j < nk; j += F32_NT) lg[j] = lg[j] / sum;
  __syncthreads();
  for (int d = threadIdx.x; d < hd; d += F32_NT) {
    float acc = 0.f;
    for (int j = 0; j < Sp; ++j) acc = fmaf(lg[j], vp[((size_t)kvh * Sp + j) * hd + d], acc);
    for (int j = 0; j < Ts; ++j) acc = fmaf(lg[Sp + j], vs[(size_t)j * s_ld + kvh * hd + d], acc);
    out[(size_t)t * o_ld + h * hd + d] = acc;
  }
}

// h[t][i] = gelu_tanh(gu[t][i]) * gu[t][F + i]
__global__ void f32_geglu_kernel(const float* __restrict__ gu, int F, int rows, float* __restrict__ hout) {
  const size_t n = (size_t)rows * F;
  const float c = 0.7978845608028654f;  // sqrt(2 / pi)
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const size_t t = e / F, i = e % F;
    const float x = gu[t * 2 * F + i], u = gu[t * 2 * F + F + i];
    const float g = 0.5f * x * (1.0f + tanhf(c * (x + 0.044715f * x * x * x)));
    hout[e] = g * u;
  }
}

// x[t][i] = x[t][i] + y[t][i] (gate null) or x[t][i] + y[t][i] * gate[i]
__global__ void f32_residual_kernel(float* __restrict__ x, const float* __restrict__ y,
                                    const float* __restrict__ gate, int W, int rows) {
  const size_t n = (size_t)rows * W;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const float yy = gate ? y[e] * gate[e % W] : y[e];
    x[e] = x[e] + yy;
  }
}

// x = x + dt * v
__global__ void f32_euler_kernel(float* __restrict__ x, const float* __restrict__ v, float dt, int n) {
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) x[e] = x[e] + dt * v[e];
}

int ew_grid(size_t n) { return (int)std::min<size_t>((n + 255) / 256, 4096); }

}  // namespace

struct F32Lin {
  const float* w = nullptr;
  const float* b = nullptr;
  int N = 0, K = 0;
};
struct F32Layer {
  F32Lin q[2], k[2], v[2], o[2], gu[2], dn[2], mod_in, mod_post;
  const float* ln_in0 = nullptr;
  const float* ln_post0 = nullptr;
};

struct F32Model {
  int W0, F0, W1, F1, D, H, KV, HD, P, T, A, S;
  float eps;
  bool bound = false;
  // the matrix-core kernels (gemm_f32.hip) take these widths and weight pointers; else the general ones
  bool shape_ok = false, fast = false;
  std::vector<F32Tab> tab;  // the 2 D + 1 modulations' weights and biases
  // the loop and the chunk as captured graphs over the model's own buffers (MLCV_OPT_USE_GRAPH): the
  // inputs are staged into them and the caller's cache is reached through kvp, so a graph serves
  // every call until the parameters are bound again
  bool use_graph = true;
  hipGraphExec_t g_loop = nullptr, g_chunk = nullptr;
  hipStream_t cap = nullptr;
  const float** kvp = nullptr;  // device: {keys, values} of the loop's call
  int SB = 1;                   // steps whose modulations are made in one go
  std::vector<F32Layer> layers;
  F32Lin final_mod, ain, aout, tin, tout;
  std::vector<void*> owned;
  // prefill
  float *px, *pxn, *pq, *pk, *pv, *pattn, *po, *pgu, *ph, *pcos, *psin, *mask;
  // the chunk's own cache
  float *ckeys, *cvalues;
  // step
  float *x, *xn, *q, *k, *v, *attn, *o, *gu, *h, *cond, *tmp, *mods, *vout, *x32;
  float *scos, *ssin, *smask, *te;
  float* aws = nullptr;  // split partials of the attention

  ~F32Model() {
    for (void* p : owned) (void)hipFree(p);
    if (kvp) (void)hipFree(kvp);
    drop_graphs();
    if (cap) (void)hipStreamDestroy(cap);
  }
  void drop_graphs() {
    for (hipGraphExec_t* g : {&g_loop, &g_chunk}) {
      if (*g) (void)hipGraphExecDestroy(*g);
      *g = nullptr;
    }
  }
  int alloc(float** p, size_t n) {
    MLCV_HIP(hipMalloc(reinterpret_cast<void**>(p), std::max<size_t>(n, 1) * sizeof(float)));
    owned.push_back(*p);
    MLCV_HIP(hipMemset(*p, 0, std::max<size_t>(n, 1) * sizeof(float)));
    return 0;
  }
};

namespace {

int gemm(const float* X, int ldx, const F32Lin& l, float* Y, int ldy, int M, int act, hipStream_t st,
         bool bias = true) {
  const dim3 grid((l.N + 63) / 64, (M + 63) / 64);
  f32_gemm_kernel<<<grid, F32_NT, 0, st>>>(X, ldx, l.w, bias ? l.b : nullptr, Y, ldy, M, l.N, l.K, act);
  MLCV_HIP(hipGetLastError());
  return 0;
}
int attn(const float* q, int q_ld, const F32Model& m, const float* kp, const float* vp, int Sp, const float* mask,
         const float* ks, const float* vs, int s_ld, int Ts, float* out, int rows, hipStream_t st) {
  const size_t lds = (size_t)(m.HD + Sp + Ts) * sizeof(float);
  MLCV_REQUIRE(lds <= 64 * 1024, "float32 attention: too many keys");
  f32_attn_kernel<<<dim3(rows, m.H), F32_NT, lds, st>>>(q, q_ld, m.H, m.KV, m.HD, kp, vp, Sp, mask, ks, vs, s_ld,
                                                        Ts, out, m.H * m.HD);
  MLCV_HIP(hipGetLastError());
  return 0;
}
int norm(const float* x, int W, const float* w, const float* mod, float eps, float* out, int rows, hipStream_t st) {
  f32_norm_kernel<<<rows, F32_NT, 0, st>>>(x, W, w, mod, eps, out);
  MLCV_HIP(hipGetLastError());
  return 0;
}
int residual(float* x, const float* y, const float* gate, int W, int rows, hipStream_t st) {
  f32_residual_kernel<<<ew_grid((size_t)rows * W), 256, 0, st>>>(x, y, gate, W, rows);
  MLCV_HIP(hipGetLastError());
  return 0;
}

bool f32_aligned(std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if ((reinterpret_cast<uintptr_t>(p) & 15) != 0) return false;
  return true;
}

F32Op lin_op(const float* x, int ldx, int M, const F32Lin& l, int epi, float* out, int ldo) {
  F32Op a{};
  a.x = x;
  a.ldx = ldx;
  a.M = M;
  a.K = l.K;
  a.N = l.N;
  a.w[0] = l.w;
  a.b = l.b;
  a.epi = epi;
  a.out = out;
  a.ldo = ldo;
  return a;
}

// q, k and v of one expert over its rows in one product: q roped and scaled to q [M][nq], k roped and v
// to element (m, head, d) at m * kv_m + head * kv_h + d.  with_q false: k and v alone.
F32Op qkv_op(const F32Model& m, const F32Lin& q, const F32Lin& k, const F32Lin& v, bool with_q, const float* x, int M,
             float* qo, float* ko, float* vo, int kv_m, size_t kv_h, const float* cs, const float* sn) {
  F32Op a{};
  a.x = x;
  a.ldx = a.K = k.K;
  a.M = M;
  a.nq = with_q ? q.N : 0;
  a.nkv = k.N;
  a.N = a.nq + 2 * a.nkv;
  a.w[0] = q.w;
  a.w[1] = k.w;
  a.w[2] = v.w;
  a.epi = FE_QKV;
  a.qo = qo;
  a.ko = ko;
  a.vo = vo;
  a.hd = m.HD;
  a.kv_m = kv_m;
  a.kv_h = kv_h;
  a.cos = cs;
  a.sin = sn;
  a.qscale = 1.0f / std::sqrt((float)m.HD);
  a.eps = m.eps;
  return a;
}

// kv_off: with kp null, the cache slices at m.kvp[0 / 1] + kv_off
int fast_attn(const F32Model& m, const float* q, int rows, const float* kp, const float* vp, size_t kv_off,
              const float* mask, const float* ks, const float* vs, int Ts, float* out, hipStream_t st) {
  F32Attn a{};
  a.q = q;
  a.q_ld = a.o_ld = m.H * m.HD;
  a.Tq = rows;
  a.H = m.H;
  a.KV = m.KV;
  a.hd = m.HD;
  a.kp = kp;
  a.vp = vp;
  a.kv = kp ? nullptr : m.kvp;
  a.kv_off = kv_off;
  a.Sp = m.P;
  a.mask = mask;
  a.ks = ks;
  a.vs = vs;
  a.s_ld = m.KV * m.HD;
  a.Ts = Ts;
  a.out = out;
  a.ws = m.aws;
  return f32_attn_launch(a, st);
}

// the time MLP and every modulation of `steps` time embeddings te [steps][W1] into mods
// [steps][2 D + 1][3 W1]
int f32_mods(F32Model& m, const float* te, int steps, hipStream_t st) {
  const int W1 = m.W1, nm = 2 * m.D + 1;
  F32Op a = lin_op(te, W1, steps, m.tin, FE_STORE, m.tmp, W1);
  a.act = 1;
  MLCV_TRY(f32_gemm_launch(a, st));
  a = lin_op(m.tmp, W1, steps, m.tout, FE_STORE, m.cond, W1);
  a.act = 1;
  MLCV_TRY(f32_gemm_launch(a, st));
  a = lin_op(m.cond, W1, steps, m.final_mod, FE_STORE, m.mods, nm * 3 * W1);
  a.tab = m.tab.data();
  a.ntab = nm;
  a.tab_stride = (size_t)3 * W1;
  return f32_gemm_launch(a, st);
}

// one velocity evaluation (keys null: the cache at m.kvp) of x_t with the modulations mods [2 D + 1][3 W1]: into v_out, or (x32
// non-null) the Euler update x32 += dt * v
int f32_velocity(F32Model& m, const float* keys, const float* values, const float* x_t, const float* mods,
                 const float* cs, const float* sn, const float* pmask, float* v_out, float* x32, float dt,
                 hipStream_t st) {
  const int T = m.T, W1 = m.W1, nq = m.H * m.HD, nkv = m.KV * m.HD;
  const size_t kvs = (size_t)m.KV * m.P * m.HD;
  MLCV_TRY(f32_gemm_launch(lin_op(x_t, m.A, T, m.ain, FE_STORE, m.x, W1), st));
  for (int L = 0; L < m.D; ++L) {
    const F32Layer& ly = m.layers[L];
    const float* mi = mods + (size_t)(2 * L) * 3 * W1;
    const float* mp = mi + 3 * W1;
    F32Op a = qkv_op(m, ly.q[1], ly.k[1], ly.v[1], true, m.x, T, m.q, m.k, m.v, nkv, m.HD, cs, sn);
    a.mod = mi;
    a.xn = m.xn;
    MLCV_TRY(f32_gemm_launch(a, st));
    MLCV_TRY(fast_attn(m, m.q, T, keys ? keys + L * kvs : nullptr, keys ? values + L * kvs : nullptr, L * kvs, pmask, m.k, m.v, T, m.attn, st));
    a = lin_op(m.attn, nq, T, ly.o[1], FE_RES, m.x, W1);
    a.gate = mi + 2 * W1;
    MLCV_TRY(f32_gemm_launch(a, st));
    a = lin_op(m.x, W1, T, ly.gu[1], FE_GEGLU, m.h, m.F1);
    a.F = m.F1;
    a.mod = mp;
    a.xn = m.xn;
    a.eps = m.eps;
    MLCV_TRY(f32_gemm_launch(a, st));
    a = lin_op(m.h, m.F1, T, ly.dn[1], FE_RES, m.x, W1);
    a.gate = mp + 2 * W1;
    MLCV_TRY(f32_gemm_launch(a, st));
  }
  F32Op a = lin_op(m.x, W1, T, m.aout, x32 ? FE_EULER : FE_STORE, x32 ? x32 : v_out, m.A);
  a.mod = mods + (size_t)(2 * m.D) * 3 * W1;
  a.xn = m.xn;
  a.eps = m.eps;
  a.dt = dt;
  return f32_gemm_launch(a, st);
}

// the prefix layers over px; the last one gives its keys and values only (nothing reads the rest)
int f32_prefix(F32Model& m, float* keys, float* values, hipStream_t st) {
  const int P = m.P, W0 = m.W0, nq = m.H * m.HD;
  const size_t kvs = (size_t)m.KV * P * m.HD;
  for (int L = 0; L < m.D; ++L) {
    const F32Layer& ly = m.layers[L];
    const bool last = L == m.D - 1;
    float *kL = keys + L * kvs, *vL = values + L * kvs;
    F32Op a = qkv_op(m, ly.q[0], ly.k[0], ly.v[0], !last, m.px, P, m.pq, kL, vL, m.HD, (size_t)P * m.HD, m.pcos, m.psin);
    a.nw = ly.ln_in0;
    a.xn = m.pxn;
    MLCV_TRY(f32_gemm_launch(a, st));
    if (last) break;
    MLCV_TRY(fast_attn(m, m.pq, P, kL, vL, 0, m.mask, nullptr, nullptr, 0, m.pattn, st));
    MLCV_TRY(f32_gemm_launch(lin_op(m.pattn, nq, P, ly.o[0], FE_RES, m.px, W0), st));
    a = lin_op(m.px, W0, P, ly.gu[0], FE_GEGLU, m.ph, m.F0);
    a.F = m.F0;
    a.nw = ly.ln_post0;
    a.xn = m.pxn;
    a.eps = m.eps;
    MLCV_TRY(f32_gemm_launch(a, st));
    MLCV_TRY(f32_gemm_launch(lin_op(m.ph, m.F0, P, ly.dn[0], FE_RES, m.px, W0), st));
  }
  return 0;
}

// the model's S Euler steps on x32 from the staged time embeddings, tables and mask
int f32_steps(F32Model& m, const float* keys, const float* values, const float* pmask, hipStream_t st) {
  const float dt = (float)(-1.0 / m.S);
  const size_t modstep = (size_t)(2 * m.D + 1) * 3 * m.W1;
  for (int i = 0; i < m.S; ++i) {
    if (i % m.SB == 0) MLCV_TRY(f32_mods(m, m.te + (size_t)i * m.W1, std::min(m.SB, m.S - i), st));
    MLCV_TRY(f32_velocity(m, keys, values, m.x32, m.mods + (i % m.SB) * modstep, m.scos, m.ssin, pmask, nullptr, m.x32,
                          dt, st));
  }
  return 0;
}

// `body` on the caller's stream: as a graph captured on the model's own stream at its first use, or
// directly (graphs off, or the caller is capturing)
template <class F>
int f32_run(F32Model& m, hipGraphExec_t& g, hipStream_t user, F&& body) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  MLCV_HIP(hipStreamIsCapturing(user, &cs));
  if (!m.use_graph || cs != hipStreamCaptureStatusNone) return body(user);
  if (!g) {
    if (!m.cap) MLCV_HIP(hipStreamCreateWithFlags(&m.cap, hipStreamNonBlocking));
    MLCV_HIP(hipStreamBeginCapture(m.cap, hipStreamCaptureModeThreadLocal));
    const int r = body(m.cap);
    hipGraph_t graph = nullptr;
    const hipError_t e = hipStreamEndCapture(m.cap, &graph);
    if (r != 0 || e != hipSuccess) {
      if (e == hipSuccess && graph) (void)hipGraphDestroy(graph);
      if (r != 0) return r;
      MLCV_HIP(e);
    }
    const hipError_t ie = hipGraphInstantiate(&g, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (ie != hipSuccess) g = nullptr;
    MLCV_HIP(ie);
  }
  MLCV_HIP(hipGraphLaunch(g, user));
  return 0;
}

__global__ void f32_set_kv_kernel(const float** kvp, const float* keys, const float* values) {
  kvp[0] = keys;
  kvp[1] = values;
}

// The general form of one velocity evaluation, for widths or pointers the matrix-core kernels do not
// take: x_t (the model's x) with the time embedding te (pi0_model.py:142-163)
int f32_step_general(F32Model& m, const float* keys, const float* values, const float* x_t, const float* te,
                const float* cs, const float* sn, const float* pmask, float* v_out, hipStream_t st) {
  const int T = m.T, W1 = m.W1, nq = m.H * m.HD, nkv = m.KV * m.HD, W3 = 3 * W1;
  const size_t kvs = (size_t)m.KV * m.P * m.HD;  // one layer's cache slice
  const float scale = 1.0f / std::sqrt((float)m.HD);
  MLCV_TRY(gemm(x_t, m.A, m.ain, m.x, W1, T, 0, st));
  MLCV_TRY(gemm(te, W1, m.tin, m.tmp, W1, 1, 1, st));
  MLCV_TRY(gemm(m.tmp, W1, m.tout, m.cond, W1, 1, 1, st));
  for (int L = 0; L < m.D; ++L) {
    MLCV_TRY(gemm(m.cond, W1, m.layers[L].mod_in, m.mods + (size_t)(2 * L) * W3, W3, 1, 0, st));
    MLCV_TRY(gemm(m.cond, W1, m.layers[L].mod_post, m.mods + (size_t)(2 * L + 1) * W3, W3, 1, 0, st));
  }
  MLCV_TRY(gemm(m.cond, W1, m.final_mod, m.mods + (size_t)(2 * m.D) * W3, W3, 1, 0, st));
  for (int L = 0; L < m.D; ++L) {
    const F32Layer& ly = m.layers[L];
    const float* mi = m.mods + (size_t)(2 * L) * W3;
    const float* mp = m.mods + (size_t)(2 * L + 1) * W3;
    MLCV_TRY(norm(m.x, W1, nullptr, mi, m.eps, m.xn, T, st));
    MLCV_TRY(gemm(m.xn, W1, ly.q[1], m.q, nq, T, 0, st, false));
    MLCV_TRY(gemm(m.xn, W1, ly.k[1], m.k, nkv, T, 0, st, false));
    MLCV_TRY(gemm(m.xn, W1, ly.v[1], m.v, nkv, T, 0, st, false));
    f32_rope_kernel<<<T, 256, 0, st>>>(m.q, nq, 0, m.H, m.HD, cs, sn, scale);
    f32_rope_kernel<<<T, 256, 0, st>>>(m.k, nkv, 0, m.KV, m.HD, cs, sn, 1.0f);
    MLCV_HIP(hipGetLastError());
    MLCV_TRY(attn(m.q, nq, m, keys + L * kvs, values + L * kvs, m.P, pmask, m.k, m.v, nkv, T, m.attn, T, st));
    MLCV_TRY(gemm(m.attn, nq, ly.o[1], m.o, W1, T, 0, st, false));
    MLCV_TRY(residual(m.x, m.o, mi + 2 * W1, W1, T, st));
    MLCV_TRY(norm(m.x, W1, nullptr, mp, m.eps, m.xn, T, st));
    MLCV_TRY(gemm(m.xn, W1, ly.gu[1], m.gu, 2 * m.F1, T, 0, st, false));
    f32_geglu_kernel<<<ew_grid((size_t)T * m.F1), 256, 0, st>>>(m.gu, m.F1, T, m.h);
    MLCV_HIP(hipGetLastError());
    MLCV_TRY(gemm(m.h, m.F1, ly.dn[1], m.o, W1, T, 0, st, false));
    MLCV_TRY(residual(m.x, m.o, mp + 2 * W1, W1, T, st));
  }
  MLCV_TRY(norm(m.x, W1, nullptr, m.mods + (size_t)(2 * m.D) * W3, m.eps, m.xn, T, st));
  return gemm(m.xn, W1, m.aout, v_out, m.A, T, 0, st);
}

}  // namespace

int f32_create(const ::mlcv_config& cfg, F32Model** out) {
  auto m = std::make_unique<F32Model>();
  m->W0 = cfg.vlm_width;
  m->F0 = cfg.vlm_mlp;
  m->W1 = cfg.ae_width;
  m->F1 = cfg.ae_mlp;
  m->D = cfg.depth;
  m->H = cfg.num_heads;
  m->KV = cfg.num_kv_heads;
  m->HD = cfg.head_dim;
  m->P = cfg.prefix_len;
  m->T = cfg.suffix_len;
  m->A = cfg.action_dim;
  m->S = cfg.num_steps;
  m->eps = cfg.rms_norm_eps;
  m->shape_ok = (m->HD == 16 || m->HD == 32 || m->HD == 64 || m->HD == 128 || m->HD == 256) && m->W0 % 8 == 0 &&
                m->F0 % 8 == 0 && m->W1 % 8 == 0 && m->F1 % 8 == 0 && m->A % 8 == 0;
  MLCV_REQUIRE(m->HD % 2 == 0 && m->H % m->KV == 0, "float32 model: head_dim even, heads a multiple of kv heads");
  MLCV_REQUIRE((size_t)(m->HD + m->P + m->T) * 4 <= 64 * 1024, "float32 model: prefix_len + suffix_len too large");
  m->SB = std::min(m->S, 64);
  const size_t SB = m->SB;
  const size_t P = m->P, T = m->T, nq = (size_t)m->H * m->HD, nkv = (size_t)m->KV * m->HD;
  const size_t kv = (size_t)m->D * nkv * P;
  F32Model& r = *m;
  for (auto [p, n] : std::initializer_list<std::pair<float**, size_t>>{
           {&r.px, P * r.W0}, {&r.pxn, P * r.W0}, {&r.pq, P * nq}, {&r.pk, P * nkv}, {&r.pv, P * nkv},
           {&r.pattn, P * nq}, {&r.po, P * r.W0}, {&r.pgu, P * 2 * r.F0}, {&r.ph, P * r.F0},
           {&r.pcos, P * r.HD / 2}, {&r.psin, P * r.HD / 2}, {&r.mask, P}, {&r.ckeys, kv}, {&r.cvalues, kv},
           {&r.x, T * r.W1}, {&r.xn, T * r.W1}, {&r.q, T * nq}, {&r.k, T * nkv}, {&r.v, T * nkv},
           {&r.attn, T * nq}, {&r.o, T * r.W1}, {&r.gu, T * 2 * r.F1}, {&r.h, T * r.F1}, {&r.cond, SB * r.W1},
           {&r.tmp, SB * r.W1}, {&r.mods, SB * (2 * r.D + 1) * 3 * r.W1}, {&r.vout, T * r.A}, {&r.x32, T * r.A},
           {&r.scos, T * r.HD / 2}, {&r.ssin, T * r.HD / 2}, {&r.smask, P}, {&r.te, (size_t)r.S * r.W1}})
    MLCV_TRY(r.alloc(p, n));
  size_t aws = 0;
  for (auto [rows, nk] : {std::pair<int, int>{r.P, r.P}, {r.T, r.P + r.T}}) {
    int ns = 1, cps = 1;
    f32_attn_plan(rows * (r.H / r.KV), r.KV, nk, &ns, &cps);
    aws = std::max(aws, f32_attn_ws_floats(r.KV, rows * (r.H / r.KV), r.HD, ns));
  }
  MLCV_TRY(r.alloc(&r.aws, aws));
  MLCV_HIP(hipMalloc(reinterpret_cast<void**>(&r.kvp), 2 * sizeof(float*)));
  // RoPE of the prefill's positions 0..P-1: radians = pos / theta^((2/hd) i) in float64
  std::vector<float> hc(P * r.HD / 2), hs(P * r.HD / 2);
  for (size_t p = 0; p < P; ++p)
    for (int i = 0; i < r.HD / 2; ++i) {
      const double rad = (double)p / std::pow((double)cfg.rope_theta, (2.0 / r.HD) * i);
      hc[p * (r.HD / 2) + i] = (float)std::cos(rad);
      hs[p * (r.HD / 2) + i] = (float)std::sin(rad);
    }
  MLCV_HIP(hipMemcpy(r.pcos, hc.data(), hc.size() * 4, hipMemcpyHostToDevice));
  MLCV_HIP(hipMemcpy(r.psin, hs.data(), hs.size() * 4, hipMemcpyHostToDevice));
  *out = m.release();
  return 0;
}

void f32_destroy(F32Model* m) { delete m; }

void f32_set_graph(F32Model& m, bool on) { m.use_graph = on; }

int f32_bind(F32Model& m, const void* const* ptrs, int count) {
  m.bound = false;
  // a replay may still be running on any stream: the call that started it did not wait
  if (m.g_loop || m.g_chunk) MLCV_HIP(hipDeviceSynchronize());
  m.drop_graphs();
  int idx = 0;
  auto f = [&]() { return reinterpret_cast<const float*>(ptrs[idx++]); };
  auto lin = [&](F32Lin& l, int N, int K, bool bias) {
    l.N = N;
    l.K = K;
    l.w = f();
    l.b = bias ? f() : nullptr;
  };
  const int nq = m.H * m.HD, nkv = m.KV * m.HD;
  const int widths[2] = {m.W0, m.W1}, mlps[2] = {m.F0, m.F1};
  m.layers.assign(m.D, F32Layer{});
  for (int L = 0; L < m.D; ++L) {  // the order of named_params (pi0_model.py:81-88)
    F32Layer& ly = m.layers[L];
    for (int e = 0; e < 2; ++e) {
      lin(ly.q[e], nq, widths[e], false);
      lin(ly.k[e], nkv, widths[e], false);
      lin(ly.v[e], nkv, widths[e], false);
      lin(ly.o[e], widths[e], nq, false);
    }
    for (int e = 0; e < 2; ++e) {
      lin(ly.gu[e], 2 * mlps[e], widths[e], false);
      lin(ly.dn[e], widths[e], mlps[e], false);
    }
    ly.ln_in0 = f();
    lin(ly.mod_in, 3 * m.W1, m.W1, true);
    ly.ln_post0 = f();
    lin(ly.mod_post, 3 * m.W1, m.W1, true);
  }
  idx++;  // backbone.final_norm.0.weight (not read by the M1 functions)
  lin(m.final_mod, 3 * m.W1, m.W1, true);
  lin(m.ain, m.W1, m.A, true);
  lin(m.aout, m.A, m.W1, true);
  lin(m.tin, m.W1, m.W1, true);
  lin(m.tout, m.W1, m.W1, true);
  MLCV_REQUIRE(idx == count, "internal: float32 parameter walk mismatch");
  for (int i = 0; i < count; ++i) MLCV_REQUIRE(ptrs[i] != nullptr, "null parameter pointer");
  m.fast = m.shape_ok;
  for (int i = 0; i < count; ++i) m.fast = m.fast && f32_aligned({ptrs[i]});
  if (m.fast) {
    m.tab.clear();
    for (const F32Layer& ly : m.layers)
      for (const F32Lin* l : {&ly.mod_in, &ly.mod_post}) m.tab.push_back({l->w, l->b});
    m.tab.push_back({m.final_mod.w, m.final_mod.b});
  }
  m.bound = true;
  return 0;
}

// prefill (pi0_model.py:128-140; prefill_e0 gemma_dual.py:334-341, attn_prefill_e0 :236-253)
int f32_prefill(F32Model& m, const void* prefix_embs, const float* prefix_mask, float* keys, void* values,
                hipStream_t st) {
  MLCV_REQUIRE(m.bound, "parameters not bound");
  const int P = m.P, W0 = m.W0, nq = m.H * m.HD, nkv = m.KV * m.HD;
  const size_t kvs = (size_t)m.KV * P * m.HD;
  float* vals = reinterpret_cast<float*>(values);
  const float scale = 1.0f / std::sqrt((float)m.HD);
  const CopyJob in[] = {{prefix_embs, m.px, (size_t)P * W0 * 4}, {prefix_mask, m.mask, (size_t)P * 4}};
  MLCV_TRY(copy_list_launch(in, 2, st));
  if (m.fast && f32_aligned({keys, values})) return f32_prefix(m, keys, vals, st);
  for (int L = 0; L < m.D; ++L) {
    const F32Layer& ly = m.layers[L];
    MLCV_TRY(norm(m.px, W0, ly.ln_in0, nullptr, m.eps, m.pxn, P, st));
    MLCV_TRY(gemm(m.pxn, W0, ly.q[0], m.pq, nq, P, 0, st, false));
    MLCV_TRY(gemm(m.pxn, W0, ly.k[0], m.pk, nkv, P, 0, st, false));
    MLCV_TRY(gemm(m.pxn, W0, ly.v[0], m.pv, nkv, P, 0, st, false));
    f32_rope_kernel<<<P, 256, 0, st>>>(m.pq, nq, 0, m.H, m.HD, m.pcos, m.psin, scale);
    f32_rope_kernel<<<P, 256, 0, st>>>(m.pk, nkv, 0, m.KV, m.HD, m.pcos, m.psin, 1.0f);
    f32_kv_write_kernel<<<ew_grid(kvs), 256, 0, st>>>(m.pk, m.pv, P, m.KV, m.HD, keys + L * kvs, vals + L * kvs);
    MLCV_HIP(hipGetLastError());
    MLCV_TRY(attn(m.pq, nq, m, keys + L * kvs, vals + L * kvs, P, m.mask, nullptr, nullptr, 0, 0, m.pattn, P, st));
    MLCV_TRY(gemm(m.pattn, nq, ly.o[0], m.po, W0, P, 0, st, false));
    MLCV_TRY(residual(m.px, m.po, nullptr, W0, P, st));
    MLCV_TRY(norm(m.px, W0, ly.ln_post0, nullptr, m.eps, m.pxn, P, st));
    MLCV_TRY(gemm(m.pxn, W0, ly.gu[0], m.pgu, 2 * m.F0, P, 0, st, false));
    f32_geglu_kernel<<<ew_grid((size_t)P * m.F0), 256, 0, st>>>(m.pgu, m.F0, P, m.ph);
    MLCV_HIP(hipGetLastError());
    MLCV_TRY(gemm(m.ph, m.F0, ly.dn[0], m.po, W0, P, 0, st, false));
    MLCV_TRY(residual(m.px, m.po, nullptr, W0, P, st));
  }
  return 0;
}

int f32_step(F32Model& m, const float* keys, const void* values, const void* x_t, const void* time_emb,
             const float* cs, const float* sn, const float* prefix_mask, float* v_out, hipStream_t st) {
  MLCV_REQUIRE(m.bound, "parameters not bound");
  const float* vals = reinterpret_cast<const float*>(values);
  const float *x = reinterpret_cast<const float*>(x_t), *te = reinterpret_cast<const float*>(time_emb);
  if (m.fast && f32_aligned({keys, vals, x, te, cs, sn, v_out})) {
    MLCV_TRY(f32_mods(m, te, 1, st));
    return f32_velocity(m, keys, vals, x, m.mods, cs, sn, prefix_mask, v_out, nullptr, 0.f, st);
  }
  return f32_step_general(m, keys, vals, x, te, cs, sn, prefix_mask, v_out, st);
}

// N Euler steps x <- x + (-1/N) v(x), x fed to each step as the model's x (pi0_model.py:165-194)
int f32_loop(F32Model& m, const float* keys, const void* values, const float* x0, const void* time_embs,
             const float* cs, const float* sn, const float* prefix_mask, float* x_out, hipStream_t st) {
  MLCV_REQUIRE(m.bound, "parameters not bound");
  const size_t n = (size_t)m.T * m.A, half = m.HD / 2;
  const float* vals = reinterpret_cast<const float*>(values);
  const float* te = reinterpret_cast<const float*>(time_embs);
  const CopyJob in[] = {{x0, m.x32, n * 4},
                        {te, m.te, (size_t)m.S * m.W1 * 4},
                        {cs, m.scos, m.T * half * 4},
                        {sn, m.ssin, m.T * half * 4},
                        {prefix_mask, m.smask, (size_t)m.P * 4}};
  MLCV_TRY(copy_list_launch(in, 5, st));
  if (m.fast && f32_aligned({keys, vals})) {
    f32_set_kv_kernel<<<1, 1, 0, st>>>(m.kvp, keys, vals);
    MLCV_HIP(hipGetLastError());
    MLCV_TRY(f32_run(m, m.g_loop, st, [&](hipStream_t s) { return f32_steps(m, nullptr, nullptr, m.smask, s); }));
  } else {
    const float dt = (float)(-1.0 / m.S);
    for (int i = 0; i < m.S; ++i) {
      MLCV_TRY(f32_step_general(m, keys, vals, m.x32, m.te + (size_t)i * m.W1, m.scos, m.ssin, m.smask, m.vout, st));
      f32_euler_kernel<<<ew_grid(n), 256, 0, st>>>(m.x32, m.vout, dt, (int)n);
      MLCV_HIP(hipGetLastError());
    }
  }
  const CopyJob out{m.x32, x_out, n * 4};
  return copy_list_launch(&out, 1, st);
}

int f32_chunk(F32Model& m, const void* prefix_embs, const float* prefix_mask, const float* x0, const void* time_embs,
              const float* cs, const float* sn, float* x_out, hipStream_t st) {
  MLCV_REQUIRE(m.bound, "parameters not bound");
  if (!m.fast) {
    MLCV_TRY(f32_prefill(m, prefix_embs, prefix_mask, m.ckeys, m.cvalues, st));
    return f32_loop(m, m.ckeys, m.cvalues, x0, time_embs, cs, sn, m.mask, x_out, st);
  }
  const size_t n = (size_t)m.T * m.A, half = m.HD / 2;
  const CopyJob in[] = {{prefix_embs, m.px, (size_t)m.P * m.W0 * 4}, {prefix_mask, m.mask, (size_t)m.P * 4},
                        {x0, m.x32, n * 4},                          {time_embs, m.te, (size_t)m.S * m.W1 * 4},
                        {cs, m.scos, m.T * half * 4},                {sn, m.ssin, m.T * half * 4}};
  MLCV_TRY(copy_list_launch(in, 6, st));
  MLCV_TRY(f32_run(m, m.g_chunk, st, [&](hipStream_t s) {
    MLCV_TRY(f32_prefix(m, m.ckeys, m.cvalues, s));
    return f32_steps(m, m.ckeys, m.cvalues, m.mask, s);
  }));
  const CopyJob out{m.x32, x_out, n * 4};
  return copy_list_launch(&out, 1, st);
}

}  // namespace mlcv
