// The float32 model's attention on the fp32 matrix cores (v_mfma_f32_16x16x4_f32): logits, softmax,
// probabilities and sums in fp32 (gemma_dual.py:97-122), the softmax in its online form over 32-key
// chunks and, where that fills the CUs, over key splits.
//
// A workgroup takes 64 query rows of one kv head (row = query head in the group * Tq + token), 16 per
// wave, and a range of key chunks.  K and V of a chunk sit in LDS (rows of hd + 4 floats: 16 rows'
// 16-byte reads, and 4 rows' 64-byte runs 4 rows apart, hit distinct banks of 64); the next chunk's
// loads are in registers meanwhile, and two workgroups share a CU (67 KB at hd 256).
// S^T[key][row] = K . Q^T leaves a lane 4 keys of one query row per 16-key tile, which is the B operand
// of O^T[d][row] += V^T . P^T (k index = lane / 16, key 4 (lane / 16) + i in the i-th of 4 products), so
// the probabilities stay in registers.
// Bound by the matrix cores: 2 x 128 products of 32 clocks per chunk and wave at hd 256.
// Measured at P = 968, 8 heads on one kv head of 256 (7.7 GFLOP, 50 us at the matrix cores' rate): 103 us
// and 10 us for the combine (75 TFLOP/s), against 1217 us for one workgroup per (row, head) with serial
// dot products from global memory, which is what other head dims still run (model_f32.hip).  Bounding the
// registers to two workgroups per CU (256 instead of 336) is part of that.
#include "f32.h"
#include "plan.h"

#pragma clang fp contract(off)

namespace mlcv {
namespace {

struct FaArgs {
  F32Attn a;
  int rows, rpad, nsplit, cps;
  float *part, *ml;
};

__device__ __forceinline__ f4 fa_mfma(float a, float b, f4 c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
#else
  return c;
#endif
}

template <int HD>
__global__ __launch_bounds__(256, 2) void f32_fa_kernel(const FaArgs p) {
  constexpr int LD = HD + 4, NS = HD / 16, PPR = HD / 4;  // PPR: 16-byte pieces per row
  constexpr int NI = (ATTN_KCH * PPR + 255) / 256;        // pieces of K (and of V) per thread and chunk
  __shared__ __attribute__((aligned(16))) float sk[ATTN_KCH * LD], sv[ATTN_KCH * LD];
  __shared__ float sm[ATTN_KCH];
  const F32Attn& a = p.a;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, g = lane >> 4;
  const int split = blockIdx.y, kvh = blockIdx.z, grp = a.H / a.KV, nk = a.Sp + a.Ts;
  const int row = blockIdx.x * ATTN_ROWS + 16 * w + r, rowc = min(row, p.rows - 1);
  const int h = kvh * grp + rowc / a.Tq, t = rowc % a.Tq;

  const float* kp = a.kv ? load_global(a.kv) + a.kv_off : a.kp;
  const float* vp = a.kv ? load_global(a.kv + 1) + a.kv_off : a.vp;
  f4 kr[NI], vr[NI];
  float mr = 0.f;
  auto load = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int it = (tid + 256 * i) % (ATTN_KCH * PPR);
      const int kj = min(c * ATTN_KCH + it / PPR, nk - 1), d = it % PPR * 4;  // past the keys: the last one
      const size_t pre = ((size_t)kvh * a.Sp + kj) * HD + d, suf = (size_t)(kj - a.Sp) * a.s_ld + kvh * HD + d;
      const bool in = kj < a.Sp;
      kr[i] = load_global(reinterpret_cast<const f4*>(in ? kp + pre : a.ks + suf));
      vr[i] = load_global(reinterpret_cast<const f4*>(in ? vp + pre : a.vs + suf));
    }
    if (tid < ATTN_KCH) {
      const int kj = c * ATTN_KCH + tid;
      mr = kj >= nk ? -INFINITY : kj < a.Sp && a.mask ? load_global(a.mask + kj) : 0.f;
    }
  };
  const int nch = (nk + ATTN_KCH - 1) / ATTN_KCH, c0 = split * p.cps, c1 = min(nch, c0 + p.cps);
  load(c0);
  f4 q[NS], o[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    q[s] = load_global(reinterpret_cast<const f4*>(a.q + (size_t)t * a.q_ld + h * HD + 16 * s + 4 * g));
    o[s] = (f4){0.f, 0.f, 0.f, 0.f};
  }
  float m_run = -INFINITY, l_run = 0.f;
  for (int c = c0; c < c1; ++c) {
    __syncthreads();  // every wave is done with the chunk before
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int it = (tid + 256 * i) % (ATTN_KCH * PPR), at = it / PPR * LD + it % PPR * 4;
      *reinterpret_cast<f4*>(sk + at) = kr[i];
      *reinterpret_cast<f4*>(sv + at) = vr[i];
    }
    if (tid < ATTN_KCH) sm[tid] = mr;
    __syncthreads();
    if (c + 1 < c1) load(c + 1);
    f4 acc[2] = {(f4){0.f, 0.f, 0.f, 0.f}, (f4){0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      f4 k[2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) k[kt] = *reinterpret_cast<const f4*>(sk + (16 * kt + r) * LD + 16 * s + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) acc[kt] = fa_mfma(k[kt][i], q[s][i], acc[kt]);
    }
    // this lane's 8 logits of row r: keys 16 kt + 4 g + i
    float x[8];
    float cmax = -INFINITY;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      x[j] = acc[j >> 2][j & 3] + sm[16 * (j >> 2) + 4 * g + (j & 3)];
      cmax = fmaxf(cmax, x[j]);
    }
    cmax = xor_max_16_32(cmax);
    const float m_new = fmaxf(m_run, cmax);
    const float ref = m_new == -INFINITY ? 0.f : m_new;  // every key so far at -inf: their exp is 0
    if (__any(m_new > m_run)) {
      const float alpha = expf(m_run - ref);
      l_run = l_run * alpha;
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[s][i] = o[s][i] * alpha;
      m_run = m_new;
    }
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      x[j] = expf(x[j] - ref);
      sum = sum + x[j];
    }
    l_run = l_run + xor_sum_16_32(sum);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float* vrow = sv + (16 * (j >> 2) + 4 * g + (j & 3)) * LD + r;
#pragma unroll
      for (int s = 0; s < NS; ++s) o[s] = fa_mfma(vrow[16 * s], x[j], o[s]);
    }
  }
  if (row >= p.rows) return;
  if (p.nsplit > 1) {
    const size_t pr = ((size_t)kvh * p.nsplit + split) * p.rpad + row;
#pragma unroll
    for (int s = 0; s < NS; ++s) *reinterpret_cast<f4*>(p.part + pr * HD + 16 * s + 4 * g) = o[s];
    if (g == 0) *reinterpret_cast<f2*>(p.ml + 2 * pr) = (f2){m_run, l_run};
    return;
  }
  float* op = a.out + (size_t)t * a.o_ld + h * HD + 4 * g;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    f4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = o[s][i] / l_run;
    *reinterpret_cast<f4*>(op + 16 * s) = v;
  }
}

// the splits of one row added in split order, 4 dims per lane; 4 rows per workgroup
__global__ __launch_bounds__(256) void f32_fa_combine_kernel(const FaArgs p) {
  const F32Attn& a = p.a;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), kvh = blockIdx.y, lane = threadIdx.x & 63, hd = a.hd;
  if (row >= p.rows) return;
  const size_t pr0 = (size_t)kvh * p.nsplit * p.rpad + row;
  float m = -INFINITY;
  for (int s = 0; s < p.nsplit; ++s) m = fmaxf(m, p.ml[2 * (pr0 + (size_t)s * p.rpad)]);
  const float ref = m == -INFINITY ? 0.f : m;
  const int d = 4 * lane;
  const bool in = d < hd;
  float l = 0.f;
  f4 acc = (f4){0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < p.nsplit; ++s) {
    const size_t pr = pr0 + (size_t)s * p.rpad;
    const f2 ml = *reinterpret_cast<const f2*>(p.ml + 2 * pr);
    const f4 o = in ? *reinterpret_cast<const f4*>(p.part + pr * hd + d) : (f4){0.f, 0.f, 0.f, 0.f};
    const float wgt = expf(ml[0] - ref);
    l = l + wgt * ml[1];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = acc[i] + wgt * o[i];
  }
  if (!in) return;
  f4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = acc[i] / l;
  const int h = kvh * (a.H / a.KV) + row / a.Tq, t = row % a.Tq;
  *reinterpret_cast<f4*>(a.out + (size_t)t * a.o_ld + h * hd + d) = v;
}

}  // namespace

int f32_attn_launch(const F32Attn& a, hipStream_t st) {
  MLCV_REQUIRE(a.Tq > 0 && a.KV > 0 && a.H % a.KV == 0 && a.Sp >= 0 && a.Ts >= 0 && a.Sp + a.Ts > 0, "float32 attention: shape");
  FaArgs p{};
  p.a = a;
  p.rows = a.Tq * (a.H / a.KV);
  p.rpad = (p.rows + ATTN_ROWS - 1) / ATTN_ROWS * ATTN_ROWS;
  f32_attn_plan(p.rows, a.KV, a.Sp + a.Ts, &p.nsplit, &p.cps);
  MLCV_REQUIRE(p.nsplit == 1 || a.ws, "float32 attention: workspace");
  p.part = a.ws;
  p.ml = a.ws + (size_t)a.KV * p.nsplit * p.rpad * a.hd;
  const dim3 grid(p.rpad / ATTN_ROWS, p.nsplit, a.KV);
  switch (a.hd) {
    case 16: f32_fa_kernel<16><<<grid, 256, 0, st>>>(p); break;
    case 32: f32_fa_kernel<32><<<grid, 256, 0, st>>>(p); break;
    case 64: f32_fa_kernel<64><<<grid, 256, 0, st>>>(p); break;
    case 128: f32_fa_kernel<128><<<grid, 256, 0, st>>>(p); break;
    case 256: f32_fa_kernel<256><<<grid, 256, 0, st>>>(p); break;
    default: MLCV_REQUIRE(false, "float32 attention: head dim");
  }
  MLCV_HIP(hipGetLastError());
  if (p.nsplit > 1) {
    f32_fa_combine_kernel<<<dim3((p.rows + 3) / 4, a.KV), 256, 0, st>>>(p);
    MLCV_HIP(hipGetLastError());
  }
  return 0;
}

}  // namespace mlcv
