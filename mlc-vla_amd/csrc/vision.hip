// SigLIP vision tower + PaliGemma multi-modal projector (siglip.py:20-120), the
// `embed_image` function (pi0_model.py:97-99): one channels-last image [S][S][C] in fp16
// -> [num_patches][projection_dim] fp16.
//
// Seven launches a layer, each a few microseconds of memory latency over the L2: LayerNorm, q/k/v,
// attention, out_proj + residual, LayerNorm, fc1 + GELU, fc2 + residual.  The linears add bias, GELU,
// residual or position embedding in their epilogues (gemm_mid.hip; fp32 accumulation, one fp16 rounding
// per op of the reference); LayerNorm keeps its statistics in fp32 (siglip.py:20-35), one wave per row
// with the row in registers.  The attention follows the reference's cast points (siglip.py:58-70) with
// the exact products of the fp16 q and k scaled in fp32 (the reference rounds q * scale to fp16), fp32
// logits and softmax, fp16 probabilities, P.V accumulated in fp32.
#include "kernels.h"

#include <algorithm>
#include <cmath>

namespace mlcv {

namespace {

// patches [np][kp]: row py * side + px, column (i * p + j) * C + c holds pixel
// (py * p + i, px * p + j, c) (siglip.py:97-107); columns past p * p * C are zero
__global__ void patchify_kernel(const _Float16* __restrict__ img, int size, int p, int C, int kp,
                                _Float16* __restrict__ out) {
  const int patch = blockIdx.x, side = size / p;
  const int py = patch / side, px = patch % side;
  for (int col = threadIdx.x; col < kp; col += blockDim.x) {
    _Float16 v = (_Float16)0.f;
    if (col < p * p * C) {
      const int c = col % C, j = (col / C) % p, i = col / (C * p);
      v = img[((size_t)(py * p + i) * size + (px * p + j)) * C + c];
    }
    out[(size_t)patch * kp + col] = v;
  }
}

// w [n][k] -> wp [n][kp], zero columns past k
__global__ void pad_cols_kernel(const _Float16* __restrict__ w, int k, int kp, _Float16* __restrict__ wp) {
  const int r = blockIdx.x;
  for (int c = threadIdx.x; c < kp; c += blockDim.x) wp[(size_t)r * kp + c] = c < k ? w[(size_t)r * k + c] : (_Float16)0.f;
}

// Prefetch workgroups beside a LayerNorm's rows and beside an attention's tiles: the whole tower (27
// layers of width 1152) takes 1754 us without either, 1720 with 128 beside the attention alone, 1743 with
// 256 beside the LayerNorms alone, 1714 with both, 1718 with 512 each.  With the LayerNorms' share on the
// CUs that fc1 and fc2 leave idle instead (at least MID_PF_MIN of them): 1588; 8 layers of 4 / 64 / 196
// patches 368 / 394 / 505 -> 328 / 365 / 474.
constexpr int LN_PF = 256, ATTN_PF = 128;
constexpr int MID_PF_MIN = 32;

enum VisEpi { VE_BIAS = 0, VE_BIAS_GELU = 1, VE_BIAS_RESIDUAL = 2, VE_BIAS_POS = 3 };

// y = fp16(y + b) on columns [0, n) of rows with stride ldy, then:
//   VE_BIAS_GELU      y = fp16(gelu_tanh(y))
//   VE_BIAS_RESIDUAL  x = fp16(x + y)            (x: the residual stream, stride ldx)
//   VE_BIAS_POS       y = fp16(y + pos[m % npos])  (position embedding, stride n)
__global__ void vis_epilogue_kernel(_Float16* __restrict__ y, int ldy, const _Float16* __restrict__ b, int n,
                                    int mode, _Float16* __restrict__ x, int ldx, const _Float16* __restrict__ pos,
                                    int npos) {
  const int m = blockIdx.x;
  if ((n & 7) == 0 && (ldy & 7) == 0 && (ldx & 7) == 0 &&
      ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(x) |
        reinterpret_cast<uintptr_t>(pos)) & 15) == 0) {
    // 16-byte pieces, the same arithmetic per element
    for (int c = 8 * threadIdx.x; c < n; c += 8 * blockDim.x) {
      const h8 yv = *reinterpret_cast<const h8*>(y + (size_t)m * ldy + c), bv = *reinterpret_cast<const h8*>(b + c);
      h8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v[e] = hadd(yv[e], bv[e]);
        if (mode == VE_BIAS_GELU) v[e] = f2h(gelu_tanh(h2f(v[e])));
      }
      if (mode == VE_BIAS_RESIDUAL) {
        h8* xp = reinterpret_cast<h8*>(x + (size_t)m * ldx + c);
        const h8 xv = *xp;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = hadd(xv[e], v[e]);
        *xp = v;
        continue;
      }
      if (mode == VE_BIAS_POS) {
        const h8 pv = *reinterpret_cast<const h8*>(pos + (size_t)(m % npos) * n + c);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = hadd(v[e], pv[e]);
      }
      *reinterpret_cast<h8*>(y + (size_t)m * ldy + c) = v;
    }
    return;
  }
  for (int c = threadIdx.x; c < n; c += blockDim.x) {
    _Float16 v = hadd(y[(size_t)m * ldy + c], b[c]);
    if (mode == VE_BIAS_GELU) v = f2h(gelu_tanh(h2f(v)));
    if (mode == VE_BIAS_RESIDUAL) {
      x[(size_t)m * ldx + c] = hadd(x[(size_t)m * ldx + c], v);
      continue;
    }
    if (mode == VE_BIAS_POS) v = hadd(v, pos[(size_t)(m % npos) * n + c]);
    y[(size_t)m * ldy + c] = v;
  }
}

// LayerNorm of one row per block: mean, then variance about it, in fp32 (two passes over
// the row), out = fp16((x - mean) / sqrt(var + eps) * w + b) with w, b in fp32
__global__ __launch_bounds__(256) void layernorm_kernel(const _Float16* __restrict__ x, const _Float16* __restrict__ w,
                                                        const _Float16* __restrict__ b, int n, float eps,
                                                        _Float16* __restrict__ out) {
  __shared__ float red[4];
  __shared__ float stat[2];
  const int r = blockIdx.x, tid = threadIdx.x;
  const _Float16* xr = x + (size_t)r * n;
  float s = 0.f;
  for (int c = tid; c < n; c += 256) s += h2f(xr[c]);
  s = wave_sum(s);
  if ((tid & 63) == 0) red[tid >> 6] = s;
  __syncthreads();
  if (tid == 0) stat[0] = (red[0] + red[1] + red[2] + red[3]) / (float)n;
  __syncthreads();
  const float mean = stat[0];
  float q = 0.f;
  for (int c = tid; c < n; c += 256) {
    const float d = h2f(xr[c]) - mean;
    q += d * d;
  }
  q = wave_sum(q);
  __syncthreads();
  if ((tid & 63) == 0) red[tid >> 6] = q;
  __syncthreads();
  if (tid == 0) stat[1] = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)n + eps);
  __syncthreads();
  const float rstd = stat[1];
  for (int c = tid; c < n; c += 256)
    out[(size_t)r * n + c] = f2h((h2f(xr[c]) - mean) * rstd * h2f(w[c]) + h2f(b[c]));
}

// LayerNorm of one row per wave, the row in registers (n % 8 == 0, n <= 512 NP, 16-byte aligned): one pass
// and no barriers.  256 rows of 1152: 4.8 us in a kernel trace, 7.7 beside the prefetch workgroups (a block per
// row, two passes: 4.8 there, without room for them).
template <int NP>
__global__ __launch_bounds__(64) void layernorm_wave_kernel(const _Float16* __restrict__ x, const _Float16* __restrict__ w,
                                                            const _Float16* __restrict__ b, int n, float eps,
                                                            _Float16* __restrict__ out, int rows, const Prefetch pf) {
  if ((int)blockIdx.x >= rows) {
    prefetch_run(pf, blockIdx.x, rows);
    return;
  }
  const int lane = threadIdx.x, np = n / 8;
  const h8* xr = reinterpret_cast<const h8*>(x + (size_t)blockIdx.x * n);
  h8 v[NP], wv[NP], bv[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = min(lane + 64 * i, np - 1);
    v[i] = xr[p];
    wv[i] = reinterpret_cast<const h8*>(w)[p];
    bv[i] = reinterpret_cast<const h8*>(b)[p];
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (lane + 64 * i < np) {
#pragma unroll
      for (int e = 0; e < 8; ++e) s += h2f(v[i][e]);
    }
  const float mean = wave_sum(s) / (float)n;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (lane + 64 * i < np) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = h2f(v[i][e]) - mean;
        q += d * d;
      }
    }
  const float rstd = 1.0f / sqrtf(wave_sum(q) / (float)n + eps);
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (lane + 64 * i < np) {
      h8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = f2h((h2f(v[i][e]) - mean) * rstd * h2f(wv[i][e]) + h2f(bv[i][e]));
      reinterpret_cast<h8*>(out + (size_t)blockIdx.x * n)[lane + 64 * i] = o;
    }
}

// Attention of one head over T tokens straight from the fused projection qkv [T][3 H hd]: a workgroup
// takes 16 QT query rows, its 4 waves every 4th chunk of 32 keys, and their online softmax states are
// merged through LDS, so one launch of (T / 16 QT) H workgroups (256 for 16 heads of 256 patches) does it.
// HP = 32 NKS >= hd: dims past hd are zeros in registers.  Per chunk: S^T[key][row] = K . q^T on
// 16x16x32 MFMAs with K from global memory in operand order, p = exp(scale s - m) to fp16 in registers,
// O^T[d][row] += V^T . p^T with V transposed through the wave's own LDS (key pairs, 36-half rows).
// Bound by latency: 2 chunks a wave.  Measured with 16 heads of 72, 256 tokens: 6.5 us (7.7 beside the
// prefetch workgroups); before, a launch each to pad the heads (5.1), attend over 4 key slices (8.4),
// combine (4.7) and unpad (4.8).
constexpr int VA_LD = 36;
template <int NKS, int QT>
__global__ __launch_bounds__(256) void vis_attn_kernel(const _Float16* __restrict__ qkv, int T, int H, int hd,
                                                       float scale, _Float16* __restrict__ out, const Prefetch pf) {
  if ((int)blockIdx.y >= H) {
    prefetch_run(pf, blockIdx.y * gridDim.x + blockIdx.x, H * gridDim.x);
    return;
  }
  constexpr int HP = 32 * NKS, NDT = HP / 16;
  constexpr int VB = HP * VA_LD * 2, OB = QT * NDT * 64 * 16;  // bytes per wave: V^T of a chunk, then its O
  __shared__ __attribute__((aligned(16))) char lds[4 * (VB > OB ? VB : OB)];
  __shared__ float ml[4][16 * QT][2];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * 16 * QT, h = blockIdx.y, ld = 3 * H * hd;
  const bool vec = (hd & 7) == 0;
  const _Float16 *q = qkv + h * hd, *k = q + H * hd, *v = k + H * hd;
  auto ld8 = [&](const _Float16* p, int t, int d) __attribute__((always_inline)) -> h8 {
    h8 z = {0, 0, 0, 0, 0, 0, 0, 0};
    const _Float16* a = p + (size_t)min(t, T - 1) * ld + d;
    if (vec) {
      if (d < hd) z = load_global(reinterpret_cast<const h8*>(a));
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (d + e < hd) z[e] = load_global(a + e);
    }
    return z;
  };
  h8 kf[2][NKS], vr[NKS][2];
  auto load = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) kf[kt][ks] = ld8(k, 32 * c + 16 * kt + r, 32 * ks + 8 * g);
#pragma unroll
    for (int i = 0; i < NKS; ++i)  // key pair r, dims 8 (g + 4 i) ..
#pragma unroll
      for (int e = 0; e < 2; ++e) vr[i][e] = ld8(v, 32 * c + 2 * r + e, 8 * (g + 4 * i));
  };
  const int nch = (T + 31) / 32;
  h8 qf[QT][NKS];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt)
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qf[qt][ks] = ld8(q, t0 + 16 * qt + r, 32 * ks + 8 * g);
  if (w < nch) load(w);
  f4 o[QT][NDT];
  float m_run[QT], l_run[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
#pragma unroll
    for (int i = 0; i < NDT; ++i) o[qt][i] = (f4){0.f, 0.f, 0.f, 0.f};
    m_run[qt] = -INFINITY;
    l_run[qt] = 0.f;
  }
  _Float16* vt = reinterpret_cast<_Float16*>(lds + w * (VB > OB ? VB : OB));
  for (int c = w; c < nch; c += 4) {
    f4 s[QT][2];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) s[qt][0] = s[qt][1] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) s[qt][kt] = mfma16x16x32(kf[kt][ks], qf[qt][ks], s[qt][kt]);
#pragma unroll
    for (int i = 0; i < NKS; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const h2 pair = {vr[i][0][e], vr[i][1][e]};
        *reinterpret_cast<h2*>(vt + (8 * (g + 4 * i) + e) * VA_LD + 2 * r) = pair;
      }
    if (c + 4 < nch) load(c + 4);
    float alpha[QT];
    h8 pb[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      float x[8], cmax = -INFINITY;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        x[j] = 32 * c + 16 * (j >> 2) + 4 * g + (j & 3) < T ? s[qt][j >> 2][j & 3] * scale : -INFINITY;
        cmax = fmaxf(cmax, x[j]);
      }
      const float m_new = fmaxf(m_run[qt], xor_max_16_32(cmax));  // finite: the chunk holds a key
      alpha[qt] = exp_hw(m_run[qt] - m_new);
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float e = exp_hw(x[j] - m_new);
        sum += e;
        pb[qt][j] = f2h(e);
      }
      l_run[qt] = l_run[qt] * alpha[qt] + xor_sum_16_32(sum);
      m_run[qt] = m_new;
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // this wave's V^T stores
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < NDT; ++i) {
      const _Float16* vp = vt + (16 * i + r) * VA_LD + 4 * g;
      const h4 a = *reinterpret_cast<const h4*>(vp), b = *reinterpret_cast<const h4*>(vp + 16);
      const h8 av = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) o[qt][i] = mfma16x16x32(av, pb[qt], o[qt][i] * alpha[qt]);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_wave_barrier();
  }
  // merge: every wave's (m, l) and O, then wave w adds up d tiles w, w + 4, ..
  __syncthreads();
  f4* ob = reinterpret_cast<f4*>(lds);
  constexpr int OW = (VB > OB ? VB : OB) / 16;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
#pragma unroll
    for (int i = 0; i < NDT; ++i) ob[w * OW + (qt * NDT + i) * 64 + lane] = o[qt][i];
    if (g == 0) {
      ml[w][16 * qt + r][0] = m_run[qt];
      ml[w][16 * qt + r][1] = l_run[qt];
    }
  }
  __syncthreads();
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int t = t0 + 16 * qt + r;
    if (t >= T) return;
    float m = ml[0][16 * qt + r][0], l = 0.f, wg[4];
#pragma unroll
    for (int i = 1; i < 4; ++i) m = fmaxf(m, ml[i][16 * qt + r][0]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      wg[i] = exp_hw(ml[i][16 * qt + r][0] - m);  // a wave without a chunk: exp(-inf) = 0
      l += wg[i] * ml[i][16 * qt + r][1];
    }
    const float inv = 1.0f / l;
    for (int i = w; i < NDT; i += 4) {
      f4 acc = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) acc += wg[q4] * ob[q4 * OW + (qt * NDT + i) * 64 + lane];
      _Float16* op = out + (size_t)t * H * hd + h * hd + 16 * i + 4 * g;
      h4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = f2h(acc[e] * inv);
      const int d = 16 * i + 4 * g;
      if ((hd & 3) == 0) {
        if (d < hd) *reinterpret_cast<h4*>(op) = y;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < hd) op[e] = y[e];
      }
    }
  }
}

int vis_attn(const _Float16* qkv, int T, int H, int hd, _Float16* out, Prefetch pf, hipStream_t st) {
  // Two row tiles a workgroup halve the reads of K and V, where that still leaves a workgroup per CU.  4
  // layers of 16 heads of 72, us, one / two: 256 patches 265 / 276, 576 patches 419 / 415, 1024 patches
  // 644 / 589, 4096 patches 3738 / 2699.  Past a head dim of 128 a CU holds one workgroup (256 registers and
  // more), so two tiles pay as soon as single ones take a second round: 3 layers of 16 heads of 160 1530 / 1329
  // at 1369 patches, of 4 heads of 256 2186 / 1519 at 4096.
  const long cus = std::max(device_cus(), 1), one = (long)(T + 15) / 16 * H, two = (long)(T + 31) / 32 * H;
  const bool wide = hd <= 128 ? two >= cus : one > cus;
  dim3 grid(wide ? (T + 31) / 32 : (T + 15) / 16, H);
  if (pf.nreg > 0) {  // whole grid rows of prefetch workgroups
    const int rows = (pf.nblocks + (int)grid.x - 1) / (int)grid.x;
    pf.nblocks = rows * (int)grid.x;
    grid.y += rows;
  }
  const float scale = (float)(1.0 / std::sqrt((double)hd));
  switch ((hd + 31) / 32) {
    case 1:
      if (wide) vis_attn_kernel<1, 2><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      else vis_attn_kernel<1, 1><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      break;
    case 2:
      if (wide) vis_attn_kernel<2, 2><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      else vis_attn_kernel<2, 1><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      break;
    case 3:
      if (wide) vis_attn_kernel<3, 2><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      else vis_attn_kernel<3, 1><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      break;
    case 4:
      if (wide) vis_attn_kernel<4, 2><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      else vis_attn_kernel<4, 1><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      break;
    case 5: case 6:
      if (wide) vis_attn_kernel<6, 2><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      else vis_attn_kernel<6, 1><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      break;
    case 7: case 8:
      if (wide) vis_attn_kernel<8, 2><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      else vis_attn_kernel<8, 1><<<grid, 256, 0, st>>>(qkv, T, H, hd, scale, out, pf);
      break;
    default: MLCV_REQUIRE(false, "vision head_dim above 256");
  }
  MLCV_HIP(hipGetLastError());
  return 0;
}

int layernorm(const _Float16* x, const _Float16* w, const _Float16* b, int rows, int n, float eps, _Float16* out,
              const Prefetch& pf, hipStream_t st) {
  const unsigned blocks = rows + (pf.nreg > 0 ? pf.nblocks : 0);
  const uintptr_t p = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(b) |
                      reinterpret_cast<uintptr_t>(out);
  if (n % 8 == 0 && (p & 15) == 0 && n <= 1536) layernorm_wave_kernel<3><<<blocks, 64, 0, st>>>(x, w, b, n, eps, out, rows, pf);
  else if (n % 8 == 0 && (p & 15) == 0 && n <= 4096) layernorm_wave_kernel<8><<<blocks, 64, 0, st>>>(x, w, b, n, eps, out, rows, pf);
  else layernorm_kernel<<<rows, 256, 0, st>>>(x, w, b, n, eps, out);
  MLCV_HIP(hipGetLastError());
  return 0;
}

}  // namespace

size_t vision_ws_bytes(const VisionCfg& v) {
  const int np = (v.image_size / v.patch_size) * (v.image_size / v.patch_size);
  const size_t kp = ((size_t)v.patch_size * v.patch_size * v.num_channels + 7) / 8 * 8;
  const size_t halfs = (size_t)np * kp + (size_t)v.hidden * kp + (size_t)np * v.hidden * 4 +
                       (size_t)np * 3 * v.hidden + (size_t)np * v.inter;
  return halfs * 2 + 512;
}

int embed_image_enqueue(const VisionCfg& v, const _Float16* const* prm, const _Float16* image, _Float16* out,
                        void* ws, size_t ws_bytes, float* gemm_ws, size_t gemm_ws_floats, unsigned* gemm_sync,
                        int gemm_sync_tiles, unsigned* gemm_err, hipStream_t st) {
  MLCV_REQUIRE(v.image_size % v.patch_size == 0 && v.hidden % v.heads == 0, "vision config");
  MLCV_REQUIRE(v.hidden / v.heads <= 256, "vision head_dim above 256");
  MLCV_REQUIRE(v.hidden % 8 == 0 && v.inter % 8 == 0 && v.proj % 4 == 0, "vision widths must be multiples of 8");
  MLCV_REQUIRE(ws_bytes >= vision_ws_bytes(v), "vision workspace too small");
  const int side = v.image_size / v.patch_size, np = side * side, H = v.hidden, hd = H / v.heads;
  const int pdim = v.patch_size * v.patch_size * v.num_channels, kp = (pdim + 7) / 8 * 8;
  _Float16* p = reinterpret_cast<_Float16*>((reinterpret_cast<uintptr_t>(ws) + 255) & ~uintptr_t(255));
  _Float16* patches = p;
  p += (size_t)np * kp;
  _Float16* wpad = p;
  p += (size_t)H * kp;
  _Float16* x = p;
  p += (size_t)np * H;
  _Float16* hn = p;
  p += (size_t)np * H;
  _Float16* ctx = p;
  p += (size_t)np * H;
  _Float16* t = p;
  p += (size_t)np * H;
  _Float16* qkv = p;
  p += (size_t)np * 3 * H;
  _Float16* u = p;
  p += (size_t)np * v.inter;
  auto gemm = [&](const _Float16* a, int lda, const _Float16* b0, const _Float16* b1, const _Float16* b2, int n1,
                  int n2, int ldb, _Float16* c, int ldc, int M, int N, int K) {
    TgArgs g{};
    g.a = a;
    g.lda = lda;
    g.b0 = b0;
    g.b1 = b1;
    g.b2 = b2;
    g.n1 = n1;
    g.n2 = n2;
    g.ldb = ldb;
    g.c = c;
    g.ldc = ldc;
    g.M = M;
    g.N = N;
    g.K = K;
    g.epi = TG_STORE;
    g.ws = gemm_ws;
    g.ws_floats = gemm_ws_floats;
    g.sync = gemm_sync;
    g.sync_tiles = gemm_sync_tiles;
    g.err = gemm_err;
    return tg_launch(g, st);
  };
  auto epi = [&](_Float16* y, int ldy, const _Float16* b, int n, int mode, _Float16* xr, const _Float16* pos) {
    vis_epilogue_kernel<<<np, 256, 0, st>>>(y, ldy, b, n, mode, xr, H, pos, np);
    MLCV_HIP(hipGetLastError());
    return 0;
  };

  // y = epilogue(a . [w0 | w1 | w2]^T + bias): fused on gemm_mid.hip's small tiles where they are the faster
  // ones (and the operands aligned), else the long-M GEMM and a pass
  auto args = [&](const _Float16* a, const _Float16* const* w, const _Float16* const* b, int nseg, int N, int K,
                  _Float16* y, int epi_mode) {
    MidArgs g{};
    g.x = a;
    g.ldx = K;
    g.M = np;
    g.K = K;
    g.N = N;
    g.n1 = nseg > 1 ? N / nseg : N;
    g.n2 = nseg > 1 ? 2 * (N / nseg) : N;
    for (int i = 0; i < 3; ++i) {
      g.w[i] = w[i < nseg ? i : 0];
      g.b[i] = b[i < nseg ? i : 0];
    }
    g.y = y;
    g.ldy = N;
    g.epi = epi_mode;
    g.pos = epi_mode == ME_POS ? prm[2] : nullptr;
    g.npos = np;
    return g;
  };
  auto small = [&](const MidArgs& g) { return mid_ok(g) && mid_worth(g); };
  auto linear = [&](const MidArgs& g) -> int {
    if (small(g)) return mid_gemm_launch(g, st);
    _Float16* dst = g.epi == ME_RESIDUAL ? t : g.y;
    MLCV_TRY(gemm(g.x, g.K, g.w[0], g.w[1], g.w[2], g.n1, g.n2, g.K, dst, g.N, np, g.N, g.K));
    const int ve = g.epi == ME_GELU ? VE_BIAS_GELU : g.epi == ME_RESIDUAL ? VE_BIAS_RESIDUAL
                   : g.epi == ME_POS ? VE_BIAS_POS : VE_BIAS;
    const int nseg = g.n1 < g.N ? 3 : 1;
    for (int s = 0; s < nseg; ++s) MLCV_TRY(epi(dst + s * g.n1, g.N, g.b[s], g.N / nseg, ve, g.y, g.pos));
    return 0;
  };
  // The weights of a linear come from HBM (a tower of 0.8 GB passes through the caches once per image),
  // which its own loads would wait out stage by stage: spare workgroups of the LayerNorm and attention
  // launches before it, which are chains of latencies themselves, have them fetched,
  auto prefetch = [&](std::initializer_list<const MidArgs*> ls, int nblocks) {
    Prefetch pf{};
    for (const MidArgs* g : ls)
      if (small(*g)) mid_prefetch_add(*g, nblocks, pf);
    return pf;
  };
  // or, better, those beside an earlier linear, on the CUs that its own tiles leave idle (64 of 256 at fc1 and
  // fc2 of 256 patches): `next`'s weights beside `g`.
  auto beside = [&](MidArgs& g, const MidArgs& next) {
    const int spare = small(g) ? mid_spare(g) : 0;
    if (spare < MID_PF_MIN) return false;
    g.pf = prefetch({&next}, spare);
    return g.pf.nreg > 0;
  };

  // patch embedding (+ bias) + position embedding
  patchify_kernel<<<np, 256, 0, st>>>(image, v.image_size, v.patch_size, v.num_channels, kp, patches);
  pad_cols_kernel<<<H, 256, 0, st>>>(prm[0], pdim, kp, wpad);
  MLCV_HIP(hipGetLastError());
  const _Float16* wp[1] = {wpad};
  MLCV_TRY(linear(args(patches, wp, prm + 1, 1, H, kp, x, ME_POS)));
  const _Float16* const* tail = prm + 3 + 16 * v.layers;  // post LN w, b; projector w, b
  const MidArgs ap = args(hn, tail + 2, tail + 3, 1, v.proj, H, out, ME_STORE);
  bool ahead = false;  // the next linear after a LayerNorm has its weights on the way
  for (int L = 0; L < v.layers; ++L) {
    const _Float16* const* lp = prm + 3 + 16 * L;  // q w,b  k w,b  v w,b  o w,b  fc1 w,b  fc2 w,b  ln1 w,b  ln2 w,b
    const _Float16 *qw[3] = {lp[0], lp[2], lp[4]}, *qb[3] = {lp[1], lp[3], lp[5]};
    const MidArgs aq = args(hn, qw, qb, 3, 3 * H, H, qkv, ME_STORE), ao = args(ctx, lp + 6, lp + 7, 1, H, H, x, ME_RESIDUAL);
    MidArgs a1 = args(hn, lp + 8, lp + 9, 1, v.inter, H, u, ME_GELU), a2 = args(u, lp + 10, lp + 11, 1, H, v.inter, x, ME_RESIDUAL);
    const bool ahead2 = beside(a1, a2);
    MLCV_TRY(layernorm(x, lp[12], lp[13], np, H, v.eps, hn, ahead ? Prefetch{} : prefetch({&aq}, LN_PF), st));
    MLCV_TRY(linear(aq));
    MLCV_TRY(vis_attn(qkv, np, v.heads, hd, ctx, prefetch({&ao, &a1}, ATTN_PF), st));
    MLCV_TRY(linear(ao));
    MLCV_TRY(layernorm(x, lp[14], lp[15], np, H, v.eps, hn, ahead2 ? Prefetch{} : prefetch({&a2}, LN_PF), st));
    MLCV_TRY(linear(a1));
    if (L + 1 < v.layers) {
      const _Float16 *nw[3] = {lp[16], lp[18], lp[20]}, *nb[3] = {lp[17], lp[19], lp[21]};  // the next layer's q/k/v
      ahead = beside(a2, args(hn, nw, nb, 3, 3 * H, H, qkv, ME_STORE));
    } else {
      ahead = beside(a2, ap);
    }
    MLCV_TRY(linear(a2));
  }
  MLCV_TRY(layernorm(x, tail[0], tail[1], np, H, v.eps, hn, ahead ? Prefetch{} : prefetch({&ap}, LN_PF), st));
  return linear(ap);
}

}  // namespace mlcv
