// The float32 model's linears on the fp32 matrix cores (v_mfma_f32_32x32x2_f32 and 16x16x4: products
// and sums in fp32, 256 flop per clock and CU, about 155 TFLOP/s), with the norm before a linear in
// the same pass (few rows; many rows: a launch before it) and the elementwise work after it in its epilogue.
//
// Two kernels over the same operands and epilogues:
// - f32_tile_kernel: many rows (prefill).  Workgroup tiles of 128 x 128 or 64 x 64, 4 waves in 2 x 2,
//   32 k per stage by buffer -> LDS DMA into two stages.  Bound by the matrix cores: a stage of a 128 x
//   128 tile is 4096 clocks of MFMA per wave against 32 KB of DMA and 16 LDS reads of 16 bytes, so two
//   stages are enough.  A lane reads 4 consecutive k of one row at a time; element i of the four is k
//   index 4 (lane / 32) + i of both operands, so one 16-byte read feeds 4 MFMAs.
// - f32_skinny_kernel: few rows (the suffix, small prefixes) or few outputs.  Bound by the weights and
//   by latency: a workgroup takes 16 weight rows and up to 64 rows of x over the whole K, its 8 waves
//   every 8th block of 32 k, straight from global memory into registers (a lane takes 8 consecutive k
//   of one row: 16 rows x 128 bytes per pair of loads), and sums the waves' products through LDS.
//
// Measured (MI355X; before: 64 x 64 tiles of FMAs with one LDS read per operand element, the norm,
// RoPE, cache, GeGLU and residual passes as launches of their own): the prefix layer at P = 968, width
// 2048, MLP 16384: gate_up 2004 -> 1100 us (118 TFLOP/s), down 1950 -> 560 us, q/k/v + RoPE + cache 560
// -> 116 us; the suffix linears of the 2-layer model (8 rows, width 128) 12 us plus 4.6 us per pass ->
// 2.2 to 5 us in all.  Two layers' prefill 13.08 -> 2.95 ms, the small model's chunk 4.04 -> 0.62 ms (1.87 and
// 0.46 ms with the attention on the matrix cores and the captured chunk).
#include "f32.h"
#include "plan.h"

#include <algorithm>

#pragma clang fp contract(off)

namespace mlcv {

int device_cus();

namespace {

typedef __attribute__((address_space(3))) void* lptr_t;

__device__ __forceinline__ f4 mfma_f32_16(float a, float b, f4 c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
#else
  return c;
#endif
}
__device__ __forceinline__ f16v mfma_f32_32(float a, float b, f16v c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
#else
  return c;
#endif
}
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t r, void* lds, int voff, int soff) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass drops the launch stubs of kernels that use it
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lptr_t)lds, 16, voff, soff, 0, 0);
#endif
}
__device__ __forceinline__ f4 ldg4(const float* p) { return load_global(reinterpret_cast<const f4*>(p)); }

// weight row of logical row n (n in [0, N))
template <int EPI>
__device__ __forceinline__ const float* w_row(const F32Op& a, const float* w0, int n) {
  if constexpr (EPI == FE_GEGLU) {
    const int s = n >> 4, r = n & 15;
    return w0 + (size_t)(r < 8 ? 8 * s + r : a.F + 8 * s + r - 8) * a.K;
  } else if constexpr (EPI == FE_QKV) {
    if (n >= a.nq + a.nkv) return a.w[2] + (size_t)(n - a.nq - a.nkv) * a.K;
    const bool k = n >= a.nq;
    const int nn = k ? n - a.nq : n, s = nn >> 4, r = nn & 15, spb = a.hd >> 4, h = s / spb, j = s % spb;
    return (k ? a.w[1] : a.w[0]) + (size_t)(h * a.hd + 8 * j + (r < 8 ? r : (a.hd >> 1) + r - 8)) * a.K;
  } else {
    return w0 + (size_t)n * a.K;
  }
}

// What an epilogue reads for the quad n .. n + 3 of row m besides the product: FE_STORE u = bias;
// FE_RES u = the old value, v = gate; FE_EULER u = the old value, v = bias; FE_QKV (q, k) u = cos, v = sin
struct EpiIn {
  f4 u, v;
};
template <int EPI>
__device__ __forceinline__ EpiIn epi_in(const F32Op& a, const float* b, const float* out, int m, int n) {
  EpiIn e{};
  if constexpr (EPI == FE_STORE) {
    if (b) e.u = ldg4(b + n);
  } else if constexpr (EPI == FE_RES || EPI == FE_EULER) {
    e.u = load_global(reinterpret_cast<const f4*>(out + (size_t)m * a.ldo + n));
    const float* g = EPI == FE_RES ? a.gate : b;
    if (g) e.v = ldg4(g + n);
  } else if constexpr (EPI == FE_QKV) {
    if (n < a.nq + a.nkv) {
      const int nn = n < a.nq ? n : n - a.nq, d = 8 * ((nn >> 4) % (a.hd >> 4)) + (n & 7), half = a.hd >> 1;
      e.u = ldg4(a.cos + (size_t)m * half + d);
      e.v = ldg4(a.sin + (size_t)m * half + d);
    }
  }
  return e;
}

// 4 consecutive outputs n .. n + 3 of row m, unpaired
template <int EPI>
__device__ __forceinline__ void epi_one(const F32Op& a, const float* b, float* out, int m, int n, f4 v,
                                        const EpiIn& e) {
  if constexpr (EPI == FE_QKV) {  // v
    const int nn = n - a.nq - a.nkv, h = nn / a.hd, d = nn % a.hd;
    *reinterpret_cast<f4*>(a.vo + (size_t)m * a.kv_m + h * a.kv_h + d) = v;
    return;
  }
  if (EPI == FE_STORE || EPI == FE_EULER) {
    if (b) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = v[i] + (EPI == FE_STORE ? e.u[i] : e.v[i]);
    }
  }
  if constexpr (EPI == FE_STORE) {
    if (a.act == 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.0f + expf(-v[i]));
    }
  } else if constexpr (EPI == FE_RES) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float y = a.gate ? v[i] * e.v[i] : v[i];
      v[i] = e.u[i] + y;
    }
  } else if constexpr (EPI == FE_EULER) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float y = a.dt * v[i];
      v[i] = e.u[i] + y;
    }
  }
  *reinterpret_cast<f4*>(out + (size_t)m * a.ldo + n) = v;
}

// outputs n .. n + 3 (the first 8 rows of a slab) and their partners n + 8 .. n + 11 of row m, of the
// paired epilogues (FE_GEGLU, FE_QKV)
template <int EPI>
__device__ __forceinline__ void epi_pair(const F32Op& a, float* out, int m, int n, f4 v, f4 vp, const EpiIn& e) {
  if constexpr (EPI == FE_GEGLU) {
    const float c = 0.7978845608028654f;  // sqrt(2 / pi)
    f4 h;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = v[i];
      const float g = 0.5f * x * (1.0f + tanhf(c * (x + 0.044715f * x * x * x)));
      h[i] = g * vp[i];
    }
    *reinterpret_cast<f4*>(out + (size_t)m * a.ldo + 8 * (n >> 4) + (n & 7)) = h;
  } else {
    if (n >= a.nq + a.nkv) {
      epi_one<EPI>(a, nullptr, out, m, n, v, e);
      epi_one<EPI>(a, nullptr, out, m, n + 8, vp, e);
      return;
    }
    const bool k = n >= a.nq;
    const int nn = k ? n - a.nq : n, s = nn >> 4, spb = a.hd >> 4, h = s / spb, d = 8 * (s % spb) + (n & 7);
    const float scale = k ? 1.0f : a.qscale;
    f4 o1, o2;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o1[i] = (v[i] * e.u[i] - vp[i] * e.v[i]) * scale;
      o2[i] = (vp[i] * e.u[i] + v[i] * e.v[i]) * scale;
    }
    float* o = k ? a.ko + (size_t)m * a.kv_m + h * a.kv_h + d : a.qo + (size_t)m * a.nq + h * a.hd + d;
    *reinterpret_cast<f4*>(o) = o1;
    *reinterpret_cast<f4*>(o + (a.hd >> 1)) = o2;
  }
}
template <int EPI>
constexpr bool epi_paired() { return EPI == FE_GEGLU || EPI == FE_QKV; }

// ---- many rows ---------------------------------------------------------------------------
constexpr int FT_BK = 32;  // k per stage: 128-byte rows in LDS, 8 pieces of 16 bytes
// row r's piece p sits in slot p ^ swz(r): the operand reads of consecutive rows hit distinct banks
__device__ __forceinline__ int ft_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

template <int BM, int BN, int EPI>
__global__ __launch_bounds__(256) void f32_tile_kernel(const F32Op a, int mtiles, int ntiles) {
  constexpr int MBW = BM / 64, NBW = BN / 64;  // 32 x 32 blocks per wave
  constexpr int STG = (BM + BN) * FT_BK * 4;
  constexpr int NAI = BM / 32, NBI = BN / 32;  // DMA instructions (8 rows each) per wave
  __shared__ __attribute__((aligned(16))) char lds[2 * STG];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lh = lane >> 5, wm = w >> 1, wn = w & 1;
  // XCD x (id % 8) owns consecutive tiles, all m tiles of an n tile together: a weight tile is
  // fetched into one L2
  const int id = blockIdx.x, xcd = id & 7, all = mtiles * ntiles, per = (all + 7) >> 3;
  const int tile = xcd * per + (id >> 3);
  if ((id >> 3) >= per || tile >= all) return;
  const int m0 = (tile % mtiles) * BM, n0 = (tile / mtiles) * BN;
  const int lr = lane >> 3, ls = lane & 7;
  constexpr int OOB = 0x7ffffff0;

  // x rows from the tile's first one; rows past M read zeros (the buffer's size)
  const int mrows = min(BM, a.M - m0);
  const __amdgpu_buffer_rsrc_t rA = dev_rsrc(a.x + (size_t)m0 * a.ldx, (uint32_t)((size_t)mrows * a.ldx * 4));
  int aoff[NAI], apc[NAI], bpc[NBI], boff[NBI], bbytes[NBI];
  const float* bbase[NBI];
#pragma unroll
  for (int i = 0; i < NAI; ++i) {
    const int r = (NAI * w + i) * 8 + lr;
    apc[i] = (ls ^ ft_swz(r)) * 4;
    aoff[i] = (r * a.ldx + apc[i]) * 4;
  }
#pragma unroll
  for (int i = 0; i < NBI; ++i) {
    const int r0 = (NBI * w + i) * 8, n = n0 + r0;  // 8 rows of one weight matrix (N % 8 == 0)
    bbase[i] = w_row<EPI>(a, a.w[0], min(n, a.N - 8));
    bbytes[i] = n < a.N ? 8 * a.K * 4 : 0;
    bpc[i] = (ls ^ ft_swz(r0 + lr)) * 4;
    boff[i] = (lr * a.K + bpc[i]) * 4;
  }
  // k past K (K % 8 == 0: a 4-float piece is inside or outside): an offset past the buffer, zeros
  auto dma = [&](int kt, int stage) __attribute__((always_inline)) {
    char* sb = lds + stage * STG;
    const int k0 = kt * FT_BK;
#pragma unroll
    for (int i = 0; i < NAI; ++i)
      lds_dma16(rA, sb + (NAI * w + i) * 1024, k0 + apc[i] < a.K ? aoff[i] : OOB, k0 * 4);
#pragma unroll
    for (int i = 0; i < NBI; ++i)
      lds_dma16(dev_rsrc(bbase[i], (uint32_t)bbytes[i]), sb + BM * 128 + (NBI * w + i) * 1024,
                k0 + bpc[i] < a.K ? boff[i] : OOB, k0 * 4);
  };

  f16v acc[NBW][MBW];
#pragma unroll
  for (int nb = 0; nb < NBW; ++nb)
#pragma unroll
    for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[nb][mb][e] = 0.f;

  const int nkt = (a.K + FT_BK - 1) / FT_BK;
  dma(0, 0);
  for (int kt = 0; kt < nkt; ++kt) {
    // this wave's DMA of stage kt has landed; after the barrier every wave's has, and no wave still
    // reads the other stage
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x70 | 0xF00);  // vmcnt(0)
    __builtin_amdgcn_s_waitcnt(0xC07F);        // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + 1 < nkt) dma(kt + 1, (kt + 1) & 1);
    const char* sa = lds + (kt & 1) * STG;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int p = 2 * s + lh;
      f4 wf[NBW], xf[MBW];
#pragma unroll
      for (int nb = 0; nb < NBW; ++nb) {
        const int r = wn * (BN / 2) + nb * 32 + l32;
        wf[nb] = *reinterpret_cast<const f4*>(sa + BM * 128 + r * 128 + ((p ^ ft_swz(r)) << 4));
      }
#pragma unroll
      for (int mb = 0; mb < MBW; ++mb) {
        const int r = wm * (BM / 2) + mb * 32 + l32;
        xf[mb] = *reinterpret_cast<const f4*>(sa + r * 128 + ((p ^ ft_swz(r)) << 4));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int nb = 0; nb < NBW; ++nb)
#pragma unroll
          for (int mb = 0; mb < MBW; ++mb) acc[nb][mb] = mfma_f32_32(wf[nb][i], xf[mb][i], acc[nb][mb]);
    }
  }

  // lane column m = l32, rows n = 8 (e / 4) + 4 lh + (e % 4): a quad and its partner 8 rows on are
  // elements 8 i .. and 8 i + 4 .. of the same lane
#pragma unroll
  for (int nb = 0; nb < NBW; ++nb)
#pragma unroll
    for (int mb = 0; mb < MBW; ++mb) {
      const int m = m0 + wm * (BM / 2) + mb * 32 + l32;
      if (m >= a.M) continue;
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        const int n = n0 + wn * (BN / 2) + nb * 32 + 8 * q + 4 * lh;
        if (n >= a.N) continue;
        const f16v& v = acc[nb][mb];
        const f4 v0 = {v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
        const f4 v1 = {v[4 * q + 4], v[4 * q + 5], v[4 * q + 6], v[4 * q + 7]};
        if constexpr (epi_paired<EPI>()) {
          epi_pair<EPI>(a, a.out, m, n, v0, v1, epi_in<EPI>(a, a.b, a.out, m, n));
        } else {
          epi_one<EPI>(a, a.b, a.out, m, n, v0, epi_in<EPI>(a, a.b, a.out, m, n));
          if (n + 8 < a.N) epi_one<EPI>(a, a.b, a.out, m, n + 8, v1, epi_in<EPI>(a, a.b, a.out, m, n + 8));
        }
      }
    }
}

// ---- few rows ------------------------------------------------------------------------------
constexpr int FS_NW = 8;  // waves: each takes every 8th block of 32 k

// NORM: 0 none, 1 RMSNorm, 2 adaRMS of the rows, in one pass over x: the product takes x (1 + scale),
// the rows' sums of squares are added up on the way, and y = product / sqrt(mean(x^2) + eps) + shift . w.
// A launch is a chain of memory latencies, so everything it reads goes out before the first wait: the
// first blocks of the weights and of x, then what the epilogue reads.
// w0, b, out: the operation's own, or those of one linear of a table.
template <int MT, int NORM, int EPI>
__device__ __forceinline__ void f32_skinny(const F32Op& a, const float* w0, const float* b, float* out) {
  __shared__ f4 red[FS_NW * MT * 64];
  __shared__ float ssq[NORM != 0 ? FS_NW * MT * 16 : 1];  // sums of squares [wave][row]
  __shared__ float shw[NORM == 2 ? FS_NW * 16 : 1];       // shift . w [wave][weight row]
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.y * 16 * MT, K = a.K;
  const float* wr = w_row<EPI>(a, w0, min(16 * (int)blockIdx.x + r, a.N - 1));
  const float* xr[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) xr[mt] = a.x + (size_t)min(m0 + 16 * mt + r, a.M - 1) * a.ldx;
  struct Blk {
    f4 w[2], x[MT][2], sc[2], sh[2];
  };
  // block c of 32 k: this lane's 8 k at 32 c + 8 g (K % 8 == 0: wholly inside or past K, then zeros)
  auto load = [&](int c, Blk& t) __attribute__((always_inline)) {
    const int k = 32 * c + 8 * g;
    const bool in = k < K;
    const int kc = in ? k : 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      t.w[i] = ldg4(wr + kc + 4 * i);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) t.x[mt][i] = ldg4(xr[mt] + kc + 4 * i);
      if constexpr (NORM == 1) t.sc[i] = ldg4(a.nw + kc + 4 * i);
      if constexpr (NORM == 2) {
        t.sc[i] = ldg4(a.mod + kc + 4 * i);
        t.sh[i] = ldg4(a.mod + K + kc + 4 * i);
      }
    }
    if (!in) {
      t.w[0] = t.w[1] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) t.x[mt][0] = t.x[mt][1] = (f4){0.f, 0.f, 0.f, 0.f};
    }
  };
  f4 acc[MT];
  float ss[MT], sw = 0.f;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    acc[mt] = (f4){0.f, 0.f, 0.f, 0.f};
    ss[mt] = 0.f;
  }
  auto mul = [&](const Blk& t) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        f4 x = t.x[mt][i];
        if constexpr (NORM != 0) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            ss[mt] = fmaf(x[e], x[e], ss[mt]);
            x[e] = x[e] * (1.0f + t.sc[i][e]);
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[mt] = mfma_f32_16(t.w[i][e], x[e], acc[mt]);
      }
      if constexpr (NORM == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) sw = fmaf(t.w[i][e], t.sh[i][e], sw);
      }
    }
  };
  const int nc = (K + 31) / 32;
  Blk t0, t1;
  int c = w;
  if (c < nc) load(c, t0);
  if (c + FS_NW < nc) load(c + FS_NW, t1);
  // waves 0 .. MT - 1 write the m tiles: lane's rows n = 4 g .. + 3 of column m = r
  const int m = m0 + 16 * w + r, n = 16 * blockIdx.x + 4 * g;
  const bool mine = w < MT && m < a.M && n < a.N && !(epi_paired<EPI>() && g >= 2);
  EpiIn ein{};
  if (mine) ein = epi_in<EPI>(a, b, out, m, n);
  while (c < nc) {  // two blocks in flight
    mul(t0);
    if (c + 2 * FS_NW < nc) load(c + 2 * FS_NW, t0);
    c += FS_NW;
    if (c >= nc) break;
    mul(t1);
    if (c + 2 * FS_NW < nc) load(c + 2 * FS_NW, t1);
    c += FS_NW;
  }
  // the waves' products, summed in wave order
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    red[(w * MT + mt) * 64 + lane] = acc[mt];
    if constexpr (NORM != 0) {
      const float s = xor_sum_16_32(ss[mt]);
      if (g == 0) ssq[(w * MT + mt) * 16 + r] = s;
    }
  }
  if constexpr (NORM == 2) {
    const float s = xor_sum_16_32(sw);
    if (g == 0) shw[w * 16 + r] = s;
  }
  __syncthreads();
  if (w >= MT) return;
  f4 v = red[w * 64 + lane];
#pragma unroll
  for (int q = 1; q < FS_NW; ++q) {
    const f4 u = red[(q * MT + w) * 64 + lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = v[i] + u[i];
  }
  if constexpr (NORM != 0) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < FS_NW; ++q) s = s + ssq[(q * MT + w) * 16 + r];
    const float den = sqrtf(s / (float)K + a.eps);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = v[i] / den;
      if constexpr (NORM == 2) {
        float sh = 0.f;
#pragma unroll
        for (int q = 0; q < FS_NW; ++q) sh = sh + shw[q * 16 + 4 * g + i];
        v[i] = v[i] + sh;
      }
    }
  }
  if constexpr (epi_paired<EPI>()) {
    f4 vp;
#pragma unroll
    for (int i = 0; i < 4; ++i) vp[i] = __shfl_xor(v[i], 32);  // rows 8 on
    if (mine) epi_pair<EPI>(a, out, m, n, v, vp, ein);
  } else {
    if (mine) epi_one<EPI>(a, b, out, m, n, v, ein);
  }
}

template <int MT, int NORM, int EPI>
__global__ __launch_bounds__(64 * FS_NW) void f32_skinny_kernel(const F32Op a) {
  f32_skinny<MT, NORM, EPI>(a, a.w[0], a.b, a.out);
}

// The linears of a table, grid z.  The pointers are kernel arguments, as every other launch's: a launch
// that a caller has captured keeps the weights it was captured with.
constexpr int FS_TAB = 64;  // linears per launch
struct F32Tabs {
  F32Tab t[FS_TAB];
};
template <int MT>
__global__ __launch_bounds__(64 * FS_NW) void f32_skinny_tab_kernel(const F32Op a, const F32Tabs tabs) {
  const int z = blockIdx.z;
  f32_skinny<MT, 0, FE_STORE>(a, tabs.t[z].w, tabs.t[z].b, a.out + z * a.tab_stride);
}

// one row per workgroup: xn = x / sqrt(mean(x^2) + eps), then * (1 + w) or * (1 + mod) + mod[K + ..]
__global__ __launch_bounds__(256) void f32_rows_norm_kernel(const float* __restrict__ x, int ldx, int K,
                                                            const float* __restrict__ nw,
                                                            const float* __restrict__ mod, float eps,
                                                            float* __restrict__ out) {
  __shared__ float red[4];
  const float* xr = x + (size_t)blockIdx.x * ldx;
  float ss = 0.f;
  for (int k = 4 * threadIdx.x; k < K; k += 1024) {
    const f4 v = ldg4(xr + k);
#pragma unroll
    for (int i = 0; i < 4; ++i) ss = ss + v[i] * v[i];
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float dn = sqrtf((((red[0] + red[1]) + red[2]) + red[3]) / (float)K + eps);
  float* o = out + (size_t)blockIdx.x * K;
  for (int k = 4 * threadIdx.x; k < K; k += 1024) {
    const f4 v = ldg4(xr + k), sc = ldg4((nw ? nw : mod) + k);
    f4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float xn = v[i] / dn;
      y[i] = xn * (1.0f + sc[i]);
    }
    if (!nw) {
      const f4 sh = ldg4(mod + K + k);
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = y[i] + sh[i];
    }
    *reinterpret_cast<f4*>(o + k) = y;
  }
}

template <int EPI>
int tile_launch(const F32Op& a, int bm, hipStream_t st) {
  const int mt = (a.M + bm - 1) / bm, nt = (a.N + bm - 1) / bm;
  const unsigned blocks = (unsigned)((mt * nt + 7) / 8 * 8);
  if (bm == 128) f32_tile_kernel<128, 128, EPI><<<blocks, 256, 0, st>>>(a, mt, nt);
  else f32_tile_kernel<64, 64, EPI><<<blocks, 256, 0, st>>>(a, mt, nt);
  MLCV_HIP(hipGetLastError());
  return 0;
}

template <int NORM, int EPI>
int skinny_launch(const F32Op& a, int mt, hipStream_t st) {
  const dim3 grid((a.N + 15) / 16, (a.M + 16 * mt - 1) / (16 * mt));
  if (mt == 1) f32_skinny_kernel<1, NORM, EPI><<<grid, 64 * FS_NW, 0, st>>>(a);
  else if (mt == 2) f32_skinny_kernel<2, NORM, EPI><<<grid, 64 * FS_NW, 0, st>>>(a);
  else f32_skinny_kernel<4, NORM, EPI><<<grid, 64 * FS_NW, 0, st>>>(a);
  MLCV_HIP(hipGetLastError());
  return 0;
}

int tab_launch(const F32Op& in, int mt, hipStream_t st) {
  for (int i = 0; i < in.ntab; i += FS_TAB) {
    F32Op a = in;
    F32Tabs tabs{};
    const int n = std::min(FS_TAB, in.ntab - i);
    std::copy(in.tab + i, in.tab + i + n, tabs.t);
    a.out = in.out + i * in.tab_stride;
    a.tab = nullptr;  // the host's
    const dim3 grid((a.N + 15) / 16, (a.M + 16 * mt - 1) / (16 * mt), n);
    if (mt == 1) f32_skinny_tab_kernel<1><<<grid, 64 * FS_NW, 0, st>>>(a, tabs);
    else if (mt == 2) f32_skinny_tab_kernel<2><<<grid, 64 * FS_NW, 0, st>>>(a, tabs);
    else f32_skinny_tab_kernel<4><<<grid, 64 * FS_NW, 0, st>>>(a, tabs);
    MLCV_HIP(hipGetLastError());
  }
  return 0;
}

}  // namespace

int f32_gemm_launch(const F32Op& in, hipStream_t st) {
  F32Op a = in;
  MLCV_REQUIRE(a.x && a.M > 0 && a.K > 0 && a.N > 0 && a.K % 8 == 0 && a.N % 8 == 0 && a.ldx % 4 == 0,
               "float32 linear: shape");
  MLCV_REQUIRE(!a.tab || (a.ntab > 0 && a.epi == FE_STORE && !a.nw && !a.mod), "float32 linear: table");
  const int cus = std::max(device_cus(), 1);
  const int bm = f32_tile(a.M, a.N, a.tab != nullptr, cus);
  int norm = a.nw ? 1 : a.mod ? 2 : 0;
  const bool fuse = bm == 0;  // in the skinny kernel's one pass; a launch before the tiles
  if (norm != 0 && !fuse) {
    MLCV_REQUIRE(a.xn, "float32 linear: no room for the normalised rows");
    f32_rows_norm_kernel<<<a.M, 256, 0, st>>>(a.x, a.ldx, a.K, a.nw, a.mod, a.eps, a.xn);
    MLCV_HIP(hipGetLastError());
    a.x = a.xn;
    a.ldx = a.K;
    norm = 0;
  }
  if (bm) {
    switch (a.epi) {
      case FE_STORE: return tile_launch<FE_STORE>(a, bm, st);
      case FE_QKV: return tile_launch<FE_QKV>(a, bm, st);
      case FE_RES: return tile_launch<FE_RES>(a, bm, st);
      case FE_GEGLU: return tile_launch<FE_GEGLU>(a, bm, st);
      case FE_EULER: return tile_launch<FE_EULER>(a, bm, st);
      default: MLCV_REQUIRE(false, "float32 linear: epilogue");
    }
  }
  // m tiles of 16 rows per workgroup: up to 4, fewer while the grid would leave CUs idle
  int mt = a.M <= 16 ? 1 : a.M <= 32 ? 2 : 4;
  while (mt > 1 && (long)((a.N + 15) / 16) * ((a.M + 16 * mt - 1) / (16 * mt)) < cus) mt >>= 1;
  if (a.tab) return tab_launch(a, mt, st);
  switch (a.epi) {
    // the pairs of norm and epilogue that the model has
    case FE_STORE:
      if (norm == 0) return skinny_launch<0, FE_STORE>(a, mt, st);
      if (norm == 2) return skinny_launch<2, FE_STORE>(a, mt, st);
      break;
    case FE_QKV:
      if (norm == 1) return skinny_launch<1, FE_QKV>(a, mt, st);
      if (norm == 2) return skinny_launch<2, FE_QKV>(a, mt, st);
      break;
    case FE_RES:
      if (norm == 0) return skinny_launch<0, FE_RES>(a, mt, st);
      break;
    case FE_GEGLU:
      if (norm == 1) return skinny_launch<1, FE_GEGLU>(a, mt, st);
      if (norm == 2) return skinny_launch<2, FE_GEGLU>(a, mt, st);
      break;
    case FE_EULER:
      if (norm == 2) return skinny_launch<2, FE_EULER>(a, mt, st);
      break;
  }
  MLCV_REQUIRE(false, "float32 linear: norm and epilogue");
}

}  // namespace mlcv
