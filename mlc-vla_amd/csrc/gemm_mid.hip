// fp16 linears over a few hundred rows (an image's patches, short prefixes): y = x . w^T on
// v_mfma_f32_32x32x16_f16 with the bias, GELU, residual or position add in the epilogue.
//
// At these sizes a launch is bound by how fast a CU's operand tiles come out of the L2 (about 45 bytes
// per clock and CU, also into LDS), by the latency of the first ones and by LDS reads, not by the matrix
// cores.  So:
// - the tile is the one of the four below with the least operand rows per CU (mid_plan), and K is never
//   split over workgroups;
// - the waves of a workgroup share out K, 64 k at a time, and each multiplies the whole tile: a wave
//   moves its own k into its own LDS ring (buffer -> LDS DMA, row-major rows to MFMA operand order) and
//   reads every byte once, so there is no barrier in the loop and half to a quarter of the LDS reads of
//   waves that own a block each (which were half of such a loop's time).  The waves' sums meet in LDS;
// - what the epilogue reads, and in the launches before the weights themselves (mid_prefetch_add), goes
//   out first.
// Measured (256 rows, the image tower's layer; kernel times with the weights in the caches, us; before:
// 128 x 128 tiles over 3 K slices that met in the kernel, then an epilogue launch of 3 to 5 us per
// matrix): q/k/v 1152 -> 3456 in 8.8 (16.8 + 3 x 4.7), out_proj 1152 -> 1152 in 6.4 (14.2 + 4.7), fc1
// 1152 -> 4304 in 11.8 (20.1 + 4.7), fc2 4304 -> 1152 in 14.9 (20.1 + 4.7).  Tried at these sizes: 16 waves
// that own 32 x 32 blocks of a shared ring (fc1 10.6, out_proj 7.5, the tower 1718 us against 1714),
// K split over 4 waves of a 128 x 64 tile 2 (fc1 17.1), operands through registers instead of DMA (the
// tower 2022), each workgroup prefetching its own weights first (1893 against 1826 then).
#include "kernels.h"

#include <algorithm>

namespace mlcv {

namespace {

typedef __attribute__((address_space(3))) void* lptr_t;

__device__ __forceinline__ void mid_dma16(__amdgpu_buffer_rsrc_t r, void* lds, int voff, int soff) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass drops the launch stubs of kernels that use it
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lptr_t)lds, 16, voff, soff, 0, 0);
#endif
}
template <int N>
__device__ __forceinline__ void mid_vm_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x70 | 0xF00);
  asm volatile("" ::: "memory");
}
// A stage holds 64 k of the tile's rows, 128 bytes each; row r's 16-byte piece p sits in slot p ^
// swz(r), so the MFMA operand reads of consecutive rows hit distinct banks (on 32 and on 64)
__device__ __forceinline__ int mid_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

template <int BM, int BN, int NW, int NST, int EPI>
__global__ __launch_bounds__(64 * NW) void mid_gemm_kernel(const MidArgs a, int mtiles, int ntiles) {
  constexpr int MB = BM / 32, NB = BN / 32, NBLK = MB * NB;      // 32 x 32 blocks
  constexpr int STG = (BM + BN) * 128, NI = (BM + BN) / 8;       // DMA instructions (8 rows) per stage
  constexpr int NQ = NBLK * 4 / NW;                              // epilogue quads (4 n of 64 lanes) per wave
  static_assert(NQ * NW == NBLK * 4 && NW * NST * STG <= 160 * 1024 && NBLK * 4096 <= NST * STG, "LDS");
  static_assert((NST - 1) * NI < 64, "vmcnt range");
  __shared__ __attribute__((aligned(16))) char lds[NW * NST * STG];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  // n tile j runs on XCD j % 8 (workgroups are dealt to the XCDs round-robin by id), all its m tiles:
  // a weight tile is fetched into one L2, and an earlier launch can have it fetched there
  const int tiles = (ntiles + 7) / 8 * 8 * mtiles;
  if ((int)blockIdx.x >= tiles) {
    prefetch_run(a.pf, blockIdx.x, tiles);
    return;
  }
  const int j8 = blockIdx.x >> 3, tn = (blockIdx.x & 7) + 8 * (j8 / mtiles);
  if (tn >= ntiles) return;
  const int m0 = (j8 % mtiles) * BM, n0 = tn * BN;
  const int lr = lane >> 3, ls = lane & 7;
  constexpr int OOB = 0x7ffffff0;

  // plain selects: an indexed read of the argument arrays becomes a memory load per use
  const _Float16 *w0 = a.w[0], *w1 = a.w[1], *w2 = a.w[2], *b0 = a.b[0], *b1 = a.b[1], *b2 = a.b[2];
  const int n1 = a.n1, n2 = a.n2;
  // what the epilogue reads, from clamped addresses without branches (a join would wait for them):
  // quad (block, q) holds rows n = 32 nb + 8 q + 4 lh .. + 3 of column m = 32 mb + l32
  auto quad = [&](int i, int& m, int& n) __attribute__((always_inline)) {
    const int u = w + NW * i, blk = u >> 2;
    m = m0 + 32 * (blk % MB) + l32;
    n = n0 + 32 * (blk / MB) + 8 * (u & 3) + 4 * lh;
  };
  h4 bv[NQ], rv[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    int m, n;
    quad(i, m, n);
    m = min(m, a.M - 1);
    n = min(n, a.N - 4);
    const _Float16* b = n < n1 ? b0 : n < n2 ? b1 : b2;
    const _Float16* any = n < n1 ? w0 : n < n2 ? w1 : w2;  // no bias: some valid halfs, not used
    bv[i] = load_global(reinterpret_cast<const h4*>((b ? b : any) + n - (n < n1 ? 0 : n < n2 ? n1 : n2)));
    if constexpr (EPI == ME_RESIDUAL) rv[i] = load_global(reinterpret_cast<const h4*>(a.y + (size_t)m * a.ldy + n));
    if constexpr (EPI == ME_POS) rv[i] = load_global(reinterpret_cast<const h4*>(a.pos + (size_t)(m % a.npos) * a.N + n));
  }
  // rows past M and N read zeros (the buffers' sizes); 8 rows of weights are of one matrix
  const __amdgpu_buffer_rsrc_t rx =
      dev_rsrc(a.x + (size_t)m0 * a.ldx, (uint32_t)(((size_t)(min(BM, a.M - m0) - 1) * a.ldx + a.K) * 2));
  __amdgpu_buffer_rsrc_t rw[BN / 8];
#pragma unroll
  for (int i = 0; i < BN / 8; ++i) {
    const int n = n0 + 8 * i, rows = min(8, (n < n1 ? n1 : n < n2 ? n2 : a.N) - n);
    rw[i] = dev_rsrc((n < n1 ? w0 : n < n2 ? w1 : w2) + (size_t)(n < a.N ? n - (n < n1 ? 0 : n < n2 ? n1 : n2) : 0) * a.K,
                     rows > 0 ? (uint32_t)(rows * a.K * 2) : 0u);
  }
  // k past K (K % 8 == 0: a piece is inside or outside) and stages past the last: offsets past the
  // buffer, zeros; every stage issues its NI instructions, so the waits are constants.  The swizzle of
  // row 8 i + lr is (lr, i & 1).
  char* ring = lds + w * NST * STG;
  const int pe = ls ^ lr, po = pe ^ 1;  // this lane's piece in even and odd groups of 8 rows
  auto dma = [&](int kt, int stage) __attribute__((always_inline)) {
    const bool ine = kt * 64 + pe * 8 < a.K, ino = kt * 64 + po * 8 < a.K;
#pragma unroll
    for (int i = 0; i < BM / 8; ++i) {
      const int off = ((8 * i + lr) * a.ldx + ((i & 1) ? po : pe) * 8) * 2;
      mid_dma16(rx, ring + stage * STG + i * 1024, ((i & 1) ? ino : ine) ? off : OOB, kt * 128);
    }
#pragma unroll
    for (int i = 0; i < BN / 8; ++i) {
      const int off = (lr * a.K + ((i & 1) ? po : pe) * 8) * 2;
      mid_dma16(rw[i], ring + stage * STG + (BM / 8 + i) * 1024, ((i & 1) ? ino : ine) ? off : OOB, kt * 128);
    }
  };
  f16v acc[NB][MB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[nb][mb][e] = 0.f;
  const int nkt = (a.K + 63) / 64;
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < NST - 1; ++t) dma(w + t * NW, t);
  const int swz = mid_swz(l32);
  int st = 0;
  for (int kt = w; kt < nkt; kt += NW) {
    // the next stage's DMA goes into the stage read last (its reads have returned), then this one's
    // has landed once at most the NST - 1 stages after it are in flight
    const int sn = st == 0 ? NST - 1 : st - 1;
    dma(kt + (NST - 1) * NW, sn);
    mid_vm_wait<(NST - 1) * NI>();
    __builtin_amdgcn_sched_barrier(0);
    const char* sb = ring + st * STG;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int p = ((2 * ks + lh) ^ swz) << 4;
      h8 wf[NB], xf[MB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) wf[nb] = *reinterpret_cast<const h8*>(sb + (BM + 32 * nb + l32) * 128 + p);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) xf[mb] = *reinterpret_cast<const h8*>(sb + (32 * mb + l32) * 128 + p);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = mfma32x32x16(wf[nb], xf[mb], acc[nb][mb]);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_sched_barrier(0);
    st = st + 1 == NST ? 0 : st + 1;
  }
  mid_vm_wait<0>();  // the zero-filling DMA past the K range
  // the waves' sums through their own rings: [block][q][lane] f4, added in wave order
  f4* mine = reinterpret_cast<f4*>(ring);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f16v& v = acc[nb][mb];
        mine[((nb * MB + mb) * 4 + q) * 64 + lane] = (f4){v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
      }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    int m, n;
    quad(i, m, n);
    f4 v = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < NW; ++g) {
      const f4 u = reinterpret_cast<const f4*>(lds + g * NST * STG)[(w + NW * i) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += u[e];
    }
    if (m >= a.M || n >= a.N) continue;
    const bool has_b = (n < n1 ? b0 : n < n2 ? b1 : b2) != nullptr;
    h4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      _Float16 t = f2h(v[e]);
      if (has_b) t = hadd(t, bv[i][e]);
      if constexpr (EPI == ME_GELU) t = f2h(gelu_tanh_hw(h2f(t)));
      if constexpr (EPI == ME_RESIDUAL || EPI == ME_POS) t = hadd(rv[i][e], t);
      y[e] = t;
    }
    *reinterpret_cast<h4*>(a.y + (size_t)m * a.ldy + n) = y;
  }
}

template <int BM, int BN, int NW, int NST>
int launch(const MidArgs& a, hipStream_t st) {
  const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN;
  const unsigned blocks = (unsigned)((nt + 7) / 8 * 8 * mt + (a.pf.nreg > 0 ? a.pf.nblocks : 0));
  switch (a.epi) {
    case ME_STORE: mid_gemm_kernel<BM, BN, NW, NST, ME_STORE><<<blocks, 64 * NW, 0, st>>>(a, mt, nt); break;
    case ME_GELU: mid_gemm_kernel<BM, BN, NW, NST, ME_GELU><<<blocks, 64 * NW, 0, st>>>(a, mt, nt); break;
    case ME_RESIDUAL: mid_gemm_kernel<BM, BN, NW, NST, ME_RESIDUAL><<<blocks, 64 * NW, 0, st>>>(a, mt, nt); break;
    case ME_POS: mid_gemm_kernel<BM, BN, NW, NST, ME_POS><<<blocks, 64 * NW, 0, st>>>(a, mt, nt); break;
    default: MLCV_REQUIRE(false, "linear epilogue");
  }
  MLCV_HIP(hipGetLastError());
  return 0;
}

// ---- linears of few rows or short K (fp16 or q4f16_1 weights) ----------------------------------
// A call of this size is a chain of latencies: the skinny kernel stages x through LDS between two barriers
// and its K slices meet at a counter in memory.  Here a workgroup owns 32 outputs of up to 64 rows over the
// whole K.  Its waves share out K 64 k at a time, operands straight from global memory into registers (a
// lane takes the same 32 k of a weight row and of an x row, so a q4 lane's 16 bytes are one group with one
// scale), two chunks in flight, and the waves' sums meet in LDS, the only barrier.  x is read once per 32
// outputs, in 16-byte pieces of 32 rows, which bounds it from K of one to four thousand on.
// Measured (one launch after another, us; before: the skinny kernel): q4 50 x 1024 x 8192 8.8 -> 6.9,
// 1 x 1024 x 8192 8.5 -> 4.1, fp16 32 x 256 x 1024 4.8 -> 2.8, 2 x 672 x 5344 13.0 -> 3.1.
template <bool Q4, int MBK>
struct LrChunk {
  h8 x[MBK][4];
  h8 w[Q4 ? 1 : 4];
  u4 q;
  _Float16 s;
};
template <bool Q4, int MBK, int NW>
__global__ __launch_bounds__(64 * NW) void lin_rows_kernel(const _Float16* __restrict__ x, int M, int K,
                                                           const _Float16* __restrict__ w,
                                                           const uint32_t* __restrict__ qw,
                                                           const _Float16* __restrict__ qs,
                                                           const _Float16* __restrict__ bias,
                                                           _Float16* __restrict__ y, int N) {
  __shared__ f4 red[NW][MBK * 4][64];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  const int n0 = blockIdx.x * 32, m0 = blockIdx.y * (32 * MBK);
  const size_t wrow = (size_t)min(n0 + l32, N - 1);
  const _Float16* xr[MBK];
#pragma unroll
  for (int mb = 0; mb < MBK; ++mb) xr[mb] = x + (size_t)min(m0 + 32 * mb + l32, M - 1) * K;
  const int nch = (K + 63) / 64;
  // q4: two neighbouring chunks a wave, whole 64-byte pieces of a row
  const bool pair = Q4 && nch > NW;
  auto chunk = [&](int i) __attribute__((always_inline)) {
    return pair ? 2 * wv + (i & 1) + 2 * NW * (i >> 1) : wv + NW * i;
  };
  auto load = [&](LrChunk<Q4, MBK>& c, int kc) __attribute__((always_inline)) {
    const int kb = min(64 * kc + 32 * lh, K - 32);
    if constexpr (Q4) {
      c.q = load_global(reinterpret_cast<const u4*>(qw + wrow * (K / 8) + kb / 8));
      c.s = load_global(qs + wrow * (K / 32) + kb / 32);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) c.w[j] = load_global(reinterpret_cast<const h8*>(w + wrow * K + kb + 8 * j));
    }
#pragma unroll
    for (int mb = 0; mb < MBK; ++mb)
#pragma unroll
      for (int j = 0; j < 4; ++j) c.x[mb][j] = load_global(reinterpret_cast<const h8*>(xr[mb] + kb + 8 * j));
  };
  f16v acc[MBK];
#pragma unroll
  for (int mb = 0; mb < MBK; ++mb)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[mb][e] = 0.f;
  auto product = [&](LrChunk<Q4, MBK>& c, int kc) __attribute__((always_inline)) {
    const h8 z = {0, 0, 0, 0, 0, 0, 0, 0};
    const bool in = 64 * kc + 32 * lh < K;  // K % 32 == 0: a lane's k are all inside or all outside
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      h8 a;
      if constexpr (Q4) {
        const h8 v = dequant_word(c.q[j], c.s);
        a = (h8){v[0], v[2], v[4], v[6], v[1], v[3], v[5], v[7]};
      } else {
        a = c.w[j];
      }
      a = in ? a : z;
#pragma unroll
      for (int mb = 0; mb < MBK; ++mb) acc[mb] = mfma32x32x16(a, in ? c.x[mb][j] : z, acc[mb]);
    }
  };
  LrChunk<Q4, MBK> c0, c1;
  if (chunk(0) < nch) load(c0, chunk(0));
  if (chunk(1) < nch) load(c1, chunk(1));
  for (int i = 0; chunk(i) < nch; i += 2) {
    product(c0, chunk(i));
    if (chunk(i + 2) < nch) load(c0, chunk(i + 2));
    if (chunk(i + 1) < nch) {
      product(c1, chunk(i + 1));
      if (chunk(i + 3) < nch) load(c1, chunk(i + 3));
    }
  }
#pragma unroll
  for (int mb = 0; mb < MBK; ++mb)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f16v& v = acc[mb];
      red[wv][4 * mb + q][lane] = (f4){v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
    }
  __syncthreads();
  for (int u = wv; u < 4 * MBK; u += NW) {  // quad u: outputs n .. n + 3 of row m, added in wave order
    const int m = m0 + 32 * (u >> 2) + l32, n = n0 + 8 * (u & 3) + 4 * lh;
    h4 bv = {0, 0, 0, 0};
    if (bias) bv = load_global(reinterpret_cast<const h4*>(bias + min(n, N - 4)));
    f4 v = red[0][u][lane];
#pragma unroll
    for (int g = 1; g < NW; ++g) v += red[g][u][lane];
    if (m >= M || n >= N) continue;
    h4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = f2h(v[e]);
      if (bias) o[e] = hadd(o[e], bv[e]);
    }
    *reinterpret_cast<h4*>(y + (size_t)m * N + n) = o;
  }
}

template <bool Q4>
int lin_rows_q(const LinRows& a, hipStream_t st) {
  const bool one = a.M <= 32, deep = a.K > 512;
  const dim3 grid((a.N + 31) / 32, one ? 1 : (a.M + 63) / 64);
  if (one && deep) lin_rows_kernel<Q4, 1, 8><<<grid, 512, 0, st>>>(a.x, a.M, a.K, a.w, a.qw, a.qs, a.b, a.y, a.N);
  else if (one) lin_rows_kernel<Q4, 1, 4><<<grid, 256, 0, st>>>(a.x, a.M, a.K, a.w, a.qw, a.qs, a.b, a.y, a.N);
  else if (deep) lin_rows_kernel<Q4, 2, 8><<<grid, 512, 0, st>>>(a.x, a.M, a.K, a.w, a.qw, a.qs, a.b, a.y, a.N);
  else lin_rows_kernel<Q4, 2, 4><<<grid, 256, 0, st>>>(a.x, a.M, a.K, a.w, a.qw, a.qs, a.b, a.y, a.N);
  MLCV_HIP(hipGetLastError());
  return 0;
}

}  // namespace

// pieces of 16 bytes, quads of outputs, the grid
bool lin_rows_ok(const LinRows& a) {
  const uintptr_t p = reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.w) | reinterpret_cast<uintptr_t>(a.qw);
  const uintptr_t p8 = reinterpret_cast<uintptr_t>(a.y) | reinterpret_cast<uintptr_t>(a.b);
  return a.M > 0 && a.N > 0 && a.K > 0 && a.K % 32 == 0 && a.N % 4 == 0 && (p & 15) == 0 && (p8 & 7) == 0 &&
         (reinterpret_cast<uintptr_t>(a.qs) & 1) == 0 && (a.M + 63) / 64 <= 65535;
}

int lin_rows_launch(const LinRows& a, hipStream_t st) {
  MLCV_REQUIRE(lin_rows_ok(a), "linear: shape or alignment");
  return a.qw ? lin_rows_q<true>(a, st) : lin_rows_q<false>(a, st);
}

// rows of 16 bytes for the DMA, quads of outputs; the last two lines: the grid, and buffers' offsets in 32 bits
bool mid_ok(const MidArgs& a) {
  uintptr_t p = reinterpret_cast<uintptr_t>(a.x);
  for (int s = 0; s < 3; ++s) p |= reinterpret_cast<uintptr_t>(a.w[s]);
  uintptr_t p8 = reinterpret_cast<uintptr_t>(a.y) | reinterpret_cast<uintptr_t>(a.pos);
  for (int s = 0; s < 3; ++s) p8 |= reinterpret_cast<uintptr_t>(a.b[s]);
  return a.M > 0 && a.N > 0 && a.K > 0 && a.K % 8 == 0 && a.ldx % 8 == 0 && a.ldy % 4 == 0 && a.N % 4 == 0 &&
         (a.n1 % 8 == 0 || a.n1 >= a.N) && (a.n2 % 8 == 0 || a.n2 >= a.N) && (p & 15) == 0 && (p8 & 7) == 0 &&
         (size_t)((a.N + 31) / 32 + 7) * ((a.M + 31) / 32) < (1u << 23) &&  // the grid
         (size_t)a.ldx * 256 < (1u << 30) && (size_t)a.K * 16 < (1u << 30);
}

int mid_spare(const MidArgs& a) {
  constexpr int BMS[4] = {64, 64, 32, 32}, BNS[4] = {96, 64, 64, 32};  // MidTile
  const int cus = std::max(device_cus(), 1), plan = mid_plan(a.M, a.N, cus);
  const long mt = (a.M + BMS[plan] - 1) / BMS[plan], nt = (a.N + BNS[plan] - 1) / BNS[plan];
  return (int)std::max(0L, cus - (nt + TG_NXCD - 1) / TG_NXCD * TG_NXCD * mt);
}

bool mid_worth(const MidArgs& a) { return mid_vs_tile(a.M, a.N, a.K, std::max(device_cus(), 1)); }

void mid_prefetch_add(const MidArgs& a, int nblocks, Prefetch& pf) {
  if (!mid_ok(a)) return;
  const int plan = mid_plan(a.M, a.N, std::max(device_cus(), 1));
  const int bn = plan == MID_64x96 ? 96 : plan == MID_32x32 ? 32 : 64;
  const int lo[3] = {0, a.n1, a.n2}, hi[3] = {std::min(a.n1, a.N), std::min(a.n2, a.N), a.N};
  for (int s = 0; s < 3 && pf.nreg < PF_MAX_REGIONS; ++s) {
    // whole n tiles of the segment (a tail shorter than a tile is left to the launch itself), 64-byte lines
    const size_t slab = (size_t)bn * a.K * 2;
    const int n = (hi[s] - lo[s]) / bn;
    if (n > 0 && slab % 64 == 0 && slab < (1u << 30)) {
      pf.r[pf.nreg++] = PfRegion{reinterpret_cast<const char*>(a.w[s]), (int)slab, n, (lo[s] / bn) & 7, 0};
      pf.nblocks = nblocks;
    }
  }
}

int mid_gemm_launch(const MidArgs& a, hipStream_t st) {
  MLCV_REQUIRE(mid_ok(a), "linear: shape or alignment");
  switch (mid_plan(a.M, a.N, std::max(device_cus(), 1))) {
    case MID_64x96: return launch<64, 96, 4, 2>(a, st);
    case MID_64x64: return launch<64, 64, 4, 2>(a, st);
    case MID_32x64: return launch<32, 64, 4, 3>(a, st);
    default: return launch<32, 32, 4, 4>(a, st);
  }
}

}  // namespace mlcv
