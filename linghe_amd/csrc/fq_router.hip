// RMSNorm + router GEMM + 1x128 quant
// (linghe/utils/norm.py:616-784, output_mode 0; kernel :616-687):
//   r = rsqrt(mean(x^2) + eps);  y = (x*r)*gamma  (fp32)
//   y_bf16 = bf16(y);  logits = y @ W^T (fp32);  q, s = 1x128 quant of y
//
// The only contraction on this path, so the only place MFMA is used.  r is a per-row factor of
// y, hence of the logits:
//   logits[m, :] = r[m] * sum_k (x[m,k] * gamma[k]) * W[:, k]
// z = x * gamma is EXACT in fp32 (two 8-bit significands) and so is its split z = hi + lo into
// two bf16 values; W is bf16 already, and the two products go through the bf16 matrix
// instructions with fp32 accumulation: bf16 products are exact in fp32, so the result carries
// only the rounding of the fp32 accumulation and one final multiplication by r, and the
// contraction does not wait for the statistic.
//
// An fp32 router weight (what Megatron keeps) is split the same way, W = hi + lo with
// hi = bf16(W), lo = bf16(W - hi) (what is left is below 2^-17 |W|): two planes, four products
// into the same accumulators.
//
// The kernels below share the work out over (row tile, column chunk) pairs; the workgroups of
// one row tile sit on one XCD (router_tile), so that the chunks' walks over K read x from memory
// once and else from that XCD's L2.  But for the calls of few tiles, whose workgroups take a slice of K each and leave the
// rows to a second kernel (router_slices), each of them walks all of K for its columns of the logits,
// accumulating the row statistic beside it, and then writes y, the codes and the scales for its
// share of the K / 128 quantisation groups, re-reading that part of x: from the L2 where the XCD's
// row tiles and the weight still fit it (8192 x 256 x 2048 fetched 63.6 MB past the L2s where x and one weight per
// XCD are 42; 49.9 with quantising waves of their own, which do so beside the products).
#include <algorithm>
#include <climits>
#include <type_traits>

#include "fq_device.hpp"
#include "fq_launch.h"
#include "fq_policy.hpp"

namespace fq {

// cache hints: fq_policy.hpp

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

// W [N, K] -> B operands in the order the main kernels read them: one 16-byte piece per (k
// block of 128, 32-column tile, k step, lane), so that every B load of a wave is 1 KB of
// contiguous memory.  (Read straight from the row-major matrix, each lane of such a load would
// touch a cache line of its own.)  Piece j of lane l holds columns 64 (l / 32) + 8 j .. + 7 of
// the k block of row l % 32 of its tile.  With an fp32 weight the tiles come in pairs: bf16(W) of 32
// columns, then bf16 of the rest.
// A workgroup packs 16 rows of a k block: 16 lanes read a row's 128 columns as one run, and an fp32
// weight is read once for both of its tiles.  (With a thread per packed piece every load of a wave
// touched 64 lines, each of them again in a second workgroup, and an fp32 weight was read twice: us thread per
// piece / now, bf16 256 x 2048 2.22 / 1.87, 512 x 7168 5.73 / 4.80, fp32 256 x 4096 3.71 / 2.91.)
template <bool FP32W>
__global__ __launch_bounds__(256) void pack_router_weight_kernel(const void* __restrict__ wr,
                                                                 uint4* __restrict__ packed, int K, int n_halves) {
  const int kb = wg_x() / n_halves;
  const int n = (wg_x() - kb * n_halves) * 16 + (tid_x() >> 4);  // row of W
  const int c = tid_x() & 15;                                    // piece of its 128 columns
  const int vtiles = (n_halves >> 1) * (FP32W ? 2 : 1);
  const int tile = (n >> 5) * (FP32W ? 2 : 1);
  const int64_t at = (int64_t)n * K + kb * kGroup + c * 8;
  uint4* dst = packed + (((int64_t)kb * vtiles + tile) * 8 + (c & 7)) * 64 + (c >> 3) * 32 + (n & 31);
  if constexpr (!FP32W) {
    *dst = *(const uint4*)((const uint16_t*)wr + at);
  } else {
    const float4* src = (const float4*)((const float*)wr + at);
    const float4 a = src[0], b = src[1];
    float w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    const uint4 hi = pack8_bf16(w);
    float back[8], lo[8];
    unpack8(hi, back);
#pragma unroll
    for (int i = 0; i < 8; ++i) lo[i] = w[i] - back[i];
    dst[0] = hi;
    dst[8 * 64] = pack8_bf16(lo);
  }
}

struct RouterArgs {
  const uint16_t* x;      // [M, K]
  const uint16_t* gamma;  // [K]
  const uint4* w;         // packed
  uint16_t* y;            // [M, K]
  float* rstd;            // [M]
  float* logits;          // [M, N]
  uint8_t* q;             // [M, K]
  float* s;               // [K / 128, M]
  int M, K, N;
  int chunks;  // column chunks, i.e. workgroups per row tile
  float eps;
};

// workgroup -> (row tile, column chunk): workgroup i runs on XCD i % 8, so eight row tiles go
// round the XCDs and the chunks of one tile follow each other there; the last tiles % 8 row tiles do the same
// in a narrower round
__device__ __forceinline__ void router_tile(int tiles, int chunks, int& tile, int& chunk) {
  const int i = (int)wg_x();
  const int full = (tiles & ~7) * chunks;
  if (i < full) {
    const int r = i >> 3;
    chunk = r % chunks;
    tile = (r / chunks) * 8 + (i & 7);
  } else {
    const int left = tiles & 7;
    chunk = (i - full) / left;
    tile = (tiles & ~7) + (i - full) % left;
  }
}

// the two exact terms of x * gamma of 8 columns, as matrix operands
__device__ __forceinline__ void router_split(const uint4& xr, const uint4& gr, uint4& hi, uint4& lo) {
  float a[8], g[8], z[8], back[8];
  unpack8(xr, a);
  unpack8(gr, g);
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = a[i] * g[i];
  hi = pack8_bf16(z);
  unpack8(hi, back);
#pragma unroll
  for (int i = 0; i < 8; ++i) back[i] = z[i] - back[i];
  lo = pack8_bf16(back);
}

// y, codes and scale of 8 columns; the 16 lanes of a DPP row (the first of them names the scale's place)
// hold one quantisation group
template <int KIND, bool ROUND>
__device__ __forceinline__ void router_emit(uint16_t* y, uint8_t* q, float* s, bool first, const uint4& xr,
                                            const uint4& gr, float r) {
  float a[8], g[8], yv[8], m = 0.f;
  unpack8(xr, a);
  unpack8(gr, g);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    yv[i] = (a[i] * r) * g[i];
    m = fmaxf(m, fabsf(yv[i]));
  }
  m = row16_max(m);
  const float sc = make_scale<KIND, ROUND>(m);
  store16<Policy::kStoreHintRouter>(y, pack8_bf16(yv));
  store8<Policy::kStoreHintRouter>(q, quantize8<KIND, ROUND>(yv, make_quantum<ROUND>(sc)));
  if (first) store_f32(s, sc);
}

// A row whose squares overflow has the statistic 0, so y = (x * 0) * gamma is 0 where x and gamma are finite and
// NaN where they are not, and so are its logits.  The products taken before the statistic is known can say neither
// (x * gamma * W overflows): the factor of such a row's logits is 0 or NaN by its values, and 0 stands
// for the result itself.
__device__ __forceinline__ bool router_nonfinite(const uint4& v) {  // any of 8 bf16
  auto pair = [](unsigned w) { return (w & 0x7f80u) == 0x7f80u || (w & 0x7f800000u) == 0x7f800000u; };
  return pair(v.x) || pair(v.y) || pair(v.z) || pair(v.w);
}
constexpr unsigned kNanBits = 0x7fc00000u;  // as bits throughout: the compiler may take a float for not NaN
__device__ __forceinline__ float router_logit(float v, unsigned factor) {
  return __uint_as_float(factor == 0 ? 0u : __float_as_uint(v * __uint_as_float(factor)));
}

// the factor of a row that the 16 lanes of a DPP row share: r is its statistic, x the lane's first piece, gamma in LDS
__device__ __forceinline__ unsigned router_factor(float r, const uint16_t* x, const uint4* gamma, int kblocks) {
  unsigned factor = __float_as_uint(r);
  if (factor == 0) {
    bool bad = false;
#pragma unroll 1
    for (int kb = 0; kb < kblocks; ++kb)
      bad |= router_nonfinite(*(const uint4*)(x + kb * kGroup)) || router_nonfinite(gamma[kb * 16]);
    if (row16_max(bad ? 1.f : 0.f) > 0.f) factor = kNanBits;
  }
  return factor;
}

// EMIT k blocks of the lane's piece of ROWS rows; blocks beyond the last repeat it
template <int EMIT, int ROWS>
__device__ __forceinline__ void router_fetch_share(const RouterArgs& p, int row, int row_step, int cg, int k0,
                                                   uint4 (&xe)[EMIT][ROWS]) {
#pragma unroll
  for (int d = 0; d < EMIT; ++d)
#pragma unroll
    for (int u = 0; u < ROWS; ++u)
      xe[d][u] = *(const uint4*)(p.x + (int64_t)(row + u * row_step) * p.K + min(k0 + d, p.K / kGroup - 1) * kGroup +
                                 cg * 8);
}

// y, codes and scales of k blocks q0 .. q1 - 1, EMIT at a time (no load waits behind a store); the first are in xe
template <int KIND, bool ROUND, int EMIT, int ROWS>
__device__ __forceinline__ void router_emit_share(const RouterArgs& p, const uint4* gamma, int row, int row_step, int cg,
                                                  int q0, int q1, const float (&rs)[ROWS], uint4 (&xe)[EMIT][ROWS]) {
#pragma unroll 1
  for (int k0 = q0; k0 < q1; k0 += EMIT) {
    if (k0 > q0) router_fetch_share(p, row, row_step, cg, k0, xe);
    const int64_t at = (int64_t)row * p.K + k0 * kGroup + cg * 8;
    const int64_t step = (int64_t)row_step * p.K;
    float* s = p.s + (int64_t)k0 * p.M + row;
#pragma unroll
    for (int d = 0; d < EMIT; ++d) {
      if (k0 + d < q1) {
        const uint4 g = gamma[(k0 + d) * 16 + cg];
#pragma unroll
        for (int u = 0; u < ROWS; ++u)
          router_emit<KIND, ROUND>(p.y + at + u * step + d * kGroup, p.q + at + u * step + d * kGroup,
                                   s + (int64_t)d * p.M + u * row_step, cg == 0, xe[d][u], g, rs[u]);
      }
    }
  }
}

__device__ __forceinline__ bf16x8_t operand(const uint4& v) { return __builtin_bit_cast(bf16x8_t, v); }

// ---------------------------------------------------------------------------
// 64 rows x 64 VT operand columns per workgroup of eight waves: 64 VT logits of a bf16 weight, 64 of an
// fp32 one (VT = 2, its two planes).  Per 128-wide k block the threads turn 64 x 128 values of x
// into A operands in LDS (2 rows x 8 columns each) while the matrix cores work on the block before
// (double-buffered, one barrier per block).  Wave (wc, kq) multiplies all 64 rows by 32 VT operand columns
// over a quarter of the block's k, so that A is read from LDS twice per block (64 KB) and W from the L2
// once (32 KB with VT = 2; an XCD's CUs share about 35 B a clock each); the four k quarters are
// added up through LDS at the end.
// Bound by instruction issue: per k block about 1000 clocks of matrix instructions and 900 of operand
// arithmetic on each SIMD, partly on top of each other, and per block of the second part 1600 clocks of
// normalising and quantising.  us of the kernel (former 32-row workgroups with all of W each / these): 4096 x 256 x 4096
// with an fp32 weight 81 / 48, 8192 x 256 x 2048 bf16 34.3 / 34.3, 4096 x 512 x 4096 bf16 82 / 49,
// 16384 x 128 x 2048 bf16 59 / 50; with VT = 1 4096 x 256 x 2048 27.3 / 21.1.
// ---------------------------------------------------------------------------
constexpr int kRouterRows = 64;

struct RouterShared {
  uint4 a[2][2][2][8][64];  // [buffer][hi, lo][32-row tile][k step][lane slot]; afterwards the partial sums
  uint4 gamma[8192 / 8];
  unsigned factor[kRouterRows];  // of a row's logits: the bits of its statistic, or see router_logit
};

// The order of a k block's instructions: operand reads, then the matrix instructions with the next
// block's operand arithmetic between them.  (Left alone the compiler puts the arithmetic behind
// all of them, and as the waves of a SIMD go in step, matrix cores and arithmetic units take turns:
// 80 instead of 87 us at 4096 x 256 x 7168.)
template <int VT>
__device__ __forceinline__ void router_interleave() {
  constexpr int kValu = 0x2, kMfma = 0x8, kVmemRead = 0x20, kDsRead = 0x100, kDsWrite = 0x200;
  __builtin_amdgcn_sched_group_barrier(kDsRead, 5, 0);
  __builtin_amdgcn_sched_group_barrier(kValu, 12, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int m = 0; m < 2 * VT; ++m) {
      __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
      __builtin_amdgcn_sched_group_barrier(kValu, 10 / VT, 0);
    }
    if (i < 1) __builtin_amdgcn_sched_group_barrier(kDsRead, 4, 0);
    if (i < 1 + VT) __builtin_amdgcn_sched_group_barrier(kVmemRead, 2, 0);
    if (i > 0) __builtin_amdgcn_sched_group_barrier(kDsWrite, 2, 0);
  }
}

template <int KIND, bool ROUND, bool FP32W, int VT>
__global__ __launch_bounds__(512) void rmsnorm_router_quant_kernel(RouterArgs p) {
  __shared__ RouterShared sh;
  const int lane = tid_x() & 63;
  const int wave = uniform32(tid_x() >> 6);
  const int kq = wave & 3, wc = wave >> 2;
  const int cg = tid_x() & 15, rg = tid_x() >> 4;
  const int kblocks = p.K / kGroup;
  int tile, chunk;
  router_tile((p.M + kRouterRows - 1) / kRouterRows, p.chunks, tile, chunk);
  // rows that do not fill a tile are worked on twice, with the same results, by the last two tiles
  const int row0 = min(tile * kRouterRows, p.M - kRouterRows);
  const uint16_t* xrow = p.x + (int64_t)(row0 + rg) * p.K + cg * 8;
  const int64_t half_tile = (int64_t)32 * p.K;

  constexpr int kRing = 4;                // k blocks of x and W in flight or in use
  constexpr int NACC = FP32W ? 1 : VT;    // 32-column result tiles of a wave
  uint4 xr[kRing][2], b[kRing][VT][2];    // b: [slot][operand tile][k step]
  floatx16_t acc[2][NACC];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int t = 0; t < NACC; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[rt][t][v] = 0.f;
  double ss[2] = {0.0, 0.0};

  const int vtiles = p.N / 32 * (FP32W ? 2 : 1);
  const uint4* wlane = p.w + ((int64_t)(chunk * 2 + wc) * VT * 8 + kq * 2) * 64 + lane;
  auto fetch_w = [&](int kb, uint4 (&d)[VT][2]) {
    const uint4* at = wlane + (int64_t)min(kb, kblocks - 1) * vtiles * 512;
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int j = 0; j < 2; ++j) d[t][j] = at[t * 512 + j * 64];
  };
  auto fetch_x = [&](int kb, uint4 (&d)[2]) {
    const uint16_t* at = xrow + min(kb, kblocks - 1) * kGroup;
    d[0] = *(const uint4*)at;
    d[1] = *(const uint4*)(at + half_tile);
  };
  // the row position is XORed with the k step so that the 16-byte LDS writes of the eight lanes
  // of a row group fall into different banks
  const int aj = cg & 7;
  const int aslot = (cg >> 3) * 32 + (rg ^ aj);
  auto produce = [&](int kb, const uint4 (&xk)[2]) {
    const uint4 g = sh.gamma[kb * 16 + cg];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      ss[u] += (double)sumsq8(xk[u]);
      uint4 hi, lo;
      router_split(xk[u], g, hi, lo);
      sh.a[kb & 1][0][u][aj][aslot] = hi;
      sh.a[kb & 1][1][u][aj][aslot] = lo;
    }
  };
  auto multiply = [&](int buf, const uint4 (&w)[VT][2]) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int step = kq * 2 + j;
      const int slot = (lane & 32) + ((lane & 31) ^ step);
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const bf16x8_t hi = operand(sh.a[buf][0][rt][step][slot]);
        const bf16x8_t lo = operand(sh.a[buf][1][rt][step][slot]);
#pragma unroll
        for (int t = 0; t < VT; ++t) {
          floatx16_t& c = acc[rt][FP32W ? 0 : t];
          c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, operand(w[t][j]), c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, operand(w[t][j]), c, 0, 0, 0);
        }
      }
    }
  };

  // gamma (at most 1024 pieces) is asked for first, so that waiting for it waits for nothing else
  uint4 g2[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    g2[i] = *(const uint4*)(p.gamma + min((int)tid_x() + 512 * i, kblocks * 16 - 1) * 8);
#pragma unroll
  for (int d = 0; d < kRing; ++d) fetch_x(d, xr[d]);
#pragma unroll
  for (int d = 0; d < kRing - 1; ++d) fetch_w(d, b[d]);
#pragma unroll
  for (int i = 0; i < 2; ++i) sh.gamma[tid_x() + 512 * i] = g2[i];
  __syncthreads();
  produce(0, xr[0]);
  fetch_x(kRing, xr[0]);
  __syncthreads();
  // rings of kRing operand sets: a set is refilled in place once it was used.  Fetches beyond the last block
  // repeat it; all but the last 1 .. kRing blocks run without a condition
  int kb = 0;
#pragma unroll 1
  for (; kb + kRing < kblocks; kb += kRing) {
#pragma unroll
    for (int d = 0; d < kRing; ++d) {
      fetch_w(kb + d + kRing - 1, b[(d + kRing - 1) % kRing]);
      multiply(d & 1, b[d]);
      produce(kb + d + 1, xr[(d + 1) % kRing]);
      fetch_x(kb + d + 1 + kRing, xr[(d + 1) % kRing]);
      router_interleave<VT>();
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);  // the order is laid out block by block
    }
  }
#pragma unroll
  for (int d = 0; d < kRing; ++d) {
    if (kb + d < kblocks) {
      if (d == 0) fetch_w(kb + kRing - 1, b[kRing - 1]);
      multiply(d & 1, b[d]);
      if (kb + d + 1 < kblocks) produce(kb + d + 1, xr[(d + 1) % kRing]);
      __syncthreads();
    }
  }

  // ---- this workgroup's share of the quantisation groups: its first rows of x leave now
  const int q0 = chunk * kblocks / p.chunks;
  const int q1 = (chunk + 1) * kblocks / p.chunks;
  uint4 xe[4 * NACC][2];
  router_fetch_share(p, row0 + rg, 32, cg, q0, xe);

  // ---- statistic
  float rs[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    rs[u] = 1.0f / sqrtf((float)row16_sum_d(ss[u]) / (float)p.K + p.eps);
    const unsigned factor = router_factor(rs[u], xrow + u * half_tile, sh.gamma + cg, kblocks);
    if (cg == 0) {
      sh.factor[u * 32 + rg] = factor;
      if (chunk == 0) p.rstd[row0 + u * 32 + rg] = rs[u];
    }
  }

  // ---- the four k quarters: waves kq and kq ^ 2 exchange a row tile, then kq and kq ^ 1 half of
  // what they hold, so that all eight waves end up with an equal part of the sums
  floatx4_t* part = (floatx4_t*)&sh.a[0][0][0][0][0];
  auto quarter = [](const floatx16_t& c, int i) {
    floatx4_t o = {c[4 * i], c[4 * i + 1], c[4 * i + 2], c[4 * i + 3]};
    return o;
  };
  // (by value: a conditional between array elements would choose between addresses, and the
  // arrays would leave the registers)
  auto pick = [](bool first, floatx4_t a, floatx4_t c) { return first ? a : c; };
  const bool upper = kq >> 1, odd = kq & 1;
#pragma unroll
  for (int t = 0; t < NACC; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      part[((wave * NACC + t) * 4 + i) * 64 + lane] = pick(upper, quarter(acc[0][t], i), quarter(acc[1][t], i));
  __syncthreads();
  floatx4_t sum[NACC * 4];
#pragma unroll
  for (int t = 0; t < NACC; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      sum[t * 4 + i] = pick(upper, quarter(acc[1][t], i), quarter(acc[0][t], i)) +
                       part[(((wave ^ 2) * NACC + t) * 4 + i) * 64 + lane];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NACC * 2; ++i)
    part[(wave * NACC * 2 + i) * 64 + lane] = pick(odd, sum[i], sum[NACC * 2 + i]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NACC * 2; ++i) {
    const floatx4_t v = pick(odd, sum[NACC * 2 + i], sum[i]) + part[((wave ^ 1) * NACC * 2 + i) * 64 + lane];
    // register r of a 32x32 result holds row (r / 4) * 8 + (lane / 32) * 4 + r % 4, column lane % 32
    const int i4 = (odd ? NACC * 2 : 0) + i;
    const int row = (upper ? 32 : 0) + (i4 & 3) * 8 + (lane >> 5) * 4;
    const int col = ((chunk * 2 + wc) * NACC + (i4 >> 2)) * 32 + (lane & 31);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      p.logits[(int64_t)(row0 + row + e) * p.N + col] = router_logit(v[e], sh.factor[row + e]);
  }

  router_emit_share<KIND, ROUND>(p, sh.gamma, row0 + rg, 32, cg, q0, q1, rs, xe);
}

// ---------------------------------------------------------------------------
// 32 rows x 32 WAVES NACC logits per workgroup: all logits of the rows wherever N is 128, 256 or (bf16) 512, so that
// x becomes operands once. Wave w multiplies the 32 rows by its own VT operand tiles (NACC of logits: VT, or
// one for the two planes of an fp32 weight) over all of K; nothing is exchanged at the end.
// W operands come in sets of half a k block (whole blocks cost 165-175 registers instead of 127 with 256 logits, and the
// second workgroup on a CU: 16384 x 256 x 1024 36.7 / 33.0 us). Three workgroups fit a CU with 128 logits, two with 256
// of a bf16 weight, one otherwise. Bound by instruction issue like the kernel above, W read per 32 instead of 64 rows;
// us of the 64-row form / this: 4224 x 512 x 1024 29.5 / 22.1, 16384 x 256 x 1024 40.0 / 33.5, fp32 4224 x 256 x 1024
// 26.8 / 21.2.
// ---------------------------------------------------------------------------
template <int KIND, bool ROUND, bool FP32W, int VT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, WAVES == 4 ? 3 : 2) void rmsnorm_router_quant_32_rows_kernel(RouterArgs p) {
  constexpr int kRows = 32;
  constexpr int RPT = 8 / WAVES;        // rows per thread
  constexpr int NACC = FP32W ? 1 : VT;  // 32-column result tiles of a wave
  constexpr int SETS = 2, STEPS = 8 / SETS;  // sets of W operands per k block, k steps of a set
  __shared__ struct {
    uint4 a[2][2][8][64];  // [buffer][hi, lo][k step][lane slot]
    uint4 gamma[8192 / 8];
    unsigned factor[kRows];
  } sh;
  const int lane = tid_x() & 63;
  const int wave = uniform32(tid_x() >> 6);
  const int cg = tid_x() & 15, rg = tid_x() >> 4;
  const int kblocks = p.K / kGroup;
  int tile, chunk;
  router_tile(p.M / kRows, p.chunks, tile, chunk);
  const int row0 = tile * kRows;
  const uint16_t* xrow = p.x + (int64_t)(row0 + rg) * p.K + cg * 8;
  const int64_t row_step = (int64_t)(4 * WAVES) * p.K;

  constexpr int kRing = 4;                // k blocks of x in flight or in use
  uint4 xr[kRing][RPT], b[2][VT][STEPS];  // b: two sets of W operands, one in use, one in flight
  // the products of the leading terms by k parity, all others in an accumulator of their own: shorter chains of roundings
  floatx16_t lead[NACC][2], rest[NACC];
#pragma unroll
  for (int t = 0; t < NACC; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) lead[t][0][v] = lead[t][1][v] = rest[t][v] = 0.f;
  double ss[RPT];
#pragma unroll
  for (int u = 0; u < RPT; ++u) ss[u] = 0.0;

  const int vtiles = p.N / 32 * (FP32W ? 2 : 1);
  const uint4* wlane = p.w + (int64_t)(chunk * WAVES + wave) * VT * 512 + lane;
  auto fetch_w = [&](int kb, int set, uint4 (&d)[VT][STEPS]) {
    const uint4* at = wlane + (int64_t)min(kb, kblocks - 1) * vtiles * 512 + set * STEPS * 64;
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int j = 0; j < STEPS; ++j) d[t][j] = at[t * 512 + j * 64];
  };
  auto fetch_x = [&](int kb, uint4 (&d)[RPT]) {
#pragma unroll
    for (int u = 0; u < RPT; ++u) d[u] = *(const uint4*)(xrow + u * row_step + min(kb, kblocks - 1) * kGroup);
  };
  const int aj = cg & 7;  // the row position is XORed with the k step as in the kernel above
  auto produce = [&](int kb, const uint4 (&xk)[RPT]) {
    const uint4 g = sh.gamma[kb * 16 + cg];
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      ss[u] += (double)sumsq8(xk[u]);
      uint4 hi, lo;
      router_split(xk[u], g, hi, lo);
      const int slot = (cg >> 3) * 32 + ((rg + u * 4 * WAVES) ^ aj);
      sh.a[kb & 1][0][aj][slot] = hi;
      sh.a[kb & 1][1][aj][slot] = lo;
    }
  };
  auto multiply = [&](int buf, int set, const uint4 (&w)[VT][STEPS]) {
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
      const int step = set * STEPS + j;
      const int slot = (lane & 32) + ((lane & 31) ^ step);
      const bf16x8_t hi = operand(sh.a[buf][0][step][slot]);
      const bf16x8_t lo = operand(sh.a[buf][1][step][slot]);
#pragma unroll
      for (int t = 0; t < VT; ++t) {
        const bf16x8_t wt = operand(w[t][j]);
        if (!FP32W || t == 0) {
          floatx16_t& c = lead[FP32W ? 0 : t][step & 1];
          c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, wt, c, 0, 0, 0);
        } else {
          rest[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, wt, rest[0], 0, 0, 0);
        }
        floatx16_t& c = rest[FP32W ? 0 : t];
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, wt, c, 0, 0, 0);
      }
    }
  };

#pragma unroll
  for (int d = 0; d < kRing; ++d) fetch_x(d, xr[d]);
  fetch_w(0, 0, b[0]);
  for (int i = tid_x(); i < kblocks * 16; i += 64 * WAVES) sh.gamma[i] = *(const uint4*)(p.gamma + i * 8);
  __syncthreads();
  produce(0, xr[0]);
  fetch_x(kRing, xr[0]);
  __syncthreads();
#pragma unroll 1
  for (int kb = 0; kb < kblocks; kb += kRing) {
#pragma unroll
    for (int d = 0; d < kRing; ++d) {
      if (kb + d < kblocks) {
#pragma unroll
        for (int set = 0; set < SETS; ++set) {
          fetch_w(kb + d + (set + 1) / SETS, (set + 1) % SETS, b[(set + 1) & 1]);
          multiply(d & 1, set, b[set & 1]);
        }
        if (kb + d + 1 < kblocks) {
          produce(kb + d + 1, xr[(d + 1) % kRing]);
          fetch_x(kb + d + 1 + kRing, xr[(d + 1) % kRing]);
        }
        __syncthreads();
      }
    }
  }

  const int q0 = chunk * kblocks / p.chunks, q1 = (chunk + 1) * kblocks / p.chunks;
  uint4 xe[8 / RPT][RPT];
  router_fetch_share(p, row0 + rg, 4 * WAVES, cg, q0, xe);
  float rs[RPT];
#pragma unroll
  for (int u = 0; u < RPT; ++u) {
    rs[u] = 1.0f / sqrtf((float)row16_sum_d(ss[u]) / (float)p.K + p.eps);
    const unsigned factor = router_factor(rs[u], xrow + u * row_step, sh.gamma + cg, kblocks);
    if (cg == 0) {
      sh.factor[u * 4 * WAVES + rg] = factor;
      if (chunk == 0) p.rstd[row0 + u * 4 * WAVES + rg] = rs[u];
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NACC; ++t) {
    const int col = ((chunk * WAVES + wave) * NACC + t) * 32 + (lane & 31);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      // register v of a 32x32 result holds row (v / 4) * 8 + (lane / 32) * 4 + v % 4, column lane % 32
      const int row = (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
      p.logits[(int64_t)(row0 + row) * p.N + col] =
          router_logit((lead[t][0][v] + lead[t][1][v]) + rest[t][v], sh.factor[row]);
    }
  }
  router_emit_share<KIND, ROUND>(p, sh.gamma, row0 + rg, 4 * WAVES, cg, q0, q1, rs, xe);
}

// ---------------------------------------------------------------------------
// Few rows: 16 rows x 32 logits per workgroup.  Every wave takes whole k blocks of its own (block
// number modulo 8) and makes the A operands in its registers, so there is neither an LDS round
// trip nor a barrier in the walk over K; the eight partial results meet in LDS at the end.
// Latency bound: 512 x 256 x 2048 24.1 -> 8.2 us, 512 x 256 x 7168 82 -> 19.5 (32-row workgroups before).
// ---------------------------------------------------------------------------
constexpr int kRouterFewRows = 16;

template <int KIND, bool ROUND, bool FP32W>
__global__ __launch_bounds__(512) void rmsnorm_router_quant_few_rows_kernel(RouterArgs p) {
  constexpr int NV = FP32W ? 2 : 1;  // operand tiles of 32 columns
  __shared__ float part[8][512];
  __shared__ double ssum[32][16];
  __shared__ float srstd[16];
  const int lane = tid_x() & 63;
  const int wave = uniform32(tid_x() >> 6);
  const int kblocks = p.K / kGroup;
  int tile, chunk;
  router_tile(p.M / kRouterFewRows, p.chunks, tile, chunk);
  const int row0 = tile * kRouterFewRows;
  const int r = lane & 15, g = lane >> 4;
  // lane group g of k step s holds 8-column piece 2 s + g % 2 of half g / 2 of the k block
  const int col0 = (g >> 1) * 64 + (g & 1) * 8;
  const uint16_t* xl = p.x + (int64_t)(row0 + r) * p.K + col0;
  const uint16_t* gl = p.gamma + col0;
  const int vtiles = p.N / 32 * NV;
  const uint4* wl = p.w + ((int64_t)chunk * NV * 8 + (g & 1)) * 64 + (g >> 1) * 32 + r;

  floatx4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  double ss = 0.0;
  uint4 xr[2][4], gr[2][4], b[2][NV][4][2];
  auto fetch = [&](int kb, uint4 (&xd)[4], uint4 (&gd)[4], uint4 (&bd)[NV][4][2]) {
    const int k = min(kb, kblocks - 1);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      xd[s] = *(const uint4*)(xl + k * kGroup + s * 16);
      gd[s] = *(const uint4*)(gl + k * kGroup + s * 16);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) bd[v][s][t] = wl[((int64_t)k * vtiles + v) * 512 + s * 128 + t * 16];
  };
  auto multiply = [&](const uint4 (&xd)[4], const uint4 (&gd)[4], const uint4 (&bd)[NV][4][2]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      ss += (double)sumsq8(xd[s]);
      uint4 hi, lo;
      router_split(xd[s], gd[s], hi, lo);
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(operand(hi), operand(bd[v][s][t]), acc[t], 0, 0, 0);
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(operand(lo), operand(bd[v][s][t]), acc[t], 0, 0, 0);
        }
    }
  };
  fetch(wave, xr[0], gr[0], b[0]);
#pragma unroll 1
  for (int kb = wave; kb < kblocks; kb += 16) {
    fetch(kb + 8, xr[1], gr[1], b[1]);
    multiply(xr[0], gr[0], b[0]);
    if (kb + 8 < kblocks) {
      fetch(kb + 16, xr[0], gr[0], b[0]);
      multiply(xr[1], gr[1], b[1]);
    }
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) *(floatx4_t*)&part[wave][t * 256 + lane * 4] = acc[t];
  ssum[wave * 4 + g][r] = ss;
  __syncthreads();
  if (tid_x() < 16) {
    double total = 0.0;
#pragma unroll
    for (int i = 0; i < 32; ++i) total += ssum[i][tid_x()];
    const float rs = 1.0f / sqrtf((float)total / (float)p.K + p.eps);
    srstd[tid_x()] = rs;
    if (chunk == 0) p.rstd[row0 + tid_x()] = rs;
  }
  __syncthreads();
  {
    // register e of a 16x16 result holds row (lane / 16) * 4 + e, column lane % 16
    const int col = tid_x() & 31, row = tid_x() >> 5;
    const int at = (col >> 4) * 256 + ((row >> 2) * 16 + (col & 15)) * 4 + (row & 3);
    float v = part[0][at];
#pragma unroll
    for (int i = 1; i < 8; ++i) v += part[i][at];
    unsigned factor = __float_as_uint(srstd[row]);
    bool bad = false;
    if (factor == 0) {
#pragma unroll 1
      for (int c = col * 8; c < p.K; c += 256)
        bad |= router_nonfinite(*(const uint4*)(p.x + (int64_t)(row0 + row) * p.K + c)) ||
               router_nonfinite(*(const uint4*)(p.gamma + c));
    }
    if ((uint32_t)(__ballot(bad) >> (lane & 32))) factor = kNanBits;  // 32 lanes have one row
    p.logits[(int64_t)(row0 + row) * p.N + chunk * 32 + col] = router_logit(v, factor);
  }
  const int q0 = chunk * kblocks / p.chunks, q1 = (chunk + 1) * kblocks / p.chunks;
  const int cg = tid_x() & 15;
  for (int i = tid_x() >> 4; i < (q1 - q0) * 16; i += 32) {
    const int row = i & 15, kb = q0 + (i >> 4);
    const int c = kb * kGroup + cg * 8;
    const int64_t at = (int64_t)(row0 + row) * p.K + c;
    router_emit<KIND, ROUND>(p.y + at, p.q + at, p.s + (int64_t)kb * p.M + row0 + row, cg == 0,
                             *(const uint4*)(p.x + at), *(const uint4*)(p.gamma + c), srstd[row]);
  }
}

// The role of a wave that multiplies nothing: statistic, y, codes and scales of the tile's rows 4 batch .. 4 batch + 3,
// then of batch + step and so on, 16 lanes a row.
template <int KIND, bool ROUND>
__device__ __forceinline__ void router_rows(const RouterArgs& p, int row0, int batch, int step) {
  constexpr int kHeld = 16, kStep = 4;  // k blocks of a row in registers, worked on together; beyond the last: it again
  const int lane = tid_x() & 63, cg = lane & 15, kblocks = p.K / kGroup;
  const int last = (kblocks - 1) / kHeld;
#pragma unroll 1
  for (; batch < kRouterRows / 4; batch += step) {
    const int row = row0 + batch * 4 + (lane >> 4);
    const uint16_t* x = p.x + (int64_t)row * p.K + cg * 8;
    const uint16_t* gamma = p.gamma + cg * 8;
    uint4 xe[kHeld], ge[2][kStep];
    auto fetch = [&](int k0) {
#pragma unroll
      for (int d = 0; d < kHeld; ++d) xe[d] = *(const uint4*)(x + min(k0 + d, kblocks - 1) * kGroup);
    };
    auto fetch_gamma = [&](int k0, uint4 (&g)[kStep]) {
#pragma unroll
      for (int d = 0; d < kStep; ++d) g[d] = *(const uint4*)(gamma + min(k0 + d, kblocks - 1) * kGroup);
    };
    double ss = 0.0;
#pragma unroll 1
    for (int set = 0; set <= last; ++set) {
      fetch(set * kHeld);
#pragma unroll
      for (int d = 0; d < kHeld; ++d) ss += set * kHeld + d < kblocks ? (double)sumsq8(xe[d]) : 0.0;
    }
    fetch_gamma(last * kHeld, ge[0]);
    const float rs = 1.0f / sqrtf((float)row16_sum_d(ss) / (float)p.K + p.eps);
    if (cg == 0) p.rstd[row] = rs;
    // the last set, which is in registers, first
#pragma unroll 1
    for (int i = 0; i <= last; ++i) {
      const int k0 = (i == 0 ? last : i - 1) * kHeld;
      if (i > 0) {
        fetch(k0);
        fetch_gamma(k0, ge[0]);
      }
#pragma unroll
      for (int g = 0; g < kHeld / kStep; ++g) {
        if (k0 + g * kStep < kblocks) {
          fetch_gamma(k0 + (g + 1) * kStep, ge[(g + 1) & 1]);
#pragma unroll
          for (int d = 0; d < kStep; ++d) {
            const int kb = min(k0 + g * kStep + d, kblocks - 1);
            const int64_t at = (int64_t)row * p.K + kb * kGroup + cg * 8;
            router_emit<KIND, ROUND>(p.y + at, p.q + at, p.s + (int64_t)kb * p.M + row, cg == 0, xe[g * kStep + d],
                                     ge[g & 1][d], rs);
          }
        }
      }
    }
  }
}

// the factors of a tile's rows from the squares that four waves saw of them, eight lanes a row
__device__ __forceinline__ void router_factors(const RouterArgs& p, int row0, const double (&sq)[4][2][kRouterRows],
                                               unsigned (&sfactor)[kRouterRows]) {
  const int lane = tid_x() & 63, row = tid_x() >> 3, part = tid_x() & 7;
  double total = 0.0;
#pragma unroll
  for (int i = 0; i < 8; ++i) total += sq[i >> 1][i & 1][row];
  unsigned factor = __float_as_uint(1.0f / sqrtf((float)total / (float)p.K + p.eps));
  bool bad = false;
  if (factor == 0) {
#pragma unroll 1
    for (int c = part * 8; c < p.K; c += 64)
      bad |= router_nonfinite(*(const uint4*)(p.x + (int64_t)(row0 + row) * p.K + c)) ||
             router_nonfinite(*(const uint4*)(p.gamma + c));
  }
  if ((__ballot(bad) >> (lane & 56)) & 0xff) factor = kNanBits;
  if (part == 0) sfactor[row] = factor;
}

typedef __attribute__((address_space(3))) void lds_void_t;

// 64 rows of a k block from memory into LDS, four rows an instruction; at: this lane's byte offset in each four of 16
// rows. With valid = 0 (else K) nothing is read and zeros arrive.
__device__ __forceinline__ void router_fetch_block(const uint16_t* x, int valid, int K, int block, const uint32_t (&at)[4],
                                                   uint4* slot) {
  const __amdgpu_buffer_rsrc_t from =
      __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, kRouterRows * valid * 2, 0x00027000);
#pragma unroll
  for (int i = 0; i < kRouterRows / 4; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (lds_void_t*)(slot + i * 64), 16, at[i & 3],
                                             block * kGroup * 2 + (i >> 2) * 32 * K, 0, 0);
}

// ---------------------------------------------------------------------------
// 64 rows x 128 logits of a bf16 weight per workgroup of eight waves in two roles. Four multiply, each over every fourth k
// block for all of the logits: x comes straight into LDS two blocks ahead, becomes operands in the wave's registers one
// product group ahead, W half a block ahead; they share nothing until their sums meet at the end. The other four normalise
// and quantise the workgroup's share of the tile's rows meanwhile (router_rows).
// Bound by the instructions of the multiplying waves, one on a SIMD: 256 clocks of matrix instructions and about 220 of
// operand arithmetic per 32 rows x 16 columns x 128 logits, which overlap in part (by themselves 23 us of 32 at
// 8192 x 256 x 2048; the rows by themselves 17). us of the 64 x 128 kernel above / this: 8192 x 256 x 2048 34.4 / 31.6,
// x 4096 65.1 / 57.4, x 7168 107.9 / 93.8, 4096 x 512 x 2048 27.3 / 25.0, 3072 x 512 x 1536 20.3 / 16.6, x 4096 43.0 / 38.8;
// logits' error against 64 bits over 50 inputs 1.00 of that kernel's.
// ---------------------------------------------------------------------------
template <int KIND, bool ROUND>
__global__ __launch_bounds__(512) void rmsnorm_router_quant_two_roles_kernel(RouterArgs p) {
  // two k blocks of each multiplying wave, a row's 16 pieces XORed with its number; afterwards the partial sums of the first
  // and the second 32 rows. (Two arrays: the compiler tells the loads into one from those into the other.)
  __shared__ uint4 a0[4][kRouterRows * 16];
  __shared__ uint4 a1[4][kRouterRows * 16];
  __shared__ uint4 sgamma[4][256];          // of the k blocks of a multiplying wave
  __shared__ double sq[4][2][kRouterRows];  // squares of a row: by wave and by half of its lanes
  __shared__ unsigned sfactor[kRouterRows];
  const int lane = tid_x() & 63;
  const int wave = uniform32(tid_x() >> 6);
  const int kblocks = p.K / kGroup;
  int tile, chunk;
  router_tile((p.M + kRouterRows - 1) / kRouterRows, p.chunks, tile, chunk);
  const int row0 = min(tile * kRouterRows, p.M - kRouterRows);
  const int r = lane & 31, h = lane >> 5;

  if (wave < 4) {
    // ---- 64 rows x 128 logits over k blocks wave, wave + 4, .. (K is 512 or more: every wave has one)
    const int stages = (kblocks - wave + 3) >> 2;
    const int vtiles = p.N / 32;
    const uint4* w = p.w + (int64_t)chunk * 4 * 512;
    const uint16_t* x = p.x + (int64_t)row0 * p.K;
    auto block = [&](int s) { return min(wave + 4 * s, kblocks - 1); };
    u32x4_t g4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      g4[i] = *(const u32x4_t*)(p.gamma + block(4 * i + (lane >> 4)) * kGroup + (lane & 15) * 8);
    uint32_t at[4];  // rows 4 i + lane / 16 of 16, in bytes
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * i + (lane >> 4);
      at[i] = (uint32_t)(row * p.K + (((lane & 15) ^ row) * 8)) * 2u;
    }
    auto fetch_x = [&](int s, uint4* slot) {
      router_fetch_block(x, s < stages ? p.K : 0, p.K, block(s), at, slot);
      __builtin_amdgcn_sched_barrier(0);
    };
    uint4 b[4][4];
    auto fetch_w = [&](int s, int j, uint4 (&d)[4]) {
      const uint4* from = w + ((int64_t)block(s) * vtiles * 8 + j) * 64;
#pragma unroll
      for (int t = 0; t < 4; ++t) d[t] = from[t * 512 + lane];
    };
    floatx16_t acc[2][4];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[rt][t][v] = 0.f;
    double ss[2] = {0.0, 0.0};
    fetch_x(0, a0[wave]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      __builtin_amdgcn_sched_barrier(0);
      fetch_w(0, j, b[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
    fetch_x(1, a1[wave]);
#pragma unroll
    for (int i = 0; i < 4; ++i) *(u32x4_t*)&sgamma[wave][i * 64 + lane] = g4[i];

    uint4 hi[2], lo[2], raw[2], gr[2];
    auto load = [&](const uint4* slot, int j, int rt) {
      uint32_t lane_at = (uint32_t)(r * 256 + ((8 * h) ^ (r & 15)) * 16);
      asm volatile("" : "+v"(lane_at));  // (one register, not one per slot, k step and row tile)
      return *(const uint4*)((const char*)slot + rt * 8192 + (lane_at ^ (j * 16)));
    };
    auto gamma_of = [&](int s, int j) { return sgamma[wave][(s & 15) * 16 + 8 * h + j]; };
    // sixteen groups of products, 32 rows and a k step each: the products of group u, the operands of u + 1, the reads of
    // u + 2. (Laid out group by group: the waits count the loads behind the one they are for.)
    auto stage = [&](int s, const uint4* slot, const uint4* next) {
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int j = u >> 1, rt = u & 1, j2 = ((u + 2) & 15) >> 1;
        __builtin_amdgcn_sched_barrier(0);
        const uint4 raw2 = load(u < 14 ? slot : next, j2, rt);
        if (rt == 0) gr[(j + 1) & 1] = gamma_of(u < 14 ? s : s + 1, j2);
        __builtin_amdgcn_sched_barrier(0);
        const bf16x8_t ah = operand(hi[u & 1]), al = operand(lo[u & 1]);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          floatx16_t& c = acc[rt][t];
          c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, operand(b[j & 3][t]), c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, operand(b[j & 3][t]), c, 0, 0, 0);
        }
        const double squares = (double)sumsq8(raw[(u + 1) & 1]);
        ss[(u + 1) & 1] += u < 15 || s + 1 < stages ? squares : 0.0;
        router_split(raw[(u + 1) & 1], gr[((u + 1) >> 1) & 1], hi[(u + 1) & 1], lo[(u + 1) & 1]);
        raw[u & 1] = raw2;
        __builtin_amdgcn_sched_barrier(0);
        if (rt == 1) fetch_w(j < 4 ? s : s + 1, (j + 4) & 7, b[j & 3]);
      }
    };
    raw[0] = load(a0[wave], 0, 0);
    raw[1] = load(a0[wave], 0, 1);
    gr[0] = gamma_of(0, 0);
    ss[0] += (double)sumsq8(raw[0]);
    router_split(raw[0], gr[0], hi[0], lo[0]);
#pragma unroll 1
    for (int s = 0; s + 1 < stages; s += 2) {
      stage(s, a0[wave], a1[wave]);
      fetch_x(s + 2, a0[wave]);
      stage(s + 1, a1[wave], a0[wave]);
      fetch_x(s + 3, a1[wave]);
    }
    if (stages & 1) stage(stages - 1, a0[wave], a1[wave]);
    __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      sq[wave][h][rt * 32 + r] = ss[rt];
      floatx4_t* part = (floatx4_t*)(rt == 0 ? a0[wave] : a1[wave]);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          part[(t * 4 + i) * 64 + lane] =
              floatx4_t{acc[rt][t][4 * i], acc[rt][t][4 * i + 1], acc[rt][t][4 * i + 2], acc[rt][t][4 * i + 3]};
    }
  } else {
    router_rows<KIND, ROUND>(p, row0, chunk * 4 + wave - 4, p.chunks * 4);
  }
  __syncthreads();
  router_factors(p, row0, sq, sfactor);
  __syncthreads();
  const floatx4_t* sums = (const floatx4_t*)(wave < 4 ? &a0[0][0] : &a1[0][0]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int set = (wave & 3) * 4 + i;  // of 16 sets of four rows and 32 columns
    floatx4_t v = sums[set * 64 + lane];
#pragma unroll
    for (int k = 1; k < 4; ++k) v += sums[k * (kRouterRows * 16) + set * 64 + lane];
    // register e of a 32x32 result holds row (e / 4) * 8 + (lane / 32) * 4 + e % 4, column lane % 32
    const int row = (wave >> 2) * 32 + (set & 3) * 8 + h * 4;
    const int col = (chunk * 4 + (set >> 2)) * 32 + r;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      p.logits[(int64_t)(row0 + row + e) * p.N + col] = router_logit(v[e], sfactor[row + e]);
  }
}

// ---------------------------------------------------------------------------
// An fp32 weight with gamma folded into it:
//   logits[m, :] = r[m] * sum_k x[m, k] * (gamma[k] * W[:, k])
// x is an operand as it lies in memory, so the two planes of gamma * W take two products instead of the four of
// (x * gamma) and W, and no operand arithmetic. The planes leave of gamma * W what those of W leave of W, where W has more
// bits than two planes hold: below 2^-17 of its size, so that the logits' error against 64 bits is the re-ordered form's
// (24-bit weights, 2.45-2.48e-6 of the logits' norm / 2.44-2.51e-6). A weight of 17 bits or fewer (fp16 values kept in fp32,
// say) loses nothing in its own planes and would in those of gamma * W (2.2e-6 for 2e-7). So a block of 64 logits and 64 columns in which a row or
// a column has more than half as many values of such a kind that the fold would cut as values of more bits (one in 128 of
// random ones is of that kind), or in which gamma * W leaves the range of bf16, keeps the planes of W, and the kernel below
// multiplies x by gamma there (fp16 values 1.4-5.7e-7 / 1.3-4.1e-7, bf16 ones 1.0-4.0e-7 / 1.0-2.8e-7: the sums' own
// rounding, more of it than where eight waves share K). The folding is done on every call: it depends on gamma. Bound by the
// latency of its loads, the choice's arithmetic and two barriers: without the choice a call takes 0.4-0.9 us less.
//
// The planes lie as the kernel below reads them: per slab of 64 columns and 32-column tile four k steps of hi, then lo,
// 64 lanes of 8 columns (16 ks + 8 (lane / 32) .. of row lane % 32); behind them a word per (64 logits, slab): 1 where W was
// kept. A workgroup has one block; 8 lanes read a row's 64 columns as one run.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void router_planes(const float (&v)[8], uint4& hi, uint4& lo) {  // the two bf16 terms
  float back[8];
  hi = pack8_bf16(v);
  unpack8(hi, back);
#pragma unroll
  for (int i = 0; i < 8; ++i) back[i] = v[i] - back[i];
  lo = pack8_bf16(back);
}

// a byte for each of four values: 1 where one of its seven lowest bits is set, that is, more than 17 bits
__device__ __forceinline__ unsigned low_bits_set(float a, float b, float c, float d) {
  const unsigned ab = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x0c0c0400);
  const unsigned cd = __builtin_amdgcn_perm(__float_as_uint(d), __float_as_uint(c), 0x04000c0c);
  return ((((ab | cd) & 0x7f7f7f7fu) + 0x7f7f7f7fu) >> 7) & 0x01010101u;
}
constexpr int kDppRowRor8 = 0x128;  // eight lanes on in a row of 16
template <int CTRL>
__device__ __forceinline__ unsigned dpp_add(unsigned v) {
  return v + (unsigned)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}

__global__ __launch_bounds__(512) void fold_router_weight_kernel(const float* __restrict__ wr,
                                                                 const uint16_t* __restrict__ gamma,
                                                                 uint4* __restrict__ folded, unsigned* __restrict__ kept,
                                                                 int K, int N) {
  // per column values of more than 17 bits, and those of fewer that the fold cuts: four columns a word
  __shared__ unsigned of_columns[4][8];
  __shared__ unsigned bad_rows;
  const int slabs = K / 64;
  const int chunk = wg_x() / slabs, slab = wg_x() - chunk * slabs;
  const int c = tid_x() & 7, row = tid_x() >> 3;  // piece of the block's 64 columns, row of 64
  const float4* src = (const float4*)(wr + (int64_t)(chunk * 64 + row) * K + slab * 64 + c * 8);
  const float4 a = src[0], b = src[1];
  const float w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  float g[8], z[8];
  unpack8(*(const uint4*)(gamma + slab * 64 + c * 8), g);
  if (tid_x() < 32) of_columns[tid_x() >> 3][c] = 0;
  if (tid_x() == 32) bad_rows = 0;
  __syncthreads();
  uint4 hi, lo;
  float largest = 0.f, smallest = __builtin_inff();
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    z[i] = w[i] * g[i];
    largest = fmaxf(largest, fabsf(z[i]));
    smallest = fminf(smallest, fabsf(z[i]));
  }
  bool bad = largest >= 0x1.ffp127f;  // rounded beyond the range
  if (__ballot(smallest < 0x1p-100f)) {  // lo may be denormal
#pragma unroll
    for (int i = 0; i < 8; ++i) bad |= (fabsf(z[i]) < 0x1p-100f) & (w[i] != 0.f) & (g[i] != 0.f);
  }
  unsigned columns[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    columns[i] = low_bits_set(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
    columns[2 + i] = low_bits_set(z[4 * i], z[4 * i + 1], z[4 * i + 2], z[4 * i + 3]) & ~columns[i];
  }
  router_planes(z, hi, lo);
  uint4* dst = folded + (((int64_t)slab * (N / 32) + chunk * 2 + (row >> 5)) * 4 + (c >> 1)) * 128 + (c & 1) * 32 + (row & 31);
  dst[0] = hi;  // (on their way while the choice is made: 4096 x 256 x 384 11.6 -> 11.3 us)
  dst[64] = lo;
  // of the row, 16 bits each
  unsigned counts = __builtin_popcount(columns[0]) + __builtin_popcount(columns[1]) +
                    ((__builtin_popcount(columns[2]) + __builtin_popcount(columns[3])) << 16);
  counts = dpp_add<kDppRowHalfMirror>(dpp_add<kDppQuadXor2>(dpp_add<kDppQuadXor1>(counts)));
#pragma unroll
  for (int i = 0; i < 4; ++i) columns[i] = dpp_add<kDppRowRor8>(columns[i]);  // of two rows
  const auto loses = [](unsigned more, unsigned cut) { return 2 * cut > more; };
  bad |= loses(counts & 0xffff, counts >> 16);
  if (__ballot(bad) && (tid_x() & 63) == 0) bad_rows = 1;
  if ((tid_x() & 8) == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) atomicAdd(&of_columns[i][c], columns[i]);
  }
  __syncthreads();
  // every wave looks at all columns: lane l at column l / 8 of piece l % 8
  const int word = (tid_x() & 63) >> 5, at = 8 * (row & 3);
  const bool bad_column = loses(of_columns[word][c] >> at & 0xff, of_columns[2 + word][c] >> at & 0xff);
  const bool keep = __ballot(bad_column) != 0 || bad_rows != 0;
  if (keep) {
    router_planes(w, hi, lo);
    dst[0] = hi;
    dst[64] = lo;
  }
  if (tid_x() == 0) kept[chunk * slabs + slab] = keep;
}

// 64 rows of a slab of 64 columns from memory into LDS, eight rows an instruction; at: this lane's byte offset in the
// first and the second eight of 16 rows. With valid = 0 (else K) nothing is read and zeros arrive.
__device__ __forceinline__ void router_fetch_slab(const uint16_t* x, int valid, int K, int slab, const uint32_t (&at)[2],
                                                  uint4* slot) {
  const __amdgpu_buffer_rsrc_t from =
      __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, kRouterRows * valid * 2, 0x00027000);
#pragma unroll
  for (int i = 0; i < kRouterRows / 8; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (lds_void_t*)(slot + i * 64), 16, at[i & 1],
                                             slab * 128 + (i >> 1) * 32 * K, 0, 0);
}

// 64 rows x 64 logits per workgroup of eight waves in two roles. Four multiply, each over every fourth slab of 64 columns
// for all of the logits, x asked for four slabs ahead and straight into LDS, W one slab ahead into registers; they share
// nothing until their sums meet at the end, so there is no barrier in the walk over K. The other four normalise and
// quantise the workgroup's share of the tile's rows meanwhile, so that y and the codes leave while the matrix cores work.
// Bound by what a CU can load: 1.5 MB at K = 4096 (W 1.0, x 0.5), which takes 20 us by itself (16 us with x in the L2),
// beside 15 us of the rows' reads and writes through the same path (counted together: 1.8 MB a CU from the L2, 56 KB a us;
// matrix cores busy 21 % of the time, vector units 31 %, the waves waiting to issue 48 % of theirs). Twice the slabs in flight or
// eight multiplying waves change nothing, 128 x 64 logits leave half of the CUs idle at 4096 rows.
// us of a call (64- or 32-row form, weight re-ordered / this, weight folded / W kept in a block of each chunk): 4096 x 256 x
// 4096 52.7 / 35.4 / 49.3, 2048 x 256 x 7168 69.3 / 50.2 / 63.7, 8192 x 256 x 2048 52.5 / 37.6 / 53.5, 4224 x 512 x 1024
// 40.6 / 28.8 / 42.0, 8192 x 128 x 2048 34.9 / 27.8 / 34.8, 1024 x 256 x 1536 17.1 / 14.9 / 20.3, 16384 x 256 x 1024
// 52.4 / 45.0 / 64.5.
// ---------------------------------------------------------------------------
template <int KIND, bool ROUND>
__global__ __launch_bounds__(512) void rmsnorm_router_quant_folded_kernel(RouterArgs p) {
  // slabs of x of each multiplying wave, a row's eight pieces XORed with half its number so that reads meet all banks;
  // afterwards the partial sums of the first and the second 32 rows. Four arrays: the compiler tells the loads into one
  // from those into another, and a read waits for its own slab only.
  __shared__ uint4 a0[4][kRouterRows * 8];
  __shared__ uint4 a1[4][kRouterRows * 8];
  __shared__ uint4 a2[4][kRouterRows * 8];
  __shared__ uint4 a3[4][kRouterRows * 8];
  __shared__ uint4 sgamma[4][256];          // of the slabs of a multiplying wave, where W was kept
  __shared__ double sq[4][2][kRouterRows];  // squares of a row: by wave and by half of its lanes
  __shared__ unsigned sfactor[kRouterRows];
  const int lane = tid_x() & 63;
  const int wave = uniform32(tid_x() >> 6);
  const int kblocks = p.K / kGroup;
  int tile, chunk;
  router_tile((p.M + kRouterRows - 1) / kRouterRows, p.chunks, tile, chunk);
  const int row0 = min(tile * kRouterRows, p.M - kRouterRows);
  const int r = lane & 31, h = lane >> 5;

  if (wave < 4) {
    // ---- 64 rows x 64 logits over slabs wave, wave + 4, .. (K is 256 or more: every wave has one)
    const int slabs = kblocks * 2;
    const int stages = (slabs - wave + 3) >> 2;
    floatx16_t acc[2][2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[rt][t][v] = 0.f;
    double ss[2] = {0.0, 0.0};
    const uint4* w = p.w + (int64_t)chunk * 1024;
    const uint16_t* x = p.x + (int64_t)row0 * p.K;
    auto slab_of = [&](int s) { return min(wave + 4 * s, slabs - 1); };
    uint32_t at[2];  // rows 8 i + lane / 8 of 16, in bytes
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = 8 * i + (lane >> 3);
      at[i] = (uint32_t)(row * p.K + (((lane & 7) ^ ((row >> 1) & 7)) * 8)) * 2u;
    }
    auto fetch_x = [&](int s, uint4* slot) {
      router_fetch_slab(x, s < stages ? p.K : 0, p.K, slab_of(s), at, slot);
    };
    uint4 b[4][4];  // [k step][tile 0 hi, lo, tile 1 hi, lo]: a set is refilled in place once it was used
    auto fetch_w = [&](int s, int ks, uint4 (&d)[4]) {
      const uint4* from = w + ((int64_t)slab_of(s) * (p.N / 32) * 8 + ks * 2) * 64;
#pragma unroll
      for (int t = 0; t < 4; ++t) d[t] = from[((t >> 1) * 8 + (t & 1)) * 64 + lane];
    };
    // the slabs whose planes are those of W itself (32 at most), one lane each
    const unsigned own = ((const unsigned*)(p.w + (int64_t)p.N * p.K / 4))[chunk * slabs + slab_of(lane & 31)];
    __builtin_amdgcn_sched_barrier(0);
    fetch_x(0, a0[wave]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      fetch_w(0, i, b[i]);
    }
    __builtin_amdgcn_sched_barrier(0);
    fetch_x(1, a1[wave]);
    fetch_x(2, a2[wave]);
    fetch_x(3, a3[wave]);
    __builtin_amdgcn_sched_barrier(0);
    const unsigned kept = (unsigned)__ballot(lane < stages && own);
    auto load = [&](const uint4* slot, int ks, int rt) {
      uint32_t lane_at = (uint32_t)(r * 128 + (h ^ ((r >> 1) & 7)) * 16);
      asm volatile("" : "+v"(lane_at));  // (one register, not one per slot, k step and row tile)
      return *(const uint4*)((const char*)slot + rt * 4096 + (lane_at ^ (ks * 32)));
    };
    // (the order of loads and products is laid out step by step: the waits count the loads behind the one they are for)
    auto walk = [&](auto kept_any) {
      constexpr bool kSplit = decltype(kept_any)::value;
      uint4 af[2][2];
      auto stage = [&](int s, const uint4* slot, const uint4* next) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
          for (int rt = 0; rt < 2; ++rt) af[(ks + 1) & 1][rt] = load(ks < 3 ? slot : next, (ks + 1) & 3, rt);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int rt = 0; rt < 2; ++rt) {
            const uint4 a = af[ks & 1][rt];
            ss[rt] += (double)sumsq8(a);
            uint4 hi = a, lo;
            if constexpr (kSplit) router_split(a, sgamma[wave][s * 8 + ks * 2 + h], hi, lo);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              floatx16_t& c = acc[rt][t >> 1];
              c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(operand(hi), operand(b[ks][t]), c, 0, 0, 0);
              if constexpr (kSplit) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(operand(lo), operand(b[ks][t]), c, 0, 0, 0);
            }
          }
          fetch_w(s + 1, ks, b[ks]);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) af[0][rt] = load(a0[wave], 0, rt);
      int s = 0;
#pragma unroll 1
      for (; s + 3 < stages; s += 4) {
        stage(s, a0[wave], a1[wave]);
        fetch_x(s + 4, a0[wave]);
        __builtin_amdgcn_sched_barrier(0);
        stage(s + 1, a1[wave], a2[wave]);
        fetch_x(s + 5, a1[wave]);
        __builtin_amdgcn_sched_barrier(0);
        stage(s + 2, a2[wave], a3[wave]);
        fetch_x(s + 6, a2[wave]);
        __builtin_amdgcn_sched_barrier(0);
        stage(s + 3, a3[wave], a0[wave]);
        fetch_x(s + 7, a3[wave]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (s < stages) stage(s, a0[wave], a1[wave]);
      if (s + 1 < stages) stage(s + 1, a1[wave], a2[wave]);
      if (s + 2 < stages) stage(s + 2, a2[wave], a3[wave]);
    };
    if (kept == 0) {
      walk(std::false_type{});
    } else {
      // 1 in the place of gamma where it is in the planes
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int slab = i * 8 + (lane >> 3);
        const uint4 one = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
        const uint4 g = *(const uint4*)(p.gamma + slab_of(slab) * 64 + (lane & 7) * 8);
        sgamma[wave][i * 64 + lane] = kept >> slab & 1 ? g : one;
      }
      walk(std::true_type{});
    }
    __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      sq[wave][h][rt * 32 + r] = ss[rt];
      floatx4_t* part = (floatx4_t*)(rt == 0 ? a0[wave] : a1[wave]);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          part[(t * 4 + i) * 64 + lane] =
              floatx4_t{acc[rt][t][4 * i], acc[rt][t][4 * i + 1], acc[rt][t][4 * i + 2], acc[rt][t][4 * i + 3]};
    }
  } else {
    router_rows<KIND, ROUND>(p, row0, chunk * 4 + wave - 4, p.chunks * 4);
  }
  __syncthreads();

  router_factors(p, row0, sq, sfactor);
  __syncthreads();
  const floatx4_t* sums = (const floatx4_t*)(wave < 4 ? &a0[0][0] : &a1[0][0]);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int set = (wave & 3) * 2 + i;  // of eight sets of four rows and 32 columns
    floatx4_t v = sums[set * 64 + lane];
#pragma unroll
    for (int k = 1; k < 4; ++k) v += sums[k * (kRouterRows * 8) + set * 64 + lane];
    // register e of a 32x32 result holds row (e / 4) * 8 + (lane / 32) * 4 + e % 4, column lane % 32
    const int row = (wave >> 2) * 32 + (set & 3) * 8 + h * 4;
    const int col = (chunk * 2 + (set >> 2)) * 32 + r;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      p.logits[(int64_t)(row0 + row + e) * p.N + col] = router_logit(v[e], sfactor[row + e]);
  }
}


// ---------------------------------------------------------------------------
// Calls whose row tiles and logits leave most of the chip without work, in two launches: the products over slices of K, as many
// as the chip has room for, then per row the sum over the slices, the statistic, y, codes and scales. What a slice leaves of a
// row's logits (fp32) lies in the row's own y and, where that is full, its own codes, which the second kernel reads before it
// writes them: no scratch, and the weight needs no re-ordering of its own ahead.
// 64 rows x 64 logits of a slice per workgroup of four waves. Per slab of 64 columns the threads turn x into its two operand
// terms and an fp32 weight into its two planes, in LDS, two slabs of both on their way; a wave multiplies 32 rows by 32 logits.
// PACKED: the weight in operand order (pack_router_weight), the same values and order of products.
// Bound by the operand arithmetic and LDS traffic of a slab (about 700 clocks each, of 500 of matrix instructions), which one
// workgroup on a CU overlaps little (two from 65 tiles on), and by two launches' latencies. us of the kernels, few-rows or 64-row form
// with its re-ordering of the weight / products + rows: 640 x 256 x 4608 fp32 6.8 + 32.8 / 15.0 + 5.6, 512 x 256 x 7168 bf16 5.9 + 19.6 /
// 12.9 + 6.3, 1024 x 512 x 4096 bf16 6.0 + 31.3 / 19.3 + 8.5. With six slices for the first (16.2) a k step for each
// wave (operands read from LDS once) took 17.8, operands loaded into registers in lane order, without LDS, 20.7.
// ---------------------------------------------------------------------------
struct RouterSliceArgs {
  RouterArgs a;
  int slices, y_slices;  // of which lie in y
};
__device__ __forceinline__ float* router_slice(const RouterSliceArgs& p, int64_t row, int slice) {
  uint8_t* in_y = (uint8_t*)(p.a.y + row * p.a.K) + (int64_t)slice * p.a.N * 4;
  uint8_t* in_q = p.a.q + row * p.a.K + (int64_t)(slice - p.y_slices) * p.a.N * 4;
  return (float*)(slice < p.y_slices ? in_y : in_q);
}

template <bool FP32W, bool PACKED>
__global__ __launch_bounds__(256) void router_slices_kernel(RouterSliceArgs p) {
  constexpr int P = FP32W ? 2 : 1;  // planes of W
  __shared__ uint4 sa[2][2][2][4][64];  // [buffer][hi, lo][32 rows][k step][lane slot]
  __shared__ uint4 sb[2][P][2][4][64];  // [buffer][plane][32 logits][k step][lane slot]
  const RouterArgs& a = p.a;
  const int tid = (int)tid_x(), lane = tid & 63;
  const int wave = uniform32(tid >> 6);
  const int c = tid & 7, r = tid >> 3;  // piece of eight columns of a slab, row (and r + 32)
  const int slice = (int)wg_x() % p.slices, tile = (int)wg_x() / p.slices;  // (with eight slices an XCD has its own part of K)
  const int col_tiles = a.N / 64;
  const int tile_m = tile / col_tiles, tile_n = tile - tile_m * col_tiles;
  const int row0 = min(tile_m * kRouterRows, a.M - kRouterRows);  // (rows that do not fill a tile are worked on twice)
  const int slabs = a.K / 64;
  const int first = slice * slabs / p.slices, last = (slice + 1) * slabs / p.slices - 1;
  struct Set {
    u32x4_t x[2], g, w[2][P];  // w: of logits r and r + 32, raw fp32 or planes
  } set[2];
  // 16 bytes at `at` of one of three arrays; nothing is read beyond the slice's last slab
  const int vtiles = a.N / 32 * P;
  const uint8_t* const w_base = (const uint8_t*)a.w + (PACKED ? (int64_t)tile_n * 2 * P * 8192 : (int64_t)tile_n * 64 * a.K * (P * 2));
  const uint32_t w_bytes = PACKED ? (uint32_t)((a.K / kGroup - 1) * vtiles + 2 * P) * 8192u : 64u * a.K * (P * 2);
  const uint32_t x_at = (uint32_t)(r * a.K + c * 8) * 2u, w_at = PACKED ? c * 1024u + r * 16u : x_at * P;
  auto load = [&](const void* base, uint32_t bytes, bool valid, uint32_t at, uint32_t from) {
    return __builtin_amdgcn_raw_buffer_load_b128(
        __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, valid ? bytes : 0, 0x00027000), at, from, 0);
  };
  auto fetch = [&](int slab, Set& d) {
    const bool valid = slab <= last;
    const uint32_t k = (uint32_t)slab * 64u, pitch = 64u * a.K;  // of 32 rows of x
#pragma unroll
    for (int u = 0; u < 2; ++u) d.x[u] = load(a.x + (int64_t)row0 * a.K, 2 * pitch, valid, x_at, u * pitch + k * 2);
    d.g = load(a.gamma, a.K * 2, valid, c * 16u, k * 2);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int v = 0; v < P; ++v)
        d.w[u][v] = PACKED ? load(w_base, w_bytes, valid, w_at, ((k >> 7) * vtiles + u * P + v) * 8192u + (k & 64) * 8u)
                           : load(w_base, w_bytes, valid, w_at + v * 16u, (u * pitch + k * 2) * P);
  };
  auto words = [](const u32x4_t& v) { return make_uint4(v[0], v[1], v[2], v[3]); };
  // (the position is XORed with the piece so that the eight lanes of a row write to different banks)
  const int slot = (c & 1) * 32 + (r ^ c), step = c >> 1;
  auto produce = [&](int buf, const Set& d) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      uint4 hi, lo;
      router_split(words(d.x[u]), words(d.g), hi, lo);
      sa[buf][0][u][step][slot] = hi;
      sa[buf][1][u][step][slot] = lo;
      if constexpr (FP32W && !PACKED) {
        float w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = __uint_as_float(d.w[u][i >> 2 & (P - 1)][i & 3]);
        router_planes(w, hi, lo);
        sb[buf][0][u][step][slot] = hi;
        sb[buf][P - 1][u][step][slot] = lo;
      } else {
#pragma unroll
        for (int v = 0; v < P; ++v) sb[buf][v][u][step][slot] = words(d.w[u][v]);
      }
    }
  };
  // the products of the leading terms apart from the others, and those of even k steps from those of odd ones: shorter chains
  // of roundings
  floatx16_t lead[2], rest;
#pragma unroll
  for (int v = 0; v < 16; ++v) lead[0][v] = lead[1][v] = rest[v] = 0.f;
  const int rt = wave & 1, ct = wave >> 1;
  auto multiply = [&](int buf) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int at = (lane & 32) + ((lane & 31) ^ (2 * ks + (lane >> 5)));
      const bf16x8_t hi = operand(sa[buf][0][rt][ks][at]), lo = operand(sa[buf][1][rt][ks][at]);
      const bf16x8_t w = operand(sb[buf][0][ct][ks][at]);
      lead[ks & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, w, lead[ks & 1], 0, 0, 0);
      rest = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, w, rest, 0, 0, 0);
      if constexpr (FP32W) {
        const bf16x8_t wl = operand(sb[buf][P - 1][ct][ks][at]);
        rest = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, wl, rest, 0, 0, 0);
        rest = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, wl, rest, 0, 0, 0);
      }
    }
  };
  fetch(first, set[0]);
  fetch(first + 1, set[1]);
  auto one = [&](int slab, int u) {
    produce(u, set[u]);
    fetch(slab + 2, set[u]);
    __syncthreads();
    multiply(u);
    __builtin_amdgcn_sched_barrier(0);  // (the next slab is not waited for earlier)
  };
  int slab = first;
#pragma unroll 1
  for (; slab < last; slab += 2) {  // (no branch inside: the waits count the loads behind the one they are for)
    one(slab, 0);
    one(slab + 1, 1);
  }
  if (slab == last) one(slab, 0);
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    // register v of a 32x32 result holds row (v / 4) * 8 + (lane / 32) * 4 + v % 4, column lane % 32
    const int row = row0 + rt * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
    router_slice(p, row, slice)[tile_n * 64 + ct * 32 + (lane & 31)] = (lead[0][v] + lead[1][v]) + rest[v];
  }
}

constexpr int kRouterSliceLogits = 1024;  // at most: four of a row for each of 256 threads
template <int NC, int KIND, bool ROUND>
__global__ __launch_bounds__(256) void router_finish_kernel(RouterSliceArgs p) {
  __shared__ double red[4];
  __shared__ unsigned nonfinite;
  const RouterArgs& a = p.a;
  const int tid = (int)tid_x();
  const int64_t row = wg_x();
  const int last = (a.K >> 3) - 1;
  uint4 raw[NC], gm[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) raw[k] = *(const uint4*)(a.x + row * a.K + min(tid + k * 256, last) * 8);
#pragma unroll
  for (int k = 0; k < NC; ++k) gm[k] = *(const uint4*)(a.gamma + min(tid + k * 256, last) * 8);
  float sum[kRouterSliceLogits / 256];
#pragma unroll
  for (int i = 0; i < kRouterSliceLogits / 256; ++i) {
    sum[i] = 0.f;
    const int n = tid + i * 256;
    if (n < a.N) {
#pragma unroll 1
      for (int s0 = 0; s0 < p.slices; s0 += 8) {
        float part[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) part[s] = router_slice(p, row, min(s0 + s, p.slices - 1))[n];
#pragma unroll
        for (int s = 0; s < 8; ++s) sum[i] += s0 + s < p.slices ? part[s] : 0.f;
      }
    }
  }
  double ss = 0.0;
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const float squares = sumsq8(raw[k]);
    ss += (double)(tid + k * 256 <= last ? squares : 0.f);
  }
  ss = wave_sum_d(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  if (tid == 0) nonfinite = 0;
  // the slices are in registers before any of the row's y and codes is written over them
#pragma unroll
  for (int i = 0; i < kRouterSliceLogits / 256; ++i) asm volatile("" : "+v"(sum[i]));
  __syncthreads();
  const float r = 1.0f / sqrtf((float)(((red[0] + red[1]) + red[2]) + red[3]) / (float)a.K + a.eps);
  unsigned factor = __float_as_uint(r);
  if (factor == 0) {  // workgroup-uniform
    bool bad = false;
#pragma unroll
    for (int k = 0; k < NC; ++k) bad |= router_nonfinite(raw[k]) || router_nonfinite(gm[k]);
    if (bad) nonfinite = 1;
    __syncthreads();
    if (nonfinite) factor = kNanBits;
  }
  if (tid == 0) a.rstd[row] = r;
#pragma unroll
  for (int i = 0; i < kRouterSliceLogits / 256; ++i) {
    const int n = tid + i * 256;
    if (n < a.N) a.logits[row * a.N + n] = router_logit(sum[i], factor);
  }
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = tid + k * 256;  // 16 lanes have a group, all of them or none a place in the row
    if (c <= last)
      router_emit<KIND, ROUND>(a.y + row * a.K + c * 8, a.q + row * a.K + c * 8, a.s + (int64_t)(c >> 4) * a.M + row,
                               (c & 15) == 0, raw[k], gm[k], r);
  }
}


int64_t rmsnorm_router_folded_scratch_bytes(int K, int N) {
  return (int64_t)N * K * 4 + (int64_t)(N / 64) * (K / 64) * 4;  // two bf16 planes, a word per block of 64 x 64
}

int64_t rmsnorm_router_scratch_bytes(int K, int N, int weight_fp32) {
  return (int64_t)N * K * (weight_fp32 ? 4 : 2);  // the bf16 planes of W in operand order
}

// W [N, K] (bf16 or fp32) -> the operand order of the main kernels.  A router weight changes once
// per optimiser step, so a caller can pack it once and reuse the result for every forward in between.
hipError_t launch_pack_router_weight(const void* wr, int weight_fp32, void* wpacked, int K, int N,
                                     hipStream_t stream) {
  const int n_halves = N / 16;  // half 32-column tiles; N and K are multiples of 128
  const dim3 grid((unsigned)((int64_t)n_halves * (K / kGroup)));
  if (weight_fp32)
    hipLaunchKernelGGL(pack_router_weight_kernel<true>, grid, dim3(256), 0, stream, wr, (uint4*)wpacked, K, n_halves);
  else
    hipLaunchKernelGGL(pack_router_weight_kernel<false>, grid, dim3(256), 0, stream, wr, (uint4*)wpacked, K, n_halves);
  return hipGetLastError();
}

struct RouterForm {
  int rows, cols;          // of a workgroup: rows of x, logits
  bool two_roles = false;  // 64 x 128 with the multiplying and the quantising waves apart
};

// which kernel, by the number of workgroups that each would have: fq_policy.hpp
static RouterForm router_form(int64_t M, int K, int N, bool weight_fp32) {
  const auto ceil_div = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t tiles = ceil_div(M, kRouterRows);
  const int kblocks = K / kGroup;
  if (M < kRouterRows || tiles * (N / 64) <= Policy::kRouterFewRowsMax) return {kRouterFewRows, 32};
  const bool narrow = !weight_fp32 && tiles * (N / 64) <= Policy::kRouterNarrowMax;
  const int cols64 = weight_fp32 || narrow ? 64 : 128;
  const bool two_roles = cols64 == 128 && N % 256 == 0 &&
                         (kblocks % 4 == 0 ? K >= Policy::kRouterTwoRolesMinK
                                           : N > 256 && K >= Policy::kRouterTwoRolesAlwaysK);
  const int cols32 = N % 512 == 0 && !weight_fp32 ? 512 : N % 256 == 0 ? 256 : 128;
  const int per_cu = cols32 == 128 ? 3 : cols32 == 256 && !weight_fp32 ? 2 : 1;
  const int64_t rounds64 = ceil_div(tiles * (N / cols64), 256);
  const int64_t slots = 256 * per_cu, workgroups32 = M / 32 * (N / cols32), rounds32 = ceil_div(workgroups32, slots);
  bool take32;
  if (per_cu == 1) {
    // in fifths of a round: one that leaves CUs free is shorter, the others' W arrives faster
    const int64_t fifths = rounds32 == 1 && rounds64 > 1 ? 3 * slots + 2 * workgroups32 : 5 * slots * rounds32;
    take32 = (kblocks + 25) * fifths <= 20 * 5 * slots * rounds64 ||
             (!weight_fp32 && !narrow && kblocks <= Policy::kRouter32ShortK);
  } else if (weight_fp32) {
    take32 = (kblocks + 10) * rounds32 <= 12 * rounds64;
  } else if (cols32 == 256) {
    take32 = narrow ? kblocks <= Policy::kRouter32ShortK : (kblocks + 12) * rounds32 <= 20 * rounds64;
  } else {
    take32 = !narrow && (kblocks + 34) * rounds32 <= 40 * rounds64;
  }
  if (two_roles && K >= Policy::kRouterTwoRolesAlwaysK) take32 = false;
  // a launch has less than 2^32 work-items; the 32-row form needs half as many as the others or less
  take32 |= tiles * (N / cols64) * 512 > (int64_t)UINT32_MAX;
  return take32 ? RouterForm{32, cols32} : RouterForm{kRouterRows, cols64, two_roles};
}

// An fp32 weight: whether folding gamma into it is the faster form. us of a call re-ordered / folded, number of 64 x 64
// workgroups behind the size. Fewer than the few-rows form takes, or half of them: 512 x 256 x 2048 (32) 13.5 / 17.5,
// 512 x 384 x 2048 (48) 21.9 / 18.0, x 7168 54.1 / 52.1, 1024 x 256 x 1536 (64) 17.2 / 15.1, x 1024 13.5 / 13.2, of which the
// re-ordering, that a caller may have done ahead, is 2.3. Short K: in one round 4096 x 256 (256) x 384 12.2 / 11.8, x 256
// 11.3 / 11.5; in more 8192 x 256 (512) x 896 26.2 / 25.1, x 768 23.8 / 23.5, x 640 20.6 / 22.1, 8192 x 512 x 896 44.3 / 42.7.
// With 128 logits a workgroup has 32 rows to quantise: 4096 x 128 x 768 15.7 / 15.7, x 1024 18.2 / 16.4, x 4096 48.5 / 40.6,
// 12288 x 128 x 896 27.3 / 28.6, x 1024 30.6 / 29.3, 8192 x 128 x 8192 126.9 / 122.5.
// (The Python entry point folds where there are no slices of K: of the calls of 41 to 64 workgroups those of a K below 1792 that
// makes three slices, and of more than 1024 logits.)
bool router_folds(int64_t M, int K, int N) {
  const int64_t workgroups = (M + kRouterRows - 1) / kRouterRows * (N / 64);
  if (M < kRouterRows || workgroups * 512 > (int64_t)UINT32_MAX) return false;
  if (N == 128 && K < 1024) return false;
  if (workgroups <= Policy::kRouterFewRowsMax)
    return N > 128 && K >= 1536 && workgroups > Policy::kRouterFewRowsMax / 2;
  return K >= (workgroups <= 256 ? 384 : 896);
}

// Slices of K of the two-launch form, 0 where a call takes another one: as many as make no more than 256 workgroups of 64 x 64
// (512 where there are more than 64 row and column tiles), as fit into y and the codes, at most 16. A few workgroups more are a
// round more (us, packed weight: 384 x 256 (24 tiles) x 4096 fp32 10 slices 14.9 / 11 17.2, 768 x 256 (48) x 4096 fp32 5
// 19.3 / 6 23.0, 1536 x 256 (96) x 4096 5 23.9 / 6 26.0). Fewer than three leave the chip idle still.
// A weight packed ahead takes the form that the weight as it is takes (same results, bit by bit), and packing it saves the
// other forms a launch. So the lines up to 64 tiles lie where the few-rows kernel alone is at most a few percent ahead (once,
// 320 x 384 x 3840, 12). It needs one round of workgroups up to 32 tiles and two up to 64. us of a packed call few-rows / slices,
// [of a call on the weight as it is], sizes that take the slices; then sizes that do not:
// up to 32 tiles, 128 logits, bf16: 128 x 128 (4) x 2048 8.7 / 8.3, 512 x 128 (16) x 3200 11.5 / 11.6, 640 x 128 (20) x 3328
// 11.7 / 12.1, 1024 x 128 (32) x 3840 13.7 / 14.0 [16.6 / 14.0], x 7168 21.7 / 18.9; 512 x 128 x 2048 9.1 / 10.1 [11.6 / 9.9],
// 1024 x 128 x 3072 10.7 / 12.6. fp32: 256 x 128 (8) x 2048 10.3 / 9.7, 512 x 128 x 2048 10.5 / 10.9 [14.2 / 10.7], 640 x 128 x
// 2560 11.6 / 12.5, 1024 x 128 x 3328 14.0 / 15.0 [18.2 / 15.0]; 512 x 128 x 1536 8.3 / 10.8, 1024 x 128 x 2048 11.1 / 11.7.
// ... more logits, bf16: 256 x 256 (16) x 3328 10.6 / 10.9, 512 x 256 (32) x 3840 12.4 / 12.6, x 4096 12.9 / 12.7 [17.1 / 12.6], x
// 7168 19.7 / 17.0, 256 x 512 (32) x 4096 (six slices) 13.0 / 13.5 [19.4 / 13.5], 320 x 384 (30) x 4096 13.0 / 14.1 [18.4 / 14.2],
// 128 x 1024 (32) x 7168 (four) 22.3 / 22.8 [30.6 / 22.6]; 512 x 256 x 2048 8.7 / 10.6 [11.8 / 10.5], x 3584 11.6 / 12.3 [15.5 / 12.1],
// 256 x 512 x 3584 (four) 11.2 / 14.6, 128 x 1024 x 4096 (three) 15.9 / 18.9 [23.3 / 18.7]. fp32: 256 x 256 x 3072 11.9 / 12.6
// [18.0 / 12.6], 512 x 256 x 3328 13.3 / 14.0 [19.5 / 13.9], x 4096 17.3 / 14.8, 256 x 512 x 3584 (four) 18.0 / 18.2 [24.8 / 18.7],
// 128 x 1024 x 4096 (three) 25.8 / 24.5; 512 x 256 x 1024 6.6 / 11.6 [10.3 / 11.6], x 3072 12.0 / 13.2 [18.2 / 13.2], 128 x 512 x 2048
// (three) 10.7 / 15.0.
// 33 to 64 tiles, bf16: 1024 x 256 (64) x 2048 14.0 / 13.0, x 3072 15.2 / 15.8 [19.5 / 15.8], 640 x 384 (60) x 3072 14.5 / 15.6
// [19.3 / 15.6], 512 x 512 (64) x 2304 (three) 14.1 / 14.8 [18.7 / 14.9]; x 2560 (three) 14.0 / 15.6. fp32: 2048 x 128 (64) x 1280
// 13.3 / 13.7, x 2048 19.9 / 16.3, 384 x 512 (48) x 2048 (three) 19.3 / 16.7; 2048 x 128 x 1024 11.8 / 12.9, 512 x 384 (48) x 1536
// (three) 13.4 / 14.3.
// Beyond, on the weight as it is, other forms / slices: 2048 x 256 (128) x 2048 22.5 / 21.2 (level with a packed weight), x 3072
// 30.5 / 22.2, 2560 x 256 (160) x 2048 22.9 / 23.8, x 4096 37.6 / 32.3, 1664 x 512 (208) x 3328 32.7 / 33.3; fp32, which fold gamma
// there, 4096 x 128 (128) x 2048 24.0 / 27.9, x 4096 52.7 / 42.8, 1536 x 256 (96) x 4096 31.1 / 34.6.
int router_slices(int64_t M, int K, int N, bool weight_fp32) {
  if (M < kRouterRows || N > kRouterSliceLogits) return 0;
  const int64_t tiles = (M + kRouterRows - 1) / kRouterRows * (N / 64);
  const int most = weight_fp32 ? (N == 128 && K >= 4096 ? 128 : 64) : (K >= 4096 ? 160 : K >= 2560 ? 128 : 64);
  if (tiles > most) return 0;
  const int64_t fill = (tiles <= 64 ? 256 : 512) / tiles;
  const int slices = (int)std::min<int64_t>({fill, K / (2 * N) + K / (4 * N), 16});
  if (slices < 3) return 0;
  int from = 0;  // least K
  if (tiles <= 32) {
    if (slices < 6 && weight_fp32) from = slices >= 4 && tiles >= 16 ? 3584 : tiles > 16 ? 3840 : INT_MAX;
    else if (slices < 6) from = slices >= 4 && tiles > 16 ? 6144 : INT_MAX;
    else if (weight_fp32 && N == 128) from = tiles <= 8 ? 1792 : tiles <= 20 ? 2048 : 3328;
    else if (weight_fp32) from = N == 256 && tiles > 16 ? 3328 : 3072;
    else if (N == 128) from = tiles <= 8 ? 2048 : tiles <= 16 ? 3200 : tiles <= 20 ? 3328 : 3840;
    else if (K < 4608 && K > (K < 4096 ? 550 : 700) * slices) from = INT_MAX;  // slices that are too long
    else from = tiles <= 16 ? 3328 : 3840;
  } else if (tiles <= 64) {
    from = weight_fp32 ? (slices >= 4 ? 1280 : 1792) : slices >= 4 || K <= 2304 ? 2048 : 3584;
  }
  return K >= from ? slices : 0;
}

template <bool FP32W, bool PACKED>
static hipError_t launch_router_slices(const RouterArgs& a, int slices, int round_scale, int kind, hipStream_t stream) {
  const RouterSliceArgs p{a, slices, std::min(slices, a.K / (2 * a.N))};
  const int64_t tiles = (int64_t)(a.M + kRouterRows - 1) / kRouterRows * (a.N / 64);
  hipLaunchKernelGGL((router_slices_kernel<FP32W, PACKED>), dim3((unsigned)(tiles * slices)), dim3(256), 0, stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
#define FQ_FINISH(NCV, KINDV, ROUNDV) \
  hipLaunchKernelGGL((router_finish_kernel<NCV, KINDV, ROUNDV>), dim3((unsigned)a.M), dim3(256), 0, stream, p)
#define FQ_FINISH_NC(KINDV, ROUNDV)                    \
  if (a.K <= 2048) FQ_FINISH(1, KINDV, ROUNDV);        \
  else if (a.K <= 4096) FQ_FINISH(2, KINDV, ROUNDV);   \
  else if (a.K <= 6144) FQ_FINISH(3, KINDV, ROUNDV);   \
  else FQ_FINISH(4, KINDV, ROUNDV);
  if (kind == kE5M2) {
    if (round_scale) { FQ_FINISH_NC(kE5M2, true) } else { FQ_FINISH_NC(kE5M2, false) }
  } else {
    if (round_scale) { FQ_FINISH_NC(kE4M3, true) } else { FQ_FINISH_NC(kE4M3, false) }
  }
#undef FQ_FINISH_NC
#undef FQ_FINISH
  return hipGetLastError();
}

// the main kernels on a weight already in operand order
hipError_t launch_rmsnorm_router_quant_packed(const void* x, const void* gamma, const void* wpacked,
                                              int weight_fp32, void* y, float* rstd, float* logits, void* q,
                                              float* s, int64_t M, int K, int N, float eps, int round_scale,
                                              int kind, hipStream_t stream) {
  if (M == 0) return hipSuccess;
  RouterArgs p{(const uint16_t*)x, (const uint16_t*)gamma, (const uint4*)wpacked, (uint16_t*)y, rstd, logits,
               (uint8_t*)q, s, (int)M, K, N, 0, eps};
  if (const int slices = router_slices(M, K, N, weight_fp32 != 0))
    return weight_fp32 ? launch_router_slices<true, true>(p, slices, round_scale, kind, stream)
                       : launch_router_slices<false, true>(p, slices, round_scale, kind, stream);
  const RouterForm f = router_form(M, K, N, weight_fp32 != 0);
  p.chunks = N / f.cols;
  const dim3 grid((unsigned)((M + f.rows - 1) / f.rows * p.chunks));
#define FQ_ROUTER_32(KINDV, ROUNDV, FP32V, VTV, WAVESV)                                                              \
  hipLaunchKernelGGL((rmsnorm_router_quant_32_rows_kernel<KINDV, ROUNDV, FP32V, VTV, WAVESV>), grid,                 \
                     dim3(64 * WAVESV), 0, stream, p)
#define FQ_ROUTER_GO(KINDV, ROUNDV, FP32V)                                                                           \
  if (f.rows == 32) {                                                                                                \
    if (f.cols == 128) FQ_ROUTER_32(KINDV, ROUNDV, FP32V, FP32V ? 2 : 1, 4);                                         \
    else if (FP32V || f.cols == 512) FQ_ROUTER_32(KINDV, ROUNDV, FP32V, 2, 8);                                       \
    else FQ_ROUTER_32(KINDV, ROUNDV, FP32V, FP32V ? 2 : 1, 8);                                                       \
  } else if (f.rows == kRouterFewRows)                                                                                                  \
    hipLaunchKernelGGL((rmsnorm_router_quant_few_rows_kernel<KINDV, ROUNDV, FP32V>), grid, dim3(512), 0, stream, p); \
  else if (!FP32V && f.two_roles)                                                                                      \
    hipLaunchKernelGGL((rmsnorm_router_quant_two_roles_kernel<KINDV, ROUNDV>), grid, dim3(512), 0, stream, p);           \
  else if (!FP32V && f.cols == 64)                                                                                     \
    hipLaunchKernelGGL((rmsnorm_router_quant_kernel<KINDV, ROUNDV, FP32V, FP32V ? 2 : 1>), grid, dim3(512), 0,       \
                       stream, p);                                                                                   \
  else                                                                                                               \
    hipLaunchKernelGGL((rmsnorm_router_quant_kernel<KINDV, ROUNDV, FP32V, 2>), grid, dim3(512), 0, stream, p);
#define FQ_ROUTER_ROUND(KINDV, FP32V)            \
  if (round_scale) {                             \
    FQ_ROUTER_GO(KINDV, true, FP32V)             \
  } else {                                       \
    FQ_ROUTER_GO(KINDV, false, FP32V)            \
  }
#define FQ_ROUTER_WEIGHT(KINDV)        \
  if (weight_fp32) {                   \
    FQ_ROUTER_ROUND(KINDV, true)       \
  } else {                             \
    FQ_ROUTER_ROUND(KINDV, false)      \
  }
  if (kind == kE5M2) {
    FQ_ROUTER_WEIGHT(kE5M2)
  } else {
    FQ_ROUTER_WEIGHT(kE4M3)
  }
#undef FQ_ROUTER_WEIGHT
#undef FQ_ROUTER_ROUND
#undef FQ_ROUTER_GO
#undef FQ_ROUTER_32
  return hipGetLastError();
}

hipError_t launch_rmsnorm_router_quant_folded(const void* x, const void* gamma, const void* wr, void* folded, void* y,
                                              float* rstd, float* logits, void* q, float* s, int64_t M, int K, int N,
                                              float eps, int round_scale, int kind, hipStream_t stream) {
  hipLaunchKernelGGL(fold_router_weight_kernel, dim3((unsigned)((N / 64) * (K / 64))), dim3(512), 0, stream,
                     (const float*)wr, (const uint16_t*)gamma, (uint4*)folded,
                     (unsigned*)((char*)folded + (int64_t)N * K * 4), K, N);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const RouterArgs p{(const uint16_t*)x, (const uint16_t*)gamma, (const uint4*)folded, (uint16_t*)y, rstd, logits,
                     (uint8_t*)q, s, (int)M, K, N, N / 64, eps};
  const dim3 grid((unsigned)((M + kRouterRows - 1) / kRouterRows * p.chunks));
#define FQ_ROUTER_FOLDED(KINDV, ROUNDV) \
  hipLaunchKernelGGL((rmsnorm_router_quant_folded_kernel<KINDV, ROUNDV>), grid, dim3(512), 0, stream, p)
  if (kind == kE5M2) {
    if (round_scale) FQ_ROUTER_FOLDED(kE5M2, true);
    else FQ_ROUTER_FOLDED(kE5M2, false);
  } else {
    if (round_scale) FQ_ROUTER_FOLDED(kE4M3, true);
    else FQ_ROUTER_FOLDED(kE4M3, false);
  }
#undef FQ_ROUTER_FOLDED
  return hipGetLastError();
}

hipError_t launch_rmsnorm_router_quant(const void* x, const void* gamma, const void* wr, int weight_fp32,
                                       void* wpacked, void* y, float* rstd, float* logits, void* q, float* s,
                                       int64_t M, int K, int N, float eps, int round_scale, int kind,
                                       hipStream_t stream) {
  if (M == 0) return hipSuccess;
  if (const int slices = router_slices(M, K, N, weight_fp32 != 0)) {  // (the weight as it is)
    const RouterArgs p{(const uint16_t*)x, (const uint16_t*)gamma, (const uint4*)wr, (uint16_t*)y, rstd, logits,
                       (uint8_t*)q, s, (int)M, K, N, 0, eps};
    return weight_fp32 ? launch_router_slices<true, false>(p, slices, round_scale, kind, stream)
                       : launch_router_slices<false, false>(p, slices, round_scale, kind, stream);
  }
  const hipError_t e = launch_pack_router_weight(wr, weight_fp32, wpacked, K, N, stream);
  if (e != hipSuccess) return e;
  return launch_rmsnorm_router_quant_packed(x, gamma, wpacked, weight_fp32, y, rstd, logits, q, s, M, K, N, eps,
                                            round_scale, kind, stream);
}

}  // namespace fq
