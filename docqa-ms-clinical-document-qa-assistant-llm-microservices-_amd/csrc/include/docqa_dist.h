// docqa_dist.h -- the fp32 / bf16 product of database rows with queries on MFMA that the flat
// index (knn.hip) and the IVF coarse quantizer (coarse.hip) share.
//
//   v[row, q] = norms[row] - 2 <x_row, q>  |  -<x_row, q>  |  <x_row, q>          (DistMode)
//
// Output layouts:
//   TILED      D[row / 32][q][row % 32] (one (tile, query) is 128 contiguous bytes, the store
//              of one MFMA tile 4 KB) and mins[q][row / 32], the least value of each tile;
//              rows past n, NaN and +inf are FLT_MAX, "missing" to the selection
//   row-major  D[q][row], no minima
//
// Three kernels.  knn_dist_kernel: 128 rows x QT queries a workgroup through an LDS-DMA ring.
// fp32 runs on v_mfma_f32_32x32x2_f32 (256 flops a clock and CU: 154 TFLOP/s measured), so a
// 64 x 64 wave tile needs 4 ds_read_b128 per 16 MFMAs of 64 clocks and is bound by the matrix
// cores from 64 queries on; QT = 32 keeps one query tile a wave and is bound by the database's bytes
// (250000 x 768 by 1 query: 134 us, 5.7 TB/s).  knn_dist_split_kernel: the flat search's fp32 products of
// 33 queries on, as bf16 parts (250000 x 768 by 256 queries, us: 778 as fp32, 550 so, of 590 GFLOP of
// bf16 at the 1.7 GHz this load runs at; by 40: 262 with the selection, now 217; 30000 x 768 by 256: 123, 100).
// knn_dist_small_kernel: 32 rows x 32 queries a workgroup with K split over
// its 4 or 8 waves, operands straight from memory: the shapes whose 128-row tiles leave CUs idle
// are bound by the latency of one K walk, which this cuts (dist_plan).
#pragma once
#include "docqa_asm.h"
#include "docqa_common.h"
#include <float.h>

namespace docqa {

enum DistMode { DIST_L2 = 0, DIST_IP = 1, DIST_DOT = 2 };

struct DistArgs {
  const void* xb;        // [n, rowbytes] database rows, fp32 or bf16
  const void* xq;        // [nq, rowbytes] queries, same type
  const float* norms;    // [n] (DIST_L2)
  float* D;
  float* mins;           // TILED: [nq, ldt]
  int n, nq, rowbytes, ldt, mode;
  const void* parts;     // the queries for knn_dist_split_kernel (knn_split_kernel's)
};

// 16-B chunk `ch` of `row` in a [rows][128 B] tile: 32-row fragment reads hit distinct banks
__device__ __forceinline__ uint32_t dist_swz(int row, int ch) {
  return (uint32_t)(row * 128 + ((ch ^ ((row >> 1) & 7)) << 4));
}

// the 32 bytes of a row that one fragment pair covers: 4 fp32 MFMAs of 2 k's (lane halves hold
// k's 4 apart, the same permutation in both operands) or one bf16 MFMA of 16.  Tiles innermost:
// consecutive MFMAs do not wait for each other's accumulator
template <bool BF16, int RI, int QI>
__device__ __forceinline__ void dist_mma(const uint4 (&a)[RI], const uint4 (&b)[QI], f32x16 (&acc)[RI][QI]) {
  if constexpr (BF16) {
#pragma unroll
    for (int i = 0; i < RI; ++i)
#pragma unroll
      for (int j = 0; j < QI; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(&a[i]),
                                                            *reinterpret_cast<const bf16x8*>(&b[j]), acc[i][j], 0, 0, 0);
  } else {
#define DOCQA_DIST_K(E)                                                                                      \
  _Pragma("unroll") for (int i = 0; i < RI; ++i) _Pragma("unroll") for (int j = 0; j < QI; ++j) acc[i][j] = \
      __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[i].E), __uint_as_float(b[j].E), acc[i][j], 0, 0, 0)
    DOCQA_DIST_K(x);
    DOCQA_DIST_K(y);
    DOCQA_DIST_K(z);
    DOCQA_DIST_K(w);
#undef DOCQA_DIST_K
  }
}

// first term of row's values, +inf for rows past the end (LDS copies it: one load a row)
__device__ __forceinline__ float dist_first(const DistArgs& p, int row) {
  return row >= p.n ? INFINITY : p.mode == DIST_L2 ? p.norms[row] : 0.f;
}

__device__ __forceinline__ float dist_factor(const DistArgs& p) {
  return p.mode == DIST_L2 ? -2.f : p.mode == DIST_IP ? -1.f : 1.f;
}

// rows row .. row + 3 (row % 4 == 0) of query q, f their first terms and c the products' factor;
// returns the least value.  TILED: values no list ever takes (+inf, NaN, rows past the end) are
// FLT_MAX; sums with 0 have no -0, so equal distances have one bit pattern
template <bool TILED>
__device__ __forceinline__ float dist_put(const DistArgs& p, int row, int q, const float4& f, float c, float d0, float d1,
                                          float d2, float d3) {
  float4 v = make_float4(f.x + c * d0, f.y + c * d1, f.z + c * d2, f.w + c * d3);
  if constexpr (TILED) {
    v.x = v.x < FLT_MAX ? v.x : FLT_MAX;
    v.y = v.y < FLT_MAX ? v.y : FLT_MAX;
    v.z = v.z < FLT_MAX ? v.z : FLT_MAX;
    v.w = v.w < FLT_MAX ? v.w : FLT_MAX;
    if (q < p.nq && (row & ~31) < p.n)
      *reinterpret_cast<float4*>(p.D + ((size_t)(row >> 5) * p.nq + q) * 32 + (row & 31)) = v;
    return fminf(fminf(v.x, v.y), fminf(v.z, v.w));
  } else {
    if (q < p.nq) {
      float* o = p.D + (size_t)q * p.n + row;
      if (row < p.n) o[0] = v.x;
      if (row + 1 < p.n) o[1] = v.y;
      if (row + 2 < p.n) o[2] = v.z;
      if (row + 3 < p.n) o[3] = v.w;
    }
    return 0.f;
  }
}

constexpr int kDistRows = 128;

// ---- fp32 as three bf16 parts.  Every value is the exact sum of three bf16 ones (8 + 8 + 8 bits, each rounded
// to nearest); of the nine products of two values the six down to 2^-16 of the largest run on the bf16 matrix
// cores, 16 times as fast as fp32's.  What is left out is 2^-25 of a product, and the sum has fewer roundings
// than an fp32 one (K / 16 x 6 for K / 2).  Against 64 bits, rms of the 10 nearest's distances, fp32 products /
// these: 100000 unit rows of 384 1.26e-7 / 1.11e-7, of 768 1.34e-7 / 1.16e-7, inner products 6.1e-8 / 5.1e-8.
__device__ __forceinline__ void dist_split(const uint4 (&x)[2], bf16x8 (&s)[3]) {
  uint32_t p[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint4& v = x[i >> 1];
    float a = __uint_as_float(i & 1 ? v.z : v.x), b = __uint_as_float(i & 1 ? v.w : v.y);
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      p[t][i] = pack2(a, b);
      a -= __uint_as_float(p[t][i] << 16);
      b -= __uint_as_float(p[t][i] & 0xffff0000u);
    }
  }
#pragma unroll
  for (int t = 0; t < 3; ++t) s[t] = __builtin_bit_cast(bf16x8, make_uint4(p[t][0], p[t][1], p[t][2], p[t][3]));
}

// A query's parts: 12 pieces of 16 bytes for 32 values (zeros past the end), piece (2 * 3 w + part 2 + h) the 8 values
// 16 w + 4 h .. + 3 and 16 w + 8 + 4 h .. + 3: what a fragment's lane half h holds of the database's fp32
inline int dist_parts_bytes(int rowbytes) { return (rowbytes + 127) / 128 * 192; }

static __global__ __launch_bounds__(256) void knn_split_kernel(const float* __restrict__ x, char* __restrict__ y, int nq, int d,
                                                        int blocks) {
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long q = e / (blocks * 4);
  const int u = (int)(e % (blocks * 4)), w = u >> 1, h = u & 1;   // 16 values' half
  if (q >= nq) return;
  uint4 v[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int k = w * 16 + g * 8 + h * 4;                         // d % 8 == 0: wholly inside or wholly past
    v[g] = k < d ? *reinterpret_cast<const uint4*>(x + q * d + k) : make_uint4(0, 0, 0, 0);
  }
  bf16x8 s[3];
  dist_split(v, s);
  char* o = y + q * (blocks * 192) + (w >> 1) * 192 + (w & 1) * 96 + h * 16;
#pragma unroll
  for (int t = 0; t < 3; ++t) *reinterpret_cast<bf16x8*>(o + t * 32) = s[t];
}

// 128 rows x QT queries a workgroup, a wave 32 rows: rows arrive as fp32 and are split once, by the wave that
// owns them (44 instructions for QT / 32 x 6 MFMAs of 32 clocks), the queries' parts as they are.  (Waves of
// 64 x 64, each row split by two: 657 us for 612 with the selection; 8 waves on 256 rows 626.)
template <int QT>
__global__ __launch_bounds__(256, 2) void knn_dist_split_kernel(DistArgs p, int nqt) {
  constexpr int QI = QT / 32, LA = kDistRows / 32, LQ = QT * 12 / 256;   // 16-B loads a thread and stage
  constexpr int SA = kDistRows * 128, STAGE = SA + QT * 192, NS = 2;   // 80 / 56 KB
  static_assert(NS * STAGE <= 80 * 1024, "two workgroups a CU");
  __shared__ __attribute__((aligned(16))) char smem[NS * STAGE];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);      // a row tile's query tiles share an XCD's L2
  const int row0 = (wg / nqt) * kDistRows, q0 = (wg % nqt) * QT;
  const int nch = p.rowbytes >> 4, nk = (nch + 7) >> 3, qbytes = nk * 192;
  const uint32_t lds = lds_u32(smem);

  const char* xt = (const char*)p.xb + (size_t)row0 * p.rowbytes;
  const char* qt = (const char*)p.parts + (size_t)q0 * qbytes;
  uint32_t off[LA], offq[LQ];
  const int lch = (tid & 7) ^ ((tid >> 4) & 7);
#pragma unroll
  for (int i = 0; i < LA; ++i)
    off[i] = (uint32_t)(min(i * 32 + (tid >> 3), p.n - 1 - row0) * p.rowbytes + lch * 16);
#pragma unroll
  for (int i = 0; i < LQ; ++i) {
    const int c = i * 256 + tid, r = c / 12;            // piece x of row r lies at x ^ (r >> 2 & 3): 16 rows' pieces
    offq[i] = (uint32_t)(min(r, p.nq - 1 - q0) * qbytes + ((c % 12) ^ ((r >> 2) & 3)) * 16);   // hit distinct banks
  }
  auto stage = [&](int kt, int buf) {
    const uint32_t base = lds + (uint32_t)(buf * STAGE + wave * 1024);
    // chunks past the row's end: its first ones, valid memory that no product reads
    const uint32_t at = kt * 8 + lch < nch ? (uint32_t)kt * 128 : 0u - (uint32_t)lch * 16;
#pragma unroll
    for (int i = 0; i < LA; ++i) glds16_off(xt, off[i] + at, __builtin_amdgcn_readfirstlane(base + (uint32_t)(i * 4096)));
#pragma unroll
    for (int i = 0; i < LQ; ++i)
      glds16_off(qt, offq[i] + (uint32_t)kt * 192, __builtin_amdgcn_readfirstlane(base + (uint32_t)(SA + i * 4096)));
  };
  const float f0 = tid < kDistRows ? dist_first(p, row0 + tid) : 0.f;   // (before the ring: its waits count loads)
  f32x16 acc[QI];
#pragma unroll
  for (int j = 0; j < QI; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;

#pragma unroll
  for (int t = 0; t < NS - 1; ++t)
    if (t < nk) stage(t, t);
  int buf = 0, kt = 0;
  auto arrive = [&]() {
    if (NS > 2 && kt + 1 < nk) wait_vmcnt<(NS - 2) * (LA + LQ)>();
    else wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ring_barrier();
    if (kt + NS - 1 < nk) stage(kt + NS - 1, buf ? buf - 1 : NS - 1);
  };
  // 16 values of the wave's rows (8 where not whole, the others 0), and of the queries
  auto read_a = [&](int w, bool whole, uint4 (&v)[2]) {
    const char* sa = smem + buf * STAGE;
#pragma unroll
    for (int g = 0; g < 2; ++g) v[g] = *reinterpret_cast<const uint4*>(sa + dist_swz(wave * 32 + l32, w * 4 + g * 2 + hh));
    if (!whole) v[1] = make_uint4(0, 0, 0, 0);
  };
  auto read_b = [&](int w, bf16x8 (&b)[QI][3]) {
    const char* sq = smem + buf * STAGE + SA;
#pragma unroll
    for (int j = 0; j < QI; ++j)
#pragma unroll
      for (int t = 0; t < 3; ++t)
        b[j][t] = *reinterpret_cast<const bf16x8*>(sq + (j * 32 + l32) * 192 +
                                                   (((w * 3 + t) * 2 + hh) ^ ((l32 >> 2) & 3)) * 16);
  };
  auto mma = [&](const bf16x8 (&a)[3], const bf16x8 (&b)[QI][3]) {
    constexpr int TA[6] = {2, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};   // the small products first
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int j = 0; j < QI; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[TA[t]], b[j][TB[t]], acc[j], 0, 0, 0);
  };
  // whole steps in a loop of their own, as above; the second half's parts are made between the first's products
  for (; kt < nch >> 3; ++kt) {
    arrive();
    uint4 v0[2], v1[2];
    bf16x8 a0[3], a1[3], b0[QI][3], b1[QI][3];
    read_a(0, true, v0);
    read_b(0, b0);
    read_a(1, true, v1);
    dist_split(v0, a0);
    __builtin_amdgcn_sched_barrier(0);
    mma(a0, b0);
    read_b(1, b1);
    dist_split(v1, a1);
#pragma unroll
    for (int i = 0; i < 3 * QI; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);          // a product
      __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);          // two vector instructions
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);          // an LDS read
      __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    mma(a1, b1);
    buf = buf + 1 == NS ? 0 : buf + 1;
  }
  if (kt < nk) {
    arrive();
    const int left = (nch - kt * 8) >> 1;               // 8 values each
    for (int u = 0; u < left; u += 2) {
      uint4 v[2];
      bf16x8 a[3], b[QI][3];
      read_a(u >> 1, u + 1 < left, v);
      read_b(u >> 1, b);
      dist_split(v, a);
      mma(a, b);
    }
  }

  // values that came out infinite or NaN (the parts of such an operand, or a large one's products, do) are
  // what fp32 products make them, straight from memory
#pragma unroll
  for (int j = 0; j < QI; ++j) {
    bool bad = false;
#pragma unroll
    for (int r = 0; r < 16; ++r) bad = bad || !(fabsf(acc[j][r]) < INFINITY);
    if (!__any(bad)) continue;
    f32x16 e[1][1];
#pragma unroll
    for (int r = 0; r < 16; ++r) e[0][0][r] = 0.f;
    const char* ar = xt + (size_t)min(wave * 32 + l32, p.n - 1 - row0) * p.rowbytes + hh * 16;
    const char* br = (const char*)p.xq + (size_t)min(q0 + j * 32 + l32, p.nq - 1) * p.rowbytes + hh * 16;
    for (int g = 0; g < p.rowbytes; g += 32) {
      const uint4 a[1] = {*reinterpret_cast<const uint4*>(ar + g)}, b[1] = {*reinterpret_cast<const uint4*>(br + g)};
      dist_mma<false, 1, 1>(a, b, e);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (!(fabsf(acc[j][r]) < INFINITY)) acc[j][r] = e[0][0][r];
  }

  __syncthreads();                                      // the ring is free: the rows' first terms
  float* first = reinterpret_cast<float*>(smem);
  if (tid < kDistRows) first[tid] = f0;
  __syncthreads();
  const float c = dist_factor(p);
  const int lt = wave * 32, tile = row0 + lt;
#pragma unroll
  for (int j = 0; j < QI; ++j) {
    const int q = q0 + j * 32 + l32;
    float mn = FLT_MAX;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 f = *reinterpret_cast<const float4*>(first + lt + 8 * g + 4 * hh);
      mn = fminf(mn, dist_put<true>(p, tile + 8 * g + 4 * hh, q, f, c, acc[j][4 * g], acc[j][4 * g + 1],
                                    acc[j][4 * g + 2], acc[j][4 * g + 3]));
    }
    mn = fminf(mn, __shfl_xor(mn, 32, 64));
    if (hh == 0 && q < p.nq && tile < p.n) p.mins[(size_t)q * p.ldt + (tile >> 5)] = mn;
  }
}

template <int QT, bool BF16, bool TILED>
__global__ __launch_bounds__(256, 2) void knn_dist_kernel(DistArgs p, int nqt) {
  constexpr int NS = QT == 128 ? 2 : 3;                 // ring stages: 64 / 72 / 60 KB, two workgroups a CU
  constexpr int WR = QT == 128 ? 2 : 4;                 // waves along the rows
  constexpr int RI = kDistRows / WR / 32, QI = QT * WR / 4 / 32;
  constexpr int LA = kDistRows / 32, LQ = QT / 32;      // 16-B loads a thread and stage
  constexpr int STAGE = (kDistRows + QT) * 128;
  __shared__ __attribute__((aligned(16))) char smem[NS * STAGE];
  __shared__ __attribute__((aligned(16))) float first[kDistRows];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);      // a row tile's query tiles share an XCD's L2
  const int row0 = (wg / nqt) * kDistRows, q0 = (wg % nqt) * QT;
  const int wr = wave % WR, wq = wave / WR;
  const int nch = p.rowbytes >> 4, nk = (nch + 7) >> 3;
  const uint32_t lds = lds_u32(smem);

  // per-lane source offsets from the tile's first row and query; past the end: the last row again
  const char* xt = (const char*)p.xb + (size_t)row0 * p.rowbytes;
  const char* qt = (const char*)p.xq + (size_t)q0 * p.rowbytes;
  uint32_t off[LA + LQ];
  const int lch = (tid & 7) ^ ((tid >> 4) & 7);          // logical chunk: (row >> 1) & 7 of every row of this thread
#pragma unroll
  for (int i = 0; i < LA + LQ; ++i) {
    const int r = (i < LA ? i : i - LA) * 32 + (tid >> 3);
    off[i] = (uint32_t)((i < LA ? min(r, p.n - 1 - row0) : min(r, p.nq - 1 - q0)) * p.rowbytes + lch * 16);
  }
  auto stage = [&](int kt, int buf) {
    const uint32_t base = lds + (uint32_t)(buf * STAGE + wave * 1024);
    // chunks past the row's end: its first ones, valid memory that no product reads
    const uint32_t at = kt * 8 + lch < nch ? (uint32_t)kt * 128 : 0u - (uint32_t)lch * 16;
#pragma unroll
    for (int i = 0; i < LA + LQ; ++i)
      glds16_off(i < LA ? xt : qt, off[i] + at, __builtin_amdgcn_readfirstlane(base + (uint32_t)(i * 4096)));
  };

  if (tid < kDistRows) first[tid] = dist_first(p, row0 + tid);   // (before the ring: its waits count loads)
  f32x16 acc[RI][QI];
#pragma unroll
  for (int i = 0; i < RI; ++i)
#pragma unroll
    for (int j = 0; j < QI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

#pragma unroll
  for (int t = 0; t < NS - 1; ++t)
    if (t < nk) stage(t, t);
  int buf = 0, kt = 0;
  auto arrive = [&]() {
    // the loads of stage kt have landed (those of the NS - 2 later stages may be in flight), and
    // every wave is done with the buffer that the next stage overwrites
    if (NS > 2 && kt + 1 < nk) wait_vmcnt<(NS - 2) * (LA + LQ)>();
    else wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ring_barrier();
    if (kt + NS - 1 < nk) stage(kt + NS - 1, buf ? buf - 1 : NS - 1);
  };
  auto group = [&](int u) {
    const char* sa = smem + buf * STAGE;
    const char* sq = sa + kDistRows * 128;
    uint4 a[RI], b[QI];
#pragma unroll
    for (int i = 0; i < RI; ++i)
      a[i] = *reinterpret_cast<const uint4*>(sa + dist_swz((wr * RI + i) * 32 + l32, u * 2 + hh));
#pragma unroll
    for (int j = 0; j < QI; ++j)
      b[j] = *reinterpret_cast<const uint4*>(sq + dist_swz((wq * QI + j) * 32 + l32, u * 2 + hh));
    dist_mma<BF16, RI, QI>(a, b, acc);
  };
  // whole 128-byte steps in a loop of their own: with a branch for the row's end in it hipcc
  // copied all accumulators twice a step behind a full MFMA drain (250000 x 256: 878 us)
  for (; kt < nch >> 3; ++kt) {
    arrive();
#pragma unroll
    for (int u = 0; u < 4; ++u) group(u);
    buf = buf + 1 == NS ? 0 : buf + 1;
  }
  if (kt < nk) {
    arrive();
    for (int u = 0; u < (nch - kt * 8) >> 1; ++u) group(u);
  }

  // lane: query l32 of its tile; registers 4g .. 4g + 3: rows 8g + 4hh .. + 3
  const float c = dist_factor(p);
#pragma unroll
  for (int i = 0; i < RI; ++i) {
    const int lt = (wr * RI + i) * 32, tile = row0 + lt;
#pragma unroll
    for (int j = 0; j < QI; ++j) {
      const int q = q0 + (wq * QI + j) * 32 + l32;
      float mn = FLT_MAX;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 f = *reinterpret_cast<const float4*>(first + lt + 8 * g + 4 * hh);
        mn = fminf(mn, dist_put<TILED>(p, tile + 8 * g + 4 * hh, q, f, c, acc[i][j][4 * g], acc[i][j][4 * g + 1],
                                       acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]));
      }
      if constexpr (TILED) {
        mn = fminf(mn, __shfl_xor(mn, 32, 64));
        if (hh == 0 && q < p.nq && tile < p.n) p.mins[(size_t)q * p.ldt + (tile >> 5)] = mn;
      }
    }
  }
}

template <bool BF16, bool TILED, int NW>
__global__ __launch_bounds__(64 * NW) void knn_dist_small_kernel(DistArgs p, int nqt) {
  __shared__ __attribute__((aligned(16))) float part[NW][32][36];    // [wave][query][row], rows padded
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, hh = lane >> 5;
  const int row0 = (blockIdx.x / nqt) * 32, q0 = (blockIdx.x % nqt) * 32;
  const char* xr = (const char*)p.xb + (size_t)min(row0 + l32, p.n - 1) * p.rowbytes + hh * 16;
  const char* qr = (const char*)p.xq + (size_t)min(q0 + l32, p.nq - 1) * p.rowbytes + hh * 16;
  // this wave's 32-byte groups of K
  const int ng = p.rowbytes >> 5, per = (ng + NW - 1) / NW;
  const int g0 = min(ng, wave * per), g1 = min(ng, g0 + per);
  f32x16 acc2[1][1];
  f32x16& acc = acc2[0][0];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  constexpr int U = 12;                                // groups in flight: 96 registers
  for (int g = g0; g < g1; g += U) {
    uint4 a[U][1], b[U][1];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int at = min(g + u, g1 - 1) * 32;          // past the end: valid memory, not used
      a[u][0] = *reinterpret_cast<const uint4*>(xr + at);
      b[u][0] = *reinterpret_cast<const uint4*>(qr + at);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (g + u < g1) dist_mma<BF16, 1, 1>(a[u], b[u], acc2);
  }
#pragma unroll
  for (int g = 0; g < 4; ++g)
    *reinterpret_cast<float4*>(&part[wave][l32][8 * g + 4 * hh]) =
        make_float4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]);
  __syncthreads();
  // thread: 4 rows of one query; the 8 threads of a query are neighbours
  if (tid >= 256) return;
  const int q = tid >> 3, r = (tid & 7) * 4;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < NW; w += 2)
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += part[w][q][r + e] + part[w + 1][q][r + e];
  const float4 f = make_float4(dist_first(p, row0 + r), dist_first(p, row0 + r + 1), dist_first(p, row0 + r + 2),
                               dist_first(p, row0 + r + 3));
  float mn = dist_put<TILED>(p, row0 + r, q0 + q, f, dist_factor(p), v[0], v[1], v[2], v[3]);
  if constexpr (TILED) {
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) mn = fminf(mn, __shfl_xor(mn, o, 64));
    if ((tid & 7) == 0 && q0 + q < p.nq) p.mins[(size_t)(q0 + q) * p.ldt + (row0 >> 5)] = mn;
  }
}

// queries of a workgroup's tile, 0: the small kernel.  The small kernel where its workgroups are
// about one a CU and a K walk is long enough to be worth cutting (us, small / 32-wide: fp32 d 384
// 8192 rows x 32 queries, 256 workgroups, 6.8 / 10.5, 2647 x 128, 332 of them, 9.5 / 10.2, 16384 x 33,
// 1024 of them, 18.1 / 10.5; bf16 d 768 2647 x 1 4.2 / 5.8, d 384 2647 x 33 5.2 / 4.3); else the
// widest tile that still has two workgroups a CU (32 as fp32 / 64 / 128 as parts, whole searches, fp32 d 384:
// 8192 x 256 31.6 / 32.2 / 36.9; 16384 x 256 47.7 / 40.6 / 41.2; 32768 x 256 76.8 / 60.0 / 55.1; d 768, 65536 x 48
// 71 / 59 / 78, x 100 126 / 95 / 84).
inline int dist_plan(int n, int nq, int rowbytes) {
  const long long rt = (n + kDistRows - 1) / kDistRows;
  if ((long long)((n + 31) / 32) * ((nq + 31) / 32) <= 320 && rowbytes >= 1024) return 0;
  for (int qt = 128; qt > 32; qt >>= 1)
    if (nq > qt / 2 && rt * ((nq + qt - 1) / qt) >= 512) return qt;
  return 32;
}

template <bool BF16, bool TILED>
inline void dist_launch(const DistArgs& p, hipStream_t s) {
  const int qt = dist_plan(p.n, p.nq, p.rowbytes);
  const int rt = (p.n + kDistRows - 1) / kDistRows;
  auto nt = [&](int w) { return (p.nq + w - 1) / w; };
  if (qt >= 64) {
    if constexpr (TILED && !BF16) {
      if (qt == 128) knn_dist_split_kernel<128><<<rt * nt(128), 256, 0, s>>>(p, nt(128));
      else knn_dist_split_kernel<64><<<rt * nt(64), 256, 0, s>>>(p, nt(64));
    } else {
      if (qt == 128) knn_dist_kernel<128, BF16, TILED><<<rt * nt(128), 256, 0, s>>>(p, nt(128));
      else knn_dist_kernel<64, BF16, TILED><<<rt * nt(64), 256, 0, s>>>(p, nt(64));
    }
  }
  else if (qt == 32) knn_dist_kernel<32, BF16, TILED><<<rt * nt(32), 256, 0, s>>>(p, nt(32));
  // 4 waves while each has its share of a row in flight at once, else 8 (fp32, 2647 rows by 32
  // queries, 4 / 8 waves: d 384 6.5 / 8.5 us, d 768 10.3 / 9.1)
  else if (p.rowbytes <= 4 * 12 * 32) knn_dist_small_kernel<BF16, TILED, 4><<<((p.n + 31) / 32) * nt(32), 256, 0, s>>>(p, nt(32));
  else knn_dist_small_kernel<BF16, TILED, 8><<<((p.n + 31) / 32) * nt(32), 512, 0, s>>>(p, nt(32));
}

}  // namespace docqa
