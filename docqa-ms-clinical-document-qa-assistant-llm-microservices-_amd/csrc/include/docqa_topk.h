// docqa_topk.h -- top-K selection and the merge of partial lists that the flat and IVF-PQ search
// kernels share.  Smaller is better throughout (inner-product scores are negated by the
// producers); ties break towards the lower candidate id.
#pragma once
#include "docqa_common.h"
#include <float.h>

namespace docqa {

// insertion network over a sorted register list (static indices only: no scratch)
template <int K>
__device__ __forceinline__ void topk_insert(float (&td)[K], int (&ti)[K], float d, int id) {
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const bool sw = d < td[i] || (d == td[i] && id < ti[i]);
    const float nd = sw ? td[i] : d;
    const int ni = sw ? ti[i] : id;
    td[i] = sw ? d : td[i];
    ti[i] = sw ? id : ti[i];
    d = nd;
    id = ni;
  }
}

// order-preserving uint32 key of a float: a < b  <=>  fkey(a) < fkey(b)
__device__ __forceinline__ uint32_t fkey(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// Block-wide top-K of the union of every thread's register list (td, ti: any order,
// FLT_MAX / -1 padding): the K smallest (distance, id) pairs, ties towards the lower id
// (ids compared unsigned, so -1 padding loses every tie), written to out_d / out_i [K] in
// ascending order.  Bisection on the composite key (fkey(distance), id) with block-wide
// counts -- ~32 rounds of K compares and one reduction each (the id round only when the
// K-th distance is tied) -- then one compaction and a rank placement by K threads.  Replaces
// a 256-leaf tree of K-long insertion networks (8 serial levels of K x K compare-swaps:
// at K = 64 it dominated the IVF-PQ scan with exact-refine candidate counts).
// lds: >= topk_select_lds(K) bytes of LDS scratch; every thread of the block must call it.
constexpr size_t topk_select_lds(int K) { return (size_t)K * 8 + 64; }

template <int K, int NT>
__device__ void block_select_topk(const float (&td)[K], const int (&ti)[K], float* __restrict__ out_d,
                                  int* __restrict__ out_i, unsigned char* lds) {
  constexpr int NW = NT / 64;
  static_assert(NT % 64 == 0 && NW <= 8 && K <= NT, "block_select_topk geometry");
  float* cd = reinterpret_cast<float*>(lds);               // [K] compacted candidates
  int* ci = reinterpret_cast<int*>(lds + K * 4);           // [K]
  int* red = reinterpret_cast<int*>(lds + K * 8);          // [NW] partial counts, [NW] fill
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t key[K];
#pragma unroll
  for (int i = 0; i < K; ++i) key[i] = fkey(td[i]);
  auto total = [&](int c) -> int {                         // block sum (uniform result)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    __syncthreads();                                       // the previous round's reads of red
    if (lane == 0) red[wave] = c;
    __syncthreads();
    int t = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) t += red[w];
    return t;
  };
  // smallest T with #{key <= T} >= K
  uint32_t lo = 0, hi = 0xffffffffu;
  while (lo < hi) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    int c = 0;
#pragma unroll
    for (int i = 0; i < K; ++i) c += key[i] <= mid;
    if (total(c) >= K) hi = mid;
    else lo = mid + 1;
  }
  const uint32_t T = lo;
  int cb = 0, ce = 0;
#pragma unroll
  for (int i = 0; i < K; ++i) { cb += key[i] < T; ce += key[i] <= T; }
  const int below = total(cb);
  uint32_t U = 0xffffffffu;
  if (total(ce) > K) {                                     // tied at T: smallest id bound
    uint32_t ilo = 0, ihi = 0xffffffffu;
    while (ilo < ihi) {
      const uint32_t mid = ilo + ((ihi - ilo) >> 1);
      int c = 0;
#pragma unroll
      for (int i = 0; i < K; ++i) c += key[i] == T && (uint32_t)ti[i] <= mid;
      if (below + total(c) >= K) ihi = mid;
      else ilo = mid + 1;
    }
    U = ilo;
  }
  // compaction: the `below` entries under T first (they all fit), then the tied ones up to
  // K -- in one pass a run of FLT_MAX / -1 padding (tied at T when fewer than K entries are
  // real) could take the slots of real entries
  __syncthreads();
  if (tid == 0) red[NW] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < K; ++i)
    if (key[i] < T) {
      const int p = atomicAdd(&red[NW], 1);
      cd[p] = td[i];
      ci[p] = ti[i];
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < K; ++i)
    if (key[i] == T && (uint32_t)ti[i] <= U) {
      const int p = atomicAdd(&red[NW], 1);                // padding duplicates may exceed K
      if (p < K) { cd[p] = td[i]; ci[p] = ti[i]; }
    }
  __syncthreads();
  if (tid < K) {
    const float v = cd[tid];
    const uint32_t kv = fkey(v), iv = (uint32_t)ci[tid];
    int r = 0;
    for (int m = 0; m < K; ++m) {
      const uint32_t km = fkey(cd[m]), im = (uint32_t)ci[m];
      r += km < kv || (km == kv && (im < iv || (im == iv && m < tid)));
    }
    out_d[r] = v;
    out_i[r] = ci[tid];
  }
  __syncthreads();
}

// ---- selection by 64-bit keys (order image of the distance, id): keys order as (distance, id)
// does, ids compared unsigned, so any order of arrival selects the same candidates
typedef unsigned long long u64;
constexpr int kCandBuf = 1024;   // candidates a workgroup holds

__device__ __forceinline__ u64 cand_key(float v, uint32_t id) { return ((u64)fkey(v) << 32) | id; }
__device__ __forceinline__ float key_value(u64 k) {
  const uint32_t t = (uint32_t)(k >> 32);
  return __uint_as_float((t & 0x80000000u) ? (t & 0x7fffffffu) : ~t);
}

// buf[0, n) of kCandBuf unique keys -> its K least in ascending order at buf[0, min(n, K)).  Few
// entries: every entry counts those below it; many: bitonic sort.  All 256 threads call it.
__device__ __forceinline__ void keep_best(u64* buf, int n, int K) {
  const int tid = threadIdx.x;
  if (n <= 256) {
    const u64 mine = tid < n ? buf[tid] : ~0ull;
    int r = 0;
    for (int j = 0; j < n; ++j) r += buf[j] < mine;
    __syncthreads();
    if (tid < n && r < K) buf[r] = mine;
    __syncthreads();
    return;
  }
  int P = 512;
  while (P < n) P <<= 1;
  for (int i = n + tid; i < P; i += 256) buf[i] = ~0ull;
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = tid; i < P / 2; i += 256) {
        const int a = 2 * i - (i & (j - 1)), b = a + j;
        const u64 x = buf[a], y = buf[b];
        if ((x > y) == ((a & k) == 0)) { buf[a] = y; buf[b] = x; }
      }
      __syncthreads();
    }
}

// Of the 256 threads' values, each the least of a share of its own: the K-th least (K <= 256),
// which bounds the K-th least of all shares from above; FLT_MAX where fewer threads have one.
// tm: 256 floats of LDS, 16-byte aligned.  All 256 threads call it.
__device__ __forceinline__ float bound_of_minima(float mine, int K, float* tm, float* out) {
  const int tid = threadIdx.x;
  tm[tid] = mine;
  if (tid == 0) *out = FLT_MAX;
  __syncthreads();
  int r = 0;
  for (int j = 0; j < 256; j += 4) {
    const float4 o = *reinterpret_cast<const float4*>(tm + j);
    r += (o.x < mine || (o.x == mine && j < tid)) + (o.y < mine || (o.y == mine && j + 1 < tid)) +
         (o.z < mine || (o.z == mine && j + 2 < tid)) + (o.w < mine || (o.w == mine && j + 3 < tid));
  }
  if (r == K - 1) *out = mine;
  __syncthreads();
  return *out;
}

// Merge a query's partial lists: ws_d / ws_i [nq][cnt], any order, FLT_MAX where nothing is; ids
// are positions that idmap translates to stored 64-bit ids.  Grid: queries.  The bound of the
// threads' minima leaves little more than k_out entries to order (64 lists of 64: 89 us as a
// bisection over 64 registers a thread, 6 us so).
static __global__ __launch_bounds__(256) void topk_merge_kernel(const float* __restrict__ ws_d, const int* __restrict__ ws_i,
                                                                int cnt, int k_out, float* __restrict__ out_d,
                                                                int64_t* __restrict__ out_i,
                                                                const int64_t* __restrict__ idmap) {
  __shared__ u64 buf[kCandBuf];
  __shared__ __attribute__((aligned(16))) float tm[256];
  __shared__ float s_b;
  __shared__ int s_n;
  const int q = blockIdx.x, tid = threadIdx.x;
  const float* dq = ws_d + (size_t)q * cnt;
  const int* iq = ws_i + (size_t)q * cnt;
  float mine = FLT_MAX;
  for (int c = tid; c < cnt; c += 256) mine = fminf(mine, dq[c]);
  if (tid == 0) s_n = 0;
  float most = bound_of_minima(mine, k_out, tm, &s_b);
  for (int c = tid; c < cnt; c += 256) {
    const float v = dq[c];
    if (v <= most && v < FLT_MAX) {
      const int at = atomicAdd(&s_n, 1);
      if (at < kCandBuf) buf[at] = cand_key(v, (uint32_t)iq[c]);
    }
  }
  __syncthreads();
  int n = s_n;
  if (n > kCandBuf) {            // equal distances by the thousand: in parts
    __syncthreads();
    n = 0;
    u64 bound = cand_key(most, 0xffffffffu);
    for (int c0 = 0; c0 < cnt; c0 += 256) {
      if (tid == 0) s_n = n;
      __syncthreads();
      const float v = c0 + tid < cnt ? dq[c0 + tid] : FLT_MAX;
      if (v < FLT_MAX) {
        const u64 key = cand_key(v, (uint32_t)iq[c0 + tid]);
        if (key <= bound) buf[atomicAdd(&s_n, 1)] = key;
      }
      __syncthreads();
      n = s_n;
      if (n > kCandBuf - 256) {
        keep_best(buf, n, k_out);
        n = k_out;
        bound = buf[k_out - 1];
      }
      __syncthreads();
    }
  }
  keep_best(buf, n, k_out);
  if (tid < k_out) {
    const bool ok = tid < n;
    const u64 key = ok ? buf[tid] : 0;
    out_d[(size_t)q * k_out + tid] = ok ? key_value(key) : FLT_MAX;
    out_i[(size_t)q * k_out + tid] = ok ? idmap[(uint32_t)key] : -1;
  }
}

}  // namespace docqa
