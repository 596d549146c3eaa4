// knn.hip -- exact brute-force k-nearest-neighbour search (FAISS IndexFlatL2 / IndexFlatIP
// semantics): distances on MFMA (docqa_dist.h), then a selection that reads almost none of them.
//
// Reference parity: FAISS IndexFlatL2 search through the LangChain retriever
// (llm-qa/main.py:101, k=3) over the 649 x 384 fp32 index written by
// semantic-indexer/indexer.py:27,41.  FAISS returns squared L2 distances
// ||x||^2 + ||y||^2 - 2 x.y in ascending order and int64 labels (-1 = missing).
//
// Selection.  The product kernel leaves every distance in a workspace and the least distance of
// each 32-row tile beside it.  The K-th least of any K tile minima bounds the K-th best distance
// from above, so a query's workgroup reads its minima (1 / 32 of the distances), bounds, and
// fetches only the tiles whose minimum is within the bound -- about K of them.  Candidates are
// ordered by (distance, row), so ties go to the lower row whatever order they arrive in.  Bound by
// the product, fp32: 250,000 x 768, 256 queries, k 10 takes 809 us, and 3780 us when 32 queries at
// a time read the rows uncoalesced and every lane kept a K-long sorted list; 2647 x 384, one
// query, k 3 takes 17 us, 83 before (6 workgroups, ||q||^2 summed by one thread).
//
// Batches whose distances exceed the workspace run in pieces: queries are independent, row
// pieces carry their K best along as (distance, row) pairs.
#include "docqa_dist.h"
#include "docqa_topk.h"

using namespace docqa;

namespace {

constexpr int kMaxK = 64;
constexpr int kTiles = 1024;    // tile list
// up to here, and where tile minima do not single tiles out (T <= 4 K), a query's workgroup reads
// every distance: 32 tiles, K 64: 156 -> 10 us a launch of 64 queries; 83 tiles, K 3 takes 9.7 us
// from the minima and 12.7 us so
constexpr int kFewTiles = 128;

// One query's K best of a piece of rows [row0, row0 + 32 T) and of those carried from earlier
// pieces.  Grid: queries.
__global__ __launch_bounds__(256) void knn_select_kernel(const float* __restrict__ D, const float* __restrict__ mins,
                                                         int T, int ldt, int nq, int K, uint32_t row0,
                                                         u64* __restrict__ carry, bool first, bool last,
                                                         const float* __restrict__ xq, int d, bool ip,
                                                         float* __restrict__ out_d, int64_t* __restrict__ out_i,
                                                         int64_t id_offset) {
  __shared__ u64 buf[kCandBuf];
  __shared__ int list[kTiles];
  __shared__ __attribute__((aligned(16))) float tm[256];
  __shared__ int s_n, s_t;
  __shared__ float s_qn[4], s_b;
  const int q = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* mq = mins + (size_t)q * ldt;
  // few tiles: the bound comes from the distances themselves, each thread's share of them; many:
  // from the tiles' minima
  const bool few = T <= kFewTiles && T <= 4 * K;
  auto dist_at = [&](int e) { return D[((size_t)(e >> 5) * nq + q) * 32 + (e & 31)]; };
  float mine = FLT_MAX;
  if (few)
    for (int e = tid; e < T * 32; e += 256) mine = fminf(mine, dist_at(e));
  else
    for (int t = tid; t < T; t += 256) mine = fminf(mine, mq[t]);
  if (tid == 0) s_t = 0;
  if (wave == 0) {                                       // carried keys: ascending, ~0 where there are fewer
    const u64 key = !first && lane < K ? carry[(size_t)q * K + lane] : ~0ull;
    buf[lane] = key;
    const u64 there = __ballot(key != ~0ull);
    if (lane == 0) s_n = (int)__popcll(there);
  }
  if (last && !ip) {
    float s = 0.f;
    for (int c = tid; c < d; c += 256) s += xq[(size_t)q * d + c] * xq[(size_t)q * d + c];
    s = wave_sum(s);
    if (lane == 0) s_qn[wave] = s;
  }
  float most = bound_of_minima(mine, K, tm, &s_b);
  int n = s_n;                                           // candidates held (uniform)
  u64 bound = min(cand_key(most, 0xffffffffu), buf[K - 1]);   // carried rows are the lower ones: ties are theirs
  most = fminf(most, key_value(buf[K - 1]));
  bool done = false;
  if (few) {
    for (int e = tid; e < T * 32; e += 256) {
      const float v = dist_at(e);
      const u64 key = cand_key(v, row0 + (uint32_t)e);
      if (v < FLT_MAX && key < bound) {
        const int at = atomicAdd(&s_n, 1);
        if (at < kCandBuf) buf[at] = key;
      }
    }
    __syncthreads();
    done = s_n <= kCandBuf;
    if (done) n = s_n;
    __syncthreads();
    if (!done && tid == 0) s_n = n;                      // equal rows by the hundred: the general way
  }
  // tiles within the bound; a list that overflows (equal rows by the thousand) is taken in parts
  int step = T;
  if (!done)
    for (int t = tid; t < T; t += 256)
      if (mq[t] <= most && mq[t] < FLT_MAX) {
        const int at = atomicAdd(&s_t, 1);
        if (at < kTiles) list[at] = t;
      }
  __syncthreads();
  if (s_t > kTiles) step = kTiles;
  for (int t0 = 0; t0 < T && !done; t0 += step) {
    if (step != T) {
      __syncthreads();
      if (tid == 0) s_t = 0;
      __syncthreads();
      for (int t = t0 + tid; t < min(T, t0 + step); t += 256)
        if (mq[t] <= most && mq[t] < FLT_MAX) list[atomicAdd(&s_t, 1)] = t;
      __syncthreads();
    }
    const int cnt = s_t;
    for (int i0 = 0; i0 < cnt; i0 += 8) {
      const int i = i0 + (tid >> 5);
      if (i < cnt) {
        const int t = list[i];
        const float v = D[((size_t)t * nq + q) * 32 + (tid & 31)];
        const u64 key = cand_key(v, row0 + (uint32_t)t * 32 + (tid & 31));
        if (v < FLT_MAX && key < bound) buf[atomicAdd(&s_n, 1)] = key;
      }
      __syncthreads();
      n = s_n;
      __syncthreads();                                   // (read by all before the next group counts on)
      if (n > kCandBuf - 256) {
        keep_best(buf, n, K);
        n = K;                                           // (n > K here)
        bound = buf[K - 1];
        if (tid == 0) s_n = K;
        __syncthreads();
      }
    }
    most = key_value(bound);
  }
  __syncthreads();
  keep_best(buf, n, K);
  if (tid < K) {
    const u64 key = tid < n ? buf[tid] : ~0ull;
    if (!last) {
      carry[(size_t)q * K + tid] = key;
    } else {
      const float v = key_value(key);
      const bool ok = key != ~0ull;
      const float qn = ip ? 0.f : (s_qn[0] + s_qn[1]) + (s_qn[2] + s_qn[3]);
      out_d[(size_t)q * K + tid] = ok ? (ip ? -v : v + qn) : (ip ? -FLT_MAX : FLT_MAX);
      out_i[(size_t)q * K + tid] = ok ? (int64_t)(uint32_t)key + id_offset : -1;
    }
  }
}

// bf16 database: the queries are rounded once to its type
__global__ __launch_bounds__(256) void knn_round_kernel(const float* __restrict__ x, uint16_t* __restrict__ y, size_t n8) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  float f[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = x[i * 8 + e];
  reinterpret_cast<uint4*>(y)[i] = pack8(f);
}

constexpr long long kPiece = 64ll << 20;     // distances a launch may leave in the workspace: 268 MB
}  // namespace

// pieces of n rows and c queries run on the queries' bf16 parts
static bool knn_splits(int n, int c, int d, int is_bf16) { return !is_bf16 && dist_plan(n, c, d * 4) >= 64; }

// queries and rows of a piece, and the workspace in bytes (docqa_knn lays it out):
// distances, minima, carried keys, rounded queries or the parts of a piece's
void docqa_knn_plan(int N, int nq, int d, int is_bf16, int k, int* qc, int* rc, size_t* bytes) {
  const long long n32 = ((long long)N + 31) / 32 * 32;
  long long c = nq, r = n32;
  if (c * r > kPiece) {
    c = nq < 1024 ? nq : 1024;
    r = n32 < kPiece / c ? n32 : kPiece / c / 128 * 128;
    c = kPiece / r < nq ? kPiece / r : nq;
  }
  *qc = (int)c;
  *rc = (int)r;
  *bytes = (size_t)c * r * 4 + (size_t)c * (r / 32) * 4 + 16 + (size_t)c * k * 8 + (is_bf16 ? (size_t)nq * d * 2 : 0);
  if (knn_splits(*rc < N ? *rc : N, *qc, d, is_bf16)) *bytes += (size_t)*qc * dist_parts_bytes(d * 4) + 16;
}

// xb / xq 16-byte aligned; k <= 64
int docqa_knn(const void* xb, const float* norms, int N, int d, int is_bf16, const float* xq, int nq, int k,
              int metric_ip, void* ws, float* out_d, int64_t* out_i, int64_t id_offset, hipStream_t s) {
  if (nq == 0) return 0;
  if (d % (is_bf16 ? 16 : 8) != 0 || N <= 0 || k < 1 || k > kMaxK) return -1;
  if (!docqa_aligned16(xb) || !docqa_aligned16(xq) || !docqa_aligned16(ws)) return -1;
  const int rowbytes = d * (is_bf16 ? 2 : 4);
  if ((size_t)32 * rowbytes > 160 * 1024) return -2;     // the widest rows this entry point takes
  int qc, rc;
  size_t bytes;
  docqa_knn_plan(N, nq, d, is_bf16, k, &qc, &rc, &bytes);
  char* at = (char*)ws;
  float* D = (float*)at;
  at += (size_t)qc * rc * 4;
  void* q16 = at;
  if (is_bf16) {
    at += (size_t)nq * d * 2;
    const size_t n8 = (size_t)nq * d / 8;
    knn_round_kernel<<<(unsigned)((n8 + 255) / 256), 256, 0, s>>>(xq, (uint16_t*)q16, n8);
  }
  u64* carry = (u64*)at;
  at += (size_t)qc * k * 8;
  float* mins = (float*)at;
  at += (size_t)qc * (rc / 32) * 4;
  void* parts = nullptr;
  if (knn_splits(rc < N ? rc : N, qc, d, is_bf16)) parts = (void*)(((uintptr_t)at + 15) & ~(uintptr_t)15);
  for (int q0 = 0; q0 < nq; q0 += qc) {
    const int c = nq - q0 < qc ? nq - q0 : qc;
    const float* xs = xq + (size_t)q0 * d;
    if (parts) {
      const int blocks = (d + 31) / 32;
      knn_split_kernel<<<(unsigned)(((long long)c * blocks * 4 + 255) / 256), 256, 0, s>>>(xs, (char*)parts, c, d, blocks);
    }
    for (int r0 = 0; r0 < N; r0 += rc) {
      const int n = N - r0 < rc ? N - r0 : rc, T = (n + 31) / 32;
      DistArgs p{(const char*)xb + (size_t)r0 * rowbytes,
                 is_bf16 ? (const void*)((const uint16_t*)q16 + (size_t)q0 * d) : (const void*)xs,
                 metric_ip ? nullptr : norms + r0, D, mins, n, c, rowbytes, T, metric_ip ? DIST_IP : DIST_L2,
                 parts};
      if (is_bf16) dist_launch<true, true>(p, s);
      else dist_launch<false, true>(p, s);
      knn_select_kernel<<<c, 256, 0, s>>>(D, mins, T, T, c, k, (uint32_t)r0, carry, r0 == 0, n == N - r0, xs, d,
                                          metric_ip != 0, out_d + (size_t)q0 * k, out_i + (size_t)q0 * k, id_offset);
    }
  }
  DOCQA_CHECK_LAUNCH();
  return 0;
}
