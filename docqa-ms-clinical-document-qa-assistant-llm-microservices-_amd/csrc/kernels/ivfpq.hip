// ivfpq.hip -- IVF-PQ asymmetric-distance (ADC) search for the 10M-vector
// semantic-indexer configuration (bge-base 768-d, nlist coarse cells, M x 8-bit PQ on
// the residuals), FAISS IndexIVFPQ semantics (by_residual, squared L2).
//
// Work item = (query, probed list), one 256-thread workgroup each:
//   1. residual query r = q - c_list into LDS;
//   2. distance look-up table LUT[m][k] = || r_m - pq[m][k] ||^2, M x 256 fp32 in LDS
//      (the PQ codebook, M*256*dsub floats, is L2-resident and shared by every item);
//   3. stream the list's codes (M bytes per vector, 16-byte loads) from HBM: each lane
//      sums M LDS look-ups per vector and keeps a register top-K (insertion network,
//      skipped wave-wide when no lane improves);
//   4. 256 per-lane lists merge through LDS -> top-K of the item -> workspace.
// A second launch (docqa_topk.h) merges the nprobe lists of each query and maps code
// positions to the stored 64-bit ids.
//
// The coarse step (q vs nlist centroids, top-nprobe) is the flat MFMA kNN kernel.
// Reference parity: the reference only has IndexFlatL2 (semantic-indexer/indexer.py:39);
// IVF-PQ is the BASELINE.json config-2 scale-out of the same search API.
#include "docqa_asm.h"
#include "docqa_common.h"
#include "docqa_topk.h"
#include <hip/hip_fp16.h>
#include <float.h>
#include <algorithm>

using namespace docqa;

namespace {

template <int K, bool VEC16>
__global__ __launch_bounds__(256) void ivfpq_scan_kernel(
    const float* __restrict__ xq, const float* __restrict__ centroids,
    const float* __restrict__ pq, const uint8_t* __restrict__ codes,
    const int64_t* __restrict__ list_off, const int64_t* __restrict__ probes, int nprobe, int d,
    int M, int dsub, float* __restrict__ ws_d, int* __restrict__ ws_i) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* lut = smem;                 // [M][256]
  float* qr = smem + M * 256;        // [d]
  const int item = blockIdx.x;
  const int q = item / nprobe;
  const int tid = threadIdx.x;
  const int64_t list = probes[item];
  const size_t ob = (size_t)item * K;
  if (list < 0) {
    if (tid < K) { ws_d[ob + tid] = FLT_MAX; ws_i[ob + tid] = -1; }
    return;
  }
  for (int c = tid; c < d; c += 256) qr[c] = xq[(size_t)q * d + c] - centroids[(size_t)list * d + c];
  __syncthreads();
  for (int idx = tid; idx < M * 256; idx += 256) {
    const int m = idx >> 8;
    const float* cen = pq + (size_t)idx * dsub;
    const float* r = qr + m * dsub;
    float s = 0.f;
    for (int j = 0; j < dsub; ++j) {
      const float t = r[j] - cen[j];
      s += t * t;
    }
    lut[idx] = s;
  }
  __syncthreads();

  float td[K];
  int ti[K];
#pragma unroll
  for (int i = 0; i < K; ++i) { td[i] = FLT_MAX; ti[i] = -1; }
  const int64_t lo = list_off[list], hi = list_off[list + 1];
  for (int64_t base = lo; base < hi; base += 256) {
    const int64_t i = base + tid;
    float dist = FLT_MAX;
    if (i < hi) {
      const uint8_t* row = codes + i * M;
      float s = 0.f;
      if constexpr (VEC16) {
        for (int m0 = 0; m0 < M; m0 += 16) {
          const uint4 w = *reinterpret_cast<const uint4*>(row + m0);
          const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int b = 0; b < 4; ++b)
              s += lut[(m0 + e * 4 + b) * 256 + ((ws[e] >> (8 * b)) & 0xff)];
        }
      } else {
        for (int m0 = 0; m0 < M; m0 += 4) {
          const uint32_t w = *reinterpret_cast<const uint32_t*>(row + m0);
#pragma unroll
          for (int b = 0; b < 4; ++b) s += lut[(m0 + b) * 256 + ((w >> (8 * b)) & 0xff)];
        }
      }
      dist = s;
    }
    if (__any(dist < td[K - 1])) {
      if (dist < td[K - 1]) topk_insert<K>(td, ti, dist, (int)i);
    }
  }
  // block top-K of the 256 lane lists (threshold select; LUT region reused)
  __syncthreads();
  float* sd = smem;
  int* si = reinterpret_cast<int*>(smem + K);
  block_select_topk<K, 256>(td, ti, sd, si, reinterpret_cast<unsigned char*>(smem + 2 * K));
  if (tid < K) { ws_d[ob + tid] = sd[tid]; ws_i[ob + tid] = si[tid]; }
}

// PQ encoding of residuals: codes[i][m] = argmin_k || (x_i - c_assign(i))_m - pq[m][k] ||^2.
// One wave per (vector, sub-quantizer) group of 64 candidate centroids x 4 passes.
__global__ __launch_bounds__(256) void pq_encode_kernel(const float* __restrict__ x,
                                                        const float* __restrict__ centroids,
                                                        const int64_t* __restrict__ assign,
                                                        const float* __restrict__ pq, int n, int d,
                                                        int M, int dsub, uint8_t* __restrict__ codes) {
  const int lane = threadIdx.x & 63;
  const long long total = (long long)n * M;
  const long long nwaves = (long long)gridDim.x * 4;
  // grid-stride over (vector, sub-quantizer) pairs: a 10M x 64 encode is 640M wave-tasks,
  // past HIP's 2^32 work-item launch limit if launched flat
  for (long long wave = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); wave < total; wave += nwaves) {
  const int i = (int)(wave / M), m = (int)(wave % M);
  const float* xr = x + (size_t)i * d + m * dsub;
  const float* cr = centroids + (size_t)assign[i] * d + m * dsub;
  float best = FLT_MAX;
  int bi = 0;
  for (int k = lane; k < 256; k += 64) {
    const float* cen = pq + ((size_t)m * 256 + k) * dsub;
    float s = 0.f;
    for (int j = 0; j < dsub; ++j) {
      const float t = xr[j] - cr[j] - cen[j];
      s += t * t;
    }
    if (s < best) { best = s; bi = k; }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(bi, o, 64);
    if (ob < best || (ob == best && oi < bi)) { best = ob; bi = oi; }
  }
  if (lane == 0) codes[(size_t)i * M + m] = (uint8_t)bi;
  }
}

// ---------------------------------------------------------------------------------------
// Precomputed-table ADC scan (FAISS's "precomputed tables" decomposition, taken one step
// further).  For a vector x = c_l + r^ (coarse centroid + PQ reconstruction of the residual)
//     ||q - x||^2 = ||q||^2 - 2 <q, c_l>  +  ||c_l + r^||^2  -  2 sum_m <q_m, pq[m][code_m]>
//                   `---- per (q, list) ---'  `- per vector -'  `---- per query LUT -----'
// so the LUT depends on the QUERY only -- T[q][m][k] = -2 <q_m, pq[m][k]>, computed once per
// query for every probe (query_tables_kernel, fp16: 48 KB at M = 96) -- the vector term N_i = ||c_l + r^_i||^2 is stored at add time, and the list term is
// one dot product per probe (query_tables_kernel).  The old kernel rebuilt an M x 256 fp32 LUT
// from the 768 KB codebook for every (query, list) item (profiles/r4_ivfpq_bge_10m_coarse_
// kernel.log: 14.8 ms per 256-query batch at nprobe 256 before any top-k work).
// Top-k is threshold-filtered: a lane appends a candidate to an LDS buffer only when it
// beats the current K-th best; when the buffer nears capacity a radix select keeps the K
// best and tightens the threshold -- the per-vector cost no longer grows with K (the old
// K-long register insertion networks made k_factor 4 cost 24.8 vs 14.8 ms).

constexpr int kLutSub = 8;      // sub-quantizers a workgroup
constexpr int kBaseProbes = 4;  // probes a wave

// Per query, in one launch: T[q][m][k] = -2 <q_m, pq[m][k]> (fp16), kLutSub sub-quantizers a
// workgroup with a thread per k, and base[q][p] = ||q||^2 - 2 <q, c_probe(q, p)>, kBaseProbes
// probes a wave.  Grid: nq x (ceil(M / kLutSub) + ceil(nprobe / 16)).  Bound by latency and the
// codebook's and centroids' bytes from L2; as two launches of one workgroup a query this was
// 39 + 59 us at 64 queries, M 96, 64 probes of d 768, on 64 of the 256 CUs.
__global__ __launch_bounds__(256) void query_tables_kernel(const float* __restrict__ xq, const float* __restrict__ pq,
                                                           const float* __restrict__ centroids,
                                                           const int64_t* __restrict__ probes, int nprobe, int d, int M, bool pq16,
                                                           __half* __restrict__ lut, float* __restrict__ base) {
  const int q = blockIdx.x, tid = threadIdx.x, nm = (M + kLutSub - 1) / kLutSub;
  const float* x = xq + (size_t)q * d;
  if ((int)blockIdx.y < nm) {
    const int dsub = d / M, m1 = min(M, ((int)blockIdx.y + 1) * kLutSub);
    for (int m = blockIdx.y * kLutSub; m < m1; ++m) {
      const float* cen = pq + ((size_t)m * 256 + tid) * dsub;
      const float* r = x + m * dsub;
      float s = 0.f;
      int j = 0;
      if (dsub % 4 == 0 && pq16)
        for (; j < dsub; j += 4) {
          const float4 c4 = *reinterpret_cast<const float4*>(cen + j);
          s += r[j] * c4.x;
          s += r[j + 1] * c4.y;
          s += r[j + 2] * c4.z;
          s += r[j + 3] * c4.w;
        }
      for (; j < dsub; ++j) s += r[j] * cen[j];
      lut[((size_t)q * M + m) * 256 + tid] = __float2half(-2.f * s);
    }
    return;
  }
  const int lane = tid & 63, p0 = ((int)blockIdx.y - nm) * 4 * kBaseProbes + (tid >> 6) * kBaseProbes;
  const float* c[kBaseProbes];
  bool ok[kBaseProbes];
  float dot[kBaseProbes], qn = 0.f;
#pragma unroll
  for (int e = 0; e < kBaseProbes; ++e) {
    const int64_t l = p0 + e < nprobe ? probes[(size_t)q * nprobe + p0 + e] : -1;
    ok[e] = l >= 0;
    c[e] = centroids + (size_t)(ok[e] ? l : 0) * d;
    dot[e] = 0.f;
  }
  for (int i = lane; i < d; i += 64) {
    const float v = x[i];
    qn += v * v;
#pragma unroll
    for (int e = 0; e < kBaseProbes; ++e) dot[e] += v * c[e][i];
  }
  qn = wave_sum(qn);
#pragma unroll
  for (int e = 0; e < kBaseProbes; ++e) {
    const float t = wave_sum(dot[e]);
    if (lane == 0 && p0 + e < nprobe) base[(size_t)q * nprobe + p0 + e] = ok[e] ? qn - 2.f * t : FLT_MAX;
  }
}

// out[r] = ||x_r||^2, a wave a row
__global__ __launch_bounds__(256) void row_norms_kernel(const float* __restrict__ x, int64_t n, int d, float* __restrict__ out) {
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= n) return;
  float s = 0.f;
  for (int i = threadIdx.x & 63; i < d; i += 64) {
    const float v = x[(size_t)r * d + i];
    s += v * v;
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) out[r] = s;
}

// Radix select over the LDS candidate buffer: keep the K smallest of n entries (ties at
// the K-th distance taken in buffer order), compacted to [0, min(n, K)); returns the K-th
// smallest distance (FLT_MAX when n < K).  Every thread calls it; CAP / 256 entries each.  hist
// may lie in the buffer: entries are in registers while it is in use.
template <int K, int CAP>
__device__ float buf_select(float* bd, int* bi, int n, int* hist, int* ctl) {
  constexpr int P = CAP / 256;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float vd[P];
  int vi[P];
  uint32_t key[P];
#pragma unroll
  for (int e = 0; e < P; ++e) {
    const int s = tid + e * 256;
    vd[e] = s < n ? bd[s] : FLT_MAX;
    vi[e] = s < n ? bi[s] : -1;
    key[e] = s < n ? fkey(vd[e]) : 0xffffffffu;
  }
  if (n <= K) {       // nothing to drop (uniform: n is read from LDS by every thread)
    return FLT_MAX;
  }
  __syncthreads();    // every entry read: hist may overwrite them
  uint32_t prefix = 0, mask = 0;
  int need = K;       // rank (1-based) of the wanted key among those matching the prefix
#pragma unroll
  for (int shift = 24; shift >= 0; shift -= 8) {
    hist[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < P; ++e)
      if ((key[e] & mask) == prefix) atomicAdd(&hist[(key[e] >> shift) & 255], 1);
    __syncthreads();
    // inclusive scan of the 256 bins: per wave (64 bins), then the wave totals
    int v = hist[tid];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(v, o, 64);
      if (lane >= o) v += t;
    }
    if (lane == 63) ctl[wave] = v;
    __syncthreads();
    int off = 0;
    for (int w = 0; w < wave; ++w) off += ctl[w];
    const int incl = v + off, excl = incl - hist[tid];
    if (excl < need && need <= incl) { ctl[4] = tid; ctl[5] = need - excl; }
    __syncthreads();
    prefix |= (uint32_t)ctl[4] << shift;
    mask |= 255u << shift;
    need = ctl[5];
    __syncthreads();
  }
  const uint32_t T = prefix;   // the K-th smallest key; `need` of the entries equal to it are kept
  if (tid == 0) { ctl[6] = 0; ctl[7] = 0; }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < P; ++e)
    if (key[e] < T) {
      const int p = atomicAdd(&ctl[6], 1);
      bd[p] = vd[e];
      bi[p] = vi[e];
    }
  __syncthreads();
  const int below = ctl[6];
#pragma unroll
  for (int e = 0; e < P; ++e)
    if (key[e] == T) {
      const int t = atomicAdd(&ctl[7], 1);
      if (t < need) {
        bd[below + t] = vd[e];
        bi[below + t] = vi[e];
      }
    }
  __syncthreads();
  return __uint_as_float((T & 0x80000000u) ? (T & 0x7fffffffu) : ~T);
}

// A workgroup scans pc probed lists of one query: LUT -> LDS, a lane a vector.  Bound by the LDS
// gathers (M two-byte look-ups a vector), so everything else is kept out of their way: the LUT
// comes by LDS-DMA, a vector's codes are all loaded before the first look-up (a 16-byte load ahead
// of every 16 look-ups waited for memory six times a vector), list bounds of 16 probes at once,
// and the buffers leave room for three workgroups a CU at M = 96 (53.5 KB each).
// 64 queries x 64 lists of 488 vectors, M 96: 129 -> 75 us.
constexpr int kScanBuf = 512;     // candidates buffered
constexpr int kScanMeta = 16;     // probes whose bounds are fetched together
constexpr size_t scan_lds(int M) { return (size_t)M * 512 + kScanBuf * 8 + 16 * 4 + kScanMeta * 12; }

template <int K, bool VEC16>
__global__ __launch_bounds__(256, 3) void ivfpq_scan_pt_kernel(
    const __half* __restrict__ lut, const float* __restrict__ base, const float* __restrict__ norms,
    const uint8_t* __restrict__ codes, const int64_t* __restrict__ list_off, const int64_t* __restrict__ probes,
    int nprobe, int pc, int nchunk, int M, float* __restrict__ ws_d, int* __restrict__ ws_i) {
  constexpr int CAP = kScanBuf;
  extern __shared__ __attribute__((aligned(16))) unsigned char pt_smem[];
  __half* slut = reinterpret_cast<__half*>(pt_smem);                  // [M][256]
  float* bd = reinterpret_cast<float*>(pt_smem + (size_t)M * 512);    // [CAP]
  int* bi = reinterpret_cast<int*>(bd + CAP);                          // [CAP]
  int* ctl = bi + CAP;                                                 // [8] select scratch, [8] count
  int* mlo = ctl + 16;                                                 // [kScanMeta] first vector, vectors, base
  int* mcnt = mlo + kScanMeta;
  float* mb = reinterpret_cast<float*>(mcnt + kScanMeta);
  const int q = blockIdx.x / nchunk, chunk = blockIdx.x % nchunk;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  {   // the query's LUT -> LDS, 1 KB a wave instruction
    const unsigned char* src = reinterpret_cast<const unsigned char*>(lut + (size_t)q * M * 256) + lane * 16;
    const uint32_t dst = lds_u32(pt_smem);
    for (int c = wave; c < M / 2; c += 4) glds16<false>(src + c * 1024, __builtin_amdgcn_readfirstlane(dst + c * 1024));
  }
  // insertion counters rotate over three LDS words so one barrier per pass suffices: pass j
  // appends through ctl[8 + j % 3] while thread 0 clears the word pass j + 1 will use (last
  // read after pass j - 2's barrier)
  if (tid < 3) ctl[8 + tid] = 0;
  float thr = FLT_MAX;
  int fill = 0, pass = 0;   // uniform: buffered candidates, passes so far
  const int p0 = chunk * pc, p1 = min(nprobe, p0 + pc);
  for (int pb = p0; pb < p1; pb += kScanMeta) {
    const int np = min(kScanMeta, p1 - pb);
    if (pb != p0) __syncthreads();
    if (tid < np) {
      const int64_t l = probes[(size_t)q * nprobe + pb + tid];
      mb[tid] = base[(size_t)q * nprobe + pb + tid];
      const int64_t lo = l < 0 ? 0 : list_off[l], hi = l < 0 ? 0 : list_off[l + 1];
      mlo[tid] = (int)lo;
      mcnt[tid] = (int)(hi - lo);
    }
    wait_vmcnt<0>();
    __syncthreads();
    for (int p = 0; p < np; ++p) {
      const int lo = mlo[p], cnt = mcnt[p];
      const float b = mb[p];
      for (int i0 = 0; i0 < cnt; i0 += 256) {
        const int i = lo + i0 + tid;
        float dist = FLT_MAX;
        if (i0 + tid < cnt) {
          const uint8_t* row = codes + (size_t)i * M;
          float s = b + norms[i], s2 = 0.f;
          if constexpr (VEC16) {
            constexpr int NV = 6;                                  // 96 codes in registers
            for (int m1 = 0; m1 < M; m1 += 16 * NV) {
              uint4 w[NV];
#pragma unroll
              for (int v = 0; v < NV; ++v)
                if (m1 + 16 * v < M) w[v] = *reinterpret_cast<const uint4*>(row + m1 + 16 * v);
#pragma unroll
              for (int v = 0; v < NV; ++v) {
                if (m1 + 16 * v >= M) break;
                const uint32_t ws[4] = {w[v].x, w[v].y, w[v].z, w[v].w};
                const __half* t = slut + (m1 + 16 * v) * 256;
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                  for (int bb = 0; bb < 4; bb += 2) {
                    s += __half2float(t[(e * 4 + bb) * 256 + ((ws[e] >> (8 * bb)) & 0xff)]);
                    s2 += __half2float(t[(e * 4 + bb + 1) * 256 + ((ws[e] >> (8 * bb + 8)) & 0xff)]);
                  }
              }
            }
          } else {
            for (int m0 = 0; m0 < M; m0 += 4) {
              const uint32_t w = *reinterpret_cast<const uint32_t*>(row + m0);
#pragma unroll
              for (int bb = 0; bb < 4; ++bb) s += __half2float(slut[(m0 + bb) * 256 + ((w >> (8 * bb)) & 0xff)]);
            }
          }
          dist = s + s2;
        }
        int* cnt_at = ctl + 8 + pass % 3;
        if (dist < thr) {
          const int pos = fill + atomicAdd(cnt_at, 1);
          bd[pos] = dist;
          bi[pos] = i;
        }
        if (tid == 0) ctl[8 + (pass + 1) % 3] = 0;
        __syncthreads();
        fill += *cnt_at;
        ++pass;
        if (fill > CAP - 256) {                                // uniform: nearly full
          thr = buf_select<K, CAP>(bd, bi, fill, bi, ctl);
          fill = min(fill, K);
        }
      }
    }
  }
  __syncthreads();
  const int n = fill;
  buf_select<K, CAP>(bd, bi, n, bi, ctl);
  const size_t ob = ((size_t)q * nchunk + chunk) * K;
  if (tid < K) {
    const bool ok = tid < min(n, K);
    ws_d[ob + tid] = ok ? bd[tid] : FLT_MAX;
    ws_i[ob + tid] = ok ? bi[tid] : -1;
  }
}

}  // namespace

// Precomputed-table IVF-PQ search (see ivfpq_scan_pt_kernel): norms [N] = ||c_l + r^_i||^2
// (list-major, like codes); lut_ws: >= nq * M * 256 halves; base_ws: >= nq * nprobe floats;
// ws_d / ws_i: >= nq * nchunk * kpad where nchunk = ceil(nprobe / pc).
int docqa_ivfpq_search_pt(const float* xq, const float* centroids, const float* pq, const uint8_t* codes,
                          const float* norms, const int64_t* ids, const int64_t* list_off, const int64_t* probes,
                          int nq, int nprobe, int d, int M, int k, int pc, void* lut_ws, float* base_ws,
                          float* ws_d, int* ws_i, float* out_d, int64_t* out_i, hipStream_t s) {
  if (nq == 0) return 0;
  if (d % M != 0 || M % 4 != 0 || pc < 1) return -1;
  const int kp = k <= 8 ? 8 : k <= 16 ? 16 : k <= 32 ? 32 : k <= 64 ? 64 : -1;
  if (kp < 0) return -1;
  const size_t lds = scan_lds(M);
  if (lds > 160 * 1024) return -2;
  __half* lut = (__half*)lut_ws;
  query_tables_kernel<<<dim3(nq, (M + kLutSub - 1) / kLutSub + (nprobe + 4 * kBaseProbes - 1) / (4 * kBaseProbes)), 256, 0, s>>>(
      xq, pq, centroids, probes, nprobe, d, M, docqa_aligned16(pq), lut, base_ws);
  const int nchunk = (nprobe + pc - 1) / pc;
  const int grid = nq * nchunk;
  const bool v16 = M % 16 == 0;
#define DOCQA_PT(K_)                                                                                            \
  do {                                                                                                          \
    if (v16)                                                                                                    \
      ivfpq_scan_pt_kernel<K_, true><<<grid, 256, lds, s>>>(lut, base_ws, norms, codes, list_off, probes, nprobe, \
                                                            pc, nchunk, M, ws_d, ws_i);                          \
    else                                                                                                        \
      ivfpq_scan_pt_kernel<K_, false><<<grid, 256, lds, s>>>(lut, base_ws, norms, codes, list_off, probes,       \
                                                             nprobe, pc, nchunk, M, ws_d, ws_i);                 \
    topk_merge_kernel<<<nq, 256, 0, s>>>(ws_d, ws_i, nchunk * K_, k, out_d, out_i, ids);                         \
  } while (0)
  switch (kp) {
    case 8: DOCQA_PT(8); break;
    case 16: DOCQA_PT(16); break;
    case 32: DOCQA_PT(32); break;
    default: DOCQA_PT(64); break;
  }
#undef DOCQA_PT
  DOCQA_CHECK_LAUNCH();
  return 0;
}

namespace {
// Exact re-rank of IVF-PQ candidates (FAISS IndexRefineFlat): per query one workgroup of 16
// waves, a wave per candidate -- gather the stored vector (fp32 or bf16), squared L2 (IP: inner
// product) to the query, then the k best of the <= 64 candidates by rank counting (ties to the
// lower candidate slot).  Bound by the latency of the gathers: 16 waves with up to 4 candidates
// each in flight at once (VEC: 4 elements a load; 64 queries x 40 candidates of d 768 took 43 us
// with 4 waves and a candidate at a time).  out: D [nq, k] (+inf / -inf and id -1 for missing), I [nq, k].
template <bool BF16, bool IP, bool VEC>
__global__ __launch_bounds__(1024) void refine_l2_kernel(const void* __restrict__ xb, const float* __restrict__ xq,
                                                         const int64_t* __restrict__ cand, int kc, int d, int k,
                                                         int64_t ntotal, float* __restrict__ out_d,
                                                         int64_t* __restrict__ out_i) {
  __shared__ float dist[64];
  constexpr int E = VEC ? 4 : 1, R = 4;
  const int q = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* x = xq + (size_t)q * d;
  size_t row[R];
  bool ok[R];
  float s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int j = wave + 16 * r;
    const int64_t id = j < kc ? cand[(size_t)q * kc + j] : -1;
    ok[r] = id >= 0 && id < ntotal;
    row[r] = (size_t)(ok[r] ? id : 0) * d;
    s[r] = 0.f;
  }
  for (int c = lane * E; c < d; c += 64 * E) {
    float a[E];
    if constexpr (VEC) *reinterpret_cast<float4*>(a) = *reinterpret_cast<const float4*>(x + c);
    else a[0] = x[c];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (!ok[r]) continue;                               // (uniform in the wave)
      float v[E];
      if constexpr (BF16 && VEC) {
        const uint2 w = *reinterpret_cast<const uint2*>((const uint16_t*)xb + row[r] + c);
        v[0] = __uint_as_float(w.x << 16);
        v[1] = __uint_as_float(w.x & 0xffff0000u);
        v[2] = __uint_as_float(w.y << 16);
        v[3] = __uint_as_float(w.y & 0xffff0000u);
      } else if constexpr (BF16) {
        v[0] = bf2f(((const uint16_t*)xb)[row[r] + c]);
      } else if constexpr (VEC) {
        *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>((const float*)xb + row[r] + c);
      } else {
        v[0] = ((const float*)xb)[row[r] + c];
      }
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float t = v[e] - a[e];
        s[r] += IP ? v[e] * a[e] : t * t;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float t = wave_sum(s[r]);
    if (lane == 0 && wave + 16 * r < kc) dist[wave + 16 * r] = ok[r] ? (IP ? -t : t) : FLT_MAX;
  }
  __syncthreads();
  if (tid < kc) {
    const float v = dist[tid];
    int r = 0;
    for (int j = 0; j < kc; ++j) {
      const float u = dist[j];
      r += u < v || (u == v && j < tid);
    }
    if (r < k) {
      const bool ok = v != FLT_MAX;
      out_d[(size_t)q * k + r] = ok ? (IP ? -v : v) : (IP ? -INFINITY : INFINITY);
      out_i[(size_t)q * k + r] = ok ? cand[(size_t)q * kc + tid] : -1;
    }
  }
  // fewer candidates than k: the rest stays missing
  for (int r = kc + tid; r < k; r += 1024) {
    out_d[(size_t)q * k + r] = IP ? -INFINITY : INFINITY;
    out_i[(size_t)q * k + r] = -1;
  }
}
}  // namespace

int docqa_refine_flat(const void* xb, int xb_bf16, int64_t ntotal, const float* xq, const int64_t* cand, int nq,
                      int kc, int d, int k, int ip, float* out_d, int64_t* out_i, hipStream_t s) {
  if (nq == 0) return 0;
  if (kc < 1 || kc > 64 || k < 1) return -1;
  const bool vec = d % 4 == 0 && docqa_aligned16(xb) && docqa_aligned16(xq);
  auto* kern = vec ? (xb_bf16 ? (ip ? refine_l2_kernel<true, true, true> : refine_l2_kernel<true, false, true>)
                              : (ip ? refine_l2_kernel<false, true, true> : refine_l2_kernel<false, false, true>))
                   : (xb_bf16 ? (ip ? refine_l2_kernel<true, true, false> : refine_l2_kernel<true, false, false>)
                              : (ip ? refine_l2_kernel<false, true, false> : refine_l2_kernel<false, false, false>));
  kern<<<nq, 1024, 0, s>>>(xb, xq, cand, kc, d, k, ntotal, out_d, out_i);
  DOCQA_CHECK_LAUNCH();
  return 0;
}

template <int K>
static int launch_scan(const float* xq, const float* cent, const float* pq, const uint8_t* codes,
                       const int64_t* list_off, const int64_t* probes, int nq, int nprobe, int d,
                       int M, float* ws_d, int* ws_i, hipStream_t s) {
  const int dsub = d / M;
  size_t lds = (size_t)(M * 256 + d) * 4;
  const size_t merge = (size_t)K * 8 + topk_select_lds(K);
  if (merge > lds) lds = merge;
  if (lds > 160 * 1024) return -2;
  const int items = nq * nprobe;
  if (M % 16 == 0)
    ivfpq_scan_kernel<K, true><<<items, 256, lds, s>>>(xq, cent, pq, codes, list_off, probes, nprobe, d, M, dsub, ws_d, ws_i);
  else
    ivfpq_scan_kernel<K, false><<<items, 256, lds, s>>>(xq, cent, pq, codes, list_off, probes, nprobe, d, M, dsub, ws_d, ws_i);
  return 0;
}

int docqa_ivfpq_search(const float* xq, const float* centroids, const float* pq,
                       const uint8_t* codes, const int64_t* ids, const int64_t* list_off,
                       const int64_t* probes, int nq, int nprobe, int d, int M, int k,
                       float* ws_d, int* ws_i, float* out_d, int64_t* out_i, hipStream_t s) {
  if (nq == 0) return 0;
  if (d % M != 0 || M % 4 != 0) return -1;
  const int kp = k <= 4 ? 4 : k <= 8 ? 8 : k <= 16 ? 16 : k <= 32 ? 32 : k <= 64 ? 64 : -1;
  int rc;
  switch (kp) {
    case 4: rc = launch_scan<4>(xq, centroids, pq, codes, list_off, probes, nq, nprobe, d, M, ws_d, ws_i, s);
      if (!rc) topk_merge_kernel<<<nq, 256, 0, s>>>(ws_d, ws_i, nprobe * 4, k, out_d, out_i, ids);
      break;
    case 8: rc = launch_scan<8>(xq, centroids, pq, codes, list_off, probes, nq, nprobe, d, M, ws_d, ws_i, s);
      if (!rc) topk_merge_kernel<<<nq, 256, 0, s>>>(ws_d, ws_i, nprobe * 8, k, out_d, out_i, ids);
      break;
    case 16: rc = launch_scan<16>(xq, centroids, pq, codes, list_off, probes, nq, nprobe, d, M, ws_d, ws_i, s);
      if (!rc) topk_merge_kernel<<<nq, 256, 0, s>>>(ws_d, ws_i, nprobe * 16, k, out_d, out_i, ids);
      break;
    case 32: rc = launch_scan<32>(xq, centroids, pq, codes, list_off, probes, nq, nprobe, d, M, ws_d, ws_i, s);
      if (!rc) topk_merge_kernel<<<nq, 256, 0, s>>>(ws_d, ws_i, nprobe * 32, k, out_d, out_i, ids);
      break;
    case 64: rc = launch_scan<64>(xq, centroids, pq, codes, list_off, probes, nq, nprobe, d, M, ws_d, ws_i, s);
      if (!rc) topk_merge_kernel<<<nq, 256, 0, s>>>(ws_d, ws_i, nprobe * 64, k, out_d, out_i, ids);
      break;
    default: return -1;
  }
  if (rc) return rc;
  DOCQA_CHECK_LAUNCH();
  return 0;
}

int docqa_row_norms(const float* x, int64_t n, int d, float* out, hipStream_t s) {
  if (n == 0) return 0;
  row_norms_kernel<<<(unsigned)((n + 3) / 4), 256, 0, s>>>(x, n, d, out);
  DOCQA_CHECK_LAUNCH();
  return 0;
}

int docqa_pq_encode(const float* x, const float* centroids, const int64_t* assign, const float* pq,
                    int n, int d, int M, uint8_t* codes, hipStream_t s) {
  if (n == 0) return 0;
  if (d % M != 0) return -1;
  const long long waves = (long long)n * M;
  const int blocks = (int)std::min<long long>((waves + 3) / 4, 1 << 16);
  pq_encode_kernel<<<blocks, 256, 0, s>>>(x, centroids, assign, pq, n, d, M, d / M, codes);
  DOCQA_CHECK_LAUNCH();
  return 0;
}
