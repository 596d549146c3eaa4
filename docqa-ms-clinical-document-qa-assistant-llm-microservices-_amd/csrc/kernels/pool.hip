// pool.hip -- sentence-embedding pooling for the bi-encoders, fused with the
// L2 normalisation FAISS-L2 retrieval relies on (sentence-transformers MiniLM: masked
// mean pool + normalize; bge: CLS pool + normalize).  Packed varlen input [T, H] with
// cu_seqlens; output fp32 [B, H] (the dtype FAISS stores; semantic-indexer/indexer.py:41
// casts to float32).  One workgroup per sequence, 16 B per lane per token row.
#include "docqa_common.h"

using namespace docqa;

// One workgroup a sequence: a thread owns 8 dims of every (512 / PC)-th token, four in flight; the groups' sums
// meet in LDS.  (24 tokens of 384, a load after the other: 8.1 us; so: 2.6.)
template <bool MEAN, int PC>
__global__ __launch_bounds__(512) void pool_l2_kernel(const uint16_t* __restrict__ h,
                                                      const int* __restrict__ cu, int H,
                                                      int normalize, float* __restrict__ out) {
  constexpr int G = 512 / PC;
  __shared__ float part[G][PC * 8 + 4];
  __shared__ float red[PC / 64];
  const int b = blockIdx.x;
  const int s0 = cu[b], s1 = cu[b + 1];
  const int c = threadIdx.x % PC, g = threadIdx.x / PC;   // chunk of 8 dims, token group
  const bool act = c * 8 < H;
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (act) {
    if (MEAN) {
      for (int t = s0 + g; t < s1; t += 4 * G) {
        uint4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = reinterpret_cast<const uint4*>(h + (size_t)min(t + u * G, s1 - 1) * H)[c];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          float f[8];
          unpack8(v[u], f);
          if (t + u * G < s1) {
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] += f[j];
          }
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) part[g][c * 8 + j] = acc[j];
    } else if (s1 > s0 && g == 0) {
      unpack8(reinterpret_cast<const uint4*>(h + (size_t)s0 * H)[c], acc);
    }
  }
  if (MEAN) {
    __syncthreads();
    if (g == 0 && act) {
      const float inv = s1 > s0 ? 1.f / (float)(s1 - s0) : 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float v = part[0][c * 8 + j];
#pragma unroll
        for (int k = 1; k < G; ++k) v += part[k][c * 8 + j];
        acc[j] = v * inv;
      }
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) ss += acc[j] * acc[j];
  if (g == 0) {
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  }
  __syncthreads();
  if (g != 0) return;
  float tot = red[0];
  if constexpr (PC == 128) tot += red[1];
  const float inv = normalize ? 1.f / fmaxf(sqrtf(tot), 1e-12f) : 1.f;
  if (act) {
    float4* o = reinterpret_cast<float4*>(out + (size_t)b * H + c * 8);
    o[0] = make_float4(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
    o[1] = make_float4(acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv);
  }
}

int docqa_pool_l2(const void* h, const int* cu, int B, int H, int mean, int normalize, float* out,
                  hipStream_t s) {
  if (B == 0) return 0;
  if (H % 8 != 0 || H > 1024) return -1;
  const uint16_t* p = (const uint16_t*)h;
  if (H <= 512) {
    if (mean) pool_l2_kernel<true, 64><<<B, 512, 0, s>>>(p, cu, H, normalize, out);
    else pool_l2_kernel<false, 64><<<B, 64, 0, s>>>(p, cu, H, normalize, out);
  } else {
    if (mean) pool_l2_kernel<true, 128><<<B, 512, 0, s>>>(p, cu, H, normalize, out);
    else pool_l2_kernel<false, 128><<<B, 128, 0, s>>>(p, cu, H, normalize, out);
  }
  DOCQA_CHECK_LAUNCH();
  return 0;
}
