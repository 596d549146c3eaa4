// gemm.hip -- bf16 MFMA GEMM with fused epilogues for the encoder stacks
//   C[M, N] = act(A[M, K] . W[N, K]^T + bias[N]) (+ residual[M, N])
// (nn.Linear layout: weights stored [out, in]).  Epilogues: none, bias, bias+GELU(erf),
// bias+residual, and the Llama SwiGLU over 8-interleaved gate|up rows (prefill shapes whose
// 256 x 256 tiles cannot fill the chip: the 70B TP-8 gate|up shard at <= 1k tokens).  Used by the BERT encoders (MiniLM / bge / clinical-BERT): the FFN-up
// GEMM with its bias+GELU, the QKV and output projections with their biases, so no
// separate element-wise pass re-reads the [tokens, 4H] activations from HBM.
//
// Structure of the 128 x 128 kernel (cdna_hip_programming.md §5 "canonical CDNA GEMM", T1, T2, T14);
// gemm_ring_kernel below is the one for large row counts:
//   * 128x128 block tile, BK = 64, 4 waves in 2x2, each wave a 64x64 sub-tile of
//     4x4 v_mfma_f32_16x16x32_bf16 accumulators (64 fp32 registers);
//   * A and W tiles are both row-major [row][k] in LDS (W^T's k-contiguous rows are
//     exactly the B-operand fragments), double-buffered, XOR-swizzled
//     (16-B chunk ^ ((row >> 1) & 7)) so the 16-row ds_read_b128 fragment reads are
//     bank-conflict-free;
//   * register-staged global->LDS copy of tile t+1 issued before the MFMAs of tile t and
//     written after them (async-STAGE split);
//   * XCD-aware bijective block remap so neighbouring tiles share an XCD's L2;
//   * epilogue through LDS: accumulators -> fp32 tile -> coalesced 16-B rows with the
//     bias / GELU / residual applied once per output element.
// Shapes: N % 128 == 0, K % 64 == 0, any M.
#include "docqa_asm.h"
#include "docqa_common.h"
#include <type_traits>

using namespace docqa;

namespace {
constexpr int BM = 128, BN = 128, BK = 64;
typedef short i16x8 __attribute__((ext_vector_type(8)));

enum Epi { EPI_NONE = 0, EPI_BIAS = 1, EPI_BIAS_GELU = 2, EPI_BIAS_RES = 3, EPI_GLU = 4 };

__device__ __forceinline__ int sw_off(int row, int ch) {  // element offset in a [128][64] tile
  return row * BK + ((ch ^ ((row >> 1) & 7)) << 3);
}

template <int EPI>
__global__ __launch_bounds__(256) void gemm_kernel(const uint16_t* __restrict__ A,
                                                   const uint16_t* __restrict__ W,
                                                   const uint16_t* __restrict__ bias,
                                                   const uint16_t* __restrict__ res,
                                                   uint16_t* __restrict__ C, int M, int N, int K) {
  // 64 KB of double-buffered A/W tiles, reused by the epilogue's 4 x 64 x 65 fp32 staging
  __shared__ __attribute__((aligned(16))) uint16_t smem[4 * 64 * 65 * 2];
  const int nbn = N / BN, nbm = (M + BM - 1) / BM;
  const int nwg = nbn * nbm;
  const int wg = xcd_remap(blockIdx.x, nwg);
  const int bm = wg / nbn, bn = wg % nbn;
  const int row0 = bm * BM, col0 = bn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;       // 2x2 waves
  const int fr = lane & 15, fk = lane >> 4;      // fragment row / k-group

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // staging by LDS-DMA (global_load_lds, 16 B per lane): each tensor tile is 128 rows x
  // 8 chunks = 16 wave-instructions of 1 KiB, 4 per wave per tensor.  The LDS image is
  // lane-linear, so the XOR swizzle is applied to the per-lane SOURCE address (rule 21):
  // physical chunk p of the image receives logical chunk (p&7) ^ ((row>>1)&7) of its row.
  typedef __attribute__((address_space(3))) void lds_void;
  auto stage = [&](int kt, int buf) {
    uint16_t* sa = smem + buf * (2 * BM * BK);
    uint16_t* sw = sa + BM * BK;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p0 = (i * 4 + wave) * 64;          // first physical chunk of this issue
      const int p = p0 + lane;
      const int r = p >> 3;
      const int ch = (p & 7) ^ ((r >> 1) & 7);
      const int gr = min(row0 + r, M - 1);         // tail rows: valid memory, never stored
      __builtin_amdgcn_global_load_lds(A + (size_t)gr * K + kt * BK + ch * 8,
                                       (lds_void*)(sa + p0 * 8), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(W + (size_t)(col0 + r) * K + kt * BK + ch * 8,
                                       (lds_void*)(sw + p0 * 8), 16, 0, 0);
    }
  };

  const int nk = K / BK;
  stage(0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nk) stage(kt + 1, buf ^ 1);   // DMA of tile t+1 overlaps MFMAs of tile t
    const uint16_t* sa = smem + buf * (2 * BM * BK);
    const uint16_t* sw = sa + BM * BK;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {          // two 32-deep MFMA k-steps per BK
      bf16x8 af[4], bf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = wr * 64 + i * 16 + fr;
        af[i] = *reinterpret_cast<const bf16x8*>(sa + sw_off(r, ks * 4 + fk));
        const int c = wc * 64 + i * 16 + fr;
        bf[i] = *reinterpret_cast<const bf16x8*>(sw + sw_off(c, ks * 4 + fk));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }

  // ---- epilogue: stage the wave's 64x64 fp32 tile in LDS (reuse), then 16-B row stores
  float* st = reinterpret_cast<float*>(smem) + wave * (64 * 65);   // padded rows, 16.6 KB/wave
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        st[(i * 16 + fk * 4 + r) * 65 + j * 16 + fr] = acc[i][j][r];
  __syncthreads();
  if constexpr (EPI == EPI_GLU) {
    // Llama gate|up in the 8-interleaved row layout (decode GEMMs' layout): output columns
    // [16 p, 16 p + 8) are gate, [16 p + 8, 16 p + 16) up; C is [M, N / 2] =
    // silu(gate) * up, each input rounded to bf16 first (as the unfused bf16 GEMM output
    // would be).  Lane -> (row, pair p of the wave's 4)
    for (int it = 0; it < 4; ++it) {
      const int rloc = it * 16 + (lane >> 2), p = lane & 3;
      const int gr = row0 + wr * 64 + rloc;
      if (gr < M) {
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float g = bf2f(f2bf(st[rloc * 65 + p * 16 + e]));
          const float u = bf2f(f2bf(st[rloc * 65 + p * 16 + 8 + e]));
          o[e] = g / (1.f + __expf(-g)) * u;
        }
        *reinterpret_cast<uint4*>(C + (size_t)gr * (N >> 1) + ((col0 + wc * 64) >> 1) + p * 8) = pack8(o);
      }
    }
    return;
  }
  // each wave writes its own 64 rows x 64 cols: lane -> (row group, 8-col chunk)
  for (int it = 0; it < 8; ++it) {
    const int rloc = it * 8 + (lane >> 3);
    const int cch = lane & 7;
    const int gr = row0 + wr * 64 + rloc;
    const int gc = col0 + wc * 64 + cch * 8;
    if (gr < M) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = st[rloc * 65 + cch * 8 + e];
      if constexpr (EPI != EPI_NONE) {
        float b[8];
        unpack8(*reinterpret_cast<const uint4*>(bias + gc), b);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += b[e];
      }
      if constexpr (EPI == EPI_BIAS_GELU) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = gelu_erf(v[e]);
      }
      if constexpr (EPI == EPI_BIAS_RES) {
        float rr[8];
        unpack8(*reinterpret_cast<const uint4*>(res + (size_t)gr * N + gc), rr);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += rr[e];
      }
      *reinterpret_cast<uint4*>(C + (size_t)gr * N + gc) = pack8(v);
    }
  }
}

// ---- 256 rows x 128 columns a workgroup, two workgroups a CU: row counts that fill the chip.
// The 128 x 128 kernel reads 64 KB of LDS for 512 clocks of MFMA a K-step and is bound by that
// (bge-base, 30720 rows, us of QKV / O / FFN up / down: 146 / 54 / 226 / 173; here 119 / 49 / 175 /
// 140, 0.9 to 1.05 PFLOP/s, the matrix cores busy 45 % of the time at the 1.9 GHz this load runs at,
// the rest in the latency of units and epilogues).
// Here a wave owns 128 rows x 64 columns (96, with half an HA1, on 192-row tiles) (v_mfma_f32_32x32x16_bf16: 48 KB for 1024 clocks), and a
// workgroup's epilogue runs under the other one's products.
//   * K-tiles of 64 come as three units of 128 rows x 64 (whole 128-byte lines: with 64-byte rows
//     LDS-DMA moves 15 TB/s over the chip, with 128-byte ones 20 to 29) through a ring of five:
//       HA0 = the first 64 rows of both wave rows, HB = the columns, HA1 = the last 64 rows
//     phase 1 of K-tile t reads units 3t (HA0) and 3t + 1 (HB, kept in registers), phase 2 reads
//     3t + 2 (HA1); phase 1 issues unit 3t + 4 over 3t - 1, phase 2 issues 3t + 5 and 3t + 6 over
//     3t and 3t + 1, each read by every wave before the barrier that opens the phase.  At that
//     barrier two units are in flight (vmcnt(8)), two phases ahead of their reads;
//   * the MFMA's row operand is W, its column operand A: a lane holds one output row and four
//     neighbouring columns per register quad, 8-byte pieces of the bf16 tile;
//   * the tile is put together in LDS (16-B chunk ^ (row & 15): 32 rows' pieces hit distinct
//     banks) and stored in whole rows; the residual comes into the same places by LDS-DMA first
//     and is added in fp32 before the one rounding.
constexpr int WN = 128;
constexpr int UNIT = 128 * BK * 2, NUNIT = 5;         // 16 KB units of the ring, 80 KB

template <int EPI, int WM>
__global__ __launch_bounds__(256, 2) void gemm_ring_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W,
                                                           const uint16_t* __restrict__ bias,
                                                           const uint16_t* __restrict__ res, uint16_t* __restrict__ C,
                                                           int M, int N, int K) {
  __shared__ __attribute__((aligned(16))) char smem[NUNIT * UNIT];
  static_assert(NUNIT * UNIT >= WM * WN * 2, "epilogue tile");
  constexpr int WR = WM / 2, M1 = WR / 32 - 2, L1 = 2 * M1;   // a wave row; 32-row tiles and loads a thread of its HA1
  static_assert(M1 == 1 || M1 == 2, "192 or 256 rows");
  const int nbn = N / WN;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int row0 = (wg / nbn) * WM, col0 = (wg % nbn) * WN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave & 1, wc = wave >> 1;
  const int l32 = lane & 31, hh = lane >> 5;
  const uint32_t lds = lds_u32(smem);

  // four 16-B pieces a thread and unit: unit rows 32 i + tid / 8
  const char* ab = (const char*)(A + (size_t)row0 * K);
  const char* wb = (const char*)(W + (size_t)col0 * K);
  const uint32_t lch = (uint32_t)((tid & 7) ^ ((tid >> 4) & 7)) * 16;     // (row >> 1) & 7 is the thread's own
  uint32_t aoff[2][4], boff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = i * 32 + (tid >> 3);
    boff[i] = (uint32_t)r * (uint32_t)(K * 2) + lch;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int hr = h ? 32 * M1 : 64;               // rows of this half of a wave row
      aoff[h][i] = (uint32_t)min(r / hr * WR + h * 64 + r % hr, M - 1 - row0) * (uint32_t)(K * 2) + lch;
    }
  }
  // unit `part` (0 HA0, 1 HB, 2 HA1) of K-tile kt into ring slot `slot`
  auto issue = [&](int part, int kt, int slot) {
    const uint32_t d = lds + (uint32_t)(slot * UNIT + wave * 1024);
    const uint32_t k = (uint32_t)kt * (BK * 2);
#pragma unroll
    for (int i = 0; i < (part == 2 ? L1 : 4); ++i)
      glds16_off(part == 1 ? wb : ab, (part == 1 ? boff[i] : aoff[part >> 1][i]) + k,
                 __builtin_amdgcn_readfirstlane(d + i * 4096));
  };
  auto open = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ring_barrier();
  };
  // 16-B chunk `ch` of unit row `row`: 32-row fragment reads hit distinct banks
  auto frag = [&](int slot, int row, int ch) {
    return *reinterpret_cast<const bf16x8*>(smem + slot * UNIT + row * 128 + ((ch ^ ((row >> 1) & 7)) << 4));
  };

  f32x16 acc[2][2 + M1];
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int m = 0; m < 2 + M1; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[n][m][r] = 0.f;
  bf16x8 w[4][2];                                    // [16-deep k-step][n-tile] of the current K-tile
  auto phase = [&](int slot_a, int slot_b, auto part) {
    constexpr bool first = decltype(part)::value;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (first) {
#pragma unroll
        for (int n = 0; n < 2; ++n) w[ks][n] = frag(slot_b, wc * 64 + n * 32 + l32, ks * 2 + hh);
      }
      bf16x8 a[2];
#pragma unroll
      for (int m = 0; m < (first ? 2 : M1); ++m) a[m] = frag(slot_a, wr * (first ? 64 : 32 * M1) + m * 32 + l32, ks * 2 + hh);
#pragma unroll
      for (int m = 0; m < (first ? 2 : M1); ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          f32x16& c = acc[n][first ? m : 2 + m];
          c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[ks][n], a[m], c, 0, 0, 0);
        }
    }
  };

  const int nk = K / BK;
  issue(0, 0, 0);
  issue(1, 0, 1);
  issue(2, 0, 2);
  if (nk > 1) issue(0, 1, 3);
  int s0 = 0;                                        // slot of unit 3t
  auto slot = [&](int k) { return s0 + k < NUNIT ? s0 + k : s0 + k - NUNIT; };   // of unit 3t + k, k <= 4
  for (int t = 0; t < nk - 1; ++t) {
    wait_vmcnt<4 + L1>();
    open();
    issue(1, t + 1, slot(4));
    phase(slot(0), slot(1), std::true_type{});
    wait_vmcnt<8>();
    open();
    issue(2, t + 1, slot(0));
    if (t + 2 < nk) issue(0, t + 2, slot(1));
    phase(slot(2), 0, std::false_type{});
    s0 = slot(3);
  }
  wait_vmcnt<L1>();
  open();
  phase(slot(0), slot(1), std::true_type{});
  wait_vmcnt<0>();
  open();
  phase(slot(2), 0, std::false_type{});
  open();                                            // the ring is the epilogue's tile now

  // 16-B chunk of the tile that piece `it` of this thread is: row 16 it + tid / 16
  const int prow = tid >> 4, pcol = ((tid & 15) ^ prow) * 8;
  if constexpr (EPI == EPI_BIAS_RES) {
    const char* rb = (const char*)(res + (size_t)row0 * N + col0);
#pragma unroll
    for (int it = 0; it < WM / 16; ++it)
      glds16_off(rb, (uint32_t)min(16 * it + prow, M - 1 - row0) * (uint32_t)(N * 2) + pcol * 2,
                 __builtin_amdgcn_readfirstlane(lds + it * 4096 + wave * 1024));
    wait_vmcnt<0>();
    ring_barrier();
  }
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int col = wc * 64 + n * 32 + 8 * g + 4 * hh;
      float b[4] = {0.f, 0.f, 0.f, 0.f};
      if constexpr (EPI != EPI_NONE) add4(b, *reinterpret_cast<const uint2*>(bias + col0 + col));
#pragma unroll
      for (int m = 0; m < 2 + M1; ++m) {
        const int row = wr * WR + m * 32 + l32;
        uint2* at = reinterpret_cast<uint2*>(smem + row * 256 + (((col >> 3) ^ (row & 15)) << 4) + (hh << 3));
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[n][m][4 * g + e] + b[e];
        if constexpr (EPI == EPI_BIAS_GELU) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = gelu_erf(v[e]);
        }
        if constexpr (EPI == EPI_BIAS_RES) add4(v, *at);
        *at = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
      }
    }
  __syncthreads();
  uint16_t* out = C + (size_t)row0 * N + col0 + pcol;
#pragma unroll
  for (int it = 0; it < WM / 16; ++it) {
    const int r = 16 * it + prow;
    const uint4 v = *reinterpret_cast<const uint4*>(smem + it * 4096 + tid * 16);
    if (row0 + r < M) *reinterpret_cast<uint4*>(out + (size_t)r * N) = v;
  }
}

// ---- few rows: T x T tiles, K split over the workgroup's 4 waves.  Such products are bound by
// the latency of one K walk and by what a CU can fetch, so a workgroup keeps five 16 KB stages in
// flight, and each wave multiplies its quarter of every stage (a fragment read feeds T / 32 MFMAs
// where 2 x 2 waves would read twice as much); the four sums meet in LDS, and whole rows leave
// with bias, GELU or residual applied in fp32.
template <int T, int EPI>
__global__ __launch_bounds__(256, 2) void gemm_few_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W,
                                                          const uint16_t* __restrict__ bias,
                                                          const uint16_t* __restrict__ res, uint16_t* __restrict__ C,
                                                          int M, int N, int K) {
  constexpr int KB = 4096 / T;                       // k's of a stage: 16 KB of both operands
  constexpr int ROWB = KB * 2, CPR = ROWB / 16;      // bytes and 16-B chunks of a stage row
  constexpr int STAGE = 2 * T * ROWB, NS = 5, L = STAGE / 4096;
  constexpr int TI = T / 32, KS = CPR / 8;           // MFMA tiles a side, 16-deep k-steps a wave and stage
  constexpr int PITCH = T + 4;
  __shared__ __attribute__((aligned(16))) char smem[NS * STAGE];
  static_assert(4 * T * PITCH * 4 <= NS * STAGE, "partial sums");
  const int nbn = N / T;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int row0 = (wg / nbn) * T, col0 = (wg % nbn) * T;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const uint32_t lds = lds_u32(smem);
  // 16-B chunk `ch` of stage row `row`: 32-row fragment reads hit distinct banks
  auto swz = [](int row, int ch) { return CPR == 8 ? ch ^ ((row >> 1) & 7) : ch ^ (row & 15); };

  const char* ab = (const char*)(A + (size_t)row0 * K);
  const char* wb = (const char*)(W + (size_t)col0 * K);
  uint32_t off[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int r = (i * 256 + tid) / CPR, lr = r % T;               // rows of A, then of W
    off[i] = (uint32_t)(r < T ? min(lr, M - 1 - row0) : lr) * (uint32_t)(K * 2) + swz(lr, tid % CPR) * 16;
  }
  auto stage = [&](int kt, int buf) {
    const uint32_t d = lds + (uint32_t)(buf * STAGE + wave * 1024);
#pragma unroll
    for (int i = 0; i < L; ++i)
      glds16_off(i < L / 2 ? ab : wb, off[i] + (uint32_t)kt * ROWB, __builtin_amdgcn_readfirstlane(d + i * 4096));
  };

  f32x16 acc[TI][TI];
#pragma unroll
  for (int n = 0; n < TI; ++n)
#pragma unroll
    for (int m = 0; m < TI; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[n][m][r] = 0.f;
  const int nk = K / KB;
#pragma unroll
  for (int t = 0; t < NS - 1; ++t)
    if (t < nk) stage(t, t);
  int buf = 0;
  for (int kt = 0; kt < nk; ++kt) {
    // stage kt has landed: of the later ones up to NS - 2 may be in flight
    const int later = min(NS - 2, nk - 1 - kt);
    if (later == 3) wait_vmcnt<3 * L>();
    else if (later == 2) wait_vmcnt<2 * L>();
    else if (later == 1) wait_vmcnt<L>();
    else wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ring_barrier();                                  // and every wave has read what the next issue overwrites
    if (kt + NS - 1 < nk) stage(kt + NS - 1, buf ? buf - 1 : NS - 1);
    const char* sa = smem + buf * STAGE;
    const char* sw = sa + T * ROWB;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int ch = (wave * KS + ks) * 2 + hh;
      bf16x8 a[TI], w[TI];
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const int r = i * 32 + l32;
        a[i] = *reinterpret_cast<const bf16x8*>(sa + r * ROWB + swz(r, ch) * 16);
        w[i] = *reinterpret_cast<const bf16x8*>(sw + r * ROWB + swz(r, ch) * 16);
      }
#pragma unroll
      for (int n = 0; n < TI; ++n)
#pragma unroll
        for (int m = 0; m < TI; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[n], a[m], acc[n][m], 0, 0, 0);
    }
    buf = buf == NS - 1 ? 0 : buf + 1;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  ring_barrier();                                    // the ring holds the partial sums now
  float* part = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int n = 0; n < TI; ++n)
#pragma unroll
    for (int m = 0; m < TI; ++m)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(part + (wave * T + m * 32 + l32) * PITCH + n * 32 + 8 * g + 4 * hh) =
            f32x4{acc[n][m][4 * g], acc[n][m][4 * g + 1], acc[n][m][4 * g + 2], acc[n][m][4 * g + 3]};
  __syncthreads();
  constexpr int TPR = T / 8, RPI = 256 / TPR;        // threads a row, rows a pass
#pragma unroll
  for (int it = 0; it < (T + RPI - 1) / RPI; ++it) {
    const int r = it * RPI + tid / TPR, c = (tid % TPR) * 8;
    if (r >= T || row0 + r >= M) break;
    float v[8] = {};
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(part + (w * T + r) * PITCH + c + e);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[e + k] += x[k];
      }
    float b[8];
    if constexpr (EPI != EPI_NONE) {
      unpack8(*reinterpret_cast<const uint4*>(bias + col0 + c), b);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += b[e];
    }
    if constexpr (EPI == EPI_BIAS_GELU) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = gelu_erf(v[e]);
    }
    const size_t at = (size_t)(row0 + r) * N + col0 + c;
    if constexpr (EPI == EPI_BIAS_RES) {
      unpack8(*reinterpret_cast<const uint4*>(res + at), b);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += b[e];
    }
    *reinterpret_cast<uint4*>(C + at) = pack8(v);
  }
}
// ---- few rows of an encoder layer behind their LayerNorm: A = LN(X) gamma + beta (layernorm_kernel's arithmetic,
// bit for bit), made by every workgroup for its own 32 rows while its first weights are on the way, so that no
// launch stands between two products; the first column tile's workgroups also write A, the next residual.  32 x 32
// tiles, 8 waves normalise, 4 of them multiply with K split as above, A whole in LDS, W in 128-deep stages.  Bound
// by its chain of latencies; 24 rows of MiniLM, us: up 2.75 + 3.85 -> 6.35, QKV 2.75 + 3.6 -> 5.9, and the gap
// between two launches less (with 4 waves 6.7 and 6.3).
constexpr int LN_MAXK = 768;    // 80 KB of LDS, two workgroups a CU
template <int EPI, int NV>
__global__ __launch_bounds__(512) void gemm_few_ln_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ gamma,
                                                          const uint16_t* __restrict__ beta, float eps,
                                                          uint16_t* __restrict__ A, const uint16_t* __restrict__ W,
                                                          const uint16_t* __restrict__ bias, uint16_t* __restrict__ C, int M,
                                                          int N, int K) {
  constexpr int T = 32, STAGE = T * 256, NS = 4, PITCH = T + 4;
  constexpr int PANEL = T * (NV == 1 ? 512 : LN_MAXK) * 2;
  __shared__ __attribute__((aligned(16))) char smem[PANEL + NS * STAGE];
  static_assert(4 * T * PITCH * 4 <= PANEL + NS * STAGE, "partial sums");
  const int nbn = N / T;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int row0 = (wg / nbn) * T, col0 = (wg % nbn) * T;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  char* ring = smem + PANEL;
  const uint32_t lds = lds_u32(ring);
  const char* wb = (const char*)(W + (size_t)col0 * K);
  const uint32_t off = (uint32_t)(tid >> 4) * (uint32_t)(K * 2) + (uint32_t)((tid & 15) ^ ((tid >> 4) & 15)) * 16;
  auto stage = [&](int kt, int buf) {                // 16 bytes a thread
    glds16_off(wb, off + (uint32_t)kt * 256, __builtin_amdgcn_readfirstlane(lds + (uint32_t)(buf * STAGE + wave * 1024)));
  };
  const int nk = K / 128, nchunk = K >> 3;
#pragma unroll
  for (int t = 0; t < NS - 1; ++t)
    if (t < nk) stage(t, t);

  // a wave normalises 4 rows (rows past the end: the last one again, never stored)
  uint4 raw[4][NV], gr[NV], br[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = min(lane + 64 * i, nchunk - 1);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      raw[r][i] = reinterpret_cast<const uint4*>(X + (size_t)min(row0 + wave * 4 + r, M - 1) * K)[c];
    gr[i] = reinterpret_cast<const uint4*>(gamma)[c];
    br[i] = reinterpret_cast<const uint4*>(beta)[c];
  }
  float mean[4], inv[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      float v[8];
      unpack8(raw[r][i], v);
      if (lane + 64 * i < nchunk) {
#pragma unroll
        for (int j = 0; j < 8; ++j) s += v[j];
      }
    }
    mean[r] = s;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) mean[r] = wave_sum(mean[r]) / (float)K;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      float v[8];
      unpack8(raw[r][i], v);
      if (lane + 64 * i < nchunk) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float d = v[j] - mean[r];
          ss += d * d;
        }
      }
    }
    inv[r] = ss;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) inv[r] = rsqrtf(wave_sum(inv[r]) / (float)K + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = lane + 64 * i;
    if (c >= nchunk) continue;
    float g[8], b[8];
    unpack8(gr[i], g);
    unpack8(br[i], b);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = wave * 4 + r;
      float v[8], o[8];
      unpack8(raw[r][i], v);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (v[j] - mean[r]) * inv[r] * g[j] + b[j];
      const uint4 p = pack8(o);
      *reinterpret_cast<uint4*>(smem + row * (K * 2) + (((c & ~15) | ((c & 15) ^ (row & 15))) << 4)) = p;
      if (col0 == 0 && row0 + row < M) reinterpret_cast<uint4*>(A + (size_t)(row0 + row) * K)[c] = p;
    }
  }

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  int buf = 0;
  for (int kt = 0; kt < nk; ++kt) {
    // (the rows' stores, issued after the first stages, only make these waits longer)
    const int later = min(NS - 2, nk - 1 - kt);
    if (later == 2) wait_vmcnt<2>();
    else if (later == 1) wait_vmcnt<1>();
    else wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ring_barrier();
    if (kt + NS - 1 < nk) stage(kt + NS - 1, buf ? buf - 1 : NS - 1);
    if (wave < 4) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int ch = ((wave * 2 + ks) * 2 + hh) ^ (l32 & 15);
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(smem + l32 * (K * 2) + kt * 256 + ch * 16);
        const bf16x8 w = *reinterpret_cast<const bf16x8*>(ring + buf * STAGE + l32 * 256 + ch * 16);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, a, acc, 0, 0, 0);
      }
    }
    buf = buf == NS - 1 ? 0 : buf + 1;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  ring_barrier();                                    // the partial sums' place now
  float* part = reinterpret_cast<float*>(smem);
  if (wave < 4) {
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(part + (wave * T + l32) * PITCH + 8 * g + 4 * hh) =
          f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  }
  __syncthreads();
  const int r = tid >> 2, c = (tid & 3) * 8;
  if (r >= T || row0 + r >= M) return;
  float v[8] = {};
#pragma unroll
  for (int w = 0; w < 4; ++w)
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(part + (w * T + r) * PITCH + c + e);
#pragma unroll
      for (int k = 0; k < 4; ++k) v[e + k] += x[k];
    }
  float b[8];
  unpack8(*reinterpret_cast<const uint4*>(bias + col0 + c), b);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    v[e] += b[e];
    if constexpr (EPI == EPI_BIAS_GELU) v[e] = gelu_erf(v[e]);
  }
  *reinterpret_cast<uint4*>(C + (size_t)(row0 + r) * N + col0 + c) = pack8(v);
}
}  // namespace

// whether docqa_gemm_ln takes the product: as few 32 x 32 tiles as docqa_gemm gives that form
bool docqa_gemm_ln_ok(int M, int N, int K) {
  return M > 0 && N % BN == 0 && K % 128 == 0 && K <= LN_MAXK && (long long)((M + 31) / 32) * (N / 32) <= 512;
}

// C = act(A . W^T + bias), A = LN(X) gamma + beta, which is written too; epi bias or bias + GELU.  X and A differ.
int docqa_gemm_ln(const void* X, const void* gamma, const void* beta, float eps, void* A, const void* W, const void* bias,
                  void* C, int M, int N, int K, int epi, hipStream_t s) {
  if (!docqa_gemm_ln_ok(M, N, K) || (epi != EPI_BIAS && epi != EPI_BIAS_GELU) || X == A) return -1;
  for (const void* p : {X, gamma, beta, (const void*)A, W, bias, (const void*)C})
    if (!docqa_aligned16(p)) return -1;
  const int grid = (M + 31) / 32 * (N / 32);
#define DOCQA_LN(E, NV)                                                                                                   \
  gemm_few_ln_kernel<E, NV><<<grid, 512, 0, s>>>((const uint16_t*)X, (const uint16_t*)gamma, (const uint16_t*)beta, eps, \
                                                 (uint16_t*)A, (const uint16_t*)W, (const uint16_t*)bias, (uint16_t*)C, M, N, K)
  if (K <= 512) {
    if (epi == EPI_BIAS) DOCQA_LN(EPI_BIAS, 1);
    else DOCQA_LN(EPI_BIAS_GELU, 1);
  } else {
    if (epi == EPI_BIAS) DOCQA_LN(EPI_BIAS, 2);
    else DOCQA_LN(EPI_BIAS_GELU, 2);
  }
#undef DOCQA_LN
  DOCQA_CHECK_LAUNCH();
  return 0;
}

// What `tiles` ring tiles take, in eighths of a round of 512 (two workgroups a CU): alone on its CU a workgroup
// takes five of them.  A round of 192-row tiles is worth 0.8 of one of 256 (fitted to 95 launches, bge-base and
// MiniLM at 3600..34000 rows: 0.3 % off the better one on average, 256 rows alone 7 %; us of 256 / 192: QKV
// 4500 rows 25.6 / 21.4, down 22000 rows 129 / 107, up 13000 rows 79 / 85)
static long long ring_cost(long long tiles) {
  const long long rest = tiles % 512;
  return tiles / 512 * 8 + (rest == 0 ? 0 : rest <= 256 ? 5 : 8);
}

int docqa_gemm(const void* A, const void* W, const void* bias, const void* res, void* C, int M,
               int N, int K, int epi, hipStream_t s) {
  if (M == 0) return 0;
  if (N % BN != 0 || K % BK != 0) return -1;
  if (epi != EPI_NONE && epi != EPI_GLU && bias == nullptr) return -1;
  if (epi == EPI_BIAS_RES && res == nullptr) return -1;
  const int nwg = (N / BN) * ((M + BM - 1) / BM);
  const uint16_t *a = (const uint16_t*)A, *w = (const uint16_t*)W, *b = (const uint16_t*)bias,
                 *r = (const uint16_t*)res;
  uint16_t* c = (uint16_t*)C;
  // by how the tiles fill the chip (us): 32 x 32 up to two workgroups a CU (32 / 64 wide: bge QKV 128
  // rows, 288 workgroups, 5.7 / 6.3, 256 rows, 576 of them, 8.0 / 6.5), 64 x 64 up to three (64 / 128
  // wide: QKV 1024 rows, 576, 13.6 / 14.4, 1500 rows, 864, 16.6 / 14.7; O 4096 rows, 768, 13.2 / 13.5),
  // 256 x 128 from one on (128 wide / ring: QKV 4096 rows, 288, 28.1 / 25.0, 30720 rows 146 / 119;
  // FFN down, K 3072, 8192 rows, 192, 48.6 / 54.2, 19000 rows, 450, 103 / 91), of them 192 rows where
  // those end in less (see ring_cost), and where a workgroup a CU holds them but not the 128 x 128 tiles
  // (QKV 2600 rows 17.6 / 14.6, O 7000 rows 17.5 / 15.1; with 128-wide tiles below that too, or 192-row
  // tiles above it, 128 x 128 wins: O 5200 rows 13.4 / 14.1, 10500 rows 19.1 / 21.5).  Row offsets inside
  // those tiles are 32-bit
  auto tiles = [&](int tm, int tn) { return (long long)((M + tm - 1) / tm) * (N / tn); };
#define DOCQA_GEMM_EPI(KERNEL, GRID)                                                             \
  do {                                                                                           \
    const int g_ = (int)(GRID);                                                                  \
    if (epi == EPI_NONE) KERNEL(EPI_NONE)<<<g_, 256, 0, s>>>(a, w, b, r, c, M, N, K);            \
    else if (epi == EPI_BIAS) KERNEL(EPI_BIAS)<<<g_, 256, 0, s>>>(a, w, b, r, c, M, N, K);       \
    else if (epi == EPI_BIAS_GELU) KERNEL(EPI_BIAS_GELU)<<<g_, 256, 0, s>>>(a, w, b, r, c, M, N, K); \
    else KERNEL(EPI_BIAS_RES)<<<g_, 256, 0, s>>>(a, w, b, r, c, M, N, K);                        \
  } while (0)
#define DOCQA_FEW32(E) gemm_few_kernel<32, E>
#define DOCQA_FEW64(E) gemm_few_kernel<64, E>
#define DOCQA_RING(E) gemm_ring_kernel<E, 256>
#define DOCQA_RING192(E) gemm_ring_kernel<E, 192>
  if (epi < EPI_NONE || epi > EPI_GLU) return -1;
  if (epi != EPI_GLU && 256ll * (K > N ? K : N) * 2 < (1ll << 32)) {
    int kind = 0;
    if (K % 128 == 0 && tiles(32, 32) <= 512) kind = 32;
    else if (tiles(64, 64) <= 768) kind = 64;
    else if (tiles(256, WN) >= 256) kind = ring_cost(tiles(192, WN)) * 4 < ring_cost(tiles(256, WN)) * 5 ? 192 : 256;
    else if (nwg > 256 && tiles(192, WN) <= 256) kind = 192;
    if (kind == 32) DOCQA_GEMM_EPI(DOCQA_FEW32, tiles(32, 32));
    else if (kind == 64) DOCQA_GEMM_EPI(DOCQA_FEW64, tiles(64, 64));
    else if (kind == 192) DOCQA_GEMM_EPI(DOCQA_RING192, tiles(192, WN));
    else if (kind) DOCQA_GEMM_EPI(DOCQA_RING, tiles(256, WN));
    if (kind) {
      DOCQA_CHECK_LAUNCH();
      return 0;
    }
  }
  switch (epi) {
    case EPI_NONE: gemm_kernel<EPI_NONE><<<nwg, 256, 0, s>>>(a, w, b, r, c, M, N, K); break;
    case EPI_BIAS: gemm_kernel<EPI_BIAS><<<nwg, 256, 0, s>>>(a, w, b, r, c, M, N, K); break;
    case EPI_BIAS_GELU: gemm_kernel<EPI_BIAS_GELU><<<nwg, 256, 0, s>>>(a, w, b, r, c, M, N, K); break;
    case EPI_BIAS_RES: gemm_kernel<EPI_BIAS_RES><<<nwg, 256, 0, s>>>(a, w, b, r, c, M, N, K); break;
    case EPI_GLU: gemm_kernel<EPI_GLU><<<nwg, 256, 0, s>>>(a, w, b, r, c, M, N, K); break;
  }
  DOCQA_CHECK_LAUNCH();
  return 0;
}
