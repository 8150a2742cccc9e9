// o_proj after the attention: out[m][n] = bf16(sum_k x[m][k] * w[n][k]) for
// bf16 x [seq_len][cols] and w [rows][cols], f32 accumulation
// (dispatch_gemm_cols, kernels/gemm.mojo:198-225, called at
// modeling/gemma_4_moe.mojo:387-392 and :485-490 with rows = HIDDEN).
//
// Decode batches (<= 64 tokens) stream the weight: v_mfma_f32_16x16x32_bf16
// with x as the A operand (16 token rows x 32 k) and w as B (32 k x 16 output
// columns), both fragments 16-byte runs along k of one row, so w goes straight
// from HBM into registers.  They have too few output tiles to fill 256 CUs:
// gemm_cols_split_kernel gives each workgroup a slice of k loaded in one round
// trip and writes f32 partials that gemm_cols_reduce_kernel adds in slice
// order; up to 16 tokens and k of 4,096 gemm_cols_few_kernel keeps the slices in one
// workgroup.
// Larger batches run gemm_cols_tile_kernel, LDS-tiled on
// v_mfma_f32_32x32x16_bf16, in the tile shape and k splits of tile_plan.
#include <algorithm>

#include "common.hpp"
#include "launch.hpp"

namespace ifr {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kBM = 64;         // most tokens of a decode batch
constexpr int kBN = 64;         // output columns per workgroup of a decode batch
constexpr int kMaxSplits = 16;  // k slices the reduce adds

// The decode batches read w once: its loads bypass the caches' retention.
__device__ __forceinline__ uint4 load_w(const uint16_t* p) {
  const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}

// Batches past the decode sizes: a workgroup of 4 waves (2 x 2) computes a
// BM x BN tile of the output, walking k in 64-wide chunks that travel from
// memory straight into LDS (global_load_lds, no registers), three chunks
// deep: while chunk c is multiplied, c + 1 is landing and c + 2 is issued, so
// one barrier per chunk both publishes chunk c and frees the buffer that
// c + 2 goes to.  The three buffers are separate LDS objects, so the compiler
// puts no wait for the loads in flight ahead of the reads of another one.
// v_mfma_f32_32x32x16_bf16 with x as A (lane l: token l % 32, k 8*(l/32)..+7)
// and w as B (column l % 32), so a lane stores one column of 16 tokens and 32
// lanes 32 consecutive columns.
//
// LDS rows are 128 bytes (64 k); 16-byte chunk q of row r sits at q ^ ((r/2)
// & 7), so the 16 rows that a quarter of a fragment read covers lie in 16
// different 16-byte bank groups.
constexpr int kTileK = 64;   // k per LDS chunk
constexpr int kTRow = 2 * kTileK;  // LDS row bytes
constexpr int kTThreads = 256;

template <int BM, int BN, bool kSplit>
__global__ __launch_bounds__(kTThreads) __attribute__((amdgpu_waves_per_eu(1, 2)))
void gemm_cols_tile_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, uint16_t* __restrict__ out,
    float* __restrict__ part, int M, int N, int K, int k_span, int m_tiles, int n_tiles) {
  constexpr int kMB = BM / 64, kNB = BN / 64;  // 32 x 32 blocks of a wave's tile
  constexpr int kLoads = (BM + BN) / 32;       // 1 KiB loads (8 rows) a wave issues per chunk
  constexpr int kSteps = kTileK / 16;          // MFMA k steps of a chunk
  constexpr int kStepLoads = (kLoads + kSteps - 1) / kSteps;
  static_assert(kLoads < 16, "the wait count below");
  __shared__ __align__(16) uint8_t buf0[(BM + BN) * kTRow];
  __shared__ __align__(16) uint8_t buf1[(BM + BN) * kTRow];
  __shared__ __align__(16) uint8_t buf2[(BM + BN) * kTRow];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int half = lane >> 5;
  const int r32 = lane & 31;

  // Workgroups go to the 8 XCDs round robin: XCD b % 8 takes a contiguous run
  // of tiles, ordered in bands of kBand token tiles (token tile fastest inside
  // a band), so the 32 tiles that run together on one XCD read about as many
  // x rows as w rows through its L2.
  const int tiles = m_tiles * n_tiles;
  const int per = (tiles + 7) / 8;
  const int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (t >= tiles) return;  // block-uniform
  constexpr int kBand = 1024 / BM;
  const int band = t / (kBand * n_tiles), in_band = t - band * kBand * n_tiles;
  const int height = min(kBand, m_tiles - band * kBand);
  const int m0 = (band * kBand + in_band % height) * BM;
  const int n0 = (in_band / height) * BN;
  const int k0 = blockIdx.y * k_span;
  const int nk = k_span / kTileK;

  // Load i of this wave moves tile rows 8*(wave + 4i) .. +7 (x rows first, then
  // w rows): lane p row p/8, LDS chunk p % 8.  Rows past the matrix repeat its
  // last row; what they produce is not stored.
  const uint16_t* src[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int r = 8 * (wave + 4 * i) + (lane >> 3);
    const int chunk = (lane & 7) ^ ((r >> 1) & 7);
    const uint16_t* base = r < BM ? x + static_cast<int64_t>(min(m0 + r, M - 1)) * K
                                  : w + static_cast<int64_t>(min(n0 + r - BM, N - 1)) * K;
    src[i] = base + k0 + 8 * chunk;
  }
  auto load1 = [&](int i, int c, uint8_t* buf) {
    __builtin_amdgcn_global_load_lds(
        static_cast<const void*>(src[i] + static_cast<int64_t>(c) * kTileK),
        (lds_void_t*)(buf + 8 * (wave + 4 * i) * kTRow), 16, 0, 0);
  };

  f32x16_t acc[kMB][kNB];
#pragma unroll
  for (int a = 0; a < kMB; ++a)
#pragma unroll
    for (int b = 0; b < kNB; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;

  const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);
  // Fragment of 16-k step s: chunk 2s + half of row r, at (2s + half) ^ ((r/2) & 7)
  // = 2s ^ (half ^ ((r/2) & 7)): byte offset row * 128 + (lane term ^ 32 s).
  const int lane_sw = 16 * (half ^ ((r32 >> 1) & 7));
  const int a_row = (wm + r32) * kTRow;
  const int b_row = (BM + wn + r32) * kTRow;

#pragma unroll
  for (int i = 0; i < kLoads; ++i) load1(i, 0, buf0);
#pragma unroll
  for (int i = 0; i < kLoads; ++i) load1(i, min(1, nk - 1), buf1);

  auto chunk = [&](int c, const uint8_t* cur, uint8_t* next) {
    // Chunk c has landed when only chunk c + 1's loads are outstanding.
    __builtin_amdgcn_s_waitcnt(0x0F70 | kLoads);  // vmcnt(kLoads)
    // The reads of chunk c - 1 have returned before another wave may refill their
    // buffer.  Written out: the compiler waits for them only where it puts the
    // MFMAs that use them, which at 128 x 64 is partly behind the barrier.
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // Past the last chunk the loads repeat it into a buffer nothing reads, so
    // the count of outstanding loads is the same in every iteration.
    const int cn = min(c + 2, nk - 1);
    bf16x8_t af[2][kMB], bf[2][kNB];
    auto read = [&](int s, int set) {
#pragma unroll
      for (int a = 0; a < kMB; ++a)
        af[set][a] = *reinterpret_cast<const bf16x8_t*>(cur + a_row + 32 * a * kTRow +
                                                        (lane_sw ^ (32 * s)));
#pragma unroll
      for (int b = 0; b < kNB; ++b)
        bf[set][b] = *reinterpret_cast<const bf16x8_t*>(cur + b_row + 32 * b * kTRow +
                                                        (lane_sw ^ (32 * s)));
    };
    read(0, 0);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      if (s + 1 < kSteps) read(s + 1, (s + 1) & 1);
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        if (i / kStepLoads == s) load1(i, cn, next);
#pragma unroll
      for (int a = 0; a < kMB; ++a)
#pragma unroll
        for (int b = 0; b < kNB; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[s & 1][a], bf[s & 1][b],
                                                              acc[a][b], 0, 0, 0);
    }
    // The order within the chunk: step 0's fragment reads, then between the
    // MFMAs of each step the reads of the next step and the step's share of
    // the loads.
    __builtin_amdgcn_sched_group_barrier(0x100, kMB + kNB, 0);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      constexpr int kMfma = kMB * kNB, kReads = kMB + kNB;
      int reads = 0, loads = 0;
#pragma unroll
      for (int j = 0; j < kMfma; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (s + 1 < kSteps) {
          constexpr int kPer = (kReads + kMfma - 1) / kMfma;
#pragma unroll
          for (int t = 0; t < kPer; ++t)
            if (reads < kReads) {
              __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
              ++reads;
            }
        }
        constexpr int kPerL = (kStepLoads + kMfma - 1) / kMfma;
#pragma unroll
        for (int t = 0; t < kPerL; ++t)
          if (loads < kStepLoads && s * kStepLoads + loads < kLoads) {
            __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
            ++loads;
          }
      }
    }
  };
  int c = 0;
  for (; c + 3 <= nk; c += 3) {
    chunk(c, buf0, buf2);
    chunk(c + 1, buf1, buf0);
    chunk(c + 2, buf2, buf1);
  }
  if (c < nk) chunk(c, buf0, buf2);
  if (c + 1 < nk) chunk(c + 1, buf1, buf0);
  // No load may still be on its way into LDS when the workgroup ends.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // C layout: value 4j + i of a block is token 8j + 4*half + i, column r32.
#pragma unroll
  for (int a = 0; a < kMB; ++a)
#pragma unroll
    for (int b = 0; b < kNB; ++b) {
      const int n = n0 + wn + 32 * b + r32;
      if (n >= N) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = m0 + wm + 32 * a + 8 * (v >> 2) + 4 * half + (v & 3);
        if (m >= M) continue;
        const int64_t o = static_cast<int64_t>(m) * N + n;
        if constexpr (kSplit)
          part[static_cast<int64_t>(blockIdx.y) * M * N + o] = acc[a][b][v];
        else
          out[o] = static_cast<uint16_t>(f32_to_bf16_bits(acc[a][b][v]));
      }
    }
}

// Decode batches (M <= 64 tokens): one workgroup takes 64 columns and one
// 512-wide slice of k, and issues every load of the slice at once (16
// weight loads a lane straight into registers, the x slice of TM 16-row
// tiles into LDS), so the slice costs one memory round trip.  Partials f32
// [split][m][n].
template <int TM, int kSpan>
__global__ __launch_bounds__(256) void gemm_cols_split_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, float* __restrict__ part,
    int M, int N, int K) {
  constexpr int kSpanPitch = kSpan + 8;  // rows 4 banks apart
  __shared__ __align__(16) uint16_t xs[TM * 16 * kSpanPitch];
  constexpr int kXSegs = TM * 16 * (kSpan / 8) / 256;  // 16-byte x segments a thread
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int n0 = blockIdx.x * kBN + wave * 16;
  const int k0 = blockIdx.y * kSpan;
  const bool live = n0 < N;

  uint4 wr[kSpan / 32];
  if (live) {
    const uint16_t* wp = w + static_cast<int64_t>(n0 + r) * K + k0 + 8 * g;
#pragma unroll
    for (int j = 0; j < kSpan / 32; ++j) wr[j] = load_w(wp + 32 * j);
  }
  uint4 xr[kXSegs];
#pragma unroll
  for (int i = 0; i < kXSegs; ++i) {
    const int seg = threadIdx.x + 256 * i;
    const int row = seg / (kSpan / 8);
    const int col = (seg % (kSpan / 8)) * 8;
    xr[i] = *reinterpret_cast<const uint4*>(x + static_cast<int64_t>(min(row, M - 1)) * K +
                                            k0 + col);
  }
#pragma unroll
  for (int i = 0; i < kXSegs; ++i) {
    const int seg = threadIdx.x + 256 * i;
    const int row = seg / (kSpan / 8);
    const int col = (seg % (kSpan / 8)) * 8;
    *reinterpret_cast<uint4*>(&xs[row * kSpanPitch + col]) = xr[i];
  }
  __syncthreads();
  if (!live) return;

  f32x4_t acc[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) acc[t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  const uint16_t* xb = &xs[r * kSpanPitch + 8 * g];
#pragma unroll
  for (int j = 0; j < kSpan / 32; ++j) {
    const bf16x8_t b = __builtin_bit_cast(bf16x8_t, wr[j]);
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      const uint4 av = *reinterpret_cast<const uint4*>(xb + 16 * t * kSpanPitch + 32 * j);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av), b,
                                                       acc[t], 0, 0, 0);
    }
  }
  float* pz = part + static_cast<int64_t>(blockIdx.y) * M * N;
#pragma unroll
  for (int t = 0; t < TM; ++t) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = 16 * t + 4 * g + j;
      if (m < M) pz[static_cast<int64_t>(m) * N + n0 + r] = acc[t][j];
    }
  }
}

// At most 16 tokens and k of up to 4,096: a workgroup takes up to 16 columns with
// one wave per 256-wide k slice, so the slices' partials meet in LDS instead of
// memory and there is no reduce launch.  Each wave issues every load of its slice
// at once (x comes from L2: at most 128 KiB, read by every workgroup); the partials
// are added in slice order, so the bits are those of the split kernel and its reduce.
//
// What bounds it is a memory round trip and each CU's share of w, so the columns
// are spread over all 256 CUs (2,816: 11 a workgroup; lanes past them repeat the
// last).  Plain loads: a fragment load takes half of each 128-byte line, the next
// one the other half.  One token x 2816 x 4096 from HBM, launches back to back:
// split kernel and reduce 9.0 us, 16 columns with non-temporal loads 8.0, with
// plain ones 7.6, 11 columns 7.0; 16 tokens 10.6 -> 9.2.  Slices of 512, which k of
// 8,192 would take, hold 128 registers of operands where 16 waves leave 128 in all:
// 2816 x 8192 13.1 -> 13.3 us at one token and 14.5 -> 18.0 at 16, so they stay with
// the split kernel.
constexpr int kFewSpan = 256;
__global__ __launch_bounds__(64 * kMaxSplits) void gemm_cols_few_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, uint16_t* __restrict__ out,
    int M, int N, int K, int cols) {
  __shared__ float part[kMaxSplits][16][17];  // [slice][token][column]
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int n0 = blockIdx.x * cols;
  const int k0 = wave * kFewSpan + 8 * g;
  const int n = min(n0 + min(r, cols - 1), N - 1);
  const uint16_t* wp = w + static_cast<int64_t>(n) * K + k0;
  const uint16_t* xp = x + static_cast<int64_t>(min(r, M - 1)) * K + k0;
  uint4 wr[kFewSpan / 32], xr[kFewSpan / 32];
#pragma unroll
  for (int j = 0; j < kFewSpan / 32; ++j) wr[j] = *reinterpret_cast<const uint4*>(wp + 32 * j);
#pragma unroll
  for (int j = 0; j < kFewSpan / 32; ++j) xr[j] = *reinterpret_cast<const uint4*>(xp + 32 * j);
  __builtin_amdgcn_sched_barrier(0);  // every load ahead of the first MFMA
  f32x4_t acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int j = 0; j < kFewSpan / 32; ++j)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, xr[j]),
                                                  __builtin_bit_cast(bf16x8_t, wr[j]), acc, 0, 0, 0);
#pragma unroll
  for (int j = 0; j < 4; ++j) part[wave][4 * g + j][r] = acc[j];
  __syncthreads();
  const int slices = K / kFewSpan;
  for (int i = threadIdx.x; i < cols * M; i += blockDim.x) {
    const int m = i / cols, c = i - m * cols;
    if (n0 + c >= N) continue;
    float s = part[0][m][c];
    for (int z = 1; z < slices; ++z) s = s + part[z][m][c];
    out[static_cast<int64_t>(m) * N + n0 + c] = static_cast<uint16_t>(f32_to_bf16_bits(s));
  }
}

// out = bf16(part[0] + part[1] + ... + part[NS-1]), four columns a thread:
// every load issues before the first add, the adds run in split order.
template <int NS>
__global__ __launch_bounds__(256) void gemm_cols_reduce_kernel(
    const float* __restrict__ part, uint16_t* __restrict__ out, int64_t quads, int64_t mn) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= quads) return;
  float4 v[NS];
#pragma unroll
  for (int z = 0; z < NS; ++z) v[z] = reinterpret_cast<const float4*>(part + z * mn)[i];
  float4 s = v[0];
#pragma unroll
  for (int z = 1; z < NS; ++z) {
    s.x = s.x + v[z].x;
    s.y = s.y + v[z].y;
    s.z = s.z + v[z].z;
    s.w = s.w + v[z].w;
  }
  const uint32_t lo = f32_to_bf16_bits(s.x) | (f32_to_bf16_bits(s.y) << 16);
  const uint32_t hi = f32_to_bf16_bits(s.z) | (f32_to_bf16_bits(s.w) << 16);
  reinterpret_cast<uint2*>(out)[i] = make_uint2(lo, hi);
}

template <int NS>
hipError_t launch_reduce_n(const float* part, uint16_t* out, int64_t quads, int64_t mn,
                           int splits, hipStream_t stream) {
  if constexpr (NS > kMaxSplits) {
    return hipErrorInvalidValue;
  } else {
    if (splits != NS) return launch_reduce_n<NS + 1>(part, out, quads, mn, splits, stream);
    hipLaunchKernelGGL((gemm_cols_reduce_kernel<NS>),
                       dim3(static_cast<unsigned>((quads + 255) / 256)), dim3(256), 0, stream,
                       part, out, quads, mn);
    return hipGetLastError();
  }
}

// k slice of the decode kernels, or 0 when the batch takes the tile kernel.
int decode_span(int64_t M, int64_t K) {
  if (M <= 16 && K % kFewSpan == 0 && K / kFewSpan <= kMaxSplits) return kFewSpan;
  if (M <= kBM && K % 512 == 0 && K / 512 <= kMaxSplits) return 512;
  return 0;
}

template <int BM, int BN>
hipError_t launch_tile(const uint16_t* x, const uint16_t* w, uint16_t* out, float* part, int M,
                       int N, int K, int splits, hipStream_t stream) {
  const int mt = (M + BM - 1) / BM, nt = (N + BN - 1) / BN;
  const unsigned blocks = static_cast<unsigned>((mt * nt + 7) / 8) * 8;
  const dim3 grid(blocks, static_cast<unsigned>(splits));
  if (splits > 1)
    hipLaunchKernelGGL((gemm_cols_tile_kernel<BM, BN, true>), grid, dim3(kTThreads), 0, stream,
                       x, w, out, part, M, N, K, K / splits, mt, nt);
  else
    hipLaunchKernelGGL((gemm_cols_tile_kernel<BM, BN, false>), grid, dim3(kTThreads), 0, stream,
                       x, w, out, nullptr, M, N, K, K, mt, nt);
  return hipGetLastError();
}

// Tile shape and k splits of a batch past the decode sizes: the cheapest by a
// model of the launch fitted to sweeps of every shape and split over 65 to
// 16,384 tokens at N = 2816, K = 4096 and 8192.  A tile costs `us` per 1,024 of
// k and the card runs 256 of them at a time (the 64 x 64 tile three per CU, so
// its partial rounds cost their share only); splits add the reduce launch,
// their own start and the f32 partials' way out and back.  It picks the
// measured best or one within 5 % of it (12 % at 128 tokens): 128 x 64 22.2 us at
// 500 tokens (two splits of 128 x 128 21.8), 192 x 128 45.1 us at 2,000 (242 of 256 CUs;
// 256 x 128, 176 tiles, 47.9), 256 x 128 342 us at 16,384 (1,106 TFLOP/s).  Other N
// and K were not fitted but measured, 65 to 6,000 tokens against the 64 x 64 kernel
// before it: 1.05 to 4.7 times as fast at N = 1,024 x 2,048, 1.3 to 4.5 at 512 x 4,096,
// 1.4 to 4.0 at 272 x 8,192, 3.1 to 6.2 at 5,376 x 8,192, 2.5 to 4.1 at 16,384 x 1,024.
// Splits whose partials do not fit the caller's workspace are left out.
struct TilePlan {
  int bm, bn, splits;
};
TilePlan tile_plan(int64_t M, int64_t N, int64_t K, int64_t workspace_bytes) {
  struct Shape {
    int bm, bn;
    double us;
  };
  constexpr Shape kShapes[] = {
      {256, 128, 11.6}, {192, 128, 9.4}, {128, 128, 6.9}, {128, 64, 5.0}, {64, 64, 4.0}};
  TilePlan best{256, 128, 1};
  double best_us = 1e30;
  for (const Shape& sh : kShapes) {
    const int64_t tiles = ((M + sh.bm - 1) / sh.bm) * ((N + sh.bn - 1) / sh.bn);
    for (int splits = 1; splits <= kMaxSplits; splits *= 2) {
      if ((K / 128) % splits != 0 || (splits > 1 && tiles * splits > 512)) break;
      if (splits > 1 && splits * M * N * 4 > workspace_bytes) break;
      const double load = static_cast<double>(tiles * splits) / 256.0;
      const double rounds =
          sh.bm == 64 ? (load > 1.0 ? load : 1.0) : static_cast<double>((tiles * splits + 255) / 256);
      double us = rounds * sh.us * static_cast<double>(K / splits) / 1024.0;
      if (splits > 1) us += 4.0 + 0.4 * splits + static_cast<double>(splits) * M * N / 1e6;
      if (us < best_us) {
        best_us = us;
        best = {sh.bm, sh.bn, splits};
      }
    }
  }
  return best;
}

hipError_t launch_plan(const TilePlan& p, const uint16_t* x, const uint16_t* w, uint16_t* out,
                       float* part, int M, int N, int K, hipStream_t stream) {
  if (p.bm == 256) return launch_tile<256, 128>(x, w, out, part, M, N, K, p.splits, stream);
  if (p.bm == 192) return launch_tile<192, 128>(x, w, out, part, M, N, K, p.splits, stream);
  if (p.bm == 128 && p.bn == 128)
    return launch_tile<128, 128>(x, w, out, part, M, N, K, p.splits, stream);
  if (p.bm == 128) return launch_tile<128, 64>(x, w, out, part, M, N, K, p.splits, stream);
  return launch_tile<64, 64>(x, w, out, part, M, N, K, p.splits, stream);
}

}  // namespace

int64_t gemm_cols_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (const int span = decode_span(M, K))
    return span == kFewSpan ? 0 : K / span * M * N * 4;  // there the slices meet in LDS
  const int splits = tile_plan(M, N, K, INT64_MAX).splits;
  return splits > 1 ? splits * M * N * 4 : 0;
}

void gemm_cols_plan(int64_t M, int64_t N, int64_t K, int64_t workspace_bytes, int64_t* plan) {
  const int span = decode_span(M, K);
  const TilePlan p = span ? TilePlan{0, 0, static_cast<int>(K / span)}
                          : tile_plan(M, N, K, workspace_bytes);
  plan[0] = p.bm;
  plan[1] = p.bn;
  plan[2] = p.splits;
}

// Batches of more than 256 tiles of 64 x 64 run without a workspace, fewer with
// room for two splits; what the plan takes beyond that is a matter of speed (400
// tokens x 2816 x 8192: four splits 33.8 us, two 32.4, none 41.1).
int64_t gemm_cols_required_bytes(int64_t M, int64_t N, int64_t K) {
  const int64_t wanted = gemm_cols_workspace_bytes(M, N, K);
  if (decode_span(M, K)) return wanted;
  const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64);
  return tiles > 256 ? 0 : std::min(wanted, 2 * M * N * 4);
}

hipError_t launch_gemm_cols(const void* x, const void* w, void* out, float* workspace,
                            int64_t workspace_bytes, int64_t M, int64_t N, int64_t K,
                            hipStream_t stream) {
  if (M <= 0) return hipSuccess;
  const int span = decode_span(M, K);
  const TilePlan plan = span ? TilePlan{} : tile_plan(M, N, K, workspace_bytes);
  const int splits = span ? static_cast<int>(K / span) : plan.splits;
  const auto* xp = static_cast<const uint16_t*>(x);
  const auto* wp = static_cast<const uint16_t*>(w);
  auto* op = static_cast<uint16_t*>(out);
  const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
  hipError_t err;
  if (span) {
    dim3 sgrid(static_cast<unsigned>((N + kBN - 1) / kBN), static_cast<unsigned>(splits));
    const int tm = static_cast<int>((M + 15) / 16);
    if (span == kFewSpan) {
      const int cols = static_cast<int>(std::min<int64_t>(16, (N + 255) / 256));
      const dim3 fgrid(static_cast<unsigned>((N + cols - 1) / cols));
      hipLaunchKernelGGL(gemm_cols_few_kernel, fgrid, dim3(static_cast<unsigned>(64 * splits)), 0,
                         stream, xp, wp, op, m, n, k, cols);
      return hipGetLastError();
    }
    if (tm == 1) {
      hipLaunchKernelGGL((gemm_cols_split_kernel<1, 512>), sgrid, dim3(256), 0, stream, xp,
                         wp, workspace, m, n, k);
    } else if (tm == 2) {
      hipLaunchKernelGGL((gemm_cols_split_kernel<2, 512>), sgrid, dim3(256), 0, stream, xp,
                         wp, workspace, m, n, k);
    } else if (tm == 3) {
      hipLaunchKernelGGL((gemm_cols_split_kernel<3, 512>), sgrid, dim3(256), 0, stream, xp,
                         wp, workspace, m, n, k);
    } else {
      hipLaunchKernelGGL((gemm_cols_split_kernel<4, 512>), sgrid, dim3(256), 0, stream, xp,
                         wp, workspace, m, n, k);
    }
    err = hipGetLastError();
  } else {
    err = launch_plan(plan, xp, wp, op, workspace, m, n, k, stream);
    if (splits == 1) return err;
  }
  if (err != hipSuccess) return err;
  return launch_reduce_n<1>(workspace, op, M * N / 4, M * N, splits, stream);
}

}  // namespace ifr
