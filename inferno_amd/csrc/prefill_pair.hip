// Chunked causal prefill of full attention at head_dim 256 / GQA 2 (gfx950),
// pages of 16 rows and more: the walk of prefill_full_mfma_kernel
// (FlashPrefillFullKernel + PrefillMergeKernel,
// kernels/flash_attention_prefill.mojo:117-248: tiles of 16 keys from key 0, the
// biased exp, one-segment merge) with two waves on every SIMD.
//
// A row is one (query token, q head).  prefill_full_mfma_kernel gives a wave 32
// rows and all 256 output dims, 200 registers of accumulators and queries, so a
// SIMD holds one wave, and that wave pays for its LDS reads, its softmax and its
// MFMAs one after the other (7,400 cycles for 64 keys where one round of blocks runs,
// 6,450 on a full grid).
// Here two waves share the 32 rows of a row group:
//
//   scores   wave w of the pair takes keys 32 w .. +31 of the 64 staged ones (two
//            16-key tiles), S^T = K . Q^T
//   softmax  the tile maxima go through LDS; both waves then know the running
//            maximum before and after each of the four tiles, so each takes the
//            weights of its own two, scaled by the later tiles' corrections
//   P.V      wave w owns output dims 128 w .. +127 and reads the pair's weights
//            (bf16 hi + lo parts) from LDS, O^T += V^T . P^T
//
// so neither scores nor softmax are repeated, each wave needs 64 accumulators,
// and eight waves (four row groups, 64 tokens) fit a CU with 256 registers each.
//
// Left alone, all eight waves would run scores, softmax and P.V at the same time
// and want the matrix cores, the vector units and LDS in turn.  The waves of row
// groups 2 and 3 (`late`; SIMD i holds waves i and i + 4) therefore run one phase
// behind: with barriers counted from the prologue, groups 0 and 1 take the scores
// of iteration it after barrier 3 it, the others after barrier 3 it + 1, and so on.
// Of the 64-key tiles in LDS, K is single-buffered: its last reader ends at barrier
// 3 it + 2, where both halves refill it; both have waited for their loads before
// barrier 3 it + 3.  V has two buffers: V of it + 1 is loaded from barrier 3 it + 1,
// when V of it - 1 has no reader left, and is waited for before 3 it + 3 as well.
//
// Bound by the three phases' own chains: 5,500 cycles for 64 keys in one round of
// blocks, 5,930 on a full grid, the matrix cores busy for 40 % of them (a lo part in
// about every third tile).  On the full grid the clock falls with the cycles (2.31 to
// 2.17 GHz), which gives most of the gain back.  Measured on one card, 8 kv heads, from
// prefill_full_mfma_kernel: 2,000 tokens on 7,000 keys 552 -> 370 us, two chunks of
// 1,500 on 1,000 to 8,000 420 -> 376, four of 500 on 1,000 111 -> 77, 2,100 on 100
// 154 -> 98, eight of 2,048 on up to 16,384 3,042 -> 2,951.  A V load that is issued
// after P.V instead costs 10 to 20 %, waves in step 8 %.
#include <type_traits>

#include "launch.hpp"
#include "prefill_waves.hpp"

namespace ifr {
namespace {

using namespace prefill;

constexpr int kPairWaves = 8;
constexpr int kPairGroups = kPairWaves / 2;   // row groups of 32 rows
constexpr int kPairSteps = kPD / 16;          // score MFMA steps
constexpr int kPairBlocks = kPD / 2 / 32;     // 32-dim blocks of a wave
constexpr int kPairRows = kKeys / kPairWaves; // key rows a wave stages
static_assert(kPairGroups * 16 == kPrefillTokens, "one block per plan query block");

__global__ __launch_bounds__(64 * kPairWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void prefill_pair_kernel(const int32_t* __restrict__ image, const uint16_t* __restrict__ q,
                         const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
                         uint16_t* __restrict__ out, int num_q, int num_kv, int64_t kv_stride,
                         int shift, int row_mask) {
  __shared__ __align__(16) uint8_t kbuf[kTileBytes];
  __shared__ __align__(16) uint8_t vbuf[2 * kTileBytes];
  __shared__ __align__(16) uint4 phi[kPairGroups][4][64];
  __shared__ __align__(16) uint4 plo[kPairGroups][4][64];
  __shared__ __align__(16) float tmax[kPairGroups * 32][4];
  __shared__ __align__(16) float tsum[kPairGroups * 32][4];
  __shared__ __align__(16) int32_t big_flag[kPairGroups][4];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int rg = wave >> 1;  // row group
  const int w2 = wave & 1;   // wave of the pair
  const bool late = wave >= kPairWaves / 2;  // one phase behind the others
  const int r = lane & 31;   // row of the group
  const int half = lane >> 5;
  const int g = blockIdx.x % num_kv;
  const int qb = blockIdx.x / num_kv;

  const int32_t* blk = image + image[kHdrOffQBlocks] + qb * kQBlockWords;
  const int run = blk[0];
  const int t0 = blk[1];
  const int ntok = blk[2];
  const int32_t* rp = image + image[kHdrOffRuns] + run * 4;
  const int pos0 = rp[1] + (t0 - rp[0]);  // first token's position
  const int32_t* rows = image + image[kHdrOffRows] + rp[2];
  const int min_count = pos0 + 1;         // keys below are valid for every row
  const int count_max = pos0 + ntok;      // keys the block needs
  const int n_it = (count_max + kKeys - 1) / kKeys;

  // Row r of group rg: token 16 rg + r / 2, q head 2 g + r % 2.  Rows past the
  // last token repeat it and are not stored.
  const int tok_local = 16 * rg + (r >> 1);
  const bool live = tok_local < ntok;
  const int tl = min(tok_local, ntok - 1);
  const int count = min_count + tl;
  const int64_t q_row = static_cast<int64_t>(t0 + tl) * num_q + g * 2 + (r & 1);
  bf16x8_t qf[kPairSteps];
  {
    const uint16_t* qr = q + q_row * kPD + 8 * half;
#pragma unroll
    for (int s = 0; s < kPairSteps; ++s) qf[s] = *reinterpret_cast<const bf16x8_t*>(qr + 16 * s);
  }

  // Waited for here: carried into the loop as outstanding, they would put waits
  // among its MFMAs that also wait for the loads into LDS.
#pragma unroll
  for (int s = 0; s < kPairSteps; ++s) asm volatile("" : "+v"(qf[s]));

  // ---- staging: wave w moves key rows 8 w .. +7 of K and of V, two a load ----
  // K: row k's 16-byte chunk c at c ^ (k % 16); V: at c ^ 2 (k % 4).
  const int64_t row_bytes = kv_stride * 2;
  const uint32_t rb32 = static_cast<uint32_t>(row_bytes);
  const char* kg = reinterpret_cast<const char*>(kc + static_cast<int64_t>(g) * kPD);
  const char* vg = reinterpret_cast<const char*>(vc + static_cast<int64_t>(g) * kPD);
  uint32_t k_off[4], v_off[4], v_chunk[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 2 * i + half;
    k_off[i] = static_cast<uint32_t>(row) * rb32 +
               16u * static_cast<uint32_t>(r ^ ((kPairRows * wave + row) & 15)) + 1024u * (3 - i);
    v_chunk[i] = 16u * static_cast<uint32_t>(r ^ (2 * (row & 3))) + 1024u * (3 - i);
    v_off[i] = static_cast<uint32_t>(row) * rb32 + v_chunk[i];
  }
  uint8_t* kw = kbuf + wave * kPairRows * kRowBytes;
  uint8_t* vw = vbuf + wave * kPairRows * kRowBytes;
  // The wave's first key row of iteration it in the cache; past the block's last
  // key, the last 8-row group it has (pages hold whole groups).
  auto group_key = [&](int it) {
    return min(it * kKeys + kPairRows * wave, (count_max - 1) & ~(kPairRows - 1));
  };
  auto slot_of = [&](int it) -> int {
    const int key = group_key(it);
    return sload(rows + (key >> shift)) + (key & row_mask);
  };
  // Rows past the last key: K's are other rows of the page (their scores are
  // masked), V's repeat a valid one (their weights are 0, its values finite).
  auto stage_k = [&](int slot) {
    load_lds4(kg + static_cast<int64_t>(slot) * row_bytes - 3072, k_off[0], k_off[1], k_off[2],
              k_off[3], kw);
  };
  auto stage_v = [&](auto general, int it, int slot) {
    uint32_t o[4];
    const int last = count_max - 1 - group_key(it);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (general.value)
        o[i] = static_cast<uint32_t>(min(2 * i + half, last)) * rb32 + v_chunk[i];
      else
        o[i] = v_off[i];
    }
    load_lds4(vg + static_cast<int64_t>(slot) * row_bytes - 3072, o[0], o[1], o[2], o[3],
              vw + (it & 1) * kTileBytes);
  };

  // ---- per-row state, the same in both lanes of a row and both waves ----
  float m = kNegBig, l = 0.0f, S = 1.0f;
  f32x16_t acc[kPairBlocks];
#pragma unroll
  for (int b = 0; b < kPairBlocks; ++b)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[b][v] = 0.0f;

  const int slot = slot_of(0);
  int slot_next = slot_of(1);  // of the iteration after the one at hand
  stage_k(slot);
  stage_v(std::true_type{}, 0, slot);
  wait_loads<0>();
  lds_barrier();

  // K fragment s of key row 32 w2 + r: chunk 2 s + half at (2 s + half) ^ (r % 16).
  const int k_read = (32 * w2 + r) * kRowBytes + 16 * ((r & 15) ^ half);
  // Transposing V reads, as in prefill_full_mfma_kernel: even and odd 32-dim
  // blocks from two lane bases, opaque so that the blocks stay immediate offsets.
  const int vj = lane & 15;
  const int v_row = (4 * half + (vj >> 2)) * kRowBytes +
                    32 * (((lane >> 4) & 1) ^ ((vj >> 2) & 1)) + 8 * (vj & 3) +
                    64 * kPairBlocks * w2;
  int v_even = v_row + 64 * (vj >> 3);
  int v_odd1 = v_row - 64 * (vj >> 3) + 64;
  asm("" : "+v"(v_even), "+v"(v_odd1));

  // One iteration.  general: some rows may end inside it.
  auto iteration = [&](auto general, int it) {
    constexpr bool kGeneral = general.value;
    const int key0 = it * kKeys + 32 * w2 + 4 * half;
    // ---- scores ----
    if (late) stage_v(general, it + 1, slot_next);
    f32x16_t sc;
#pragma unroll
    for (int v = 0; v < 16; ++v) sc[v] = 0.0f;
    {
      constexpr int kAhead = 6;  // K reads run this many MFMAs ahead
      bf16x8_t kf[kPairSteps];
#pragma unroll
      for (int s = 0; s < kPairSteps; ++s)
        kf[s] = *reinterpret_cast<const bf16x8_t*>(kbuf + (k_read ^ (32 * s)));
#pragma unroll
      for (int s = 0; s < kPairSteps; ++s)
        sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], qf[s], sc, 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
      for (int s = 0; s < kPairSteps - kAhead; ++s) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
    }
    // The maxima below are taken by instructions that the compiler does not look
    // into, so it puts no wait states between them and the MFMAs.
    asm volatile("s_nop 15\n\ts_nop 7" : "+v"(sc));
    // Value 8 u + i of a lane is key 16 u + 8 (i / 4) + 4 half + i % 4.
    if constexpr (kGeneral) {
#pragma unroll
      for (int v = 0; v < 16; ++v) sc[v] = key0 + 8 * (v >> 2) + (v & 3) < count ? sc[v] : kNegBig;
    }
    float mx[2], lo, hi;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float sv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) sv[i] = sc[8 * u + i];
      mx[u] = max8(sv);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      pair32(mx[u], lo, hi);
      mx[u] = raw_max(lo, hi);
    }
    tmax[32 * rg + r][2 * w2 + half] = half ? mx[1] : mx[0];
    lds_barrier();
    if (late) stage_k(slot_next);
    else stage_v(general, it + 1, slot_next);
    const int slot_after = slot_of(it + 2);

    // ---- corrections and weights ----
    // total: the product of all four; after[u]: of those later than the wave's
    // tile u; ta[u]: the exp argument's offset, from the maximum after that tile.
    const float4 tm = *reinterpret_cast<const float4*>(&tmax[32 * rg + r][0]);
    const float m0 = raw_max(m, tm.x), m1 = raw_max(m0, tm.y), m2 = raw_max(m1, tm.z),
                m3 = raw_max(m2, tm.w);
    float c0 = fexp_fused_u(__builtin_fmaf(kExpA, m - m0, kExpBias));
    float c1 = fexp_fused_u(__builtin_fmaf(kExpA, m0 - m1, kExpBias));
    float c2 = fexp_fused_u(__builtin_fmaf(kExpA, m1 - m2, kExpBias));
    float c3 = fexp_fused_u(__builtin_fmaf(kExpA, m2 - m3, kExpBias));
    if constexpr (kGeneral) {
      c0 = it * kKeys < count ? c0 : 1.0f;
      c1 = it * kKeys + 16 < count ? c1 : 1.0f;
      c2 = it * kKeys + 32 < count ? c2 : 1.0f;
      c3 = it * kKeys + 48 < count ? c3 : 1.0f;
    }
    m = m3;
    const float c23 = c2 * c3;
    const float total = (c0 * c1) * c23;
    const float after[2] = {w2 ? c3 : c1 * c23, w2 ? 1.0f : c23};
    const float ta[2] = {__builtin_fmaf(-kExpA, w2 ? m2 : m0, kExpBias),
                         __builtin_fmaf(-kExpA, w2 ? m3 : m1, kExpBias)};
    float e[2][8], ts[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        e[u][i] = fexp_fused_u(__builtin_fmaf(kExpA, sc[8 * u + i], ta[u]));
        if constexpr (kGeneral)
          e[u][i] = key0 + 16 * u + 8 * (i >> 2) + (i & 3) < count ? e[u][i] : 0.0f;
      }
      ts[u] = ((e[u][0] + e[u][1]) + (e[u][2] + e[u][3])) +
              ((e[u][4] + e[u][5]) + (e[u][6] + e[u][7]));
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      pair32(ts[u], lo, hi);
      ts[u] = (lo + hi) * after[u];
    }
    tsum[32 * rg + r][2 * w2 + half] = half ? ts[1] : ts[0];
    // acc = acc_stored * S: the corrections go into S, the weights are divided
    // by it; below 2^-64 the accumulators take it over.
    float S_new = S * total;
    if (__builtin_amdgcn_ballot_w64(S_new < 0x1p-64f) != 0) {  // wave-uniform
#pragma unroll
      for (int b = 0; b < kPairBlocks; ++b) acc[b] = acc[b] * S_new;
      S_new = 1.0f;
    }
    S = S_new;
    const float inv_s = __builtin_amdgcn_rcpf(S_new);
    // P in bf16 hi parts; a tile also gets its lo parts p - hi when it draws
    // more than kLoShare of some row's l.
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float fs = after[u] * inv_s;
      float p[8];
      bf16x8_t h;
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = e[u][i] * fs;
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        const bf16x2_t hb = __builtin_convertvector(f32x2_t{p[i], p[i + 1]}, bf16x2_t);
        h[i] = hb[0];
        h[i + 1] = hb[1];
      }
      phi[rg][2 * w2 + u][lane] = __builtin_bit_cast(uint4, h);
      const bool big = __builtin_amdgcn_ballot_w64(
                           ts[u] > kLoShare * __builtin_fmaf(l, total, ts[u])) != 0;
      if (big) {  // wave-uniform
        bf16x8_t w;
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
          const bf16x2_t lb = __builtin_convertvector(
              f32x2_t{p[i] - static_cast<float>(h[i]), p[i + 1] - static_cast<float>(h[i + 1])},
              bf16x2_t);
          w[i] = lb[0];
          w[i + 1] = lb[1];
        }
        plo[rg][2 * w2 + u][lane] = __builtin_bit_cast(uint4, w);
      }
      big_flag[rg][2 * w2 + u] = big ? 1 : 0;
    }
    if (late) wait_loads<0>();
    lds_barrier();
    if (!late) stage_k(slot_next);

    // ---- P.V over this wave's dims, and l ----
    const int4 flags = *reinterpret_cast<const int4*>(&big_flag[rg][0]);
    const int flag[4] = {flags.x, flags.y, flags.z, flags.w};
    bf16x8_t ph[4], pl[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) ph[t] = __builtin_bit_cast(bf16x8_t, phi[rg][t][lane]);
    // Read whether or not the tile has lo parts: a read inside the branch would
    // be waited for on its own.
#pragma unroll
    for (int t = 0; t < 4; ++t) pl[t] = __builtin_bit_cast(bf16x8_t, plo[rg][t][lane]);
    const float4 ts4 = *reinterpret_cast<const float4*>(&tsum[32 * rg + r][0]);
    // V^T fragments a tile ahead of their MFMAs.
    bf16x8_t vf[2][kPairBlocks];
    auto read_v = [&](int t) {
#pragma unroll
      for (int b = 0; b < kPairBlocks; ++b) {
        const uint8_t* vt = vbuf + (it & 1) * kTileBytes + 16 * t * kRowBytes;
        const uint8_t* vb = (b & 1) ? vt + v_odd1 + 64 * (b - 1) : vt + v_even + 64 * b;
        const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)vb);
        const s16x4_t v1 =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(vb + 8 * kRowBytes));
        vf[t & 1][b] = __builtin_bit_cast(
            bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    read_v(0);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t < 3) read_v(t + 1);
#pragma unroll
      for (int b = 0; b < kPairBlocks; ++b)
        acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[t & 1][b], ph[t], acc[b], 0, 0, 0);
      if (__builtin_amdgcn_readfirstlane(flag[t]) != 0) {
#pragma unroll
        for (int b = 0; b < kPairBlocks; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[t & 1][b], pl[t], acc[b], 0, 0, 0);
      }
    }
    l = __builtin_fmaf(l, total, (ts4.x + ts4.y) + (ts4.z + ts4.w));
    if (!late) wait_loads<0>();
    lds_barrier();
    slot_next = slot_after;
  };
  // The keys of iterations up to it_full are valid for every row.
  const int it_full = min_count / kKeys - 1;
  if (late) lds_barrier();
  int it = 0;
  for (; it < it_full; ++it) iteration(std::false_type{}, it);
  for (; it < n_it; ++it) iteration(std::true_type{}, it);
  if (!late) lds_barrier();

  // ---- one-segment merge and bf16 store (PrefillMergeKernel) ----
  // Value 4 j + i of block b is dim 128 w2 + 32 b + 8 j + 4 half + i.
  if (!live) return;
  const float c0 = l > 0.0f ? fexp(0.0f) : 0.0f;
  const float gl = l * c0;
  const bool some = gl > 0.0f;
  const float inv_l = some ? 1.0f / gl : 0.0f;
  uint16_t* dst = out + q_row * kPD + 32 * kPairBlocks * w2 + 4 * half;
#pragma unroll
  for (int b = 0; b < kPairBlocks; ++b)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float av = (acc[b][4 * j + i] * S) * c0;
        w[i] = some ? f32_to_bf16_bits(av * inv_l) : 0u;
      }
      *reinterpret_cast<uint2*>(dst + 32 * b + 8 * j) =
          make_uint2(w[0] | (w[1] << 16), w[2] | (w[3] << 16));
    }
}

}  // namespace

// Pages hold whole tiles, and a group's row offsets fit 32 bits.
bool prefill_pair_takes(int64_t kv_stride, int page_shift) {
  return page_shift >= 4 && kv_stride <= (int64_t{1} << 25);
}

hipError_t launch_prefill_pair(const int32_t* image, int num_qblocks, const void* q,
                               const void* k, const void* v, void* output, int num_q, int num_kv,
                               int64_t kv_stride, PagedGeom geom, hipStream_t stream) {
  if (num_qblocks <= 0) return hipSuccess;
  hipLaunchKernelGGL(prefill_pair_kernel, dim3(num_qblocks * num_kv), dim3(64 * kPairWaves), 0,
                     stream, image, static_cast<const uint16_t*>(q),
                     static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v),
                     static_cast<uint16_t*>(output), num_q, num_kv, kv_stride, geom.shift,
                     geom.row_mask);
  return hipGetLastError();
}

}  // namespace ifr
