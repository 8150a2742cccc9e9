// Full-attention prefill for launches with few query rows (gfx950): the same
// walk as the query-block kernels (FlashPrefillFullKernel + PrefillMergeKernel,
// kernels/flash_attention_prefill.mojo:117-248: tiles of 16 keys from key 0,
// the biased exp, one-segment merge), split over the waves of a workgroup so
// that 32 rows (tokens x the q heads of one kv head) occupy a whole CU.
//
// A query-block kernel gives each wave 32 rows and all keys: a chunk of 512
// tokens is 64 blocks on 256 CUs, and one decoding token's block walks its
// keys with 2 of 128 rows live.  Here the NW waves of a block share 32 rows:
//
//   scores   wave w forms the NW-tile iteration's tile w:
//            S (16 keys x 32 rows) = K . Q^T      v_mfma_f32_16x16x32_bf16
//   softmax  the tile maxima go through LDS; every wave then knows the running
//            maximum before and after each tile of the iteration, so all tiles
//            of it take their weights at once, scaled by the product of the
//            later tiles' corrections
//   P.V      wave w owns D / NW output dims of all 32 rows and reads every
//            wave's weights (bf16 hi + lo parts) from LDS:
//            O^T (16 dims x 32 rows) += V^T . P^T
//
// K tiles and V column slices are private to the wave that multiplies them, so
// it refills them (global_load_lds) as soon as it has read them, without a
// barrier; the two barriers of an iteration publish the maxima and the weights.
#include <type_traits>

#include "launch.hpp"
#include "prefill_common.hpp"

namespace ifr {
namespace {

using namespace prefill;

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kNRows = 32;         // rows of a block
constexpr int kRG = kNRows / 16;   // 16-row groups

// Members of the (lane, lane ^ 16) and (lane, lane ^ 32) pairs, lower lane
// first, the same in both lanes.
__device__ __forceinline__ void pair16(float x, float& lo, float& hi) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  lo = __uint_as_float(r[0]);
  hi = __uint_as_float(r[1]);
}
__device__ __forceinline__ void pair32(float x, float& lo, float& hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  lo = __uint_as_float(r[0]);
  hi = __uint_as_float(r[1]);
}
__device__ __forceinline__ float groups_mul(float x) {
  float a, b;
  pair16(x, a, b);
  x = a * b;
  pair32(x, a, b);
  return a * b;
}
__device__ __forceinline__ float groups_add(float x) {
  float a, b;
  pair16(x, a, b);
  x = a + b;
  pair32(x, a, b);
  return a + b;
}
__device__ __forceinline__ float raw_max(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// s_waitcnt operand that waits for vmcnt <= n alone.
constexpr int vmcnt_only(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

// LDS written so far is visible to the block; the loads in flight stay in
// flight (a __syncthreads would wait for them).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int D, int G, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW / 4, NW / 4)))
void prefill_narrow_kernel(const int32_t* __restrict__ image, const uint16_t* __restrict__ q,
                           const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
                           uint16_t* __restrict__ out, int num_q, int num_kv,
                           int64_t kv_stride, int shift, int row_mask) {
  constexpr int kTok = kNRows / G;                // tokens of a block
  constexpr int kSub = kPrefillTokens / kTok;     // blocks per plan query block
  constexpr int kKI = 16 * NW;                    // keys per iteration
  constexpr int kRowB = 2 * D;                    // bytes of a K row in LDS
  constexpr int kKS = D / 32;                     // score MFMA steps
  constexpr int kDW = D / NW;                     // output dims of a wave
  constexpr int kDB = kDW / 16;                   // 16-dim blocks of it
  constexpr int kVB = 2 * kDW;                    // bytes of a V row slice in LDS
  constexpr int kPS = kKI / 32;                   // P.V MFMA steps
  constexpr int kPRow = 2 * kKI;                  // bytes of a P row in LDS
  constexpr int kKLoads = 16 * kRowB / 1024;      // 1 KiB loads of a K tile
  constexpr int kKRowsPerLoad = 1024 / kRowB;     // 2 (D = 256) or 1
  constexpr int kLPK = kVB / 16;                  // lanes per V row slice
  constexpr int kKPL = 64 / kLPK;                 // V rows per load
  constexpr int kVLoads = kKI / kKPL;
  constexpr int kTPG = NW / 4;                    // tiles per 16-lane group
  static_assert(kKLoads < 16 + 1 && kVLoads < 16 + 1 && kTPG >= 1 && kTPG <= 2, "shape");

  __shared__ __align__(16) uint8_t kbuf[NW * 16 * kRowB];
  __shared__ __align__(16) uint8_t vbuf[NW * kKI * kVB];
  __shared__ __align__(16) uint8_t phi[kNRows * kPRow];
  __shared__ __align__(16) uint8_t plo[kNRows * kPRow];
  __shared__ __align__(16) float tmax[kNRows][NW];
  __shared__ __align__(16) float tsum[kNRows][NW];
  __shared__ __align__(16) int32_t big_flag[NW];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r16 = lane & 15;
  const int grp = lane >> 4;
  const int g = blockIdx.x % num_kv;
  const int rest = blockIdx.x / num_kv;
  const int qb = rest / kSub;
  const int sub = kSub - 1 - rest % kSub;  // the longest key range first

  const int32_t* blk = image + image[kHdrOffQBlocks] + qb * kQBlockWords;
  const int run = blk[0];
  if (sub * kTok >= blk[2]) return;  // block-uniform
  const int t0 = blk[1] + sub * kTok;
  const int ntok = min(kTok, blk[2] - sub * kTok);
  const int32_t* rp = image + image[kHdrOffRuns] + run * 4;
  const int pos0 = rp[1] + (t0 - rp[0]);  // first token's position
  const int32_t* rows = image + image[kHdrOffRows] + rp[2];

  const int min_count = pos0 + 1;         // keys below are valid for every row
  const int count_max = pos0 + ntok;      // keys the block needs
  const int last_tile = (count_max - 1) >> 4;
  const int n_it = (count_max + kKI - 1) / kKI;

  // Row r of the block: token r / G, q head g * G + r % G; lane's rows are r16
  // and 16 + r16.  Rows past the last token repeat it and are not stored.
  int count[kRG];
  int64_t q_row[kRG];
  bool live[kRG];
  bf16x8_t qf[kRG][kKS];
#pragma unroll
  for (int i = 0; i < kRG; ++i) {
    const int r = 16 * i + r16;
    const int tl = min(r / G, ntok - 1);
    live[i] = r / G < ntok;
    count[i] = min_count + tl;
    q_row[i] = static_cast<int64_t>(t0 + tl) * num_q + g * G + r % G;
    const uint16_t* qr = q + q_row[i] * D + 8 * grp;
#pragma unroll
    for (int s = 0; s < kKS; ++s) qf[i][s] = *reinterpret_cast<const bf16x8_t*>(qr + 32 * s);
  }

  // ---- staging ----
  // K tile of this wave: row r's 16-byte chunk c at c ^ r (r < 16), so the 16
  // rows of a fragment read lie in 16 bank groups.  V slice: the 32-byte unit u
  // of key k at u ^ f(k), f spreading the 16 keys that a transposing read
  // touches (8*grp + 0..3) over the units of 256 bytes.
  uint8_t* kw = kbuf + wave * 16 * kRowB;
  uint8_t* vw = vbuf + wave * kKI * kVB;
  const int64_t row_bytes = kv_stride * 2;
  const char* kg = reinterpret_cast<const char*>(kc + static_cast<int64_t>(g) * D);
  const char* vg = reinterpret_cast<const char*>(vc + static_cast<int64_t>(g) * D + wave * kDW);
  auto v_swz = [](int key) -> int {
    if constexpr (kVB == 64) return (key >> 3) & 1;
    else if constexpr (kVB == 128) return ((key >> 1) & 1) | (((key >> 3) & 1) << 1);
    else return (key & 3) | (((key >> 3) & 1) << 2);
  };
  // First cache rows of the tiles of iteration it, tile t in lane t (pages hold
  // whole tiles: page_len >= 16); tiles past the last one repeat it.  Loaded an
  // iteration before the staging that uses them.
  auto tile_slots = [&](int it) -> int {
    const int key = 16 * min(it * NW + (lane & (NW - 1)), last_tile);
    return rows[key >> shift] + (key & row_mask);
  };
  auto slot_of = [&](int slots, int t) -> int64_t {
    return __builtin_amdgcn_readlane(slots, t);
  };
  const int k_lrow = lane / (64 / kKRowsPerLoad);
  const uint32_t k_off = static_cast<uint32_t>(k_lrow) * static_cast<uint32_t>(row_bytes);
  const uint32_t k_chunk = 16u * static_cast<uint32_t>((lane % (64 / kKRowsPerLoad)) ^ k_lrow);
  auto stage_k = [&](int slots) {
    // Rows past the block's last key are other rows of its page; their scores
    // are masked.
    const char* kb = kg + slot_of(slots, wave) * row_bytes;
#pragma unroll
    for (int i = 0; i < kKLoads; ++i)  // chunk ^ row, row = kKRowsPerLoad * i + k_lrow
      __builtin_amdgcn_global_load_lds(
          static_cast<const void*>(kb + i * kKRowsPerLoad * row_bytes +
                                   (k_off + (k_chunk ^ (16u * kKRowsPerLoad * i)))),
          (lds_void_t*)(kw + i * 1024), 16, 0, 0);
  };
  const int v_lrow = lane / kLPK;
  const int v_lchunk = lane % kLPK;
  // kTail: the iteration may reach past the last key; keys past it repeat a
  // valid row (their weights are 0, and its values finite).
  auto stage_v = [&](auto tail, int it, int slots) {
#pragma unroll
    for (int i = 0; i < kVLoads; ++i) {
      const int k0 = i * kKPL;  // first key of the load within the iteration
      int lrow = v_lrow;
      if constexpr (tail.value) {
        const int tile = min(it * NW + k0 / 16, last_tile);
        lrow = min(lrow, count_max - 1 - 16 * tile - (k0 & 15));
      }
      const char* vb = vg + (slot_of(slots, k0 / 16) + (k0 & 15)) * row_bytes;
      const int64_t off = static_cast<int64_t>(lrow) * row_bytes +
                          16 * (v_lchunk ^ (2 * v_swz(k0 + v_lrow)));
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(vb + off),
                                       (lds_void_t*)(vw + i * 1024), 16, 0, 0);
    }
  };

  // ---- per-row state, the same in the four lanes of a row ----
  float m[kRG], l[kRG], S[kRG];
  f32x4_t acc[kDB][kRG];
#pragma unroll
  for (int i = 0; i < kRG; ++i) {
    m[i] = kNegBig;
    l[i] = 0.0f;
    S[i] = 1.0f;
#pragma unroll
    for (int b = 0; b < kDB; ++b) acc[b][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }
  int slots = tile_slots(0);  // of the next iteration to stage
  stage_k(slots);
  stage_v(std::true_type{}, 0, slots);
  slots = tile_slots(min(1, n_it - 1));

  const int p_swz_row = kPRow == 256 ? r16 : (r16 >> 1) & 7;  // chunk swizzle of a P row
  const int k_read = r16 * kRowB;
  // Transposing read of dim block b, keys 32 s + 8 grp + 0..3 (+4): lane j of a
  // 16-lane group addresses key j / 4 of them, dims 4 (j % 4) .. +3.
  const int vkey = 8 * grp + (r16 >> 2);

  // One iteration.  general: some rows may end inside it, or the next one may
  // reach past the last key.
  auto iteration = [&](auto general, int it) {
    constexpr bool kGeneral = general.value;
    const int itn = min(it + 1, n_it - 1);
    // ---- scores of tile it * NW + wave ----
    __builtin_amdgcn_s_waitcnt(vmcnt_only(kVLoads));  // K landed
    f32x4_t sc[kRG];
    {
      bf16x8_t kf[kKS];
#pragma unroll
      for (int s = 0; s < kKS; ++s)
        kf[s] = *reinterpret_cast<const bf16x8_t*>(kw + k_read + 16 * ((4 * s + grp) ^ r16));
#pragma unroll
      for (int i = 0; i < kRG; ++i) sc[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < kKS; ++s)
#pragma unroll
        for (int i = 0; i < kRG; ++i)
          sc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[s], qf[i][s], sc[i], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, kKS, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, kKS * kRG, 0);
    }
    // The tile's rows are in registers: refill the buffer.
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    const int slots_after = tile_slots(min(it + 2, n_it - 1));
    stage_k(slots);

    // ---- tile maxima ----
    const int tile0 = (it * NW + wave) * 16;
    if constexpr (kGeneral) {
#pragma unroll
      for (int i = 0; i < kRG; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          sc[i][j] = tile0 + 4 * grp + j < count[i] ? sc[i][j] : kNegBig;
    }
#pragma unroll
    for (int i = 0; i < kRG; ++i) {
      float mx = max3_raw(sc[i][0], sc[i][1], raw_max(sc[i][2], sc[i][3]));
      float a, b;
      pair16(mx, a, b);
      mx = raw_max(a, b);
      pair32(mx, a, b);
      mx = raw_max(a, b);
      if (grp == 0) tmax[16 * i + r16][wave] = mx;
    }
    lds_barrier();

    // ---- the iteration's corrections, this tile's weights ----
    float total[kRG];
    bool big = false;
#pragma unroll
    for (int i = 0; i < kRG; ++i) {
      // Group grp of 16 lanes handles tiles kTPG * grp ..; the running maximum
      // before them comes from the other groups' maxima.
      float tm[kTPG];
      if constexpr (kTPG == 2) {
        const float2 v = *reinterpret_cast<const float2*>(&tmax[16 * i + r16][2 * grp]);
        tm[0] = v.x;
        tm[1] = v.y;
      } else {
        tm[0] = tmax[16 * i + r16][grp];
      }
      const float gmax = kTPG == 2 ? raw_max(tm[0], tm[kTPG - 1]) : tm[0];
      float lo16, hi16, lo32, hi32;
      pair16(gmax, lo16, hi16);
      const float pmax = raw_max(lo16, hi16);
      pair32(pmax, lo32, hi32);
      const float m_end = max3_raw(m[i], lo32, hi32);
      const float e1 = (grp & 1) ? lo16 : kNegBig;
      const float e2 = (grp & 2) ? lo32 : kNegBig;
      float mb = max3_raw(m[i], e1, e2);  // before the group's first tile
      float own_total = 1.0f, own_after = 1.0f, m_sel = mb;
#pragma unroll
      for (int t = 0; t < kTPG; ++t) {
        const int tile = kTPG * grp + t;  // of the iteration
        const float mn = raw_max(mb, tm[t]);
        float c = fexp_fused_u(__builtin_fmaf(kExpA, mb - mn, kExpBias));
        if constexpr (kGeneral) c = (it * NW + tile) * 16 < count[i] ? c : 1.0f;
        own_total *= c;
        own_after *= tile > wave ? c : 1.0f;
        if (t == 0 || (wave % kTPG) == t) m_sel = mn;
        mb = mn;
      }
      total[i] = groups_mul(own_total);
      const float after = groups_mul(own_after);
      // m after tile `wave`: held by group wave / kTPG.
      pair16(m_sel, lo16, hi16);
      m_sel = (wave / kTPG) & 1 ? hi16 : lo16;
      pair32(m_sel, lo32, hi32);
      const float m_w = (wave / kTPG) & 2 ? hi32 : lo32;
      m[i] = m_end;

      const float t_arg = __builtin_fmaf(-kExpA, m_w, kExpBias);
      float e[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) e[j] = fexp_fused_u(__builtin_fmaf(kExpA, sc[i][j], t_arg));
      if constexpr (kGeneral) {
#pragma unroll
        for (int j = 0; j < 4; ++j) e[j] = tile0 + 4 * grp + j < count[i] ? e[j] : 0.0f;
      }
      const float ts = groups_add((e[0] + e[1]) + (e[2] + e[3])) * after;
      big = big || ts > kLoShare * __builtin_fmaf(l[i], total[i], ts);
      // acc = acc_stored * S: the corrections go into S, the weights are
      // divided by it; below 2^-64 the accumulators take it over.
      float S_new = S[i] * total[i];
      if (__builtin_amdgcn_ballot_w64(S_new < 0x1p-64f) != 0) {  // wave-uniform
#pragma unroll
        for (int b = 0; b < kDB; ++b) acc[b][i] = acc[b][i] * S_new;
        S_new = 1.0f;
      }
      S[i] = S_new;
      const float fs = after * __builtin_amdgcn_rcpf(S_new);
      typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
      float p[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) p[j] = e[j] * fs;
      bf16x4_t h, lw;
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const bf16x2_t hb = __builtin_convertvector(f32x2_t{p[j], p[j + 1]}, bf16x2_t);
        h[j] = hb[0];
        h[j + 1] = hb[1];
        const bf16x2_t lb = __builtin_convertvector(
            f32x2_t{p[j] - static_cast<float>(hb[0]), p[j + 1] - static_cast<float>(hb[1])},
            bf16x2_t);
        lw[j] = lb[0];
        lw[j + 1] = lb[1];
      }
      const int po = (16 * i + r16) * kPRow +
                     16 * ((2 * wave + (grp >> 1)) ^ p_swz_row) + 8 * (grp & 1);
      *reinterpret_cast<uint2*>(phi + po) = __builtin_bit_cast(uint2, h);
      *reinterpret_cast<uint2*>(plo + po) = __builtin_bit_cast(uint2, lw);
      if (grp == 0) tsum[16 * i + r16][wave] = ts;
    }
    const bool any_big = __builtin_amdgcn_ballot_w64(big) != 0;
    if (lane == 0) big_flag[wave] = any_big ? 1 : 0;
    lds_barrier();

    // ---- l, and P.V over this wave's dims ----
#pragma unroll
    for (int i = 0; i < kRG; ++i) {
      float sum = 0.0f;
#pragma unroll
      for (int t = 0; t < NW; t += 4) {
        const float4 v = *reinterpret_cast<const float4*>(&tsum[16 * i + r16][t]);
        sum += (v.x + v.y) + (v.z + v.w);
      }
      l[i] = __builtin_fmaf(l[i], total[i], sum);
    }
    int any = 0;
#pragma unroll
    for (int t = 0; t < NW; t += 4) {
      const int4 v = *reinterpret_cast<const int4*>(&big_flag[t]);
      any |= (v.x | v.y) | (v.z | v.w);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(kKLoads + 1));  // V landed
    bf16x8_t vf[kPS][kDB];
#pragma unroll
    for (int s = 0; s < kPS; ++s) {
      bf16x8_t ph[kRG];
#pragma unroll
      for (int i = 0; i < kRG; ++i)
        ph[i] = *reinterpret_cast<const bf16x8_t*>(phi + (16 * i + r16) * kPRow +
                                                   16 * ((4 * s + grp) ^ p_swz_row));
#pragma unroll
      for (int b = 0; b < kDB; ++b) {
        const int ka = 32 * s + vkey, kb = ka + 4;
        const uint8_t* pa = vw + ka * kVB + 32 * (b ^ v_swz(ka)) + 8 * (r16 & 3);
        const uint8_t* pb = vw + kb * kVB + 32 * (b ^ v_swz(kb)) + 8 * (r16 & 3);
        const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)pa);
        const s16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)pb);
        vf[s][b] = __builtin_bit_cast(bf16x8_t,
                                      __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
#pragma unroll
      for (int b = 0; b < kDB; ++b)
#pragma unroll
        for (int i = 0; i < kRG; ++i)
          acc[b][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[s][b], ph[i], acc[b][i], 0, 0, 0);
    }
    // The slice is in registers: refill it.
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    stage_v(general, itn, slots);
    // The lo parts, on the same V fragments, when some row of the block draws
    // more than kLoShare of its running l from a tile of the iteration.
    if (__builtin_amdgcn_readfirstlane(any) != 0) {
#pragma unroll
      for (int s = 0; s < kPS; ++s) {
        bf16x8_t pl[kRG];
#pragma unroll
        for (int i = 0; i < kRG; ++i)
          pl[i] = *reinterpret_cast<const bf16x8_t*>(plo + (16 * i + r16) * kPRow +
                                                     16 * ((4 * s + grp) ^ p_swz_row));
#pragma unroll
        for (int b = 0; b < kDB; ++b)
#pragma unroll
          for (int i = 0; i < kRG; ++i)
            acc[b][i] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[s][b], pl[i], acc[b][i], 0, 0, 0);
      }
    }
    slots = slots_after;
  };
  // Iterations below it_full and the ones they stage lie below every row's
  // last key.
  const int it_full = min_count / kKI - 1;
  int it = 0;
  for (; it < it_full; ++it) iteration(std::false_type{}, it);
  for (; it < n_it; ++it) iteration(std::true_type{}, it);
  // No load may still be on its way into LDS when the workgroup ends.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- one-segment merge and bf16 store (PrefillMergeKernel) ----
#pragma unroll
  for (int i = 0; i < kRG; ++i) {
    if (!live[i]) continue;
    const float c0 = l[i] > 0.0f ? fexp(0.0f) : 0.0f;
    const float gl = l[i] * c0;
    const bool some = gl > 0.0f;
    const float inv_l = some ? 1.0f / gl : 0.0f;
    uint16_t* dst = out + q_row[i] * D + wave * kDW + 4 * grp;
#pragma unroll
    for (int b = 0; b < kDB; ++b) {
      uint32_t e[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float av = (acc[b][i][j] * S[i]) * c0;
        e[j] = some ? f32_to_bf16_bits(av * inv_l) : 0u;
      }
      *reinterpret_cast<uint2*>(dst + 16 * b) = make_uint2(e[0] | (e[1] << 16), e[2] | (e[3] << 16));
    }
  }
}

}  // namespace

hipError_t launch_prefill_narrow(const int32_t* image, int num_qblocks, const void* q,
                                 const void* k, const void* v, void* output, int head_dim,
                                 int num_q, int num_kv, int64_t kv_stride, PagedGeom geom,
                                 hipStream_t stream) {
  if (num_qblocks <= 0) return hipSuccess;
  const auto* qp = static_cast<const uint16_t*>(q);
  const auto* kp = static_cast<const uint16_t*>(k);
  const auto* vp = static_cast<const uint16_t*>(v);
  auto* op = static_cast<uint16_t*>(output);
  if (head_dim == 256) {
    hipLaunchKernelGGL((prefill_narrow_kernel<256, 2, 8>), dim3(num_qblocks * 4 * num_kv),
                       dim3(512), 0, stream, image, qp, kp, vp, op, num_q, num_kv, kv_stride,
                       geom.shift, geom.row_mask);
  } else {
    hipLaunchKernelGGL((prefill_narrow_kernel<512, 8, 4>), dim3(num_qblocks * 16 * num_kv),
                       dim3(256), 0, stream, image, qp, kp, vp, op, num_q, num_kv, kv_stride,
                       geom.shift, geom.row_mask);
  }
  return hipGetLastError();
}

}  // namespace ifr
