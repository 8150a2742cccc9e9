// Full-attention prefill for launches with few query rows (gfx950): the same
// walk as the query-block kernels (FlashPrefillFullKernel + PrefillMergeKernel,
// kernels/flash_attention_prefill.mojo:117-248: tiles of 16 keys from key 0,
// the biased exp, one-segment merge), split over the waves of a workgroup so
// that 32 rows (tokens x the q heads of one kv head) take four waves.
//
// A query-block kernel gives each wave 32 rows and all keys: a chunk of 512
// tokens is 64 blocks on 256 CUs, and a decoding token's block in a mixed step
// walks its keys with 2 of 128 rows live.  Here the four waves of a block share
// 32 rows:
//
//   scores   each wave takes its own 16-key tile(s) of the iteration, S = K . Q^T
//   softmax  the tile maxima go through LDS; every wave then knows the running
//            maximum before and after each tile of the iteration, so all tiles
//            of it take their weights at once, scaled by the product of the
//            later tiles' corrections
//   P.V      each wave owns a quarter of the output dims and reads every wave's
//            weights (bf16 hi + lo parts) from LDS, O^T += V^T . P^T
//
// K tiles and V column slices are private to the wave that multiplies them, so
// it refills them (global_load_lds) as soon as it has read them, without a
// barrier; the two barriers of an iteration publish the maxima and the weights.
//
// What bounds them is instruction issue: a lone wave of a SIMD issues about one
// instruction per 5 cycles and one LDS read per 24 to 34 (counted, 500 tokens on 7,013
// keys, pairs: a wave's cycles go to issuing by 51 %, to waits by 29 %, to waiting for
// the issue by 20 %; matrix cores busy 20 %).  Hence two kernels.
// prefill_narrow_pairs_kernel (head_dim 256) takes tile pairs on
// v_mfma_f32_32x32x16_bf16, 128 keys an iteration: the fewest instructions per
// key, but its LDS fills a CU.  prefill_narrow_tiles_kernel takes single tiles
// on v_mfma_f32_16x16x32_bf16, 64 keys an iteration: two blocks fit a CU at
// head_dim 256 and run under each other's waits.
//
// Measured on one card at 16 q / 8 kv heads x 256 (us, prefill_pair_kernel / pairs /
// tiles; prefill_full_mfma_kernel): 64 tokens on 7,000 271 / 136 / 186; 297.  500 on
// 7,013 284 / 140 / 186; 483.  1,000 on 7,000 304 / 282 / 238; 513.  2,000 on
// 7,000 370 / 591 / 491; 552.  32 tokens decoding at 3,000 beside a 512-token
// chunk 261 / 215 / 159; 371.  At 16 / 2 x 512
// (query-block kernel / tiles): 64 tokens 517 / 278; 500 691 / 293; 1,000 749 /
// 583; 2,000 673 / 1,233; the mixed step 624 / 298.
#include <algorithm>
#include <type_traits>

#include "launch.hpp"
#include "prefill_waves.hpp"

namespace ifr {
namespace {

using namespace prefill;

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

constexpr int kNRows = 32;        // rows of a block
constexpr int kRG = kNRows / 16;  // 16-row groups
constexpr int kNW = 4;            // waves of a block

// The sub-block (kTok tokens of a plan query block) that block number `rest`
// takes, counting only those with tokens, in plan order and the longest key
// range of a query block first: qb (-1 past the last) and sub.  The blocks
// without one then all come last, and the launch leaves them out but for a few
// (prefill_narrow_blocks).  (A grid of every query block's sub-blocks in
// order puts the single live one of each decoding token's query block on the
// same shader engine: 64 of 256 CUs did that work.)
template <int kTok>
__device__ __forceinline__ void pick_sub_block(const int32_t* image, int rest, int& qb, int& sub) {
  const int n_qb = image[kHdrNumQBlocks];
  const int32_t* blocks = image + image[kHdrOffQBlocks];
  const int lane = threadIdx.x & 63;
  qb = -1;
  sub = 0;
  for (int first = 0; first < n_qb; first += 64) {
    const int i = first + lane;
    const int cnt = i < n_qb ? (blocks[i * kQBlockWords + 2] + kTok - 1) / kTok : 0;
    int x = cnt;  // inclusive scan over the wave
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31
    const int total = __builtin_amdgcn_readlane(x, 63);
    if (rest < total) {  // wave-uniform
      const int l = __builtin_ctzll(__builtin_amdgcn_ballot_w64(x > rest));
      qb = first + l;
      sub = __builtin_amdgcn_readlane(x, l) - 1 - rest;
      return;
    }
    rest -= total;
  }
}

template <int D, int G, int kPerSimd>
__global__ __launch_bounds__(64 * kNW) __attribute__((amdgpu_waves_per_eu(kPerSimd, kPerSimd)))
void prefill_narrow_tiles_kernel(const int32_t* __restrict__ image, const uint16_t* __restrict__ q,
                           const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
                           uint16_t* __restrict__ out, int num_q, int num_kv,
                           int64_t kv_stride, int shift, int row_mask) {
  constexpr int kTok = kNRows / G;                // tokens of a block
  constexpr int kKI = 16 * kNW;                    // keys per iteration
  constexpr int kRowB = 2 * D;                    // bytes of a K row in LDS
  constexpr int kKS = D / 32;                     // score MFMA steps
  constexpr int kDW = D / kNW;                     // output dims of a wave
  constexpr int kDB = kDW / 16;                   // 16-dim blocks of it
  constexpr int kVB = 2 * kDW;                    // bytes of a V row slice in LDS
  constexpr int kPS = kKI / 32;                   // P.V MFMA steps
  constexpr int kPRow = 2 * kKI;                  // bytes of a P row in LDS
  constexpr int kKLoads = 16 * kRowB / 1024;      // 1 KiB loads of a K tile
  constexpr int kKRowsPerLoad = 1024 / kRowB;     // 2 (D = 256) or 1
  constexpr int kLPK = kVB / 16;                  // lanes per V row slice
  constexpr int kKPL = 64 / kLPK;                 // V rows per load
  static_assert(kKS % kNW == 0 && kKLoads % 4 == 0, "shape");

  __shared__ __align__(16) uint8_t kbuf[kNW * 16 * kRowB];
  __shared__ __align__(16) uint8_t vbuf[kNW * kKI * kVB];
  __shared__ __align__(16) uint8_t phi[kNRows * kPRow];
  __shared__ __align__(16) uint8_t plo[kNRows * kPRow];
  __shared__ __align__(16) float tmax[kNRows][kNW];
  __shared__ __align__(16) float tsum[kNRows][kNW];
  __shared__ __align__(16) int32_t big_flag[kNW];
  __shared__ float unused[64];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r16 = lane & 15;
  const int grp = lane >> 4;
  const int g = blockIdx.x % num_kv;
  const int rest = blockIdx.x / num_kv;
  int qb, sub;
  pick_sub_block<kTok>(image, rest, qb, sub);
  if (qb < 0) return;  // block-uniform

  const int32_t* blk = image + image[kHdrOffQBlocks] + qb * kQBlockWords;
  const int run = blk[0];
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
  // Waited for here: carried into the loop as outstanding, they would put waits
  // among its MFMAs that also wait for the loads into LDS.
#pragma unroll
  for (int i = 0; i < kRG; ++i)
#pragma unroll
    for (int s = 0; s < kKS; ++s) asm volatile("" : "+v"(qf[i][s]));

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
    if constexpr (kVB == 128) return ((key >> 1) & 1) | (((key >> 3) & 1) << 1);
    else return (key & 3) | (((key >> 3) & 1) << 2);
  };
  // First cache rows of the tiles of iteration it, tile t in lane t (pages hold
  // whole tiles: page_len >= 16); tiles past the last one repeat it.  Loaded an
  // iteration before the staging that uses them.
  auto tile_slots = [&](int it) -> int {
    const int key = 16 * min(it * kNW + (lane & (kNW - 1)), last_tile);
    return rows[key >> shift] + (key & row_mask);
  };
  auto slot_of = [&](int sl, int t) -> int64_t {
    return __builtin_amdgcn_readlane(sl, t);
  };
  // The K tile is 16 rows in kKLoads loads, 4 at a time: row kKRowsPerLoad * i +
  // k_lrow of load i, its chunk ^ the row.  Rows past the block's last key are
  // other rows of its page; their scores are masked.
  const int k_lrow = lane / (64 / kKRowsPerLoad);
  const uint32_t rb32 = static_cast<uint32_t>(row_bytes);
  uint32_t k_off[kKLoads];
#pragma unroll
  for (int i = 0; i < kKLoads; ++i) {
    const int row = kKRowsPerLoad * i + k_lrow;
    k_off[i] = static_cast<uint32_t>(row) * rb32 +
               16u * static_cast<uint32_t>((lane % (64 / kKRowsPerLoad)) ^ row) +
               1024u * (3 - i % 4);
  }
  auto stage_k4 = [&](int i4, const char* kb) {
    const int i = 4 * i4;
    load_lds4(kb - 3072, k_off[i], k_off[i + 1], k_off[i + 2], k_off[i + 3], kw + i * 1024);
  };
  auto k_base = [&](int sl) { return kg + slot_of(sl, wave) * row_bytes; };
  // Tile t of the wave's V slice of iteration it, 16 rows in kVT loads.  tail:
  // the iteration may reach past the last key; keys past it repeat a valid row
  // (their weights are 0, and its values finite).
  constexpr int kVT = 16 / kKPL;
  static_assert(kVT == 2 || kVT == 4, "V loads of a tile");
  const int v_lrow = lane / kLPK;
  uint32_t v_chunk[kVT], v_off[kVT];  // the swizzle repeats every 16 keys
#pragma unroll
  for (int i = 0; i < kVT; ++i) {
    const int row = kKPL * i + v_lrow;
    v_chunk[i] = 16u * static_cast<uint32_t>((lane % kLPK) ^ (2 * v_swz(row))) + 1024u * (kVT - 1 - i);
    v_off[i] = static_cast<uint32_t>(row) * rb32 + v_chunk[i];
  }
  auto stage_v = [&](auto tail, int t, int it, int sl) {
    const char* vb = vg + slot_of(sl, t) * row_bytes - 1024 * (kVT - 1);
    uint32_t off[kVT];
#pragma unroll
    for (int i = 0; i < kVT; ++i) {
      off[i] = v_off[i];
      if constexpr (tail.value) {
        const int last = count_max - 1 - 16 * min(it * kNW + t, last_tile);
        off[i] = static_cast<uint32_t>(min(kKPL * i + v_lrow, last)) * rb32 + v_chunk[i];
      }
    }
    const uint8_t* dst = vw + t * kVT * 1024;
    if constexpr (kVT == 2) load_lds2(vb, off[0], off[1], dst);
    else load_lds4(vb, off[0], off[1], off[2], off[3], dst);
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
  int slots = tile_slots(0);                      // of the iteration at hand
  int slots_next = tile_slots(min(1, n_it - 1));  // and of the one after it
#pragma unroll
  for (int i = 0; i < kKLoads / 4; ++i) stage_k4(i, k_base(slots));

  const int p_swz_row = (r16 >> 1) & 7;  // chunk swizzle of a P row (128 bytes)
  const int k_read = r16 * kRowB;
  // Transposing read of dim block b, keys 32 s + 8 grp + 0..3 (+4): lane j of a
  // 16-lane group addresses key j / 4 of them, dims 4 (j % 4) .. +3.
  const int vkey = 8 * grp + (r16 >> 2);

  // Where the lanes of group 0 publish a row's value; the other lanes write to
  // an unused place instead of branching.
  float* pub_max[kRG];
  float* pub_sum[kRG];
#pragma unroll
  for (int i = 0; i < kRG; ++i) {
    pub_max[i] = grp == 0 ? &tmax[16 * i + r16][wave] : &unused[lane];
    pub_sum[i] = grp == 0 ? &tsum[16 * i + r16][wave] : &unused[lane];
  }
  int p_write[kRG];
#pragma unroll
  for (int i = 0; i < kRG; ++i)
    p_write[i] = (16 * i + r16) * kPRow + 16 * ((2 * wave + (grp >> 1)) ^ p_swz_row) + 8 * (grp & 1);

  // One iteration.  general: some rows may end inside it.
  auto iteration = [&](auto general, int it) {
    constexpr bool kGeneral = general.value;
    const int tile0 = (it * kNW + wave) * 16;
    // ---- scores of tile it * kNW + wave, with the V loads of the iteration
    // between the MFMAs (its slice was read by the last P.V) ----
    wait_loads<0>();  // K landed
    f32x4_t sc[kRG];
    {
      bf16x8_t kf[kKS];
#pragma unroll
      for (int s = 0; s < kKS; ++s)
        kf[s] = *reinterpret_cast<const bf16x8_t*>(kw + k_read + 16 * ((4 * s + grp) ^ r16));
#pragma unroll
      for (int i = 0; i < kRG; ++i) sc[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < kKS; ++s) {
        if (s % (kKS / kNW) == 0) stage_v(general, s / (kKS / kNW), it, slots);
#pragma unroll
        for (int i = 0; i < kRG; ++i)
          sc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[s], qf[i][s], sc[i], 0, 0, 0);
      }
    }
    // The maxima below are taken by instructions that the compiler does not look
    // into, so it puts no wait states between them and the MFMAs.
    asm volatile("s_nop 15\n\ts_nop 7" : "+v"(sc[0]), "+v"(sc[1]));
    if constexpr (kGeneral) {
#pragma unroll
      for (int i = 0; i < kRG; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          sc[i][j] = tile0 + 4 * grp + j < count[i] ? sc[i][j] : kNegBig;
    }
    float mx[kRG];
#pragma unroll
    for (int i = 0; i < kRG; ++i)
      mx[i] = max3_raw(sc[i][0], sc[i][1], raw_max(sc[i][2], sc[i][3]));
#pragma unroll
    for (int i = 0; i < kRG; ++i) mx[i] = groups_max(mx[i]);
#pragma unroll
    for (int i = 0; i < kRG; ++i) *pub_max[i] = mx[i];
    // Also the point from which the K tile may be refilled: its reads are done.
    lds_barrier();

    // ---- the iteration's corrections and this tile's weights; the K loads of
    // the next iteration go out along the way ----
    const char* kb = k_base(slots_next);
    slots = slots_next;
    slots_next = tile_slots(min(it + 2, n_it - 1));
    int issued = 0;
    auto k_load = [&]() {
      if (issued < kKLoads / 4) stage_k4(issued++, kb);
    };
    // Group grp of 16 lanes handles tile grp; the running maximum before it comes
    // from the other groups' maxima.
    float tm[kRG];
#pragma unroll
    for (int i = 0; i < kRG; ++i) tm[i] = tmax[16 * i + r16][grp];
    k_load();
    float m_t[kRG], c[kRG];
#pragma unroll
    for (int i = 0; i < kRG; ++i) {
      float lo16, hi16, lo32, hi32;
      pair16(tm[i], lo16, hi16);
      pair32(raw_max(lo16, hi16), lo32, hi32);
      const float mb = max3_raw(m[i], (grp & 1) ? lo16 : kNegBig, (grp & 2) ? lo32 : kNegBig);
      m[i] = max3_raw(m[i], lo32, hi32);
      m_t[i] = raw_max(mb, tm[i]);
      c[i] = fexp_fused_u(__builtin_fmaf(kExpA, mb - m_t[i], kExpBias));
      if constexpr (kGeneral) c[i] = (it * kNW + grp) * 16 < count[i] ? c[i] : 1.0f;
    }
    // total: the product of all corrections; after: of those later than this
    // wave's tile; m_w: the running maximum after it (held by group `wave`).
    float total[kRG], after[kRG], m_w[kRG];
#pragma unroll
    for (int i = 0; i < kRG; ++i) {
      total[i] = groups_mul(c[i]);
      after[i] = groups_mul(grp > wave ? c[i] : 1.0f);
      float lo, hi;
      pair16(m_t[i], lo, hi);
      pair32(wave & 1 ? hi : lo, lo, hi);
      m_w[i] = wave & 2 ? hi : lo;
    }
    k_load();
    float e[kRG][4], ts[kRG];
#pragma unroll
    for (int i = 0; i < kRG; ++i) {
      const float t_arg = __builtin_fmaf(-kExpA, m_w[i], kExpBias);
#pragma unroll
      for (int j = 0; j < 4; ++j) e[i][j] = fexp_fused_u(__builtin_fmaf(kExpA, sc[i][j], t_arg));
      if constexpr (kGeneral) {
#pragma unroll
        for (int j = 0; j < 4; ++j) e[i][j] = tile0 + 4 * grp + j < count[i] ? e[i][j] : 0.0f;
      }
      k_load();
    }
    bool big = false;
    float S_new[kRG];
#pragma unroll
    for (int i = 0; i < kRG; ++i) {
      ts[i] = groups_add((e[i][0] + e[i][1]) + (e[i][2] + e[i][3])) * after[i];
      big = big || ts[i] > kLoShare * __builtin_fmaf(l[i], total[i], ts[i]);
      S_new[i] = S[i] * total[i];
    }
    // acc = acc_stored * S: the corrections go into S, the weights are divided
    // by it; below 2^-64 the accumulators take it over.
    bool small = false;
#pragma unroll
    for (int i = 0; i < kRG; ++i) small = small || S_new[i] < 0x1p-64f;
    if (__builtin_amdgcn_ballot_w64(small) != 0) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < kRG; ++i) {
#pragma unroll
        for (int b = 0; b < kDB; ++b) acc[b][i] = acc[b][i] * S_new[i];
        S_new[i] = 1.0f;
      }
    }
    const bool any_big = __builtin_amdgcn_ballot_w64(big) != 0;  // wave-uniform
    float p[kRG][4];
    bf16x4_t h[kRG];
#pragma unroll
    for (int i = 0; i < kRG; ++i) {
      S[i] = S_new[i];
      const float fs = after[i] * __builtin_amdgcn_rcpf(S_new[i]);
#pragma unroll
      for (int j = 0; j < 4; ++j) p[i][j] = e[i][j] * fs;
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const bf16x2_t hb = __builtin_convertvector(f32x2_t{p[i][j], p[i][j + 1]}, bf16x2_t);
        h[i][j] = hb[0];
        h[i][j + 1] = hb[1];
      }
      *reinterpret_cast<uint2*>(phi + p_write[i]) = __builtin_bit_cast(uint2, h[i]);
      *pub_sum[i] = ts[i];
    }
#pragma unroll
    for (int i = 0; i < kKLoads / 4; ++i) k_load();
    // The lo parts p - hi: zeros when no row draws more than kLoShare of its l
    // from the tile (its step's other tile may have some).
    uint2 lo_bits[kRG];
#pragma unroll
    for (int i = 0; i < kRG; ++i) lo_bits[i] = make_uint2(0u, 0u);
    if (any_big) {
#pragma unroll
      for (int i = 0; i < kRG; ++i) {
        bf16x4_t lw;
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
          const bf16x2_t lb = __builtin_convertvector(
              f32x2_t{p[i][j] - static_cast<float>(h[i][j]),
                      p[i][j + 1] - static_cast<float>(h[i][j + 1])},
              bf16x2_t);
          lw[j] = lb[0];
          lw[j + 1] = lb[1];
        }
        lo_bits[i] = __builtin_bit_cast(uint2, lw);
      }
    }
#pragma unroll
    for (int i = 0; i < kRG; ++i) *reinterpret_cast<uint2*>(plo + p_write[i]) = lo_bits[i];
    big_flag[wave] = any_big ? 1 : 0;
    lds_barrier();

    // ---- P.V over this wave's dims, and l ----
    int flags[kNW];
#pragma unroll
    for (int t = 0; t < kNW; t += 4) {
      const int4 v = *reinterpret_cast<const int4*>(&big_flag[t]);
      flags[t] = v.x;
      flags[t + 1] = v.y;
      flags[t + 2] = v.z;
      flags[t + 3] = v.w;
    }
    wait_loads<kKLoads>();  // V landed (the K loads came after it)
    bf16x8_t vf[kPS][kDB], ph[kPS][kRG], pl[kPS][kRG];
#pragma unroll
    for (int s = 0; s < kPS; ++s) {
#pragma unroll
      for (int i = 0; i < kRG; ++i)
        ph[s][i] = *reinterpret_cast<const bf16x8_t*>(phi + (16 * i + r16) * kPRow +
                                                      16 * ((4 * s + grp) ^ p_swz_row));
#pragma unroll
      for (int b = 0; b < kDB; ++b) {
        const int ka = 32 * s + vkey, kb2 = ka + 4;
        const uint8_t* pa = vw + ka * kVB + 32 * (b ^ v_swz(ka)) + 8 * (r16 & 3);
        const uint8_t* pb = vw + kb2 * kVB + 32 * (b ^ v_swz(kb2)) + 8 * (r16 & 3);
        const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)pa);
        const s16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)pb);
        vf[s][b] = __builtin_bit_cast(bf16x8_t,
                                      __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
#pragma unroll
      for (int b = 0; b < kDB; ++b)
#pragma unroll
        for (int i = 0; i < kRG; ++i)
          acc[b][i] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[s][b], ph[s][i], acc[b][i], 0, 0, 0);
    }
    // The lo parts on the same V fragments, for the steps with a flagged tile;
    // read in any case: a read inside the branch would be waited for on its own.
#pragma unroll
    for (int s = 0; s < kPS; ++s)
#pragma unroll
      for (int i = 0; i < kRG; ++i)
        pl[s][i] = *reinterpret_cast<const bf16x8_t*>(plo + (16 * i + r16) * kPRow +
                                                      16 * ((4 * s + grp) ^ p_swz_row));
#pragma unroll
    for (int i = 0; i < kRG; ++i) {
      float sum = 0.0f;
#pragma unroll
      for (int t = 0; t < kNW; t += 4) {
        const float4 v = *reinterpret_cast<const float4*>(&tsum[16 * i + r16][t]);
        sum += (v.x + v.y) + (v.z + v.w);
      }
      l[i] = __builtin_fmaf(l[i], total[i], sum);
    }
#pragma unroll
    for (int s = 0; s < kPS; ++s)
      if (__builtin_amdgcn_readfirstlane(flags[2 * s] | flags[2 * s + 1]) != 0) {
#pragma unroll
        for (int b = 0; b < kDB; ++b)
#pragma unroll
          for (int i = 0; i < kRG; ++i)
            acc[b][i] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[s][b], pl[s][i], acc[b][i], 0, 0, 0);
      }
    // The slice is in registers: the next iteration may refill it.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  // The keys of iterations below it_full are valid for every row.
  const int it_full = min_count / kKI;
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

constexpr int kNKeys = 32 * kNW;   // keys per iteration
constexpr int kNTiles = 2 * kNW;   // 16-key tiles per iteration

template <int D, int G>
__global__ __launch_bounds__(64 * kNW) __attribute__((amdgpu_waves_per_eu(1, 1)))
void prefill_narrow_pairs_kernel(const int32_t* __restrict__ image, const uint16_t* __restrict__ q,
                           const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
                           uint16_t* __restrict__ out, int num_q, int num_kv,
                           int64_t kv_stride, int shift, int row_mask) {
  constexpr int kTok = kNRows / G;              // tokens of a block
  constexpr int kKS = D / 16;                   // score MFMA steps
  constexpr int kRowB = 2 * D;                  // bytes of a K row
  constexpr int kDW = D / kNW;              // output dims of a wave
  constexpr int kDB = kDW / 32;                 // 32-dim blocks of it
  constexpr int kVB = 2 * kDW;                  // bytes of a V row slice in LDS
  constexpr int kKRows = 1024 / kRowB;          // K rows per 1 KiB load
  constexpr int kKLoads = 32 / kKRows;          // loads of a wave's 32 K rows
  constexpr int kLPK = kVB / 16;                // lanes per V row slice
  constexpr int kKPL = 64 / kLPK;               // V rows per load
  constexpr int kVLoads = kNKeys / kKPL;
  static_assert(kVLoads == kKS && kKLoads == kKS, "one V load per score step");

  __shared__ __align__(16) uint8_t kbuf[kNKeys * kRowB];
  __shared__ __align__(16) uint8_t vbuf[kNW * kNKeys * kVB];
  __shared__ __align__(16) uint4 phi[kNTiles][64];
  __shared__ __align__(16) uint4 plo[kNTiles][64];
  __shared__ __align__(16) float tmax[kNRows][kNTiles];
  __shared__ __align__(16) float tsum[kNRows][kNTiles];
  __shared__ __align__(16) int32_t big_flag[kNTiles];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r = lane & 31;       // row of the block
  const int half = lane >> 5;
  const int g = blockIdx.x % num_kv;
  const int rest = blockIdx.x / num_kv;
  int qb, sub;
  pick_sub_block<kTok>(image, rest, qb, sub);
  if (qb < 0) return;  // block-uniform

  const int32_t* blk = image + image[kHdrOffQBlocks] + qb * kQBlockWords;
  const int run = blk[0];
  const int t0 = blk[1] + sub * kTok;
  const int ntok = min(kTok, blk[2] - sub * kTok);
  const int32_t* rp = image + image[kHdrOffRuns] + run * 4;
  const int pos0 = rp[1] + (t0 - rp[0]);  // first token's position
  const int32_t* rows = image + image[kHdrOffRows] + rp[2];

  const int min_count = pos0 + 1;         // keys below are valid for every row
  const int count_max = pos0 + ntok;      // keys the block needs
  const int last_tile = (count_max - 1) >> 4;
  const int n_it = (count_max + kNKeys - 1) / kNKeys;

  // Row r: token r / G, q head g * G + r % G.  Rows past the last token repeat
  // it and are not stored.
  const int tl = min(r / G, ntok - 1);
  const bool live = r / G < ntok;
  const int count = min_count + tl;
  const int64_t q_row = static_cast<int64_t>(t0 + tl) * num_q + g * G + r % G;
  bf16x8_t qf[kKS];
  {
    const uint16_t* qr = q + q_row * D + 8 * half;
#pragma unroll
    for (int s = 0; s < kKS; ++s) qf[s] = *reinterpret_cast<const bf16x8_t*>(qr + 16 * s);
  }
#pragma unroll
  for (int s = 0; s < kKS; ++s) asm volatile("" : "+v"(qf[s]));  // waited for, as above

  // ---- staging ----
  // The wave's 32 K rows: row k's 16-byte chunk c at c ^ (k % 16), so the rows
  // of a fragment read lie in different bank groups.  V slice: the 32-byte
  // unit u of key k at u ^ f(k), f spreading the 16 keys that a transposing
  // read touches over the units of 256 bytes.
  uint8_t* kw = kbuf + wave * 32 * kRowB;
  uint8_t* vw = vbuf + wave * kNKeys * kVB;
  const int64_t row_bytes = kv_stride * 2;
  const uint32_t rb32 = static_cast<uint32_t>(row_bytes);
  const char* kg = reinterpret_cast<const char*>(kc + static_cast<int64_t>(g) * D);
  const char* vg = reinterpret_cast<const char*>(vc + static_cast<int64_t>(g) * D + wave * kDW);
  auto v_swz = [](int key) -> int {
    if constexpr (kVB == 128) return ((key >> 1) & 1) | (((key >> 2) & 1) << 1);
    else return key & 7;
  };
  // First cache rows of the tiles of iteration it, tile t in lane t (pages hold
  // whole tiles: page_len >= 16); tiles past the last one repeat it.  Loaded an
  // iteration before the staging that uses them.
  auto tile_slots = [&](int it) -> int {
    const int key = 16 * min(it * kNTiles + (lane & (kNTiles - 1)), last_tile);
    return rows[key >> shift] + (key & row_mask);
  };
  auto slot_of = [&](int sl, int t) -> int64_t { return __builtin_amdgcn_readlane(sl, t); };
  // A K tile is 16 rows in kTL loads, 4 at a time; row kKRows * i + k_lrow of
  // load i, its chunk ^ the row.  Rows past the block's last key are other rows
  // of its page; their scores are masked.
  constexpr int kTL = kKLoads / 2;
  const int k_lrow = lane / (64 / kKRows);
  uint32_t k_off[kTL];
#pragma unroll
  for (int i = 0; i < kTL; ++i) {
    const int row = kKRows * i + k_lrow;
    k_off[i] = static_cast<uint32_t>(row) * rb32 +
               16u * static_cast<uint32_t>((lane % (64 / kKRows)) ^ row) + 1024u * (3 - i % 4);
  }
  auto stage_k4 = [&](int i4, const char* kb) {  // loads 4 * i4 .. of the wave's two tiles
    const int i = 4 * i4 % kTL;
    load_lds4(kb - 3072, k_off[i], k_off[i + 1], k_off[i + 2], k_off[i + 3], kw + i4 * 4096);
  };
  auto k_base = [&](int sl, int t) { return kg + slot_of(sl, 2 * wave + t) * row_bytes; };
  // Tile t of the wave's V slice of iteration it, 16 rows in kVT loads.  tail:
  // the iteration may reach past the last key; keys past it repeat a valid row
  // (their weights are 0, and its values finite).
  constexpr int kVT = 16 / kKPL;
  static_assert(kVT == 2 || kVT == 4, "V loads of a tile");
  const int v_lrow = lane / kLPK;
  uint32_t v_chunk[kVT], v_off[kVT];
#pragma unroll
  for (int i = 0; i < kVT; ++i) {
    const int row = kKPL * i + v_lrow;
    v_chunk[i] = 16u * static_cast<uint32_t>((lane % kLPK) ^ (2 * v_swz(row))) + 1024u * (kVT - 1 - i);
    v_off[i] = static_cast<uint32_t>(row) * rb32 + v_chunk[i];
  }
  auto stage_v = [&](auto tail, int t, int it, int sl) {
    const char* vb = vg + slot_of(sl, t) * row_bytes - 1024 * (kVT - 1);
    uint32_t off[kVT];
#pragma unroll
    for (int i = 0; i < kVT; ++i) {
      off[i] = v_off[i];
      if constexpr (tail.value) {
        const int last = count_max - 1 - 16 * min(it * kNTiles + t, last_tile);
        off[i] = static_cast<uint32_t>(min(kKPL * i + v_lrow, last)) * rb32 + v_chunk[i];
      }
    }
    if constexpr (kVT == 2) load_lds2(vb, off[0], off[1], vw + t * 2048);
    else load_lds4(vb, off[0], off[1], off[2], off[3], vw + t * 4096);
  };

  // ---- per-row state, the same in both lanes of a row ----
  float m = kNegBig, l = 0.0f, S = 1.0f;
  f32x16_t acc[kDB];
#pragma unroll
  for (int b = 0; b < kDB; ++b)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[b][v] = 0.0f;

  int slots = tile_slots(0);                      // of the iteration at hand
  int slots_next = tile_slots(min(1, n_it - 1));  // and of the one after it
#pragma unroll
  for (int i = 0; i < kKLoads / 4; ++i) stage_k4(i, k_base(slots, 4 * i / kTL));

  const int k_read = r * kRowB + 16 * ((r & 15) ^ half);  // fragment s at k_read ^ 32 s
  // Transposing read of dim block b of a tile: lane j of 16-lane group q
  // addresses key 4 * half + j / 4 (+ 8 for the second read), dims
  // 16 * (q % 2) + 4 * (j % 4) .. +3, and gets the four keys of dim
  // 16 * (q % 2) + j: the k order of the lane's own P values.
  const int j16 = lane & 15;
  const int vkey = 4 * half + (j16 >> 2);
  const int vunit = (lane >> 4) & 1;

  // One iteration.  general: some rows may end inside it.
  auto iteration = [&](auto general, int it) {
    constexpr bool kGeneral = general.value;
    const int key0 = it * kNKeys + 32 * wave;  // of the wave's two tiles
    // ---- scores, with the V loads of the iteration between the MFMAs (the
    // slice was read by the last P.V) ----
    f32x16_t sc;
#pragma unroll
    for (int v = 0; v < 16; ++v) sc[v] = 0.0f;
    wait_loads<0>();  // K landed
    bf16x8_t kf[kKS];
#pragma unroll
    for (int s = 0; s < kKS; ++s)
      kf[s] = *reinterpret_cast<const bf16x8_t*>(kw + (k_read ^ (32 * s)));
#pragma unroll
    for (int s = 0; s < kKS; ++s) {
      if (s % (kKS / kNTiles) == 0) stage_v(general, s / (kKS / kNTiles), it, slots);
      sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], qf[s], sc, 0, 0, 0);
    }
    asm volatile("s_nop 15\n\ts_nop 7" : "+v"(sc));
    // Value 8 u + i of a lane is key 16 u + 8 (i / 4) + 4 half + i % 4.
    if constexpr (kGeneral) {
#pragma unroll
      for (int v = 0; v < 16; ++v)
        sc[v] = key0 + 8 * (v >> 2) + 4 * half + (v & 3) < count ? sc[v] : kNegBig;
    }
    float mx[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float sv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) sv[i] = sc[8 * u + i];
      mx[u] = max8(sv);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float a, b;
      pair32(mx[u], a, b);
      mx[u] = raw_max(a, b);
    }
    tmax[r][2 * wave + half] = half ? mx[1] : mx[0];
    // Also the point from which the K rows may be refilled: their reads are done.
    lds_barrier();

    // ---- the iteration's corrections and these tiles' weights; the K loads of
    // the next iteration go out along the way ----
    const char* kb0 = k_base(slots_next, 0);
    const char* kb1 = k_base(slots_next, 1);
    slots = slots_next;
    slots_next = tile_slots(min(it + 2, n_it - 1));
    int issued = 0;
    auto k_load = [&]() {
      if (issued < kKLoads / 4) {
        stage_k4(issued, 4 * issued < kTL ? kb0 : kb1);
        ++issued;
      }
    };
    // Half h of the lanes handles tiles 4 h .. 4 h + 3; the running maximum
    // before tile 4 comes from the other half's maxima.
    const float4 tm4 = *reinterpret_cast<const float4*>(&tmax[r][4 * half]);
    const float tm[4] = {tm4.x, tm4.y, tm4.z, tm4.w};
    k_load();
    float mn[4], c[4], lo, hi;
    pair32(raw_max(max3_raw(tm[0], tm[1], tm[2]), tm[3]), lo, hi);
    {
      float mb = half ? raw_max(m, lo) : m;
      m = max3_raw(m, lo, hi);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        mn[t] = raw_max(mb, tm[t]);
        c[t] = fexp_fused_u(__builtin_fmaf(kExpA, mb - mn[t], kExpBias));
        if constexpr (kGeneral)
          c[t] = (it * kNTiles + 4 * half + t) * 16 < count ? c[t] : 1.0f;
        mb = mn[t];
      }
    }
    // Of this wave's tiles a = 2 wave and b = a + 1, both held by half wave / 2:
    // the maxima after them, b's correction, and the product of the later ones.
    const float own_total = (c[0] * c[1]) * (c[2] * c[3]);
    const bool second = wave & 1;
    float own_after = (second ? 1.0f : c[2]) * (second ? 1.0f : c[3]);
    own_after = (wave >> 1) == half ? own_after : ((wave >> 1) < half ? own_total : 1.0f);
    pair32(own_total, lo, hi);
    const float total = lo * hi;
    pair32(own_after, lo, hi);
    const float after_b = lo * hi;
    pair32(second ? mn[2] : mn[0], lo, hi);
    const float m_a = wave >> 1 ? hi : lo;
    pair32(second ? mn[3] : mn[1], lo, hi);
    const float m_b = wave >> 1 ? hi : lo;
    pair32(second ? c[3] : c[1], lo, hi);
    const float after_a = after_b * (wave >> 1 ? hi : lo);
    const float after[2] = {after_a, after_b};
    const float ta[2] = {__builtin_fmaf(-kExpA, m_a, kExpBias), __builtin_fmaf(-kExpA, m_b, kExpBias)};
    float e[2][8], ts[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        e[u][i] = fexp_fused_u(__builtin_fmaf(kExpA, sc[8 * u + i], ta[u]));
        if constexpr (kGeneral)
          e[u][i] = key0 + 16 * u + 8 * (i >> 2) + 4 * half + (i & 3) < count ? e[u][i] : 0.0f;
      }
      k_load();
      ts[u] = ((e[u][0] + e[u][1]) + (e[u][2] + e[u][3])) + ((e[u][4] + e[u][5]) + (e[u][6] + e[u][7]));
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      pair32(ts[u], lo, hi);
      ts[u] = (lo + hi) * after[u];
    }
    tsum[r][2 * wave + half] = half ? ts[1] : ts[0];
    // acc = acc_stored * S: the corrections go into S, the weights are divided
    // by it; below 2^-64 the accumulators take it over.
    float S_new = S * total;
    if (__builtin_amdgcn_ballot_w64(S_new < 0x1p-64f) != 0) {  // wave-uniform
#pragma unroll
      for (int b = 0; b < kDB; ++b) acc[b] = acc[b] * S_new;
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
      phi[2 * wave + u][lane] = __builtin_bit_cast(uint4, h);
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
        plo[2 * wave + u][lane] = __builtin_bit_cast(uint4, w);
      }
      big_flag[2 * wave + u] = big ? 1 : 0;
      k_load();
    }
#pragma unroll
    for (int i = 0; i < kKLoads / 4; ++i) k_load();
    lds_barrier();

    // ---- P.V over this wave's dims, and l ----
    int flags[kNTiles];
#pragma unroll
    for (int t = 0; t < kNTiles; t += 4) {
      const int4 v = *reinterpret_cast<const int4*>(&big_flag[t]);
      flags[t] = v.x;
      flags[t + 1] = v.y;
      flags[t + 2] = v.z;
      flags[t + 3] = v.w;
    }
    // V landed: the K loads issued after it may be outstanding.
    wait_loads<kKLoads>();
    bf16x8_t vf[kNTiles][kDB];
    bf16x8_t ph[kNTiles];
#pragma unroll
    for (int t = 0; t < kNTiles; ++t) {
      ph[t] = __builtin_bit_cast(bf16x8_t, phi[t][lane]);
#pragma unroll
      for (int b = 0; b < kDB; ++b) {
        const int ka = 16 * t + vkey, kb = ka + 8;
        const int u = 2 * b + vunit;
        const uint8_t* pa = vw + ka * kVB + 32 * (u ^ v_swz(ka)) + 8 * (j16 & 3);
        const uint8_t* pb = vw + kb * kVB + 32 * (u ^ v_swz(kb)) + 8 * (j16 & 3);
        const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)pa);
        const s16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)pb);
        vf[t][b] = __builtin_bit_cast(bf16x8_t,
                                      __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    }
#pragma unroll
    for (int t = 0; t < kNTiles; ++t)
#pragma unroll
      for (int b = 0; b < kDB; ++b)
        acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[t][b], ph[t], acc[b], 0, 0, 0);
    // Read whether or not the tile has lo parts: a read inside the branch
    // would be waited for on its own.
    bf16x8_t pl[kNTiles];
#pragma unroll
    for (int t = 0; t < kNTiles; ++t) pl[t] = __builtin_bit_cast(bf16x8_t, plo[t][lane]);
    {
      const float4 v0 = *reinterpret_cast<const float4*>(&tsum[r][0]);
      const float4 v1 = *reinterpret_cast<const float4*>(&tsum[r][4]);
      l = __builtin_fmaf(l, total, ((v0.x + v0.y) + (v0.z + v0.w)) + ((v1.x + v1.y) + (v1.z + v1.w)));
    }
#pragma unroll
    for (int t = 0; t < kNTiles; ++t)
      if (__builtin_amdgcn_readfirstlane(flags[t]) != 0) {
#pragma unroll
        for (int b = 0; b < kDB; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[t][b], pl[t], acc[b], 0, 0, 0);
      }
    // The slice is in registers: the next iteration may refill it.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  // The keys of iterations below it_full are valid for every row.
  const int it_full = min_count / kNKeys;
  int it = 0;
  for (; it < it_full; ++it) iteration(std::false_type{}, it);
  for (; it < n_it; ++it) iteration(std::true_type{}, it);
  // No load may still be on its way into LDS when the workgroup ends.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- one-segment merge and bf16 store (PrefillMergeKernel) ----
  // Value 4 j + i of block b is dim 32 b + 8 j + 4 half + i.
  if (!live) return;
  const float c0 = l > 0.0f ? fexp(0.0f) : 0.0f;
  const float gl = l * c0;
  const bool some = gl > 0.0f;
  const float inv_l = some ? 1.0f / gl : 0.0f;
  uint16_t* dst = out + q_row * D + wave * kDW + 4 * half;
#pragma unroll
  for (int b = 0; b < kDB; ++b)
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

// Blocks of 32 rows (kTok tokens of a run, one kv head) that a launch needs: at most
// this many have tokens, as every run may end in a partial one.  Of every query
// block's 64 / kTok, most have none where many sequences decode, and each of those
// walks the whole plan to find that out: 2,000 sequences of up to 100 keys beside 32
// tokens 1,986 -> 271 us at 16 / 2 heads x 512, 1,065 -> 408 at 16 / 8 x 256.
int64_t prefill_narrow_blocks(int64_t num_qblocks, int64_t num_runs, int64_t seq_len,
                              int64_t num_kv, int head_dim) {
  const int64_t tok = head_dim == 256 ? 16 : 4;
  return std::min((seq_len + (tok - 1) * num_runs) / tok, kPrefillTokens / tok * num_qblocks) *
         num_kv;
}

// Which kernel takes a full-attention token plan: 0 the query-block kernel, 1
// tiles, 2 pairs.  A cost in us per 128 keys, from the measurements above: a
// launch takes its 256 (or, tiles at head_dim 256, 512) blocks at a time.  The
// query-block kernels' later rounds overlap, so beyond one round they cost their
// share of it.
int prefill_narrow_kind(int64_t num_qblocks, int64_t num_runs, int64_t seq_len, int64_t num_kv,
                        int head_dim, int64_t kv_stride, int page_shift) {
  // Pages hold whole tiles, and a tile's row offsets fit 32 bits.
  if (page_shift < 4 || kv_stride > (int64_t{1} << 25)) return 0;
  auto rounds = [](int64_t blocks, int64_t at_once) {
    return static_cast<double>((blocks + at_once - 1) / at_once);
  };
  auto block_cost = [](int64_t blocks, double one, double more) {
    return blocks <= 256 ? one : (one > more * blocks / 256.0 ? one : more * blocks / 256.0);
  };
  const int64_t live = prefill_narrow_blocks(num_qblocks, num_runs, seq_len, num_kv, head_dim);
  if (head_dim == 256) {
    const double block = block_cost(num_qblocks * num_kv, 5.1, 6.3);
    const double pairs = 2.45 * rounds(live, 256);
    const double tiles = live <= 256 ? 3.2 : 4.3 * rounds(live, 512);
    // Within 3 % the query-block kernel: what the costs leave out, a block's own start,
    // is paid by more blocks in the narrow ones (300 runs of 20 tokens on up to 50 at
    // one kv head, 7.38 against 7.35: pairs 25.7 us, prefill_pair_kernel 19.1).
    if (block <= 1.03 * std::min(pairs, tiles)) return 0;
    return pairs <= tiles ? 2 : 1;
  }
  return 5.05 * rounds(live, 256) < block_cost(4 * num_qblocks * num_kv, 11.5, 9.8) ? 1 : 0;
}

hipError_t launch_prefill_narrow(const int32_t* image, int kind, int64_t blocks, const void* q,
                                 const void* k, const void* v, void* output, int head_dim,
                                 int num_q, int num_kv, int64_t kv_stride, PagedGeom geom,
                                 hipStream_t stream) {
  if (blocks <= 0) return hipSuccess;
  const dim3 grid(static_cast<unsigned>(blocks));
  const auto* qp = static_cast<const uint16_t*>(q);
  const auto* kp = static_cast<const uint16_t*>(k);
  const auto* vp = static_cast<const uint16_t*>(v);
  auto* op = static_cast<uint16_t*>(output);
  if (head_dim == 256 && kind == 2)
    hipLaunchKernelGGL((prefill_narrow_pairs_kernel<256, 2>), grid, dim3(64 * kNW), 0, stream,
                       image, qp, kp, vp, op, num_q, num_kv, kv_stride, geom.shift,
                       geom.row_mask);
  else if (head_dim == 256)
    hipLaunchKernelGGL((prefill_narrow_tiles_kernel<256, 2, 2>), grid, dim3(64 * kNW), 0, stream,
                       image, qp, kp, vp, op, num_q, num_kv, kv_stride, geom.shift,
                       geom.row_mask);
  else
    hipLaunchKernelGGL((prefill_narrow_tiles_kernel<512, 8, 1>), grid, dim3(64 * kNW), 0, stream,
                       image, qp, kp, vp, op, num_q, num_kv, kv_stride, geom.shift,
                       geom.row_mask);
  return hipGetLastError();
}

}  // namespace ifr
