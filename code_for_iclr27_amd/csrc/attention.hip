// Attention over the packed ragged KV layout: one query block per (request, KV head) segment,
// the drop-in for the flash_attn_varlen_func call of src/lazy_recall/attention.py:15-35.
//
// Segment s (= request b * kv_heads + KV head h) owns key rows [cu[s], cu[s+1]) of the packed
// K/V buffers and `length` queries for each of its G = query_heads / kv_heads query heads. Its
// L*G query rows are numbered row = i*G + g (query i, group g). Causal masking is aligned to the
// end of the segment, as flash-attention's varlen causal mode: query i sees keys j <= i + n - L
// (n = the segment's key count); for decode (L = 1) that is every key. A row with no visible key
// outputs zeros. Softmax scale `scale`, accumulation in f32, output rounded to the input type.
//
// Calls with many query rows (prefill) run the kernel of attention_tile.hip; takes_tiles has the
// rule. Here: decode, and a few query rows on a cached prefix.
//
// Work split (flash decoding): a workgroup of four waves owns R query rows of one segment and
// one block of keys; each wave takes 12-16 KB of its K rows (wave_keys) and issues every load
// (queries, K rows, V slices) before the first use, so one memory round trip covers the wave.
// QK^T runs on v_mfma_f32_16x16x32 (the R rows padded to 16, K rows straight into the B operand,
// 16 B per lane); each wave forms its own max and exp-sum in registers, stages p in LDS and
// accumulates P*V on the VALU with each lane holding 8 elements of a V row (D/8 lanes per row).
// The four wave states merge in LDS. A segment whose keys need more than one block writes
// (max, sum, unnormalised output) partials, and a second launch merges them (one workgroup per
// segment and tile). The launch boundary orders the two: a device-scope fence per workgroup
// instead (a ticket taken by the last block) costs an L2 writeback and invalidate on every
// workgroup's XCD, and measured 4-6x slower at the cfg2 decode shape.

#include <algorithm>
#include <mutex>
#include <string>

#include "attention_tile.hpp"

namespace lr {
namespace {

// Keys per wave: 12 KB of K rows (and as many V bytes) for d64/d128, 16 KB for d256 (a whole
// number of 16-key MFMA blocks); small enough for three waves per SIMD. A call whose blocks of
// that size would not give every CU two workgroups (batch-1 decode: cfg1 has 96) takes one
// 16-key MFMA block per wave instead, so that its single round of loads spreads over the chip.
constexpr int wave_keys(int dim) { return dim == 256 ? 32 : 6144 / dim; }
constexpr int kSmallWaveKeys = 16;
constexpr int64_t kFewBlocks = 512;
// Partial states the allocation-free entry point holds (per device).
constexpr size_t kAttentionScratchBytes = size_t{16} << 20;

// The value of the lane a reduction step pairs with. Lane bits 0 and 1: that lane exactly; bits 2
// and 3: a lane of the other half of 8 or 16 lanes, the same value once the bits below are
// reduced (cross-lane reads in the vector ALU, no LDS round trip).
template <int BIT>
__device__ __forceinline__ float paired(float x) {
  constexpr int kControl = BIT == 0 ? 0xB1 : BIT == 1 ? 0x4E : BIT == 2 ? 0x141 : 0x140;
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
      0, __builtin_bit_cast(int, x), kControl, 0xF, 0xF, false));
}
// Max or sum over the 16 lanes of a row, in all of them.
template <bool kMax>
__device__ __forceinline__ float reduce16(float x) {
  auto step = [&](float y) { x = kMax ? fmaxf(x, y) : x + y; };
  step(paired<0>(x));
  step(paired<1>(x));
  step(paired<2>(x));
  step(paired<3>(x));
  return x;
}
// x plus its copy in the lane 2^BIT away (BIT 3: see paired; 4 and 5 swap whole rows).
template <int BIT>
__device__ __forceinline__ float plus_paired(float x) {
  if constexpr (BIT <= 3) {
    return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                   0, __builtin_bit_cast(int, x), 0x128, 0xF, 0xF, false));  // row_ror:8
  } else {
    const LanePair pair = lane_pair<1 << BIT>(x);
    return pair.first + pair.second;
  }
}

// Segment bounds, clamped into the key buffer, and the key blocks (of `block` keys) that the tile
// whose last query is `last_query` sees. A pending row (the decode step's own token, not yet
// appended) is key `cached` of the segment, after its cached rows.
struct SegmentKeys {
  int64_t key0;
  int cached, n, shift, key_end, needed;  // query i sees keys j <= i + shift
};
__device__ __forceinline__ SegmentKeys segment_keys(const AttnArgs& a, unsigned seg,
                                                    unsigned last_query, int block) {
  SegmentKeys k;
  int64_t key0 = a.cu[seg], n = static_cast<int64_t>(a.cu[seg + 1]) - key0;
  key0 = key0 < 0 ? 0 : (key0 > a.key_rows ? a.key_rows : key0);
  n = n < 0 ? 0 : (n > a.key_rows - key0 ? a.key_rows - key0 : n);
  k.key0 = key0;
  k.cached = static_cast<int>(n);
  k.n = k.cached + (a.pending_keys != nullptr ? 1 : 0);
  k.shift = k.n - static_cast<int>(a.length);
  const int end = static_cast<int>(last_query) + k.shift + 1;
  k.key_end = end < 0 ? 0 : (end > k.n ? k.n : end);
  // keys past splits * block are not read
  k.needed = min(static_cast<int>((static_cast<unsigned>(k.key_end) + block - 1) / block),
                 static_cast<int>(a.splits));
  return k;
}

// SEVERAL: several queries, of which a key may be hidden from some (a form of its own: the check
// below, in every decode launch's instructions, cost 32 layers 2 us of 474).
template <typename T, int D, int R, int CH, bool SEVERAL>
__global__ __launch_bounds__(kAttnThreads, D == 256 ? 2 : 3) void packed_attention_kernel(AttnArgs a) {
  static_assert(D == 64 || D == 128 || D == 256, "head dim");
  static_assert(R == 4 || R == 8, "rows per tile");
  constexpr int KS = D / 32;          // MFMA k-steps over the head dimension
  constexpr int LPK = D / 8;          // lanes per V row in the P*V phase
  constexpr int KPI = 64 / LPK;       // V rows per wave-wide load
  static_assert(CH % 16 == 0, "whole MFMA key blocks");
  constexpr int NB = CH / 16;         // 16-key MFMA blocks per wave
  constexpr int VL = CH / KPI;        // V loads (16 B) per lane
  constexpr int ITEMS = R * LPK;      // (row, 8-element slice) items of one output tile
  static_assert(ITEMS <= kAttnThreads, "one merge item per thread");
  using Vec = AttnVec<T>;
  using X8 = typename Vec::x8;
  __shared__ __align__(16) float probs[kAttnWaves][CH][R];
  __shared__ __align__(16) float wave_o[kAttnWaves][R][D];
  __shared__ float wave_ml[kAttnWaves][R][2];

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const unsigned splits = static_cast<unsigned>(a.splits), tiles = static_cast<unsigned>(a.tiles);
  const unsigned groups = static_cast<unsigned>(a.groups);
  const unsigned unit = blockIdx.x / splits, split = blockIdx.x - unit * splits;
  const unsigned seg = tiles == 1 ? unit : unit / tiles, tile = unit - seg * tiles;
  const unsigned rows = static_cast<unsigned>(a.length) * groups;
  const unsigned row0 = tile * R;
  const int rows_here = static_cast<int>(min(rows - row0, static_cast<unsigned>(R)));
  constexpr int kBlockKeys = kAttnWaves * CH;
  const SegmentKeys keys = segment_keys(a, seg, query_of(a, row0 + rows_here - 1), kBlockKeys);

  if (keys.needed == 0) {  // no visible key for any row of this tile: zeros
    if (split != 0) return;
    for (int item = tid; item < ITEMS; item += kAttnThreads) {
      const int r = item / LPK, c = item - r * LPK;
      if (r < rows_here)
        *reinterpret_cast<attn_u32x4*>(output_row<T, D>(a, seg, row0 + r) + 8 * c) =
            attn_u32x4{0u, 0u, 0u, 0u};
    }
    return;
  }
  if (static_cast<int>(split) >= keys.needed) return;  // uniform across the workgroup

  const int kb = static_cast<int>(split) * kBlockKeys + wave * CH;
  const int ke = kb + CH < keys.key_end ? kb + CH : keys.key_end;
  const int nk = kb < ke ? ke - kb : 0;
  const int m = lane & 15, j = lane >> 4;
  const int kg = lane / LPK, c = lane - kg * LPK;

  float row_max[4] = {kNegInf, kNegInf, kNegInf, kNegInf};
  float row_sum[4] = {0.f, 0.f, 0.f, 0.f};
  float acc[R][8];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[r][e] = 0.f;

  if (nk > 0) {
    const T* kbase = static_cast<const T*>(a.keys) + (keys.key0 + kb) * D;
    const T* vbase = static_cast<const T*>(a.values) + (keys.key0 + kb) * D;
    // row of wave key `key` (< nk): a cached row, or the segment's pending row
    const int cached_here = keys.cached - kb;
    auto key_row = [&](const T* base, const void* pending, int key) -> const T* {
      return key < cached_here ? base + key * D
                               : static_cast<const T*>(pending) + static_cast<int64_t>(seg) * D;
    };
    // Every load of the wave is issued before the first use: queries (A operand, row m = lane
    // & 15, k chunk j = lane >> 4), K rows (B operand, key m of each 16-key block), V slices.
    X8 qop[KS];
    {
      const bool row_ok = m < rows_here;
      const unsigned row = row0 + (row_ok ? m : 0);
      const unsigned b = seg / static_cast<unsigned>(a.kv_heads);
      const unsigned h = seg - b * static_cast<unsigned>(a.kv_heads);
      const unsigned i = query_of(a, row), g = row - i * groups;
      const T* q = static_cast<const T*>(a.queries) + b * a.q_batch +
                   static_cast<int64_t>(h * groups + g) * a.q_head + i * a.q_query + 8 * j;
      // Unconditional loads from a valid row (padding lanes read row0's) and a select after
      // them: a load under a branch is waited for inside the branch.
      attn_u32x4 raw[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) raw[ks] = load16(q + 32 * ks);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        qop[ks] = __builtin_bit_cast(X8, row_ok ? raw[ks] : attn_u32x4{0u, 0u, 0u, 0u});
    }
    attn_u32x4 kraw[NB][KS];
#pragma unroll
    for (int blk = 0; blk < NB; ++blk) {
      int key = blk * 16 + m;
      key = key < nk ? key : nk - 1;  // clamped in-range row; its score is masked below
      const T* kp = key_row(kbase, a.pending_keys, key) + 8 * j;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kraw[blk][ks] = load16(kp + 32 * ks);
    }
    attn_u32x4 vraw[VL];
#pragma unroll
    for (int u = 0; u < VL; ++u) {
      int key = kg + u * KPI;
      key = key < nk ? key : nk - 1;
      vraw[u] = load16(key_row(vbase, a.pending_values, key) + 8 * c);
    }

    // QK^T. D layout: lane holds key 16 * blk + (lane & 15) for rows 4j + r.
    int limit[4];  // causal limit of this lane's rows, relative to kb (keys <= limit seen)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      limit[r] = 4 * j + r < rows_here
                     ? static_cast<int>(query_of(a, row0 + 4 * j + r)) + keys.shift - kb : -1;
    float s[NB][4];
#pragma unroll
    for (int blk = 0; blk < NB; ++blk) {
      attn_f32x4 dot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) dot = Vec::mfma(qop[ks], __builtin_bit_cast(X8, kraw[blk][ks]), dot);
      const int key = blk * 16 + m;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[blk][r] = (key < nk && key <= limit[r]) ? dot[r] * a.scale : kNegInf;
        row_max[r] = fmaxf(row_max[r], s[blk][r]);
      }
    }
    // Row max and exp-sum over the 16 lanes that share rows 4j .. 4j + 3.
#pragma unroll
    for (int r = 0; r < 4; ++r) row_max[r] = reduce16<true>(row_max[r]);
#pragma unroll
    for (int blk = 0; blk < NB; ++blk) {
      attn_f32x4 p;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[r] = s[blk][r] == kNegInf ? 0.f
                                    : __builtin_amdgcn_exp2f((s[blk][r] - row_max[r]) * kAttnLog2e);
        row_sum[r] += p[r];
      }
      if (4 * j < R) *reinterpret_cast<attn_f32x4*>(&probs[wave][blk * 16 + m][4 * j]) = p;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) row_sum[r] = reduce16<false>(row_sum[r]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // P*V on the prefetched V slices; keys past nk carry p = 0 from a clamped row, skipped.
#pragma unroll
    for (int u = 0; u < VL; ++u) {
      const int key = kg + u * KPI;
      if (key >= nk) break;
      float v[8];
      unpack8<T>(vraw[u], v);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float p = probs[wave][key][r];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r][e] = __builtin_fmaf(p, v[e], acc[r][e]);
      }
    }
    // A masked key's p is 0, and 0 * V is NaN for a non-finite V: a wave with a non-finite sum takes
    // its rows again, over the keys that each of them sees. (Every row of a decode call sees all.)
    if constexpr (SEVERAL) {
      float poison = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < 8; ++e) poison = __builtin_fmaf(acc[r][e], 0.f, poison);
      if (__any(poison != poison)) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[r][e] = 0.f;
#pragma unroll 1
        for (int key = kg; key < nk; key += KPI) {
          float v[8];
          unpack8<T>(load16(vbase + key * D + 8 * c), v);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            if (key > static_cast<int>(query_of(a, row0 + r)) + keys.shift - kb) continue;
            const float p = probs[wave][key][r];
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[r][e] = __builtin_fmaf(p, v[e], acc[r][e]);
          }
        }
      }
    }
    // Sum the KPI lane groups (lanes c, c + LPK, ... hold the same elements).
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (LPK <= 8) acc[r][e] = plus_paired<3>(acc[r][e]);
        if constexpr (LPK <= 16) acc[r][e] = plus_paired<4>(acc[r][e]);
        acc[r][e] = plus_paired<5>(acc[r][e]);
      }
  }

  // Wave states to LDS: rows r = 4j + i are held by lanes 16j .. 16j + 15.
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r % KPI != kg) continue;
    float* wo = &wave_o[wave][r][8 * c];
    *reinterpret_cast<attn_f32x4*>(wo) = attn_f32x4{acc[r][0], acc[r][1], acc[r][2], acc[r][3]};
    *reinterpret_cast<attn_f32x4*>(wo + 4) = attn_f32x4{acc[r][4], acc[r][5], acc[r][6], acc[r][7]};
  }
  if (m == 0 && 4 * j < R) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      wave_ml[wave][4 * j + r][0] = row_max[r];
      wave_ml[wave][4 * j + r][1] = row_sum[r];
    }
  }
  __syncthreads();

  // Merge the waves: thread t < ITEMS owns row r = t / LPK, elements 8 * (t % LPK) ...
  const int r_item = tid / LPK, c_item = tid - r_item * LPK;
  MergeState st{kNegInf, 0.f, {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}};
  if (tid < ITEMS) {
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) {
      float o[8];
      const float* wo = &wave_o[w][r_item][8 * c_item];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = wo[e];
      merge_into(st, wave_ml[w][r_item][0], wave_ml[w][r_item][1], o);
    }
  }
  if (keys.needed == 1) {  // the only block of keys: normalise and write
    if (tid < ITEMS && r_item < rows_here) {
      const float inv = st.l > 0.f ? 1.0f / st.l : 0.f;
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = st.o[e] * inv;
      *reinterpret_cast<attn_u32x4*>(output_row<T, D>(a, seg, row0 + r_item) + 8 * c_item) =
          pack8<T>(o);
    }
    return;
  }

  // ---- Partial state of this block; attention_merge_kernel combines the blocks.
  const int64_t slot = static_cast<int64_t>(blockIdx.x) * R;
  if (tid < ITEMS) {
    float* po = a.part_o + (slot + r_item) * D + 8 * c_item;
    *reinterpret_cast<attn_f32x4*>(po) = attn_f32x4{st.o[0], st.o[1], st.o[2], st.o[3]};
    *reinterpret_cast<attn_f32x4*>(po + 4) = attn_f32x4{st.o[4], st.o[5], st.o[6], st.o[7]};
    if (c_item == 0) {
      a.part_ml[(slot + r_item) * 2] = st.m;
      a.part_ml[(slot + r_item) * 2 + 1] = st.l;
    }
  }
}

// Second launch: one workgroup per (segment, tile) whose keys spanned more than one block merges
// the blocks' partial states. Thread (part, item) folds blocks part, part + PARTS, ... (in that
// order, whatever U) with the loads of U blocks in flight at once; the PARTS states then meet
// in LDS.
template <typename T, int D, int R, int CH, int U>
__global__ __launch_bounds__(kAttnThreads) void attention_merge_kernel(AttnArgs a) {
  constexpr int LPK = D / 8;
  constexpr int ITEMS = R * LPK;
  constexpr int PARTS = kAttnThreads / ITEMS;
  __shared__ __align__(16) float merge_o[kAttnThreads][8];
  __shared__ float merge_ml[kAttnThreads][2];
  const int tid = threadIdx.x;
  const unsigned unit = blockIdx.x, tiles = static_cast<unsigned>(a.tiles);
  const unsigned splits = static_cast<unsigned>(a.splits);
  const unsigned seg = tiles == 1 ? unit : unit / tiles, tile = unit - seg * tiles;
  const unsigned rows = static_cast<unsigned>(a.length) * static_cast<unsigned>(a.groups);
  const unsigned row0 = tile * R;
  const int rows_here = static_cast<int>(min(rows - row0, static_cast<unsigned>(R)));
  const int part = tid / ITEMS, item = tid - part * ITEMS;
  const int r = item / LPK, cc = item - r * LPK;
  const int64_t first = static_cast<int64_t>(unit) * splits * R;
  // The first round of partial states is loaded before the segment's bounds are known (every slot
  // of the grid's splits is in the workspace; those past the needed ones are not used), so that
  // the two memory round trips overlap.
  float mk[U], lk[U];
  attn_f32x4 lo[U], hi[U];
  auto load = [&](unsigned k0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned k = k0 + u * PARTS < splits ? k0 + u * PARTS : 0;
      const int64_t at = first + static_cast<int64_t>(k) * R + r;
      mk[u] = a.part_ml[at * 2];
      lk[u] = a.part_ml[at * 2 + 1];
      lo[u] = *reinterpret_cast<const attn_f32x4*>(a.part_o + at * D + 8 * cc);
      hi[u] = *reinterpret_cast<const attn_f32x4*>(a.part_o + at * D + 8 * cc + 4);
    }
  };
  load(part);
  const unsigned needed = static_cast<unsigned>(
      segment_keys(a, seg, query_of(a, row0 + rows_here - 1), kAttnWaves * CH).needed);
  if (needed <= 1) return;  // the first launch wrote this tile's output
  MergeState total{kNegInf, 0.f, {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}};
  for (unsigned k0 = part; k0 < needed; k0 += PARTS * U) {
    if (k0 != static_cast<unsigned>(part)) load(k0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float o[8] = {lo[u][0], lo[u][1], lo[u][2], lo[u][3],
                          hi[u][0], hi[u][1], hi[u][2], hi[u][3]};
      merge_into(total, k0 + u * PARTS < needed ? mk[u] : kNegInf, lk[u], o);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) merge_o[tid][e] = total.o[e];
  merge_ml[tid][0] = total.m;
  merge_ml[tid][1] = total.l;
  __syncthreads();
  if (part != 0 || r >= rows_here) return;
  for (int p = 1; p < PARTS; ++p) {
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = merge_o[p * ITEMS + item][e];
    merge_into(total, merge_ml[p * ITEMS + item][0], merge_ml[p * ITEMS + item][1], o);
  }
  const float inv = total.l > 0.f ? 1.0f / total.l : 0.f;
  float o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = total.o[e] * inv;
  *reinterpret_cast<attn_u32x4*>(output_row<T, D>(a, seg, row0 + r) + 8 * cc) = pack8<T>(o);
}

struct AttnPlan {
  int rows_per_tile, wave_keys;
  int64_t tiles, splits, chunk, units;
};

AttnPlan plan_attention(int64_t segments, int64_t groups, int64_t length, int64_t max_keys,
                        int64_t dim) {
  AttnPlan p{};
  const int64_t rows = length * groups;
  p.rows_per_tile = rows <= 4 ? 4 : 8;
  p.tiles = ceil_div(rows, p.rows_per_tile);
  p.units = segments * p.tiles;
  // Keys one workgroup covers: four waves of wave_keys keys each.
  p.wave_keys = wave_keys(static_cast<int>(dim));
  p.chunk = kAttnWaves * p.wave_keys;
  p.splits = std::max<int64_t>(1, ceil_div(max_keys, p.chunk));
  if (p.units * p.splits < kFewBlocks && p.splits > 1) {
    p.wave_keys = kSmallWaveKeys;
    p.chunk = kAttnWaves * p.wave_keys;
    p.splits = ceil_div(max_keys, p.chunk);
  }
  return p;
}

size_t workspace_bytes(const AttnPlan& p, int64_t dim) {
  if (p.splits == 1) return 0;
  const int64_t slots = p.units * p.splits * p.rows_per_tile;
  return static_cast<size_t>(slots) * static_cast<size_t>(dim + 2) * 4;
}

// The prefill kernel's plan. Calls whose segments fit one block of the split-key kernel's keys need
// no workspace, so their keys are not split here either. Other partial states stay within the
// allocation-free entry point's array for every call that entry point accepts (its limit is the
// split-key plan's bytes, below), and within 32 MiB otherwise.
AttnTilePlan plan_tiles(int64_t segments, int64_t groups, int64_t length, int64_t max_keys,
                        int64_t dim) {
  const size_t blocks = workspace_bytes(plan_attention(segments, groups, length, max_keys, dim), dim);
  const size_t most = blocks == 0                        ? 0
                      : blocks <= kAttentionScratchBytes ? kAttentionScratchBytes
                                                         : size_t{32} << 20;
  return plan_attention_tiles(segments, groups, length, max_keys, dim, static_cast<int64_t>(most));
}

// Whether a call of several queries runs the prefill kernel (attention_tile.hip): where its estimate
// is the lower one. A call of the split-key kernel takes `call` us, less for few keys or rows; its
// blocks add up on a CU once there are more than alone / block of them, and a split call pays the
// merge and its partial states. The prefill plan's own estimate is scaled (an f16 stage takes
// longer). Fitted to 3,600 shapes (each head dimension, 2 to 64 segments, 1 to 8 groups, 2 to 256
// queries, 2 to 4,000 keys) timed with both kernels: the choice is 0.1% to 0.8% above the better one
// on average, by dimension and type. Both sides, us, split-key and tiles: 4 segments, G6, 8 queries
// on 200 keys at d256 10.8 and 14.7; 8 segments, G4, 32 queries on 300 at d64, f16, 9.9 and 12.5;
// 24 segments, G4, 2 queries on 4,000 at d128 27.4 and 20.4.
struct SplitKeyTimes {
  double call, alone, block, small_block, merge, megabyte;
};
bool takes_tiles(int64_t segments, int64_t groups, int64_t length, int64_t max_keys, int64_t dim,
                 int dtype) {
  if (length <= 1) return false;
  const SplitKeyTimes us = dim == 64    ? SplitKeyTimes{7.4, 1.2, 2.4, 0.6, 0.4, 2.5}
                           : dim == 128 ? SplitKeyTimes{7.5, 0.7, 2.2, 0.75, 1.3, 1.3}
                                        : SplitKeyTimes{7.9, 0.5, 3.7, 1.75, 2.0, 0.6};
  const AttnPlan plan = plan_attention(segments, groups, length, max_keys, dim);
  const double load = static_cast<double>(plan.units) * static_cast<double>(plan.splits) / 256.0 *
                      (plan.wave_keys == kSmallWaveKeys ? us.small_block : us.block);
  const double split_key =
      us.call - (plan.rows_per_tile == 4 ? 1.0 : 0.0) -
      0.04 * static_cast<double>(std::max<int64_t>(0, 64 - max_keys)) + std::max(us.alone, load) +
      (plan.splits > 1 ? us.merge + us.megabyte * 1e-6 * static_cast<double>(workspace_bytes(plan, dim))
                       : 0.0);
  const bool f16 = dtype == LR_DTYPE_F16;
  const double estimate = plan_tiles(segments, groups, length, max_keys, dim).us;
  const double tiles = dim == 64    ? (f16 ? 3.2 + 1.39 * estimate : 3.2 + 1.23 * estimate)
                       : dim == 128 ? (f16 ? 3.4 + 1.42 * estimate : 2.9 + 1.30 * estimate)
                                    : (f16 ? 5.1 + 1.44 * estimate : 4.2 + 1.22 * estimate);
  return tiles < split_key;
}

template <typename T, int D, int R, int CH>
int launch_attention(const AttnArgs& args, int64_t blocks, hipStream_t stream) {
  auto attend = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(kAttnThreads), 0, stream,
                       args);
  };
  if (args.length > 1) attend(packed_attention_kernel<T, D, R, CH, true>);
  else attend(packed_attention_kernel<T, D, R, CH, false>);
  if (int status = check_launch("packed_attention")) return status;
  if (args.splits == 1) return LR_OK;
  // Blocks each merging thread folds (PARTS = threads / (R * D / 8) threads share a row slice):
  // the smallest round of loads that holds them, or rounds of twelve. Nine of a cfg1 layer's 36
  // blocks in a round of nine take 0.6 us a layer less than in one of twelve, whose last loads
  // repeat a block.
  const int64_t per_part = ceil_div(args.splits, int64_t{kAttnThreads / (R * D / 8)});
  auto merge = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks / args.splits)),
                       dim3(kAttnThreads), 0, stream, args);
  };
  if (per_part <= 2) merge(attention_merge_kernel<T, D, R, CH, 2>);
  else if (per_part <= 4) merge(attention_merge_kernel<T, D, R, CH, 4>);
  else if (per_part <= 6) merge(attention_merge_kernel<T, D, R, CH, 6>);
  else if (per_part <= 9) merge(attention_merge_kernel<T, D, R, CH, 9>);
  else merge(attention_merge_kernel<T, D, R, CH, 12>);
  return check_launch("packed_attention merge");
}

template <typename T, int D, int R>
int launch_keys(const AttnArgs& args, int keys_per_wave, int64_t blocks, hipStream_t stream) {
  return keys_per_wave == kSmallWaveKeys
             ? launch_attention<T, D, R, kSmallWaveKeys>(args, blocks, stream)
             : launch_attention<T, D, R, wave_keys(D)>(args, blocks, stream);
}

template <typename T, int D>
int launch_rows(const AttnArgs& args, const AttnPlan& plan, int64_t blocks, hipStream_t stream) {
  return plan.rows_per_tile == 4 ? launch_keys<T, D, 4>(args, plan.wave_keys, blocks, stream)
                                 : launch_keys<T, D, 8>(args, plan.wave_keys, blocks, stream);
}

template <typename T>
int launch_dim(const AttnArgs& args, int64_t dim, const AttnPlan& plan, int64_t blocks,
               hipStream_t stream) {
  switch (dim) {
    case 64: return launch_rows<T, 64>(args, plan, blocks, stream);
    case 128: return launch_rows<T, 128>(args, plan, blocks, stream);
    default: return launch_rows<T, 256>(args, plan, blocks, stream);
  }
}

}  // namespace
}  // namespace lr

using namespace lr;

extern "C" size_t lr_packed_attention_workspace_bytes(int64_t segments, int64_t groups,
                                                      int64_t length, int64_t max_keys,
                                                      int64_t dim) {
  if (segments <= 0 || groups <= 0 || length <= 0 || max_keys < 0 || dim <= 0) return 0;
  const size_t split_key = workspace_bytes(plan_attention(segments, groups, length, max_keys, dim), dim);
  if (length == 1) return split_key;
  // what either type needs: which kernel runs depends on it
  const bool bf16 = takes_tiles(segments, groups, length, max_keys, dim, LR_DTYPE_BF16);
  const bool f16 = takes_tiles(segments, groups, length, max_keys, dim, LR_DTYPE_F16);
  if (!bf16 && !f16) return split_key;
  const size_t tiles =
      attention_tiles_bytes(plan_tiles(segments, groups, length, max_keys, dim), dim);
  return bf16 && f16 ? tiles : std::max(tiles, split_key);
}

extern "C" int lr_packed_attention_plan(int64_t segments, int64_t groups, int64_t length,
                                        int64_t max_keys, int64_t dim, int dtype, int64_t* plan) {
  clear_error();
  LR_REQUIRE(dim == 64 || dim == 128 || dim == 256, "Head dimension must be 64, 128 or 256");
  LR_REQUIRE(segments > 0 && groups > 0 && length > 0 && max_keys >= 0 && plan,
             "Empty attention dimensions");
  if (takes_tiles(segments, groups, length, max_keys, dim, dtype)) {
    const AttnTilePlan tiles = plan_tiles(segments, groups, length, max_keys, dim);
    plan[0] = tiles.rows;
    plan[1] = tiles.splits;
  } else {
    const AttnPlan blocks = plan_attention(segments, groups, length, max_keys, dim);
    plan[0] = blocks.rows_per_tile;
    plan[1] = blocks.splits;
  }
  return LR_OK;
}

namespace lr {
namespace {

// The checks and launches shared by the entry points.
int packed_attention(const void* queries, int64_t q_batch_stride, int64_t q_head_stride,
                     int64_t q_query_stride, const void* keys, const void* values,
                     int64_t key_rows, const int32_t* cu_seqlens_k, int64_t batch,
                     int64_t kv_heads, int64_t groups, int64_t length, int64_t dim, int dtype,
                     int64_t max_keys, float scale, void* out, void* workspace,
                     size_t workspace_size, void* stream, const void* pending_keys = nullptr,
                     const void* pending_values = nullptr) {
  LR_REQUIRE(dtype == LR_DTYPE_BF16 || dtype == LR_DTYPE_F16,
             "FlashAttention only supports fp16 and bf16 data type");
  LR_REQUIRE((pending_keys == nullptr) == (pending_values == nullptr),
             "Pending keys and values go together");
  LR_REQUIRE(pending_keys == nullptr || length == 1, "Pending rows need one query per segment");
  LR_REQUIRE(dim == 64 || dim == 128 || dim == 256, "Head dimension must be 64, 128 or 256");
  LR_REQUIRE(batch > 0 && kv_heads > 0 && groups > 0 && length > 0, "Empty attention dimensions");
  LR_REQUIRE(length <= INT32_MAX / groups, "Attention grid too large");
  LR_REQUIRE(key_rows >= 0 && max_keys >= 0, "Invalid key lengths");
  LR_REQUIRE(queries && out && cu_seqlens_k && (key_rows == 0 || (keys && values)),
             "Invalid attention buffers");
  const uintptr_t alignment = reinterpret_cast<uintptr_t>(queries) |
                              reinterpret_cast<uintptr_t>(keys) |
                              reinterpret_cast<uintptr_t>(values) |
                              reinterpret_cast<uintptr_t>(out) |
                              reinterpret_cast<uintptr_t>(pending_keys) |
                              reinterpret_cast<uintptr_t>(pending_values) |
                              static_cast<uintptr_t>((q_batch_stride | q_head_stride |
                                                      q_query_stride) * 2);
  LR_REQUIRE(alignment % 16 == 0, "Attention operands must be 16-byte aligned");
  const int64_t segments = batch * kv_heads;
  if (pending_keys != nullptr) ++max_keys;  // every segment's pending row
  const AttnPlan plan = plan_attention(segments, groups, length, max_keys, dim);
  const bool use_tiles = takes_tiles(segments, groups, length, max_keys, dim, dtype);
  AttnTilePlan tile_plan{};
  if (use_tiles) tile_plan = plan_tiles(segments, groups, length, max_keys, dim);
  const size_t needed =
      use_tiles ? attention_tiles_bytes(tile_plan, dim) : workspace_bytes(plan, dim);
  LR_REQUIRE(workspace_size >= needed && (needed == 0 || workspace != nullptr),
             "Attention workspace too small");
  LR_REQUIRE(needed == 0 || reinterpret_cast<uintptr_t>(workspace) % 256 == 0,
             "Attention workspace must be 256-byte aligned");
  // The split-key grid's limit, whichever kernel runs: a tile has at least as many rows, and a split
  // tile plan has at most 32 MiB of states, so its grid is the smaller one.
  const int64_t blocks = plan.units * plan.splits;
  LR_REQUIRE(blocks < (int64_t{1} << 31), "Attention grid too large");

  AttnArgs args{};
  args.queries = queries;
  args.q_batch = q_batch_stride;
  args.q_head = q_head_stride;
  args.q_query = q_query_stride;
  args.keys = keys;
  args.values = values;
  args.key_rows = key_rows;
  args.cu = cu_seqlens_k;
  args.kv_heads = kv_heads;
  args.groups = groups;
  args.length = length;
  args.tiles = plan.tiles;
  args.splits = plan.splits;
  args.scale = scale;
  args.out = out;
  args.pending_keys = pending_keys;
  args.pending_values = pending_values;
  const hipStream_t s = as_stream(stream);
  if (use_tiles) {
    args.tiles = tile_plan.tiles;
    args.splits = tile_plan.splits;
    if (needed) {
      args.part_ml = static_cast<float*>(workspace);
      args.part_o = args.part_ml + segments * tile_plan.tiles * tile_plan.splits * tile_plan.rows * 2;
    }
    return launch_attention_tiles(args, tile_plan, dim, dtype, s);
  }
  if (needed) {
    args.part_ml = static_cast<float*>(workspace);
    args.part_o = args.part_ml + plan.units * plan.splits * plan.rows_per_tile * 2;
  }
  return dtype == LR_DTYPE_BF16
             ? launch_dim<__bf16>(args, dim, plan, blocks, s)
             : launch_dim<_Float16>(args, dim, plan, blocks, s);
}

// Workspace of the allocation-free entry point: one fixed array per device, held from the
// library's load onto that device until the process ends. Host code never passes `scratch`
// itself to a kernel (on the host the name is only a stand-in for the symbol); it passes the
// device address hipGetSymbolAddress gives, looked up once per device.
__device__ __align__(256) unsigned char scratch[kAttentionScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_address[kMaxDevices] = {};

// The device address of `scratch` on the device that owns `stream` (the current device for the
// null stream). The first call on a device makes that device current for the lookup and then
// restores the caller's device.
int scratch_address(hipStream_t stream, void** address) {
  int device = 0;
  if (stream != nullptr) {
    LR_HIP_TRY(hipStreamGetDevice(stream, &device));
  } else {
    LR_HIP_TRY(hipGetDevice(&device));
  }
  LR_REQUIRE(device >= 0 && device < kMaxDevices, "Device ordinal out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_address[device] == nullptr) {
    int current = 0;
    LR_HIP_TRY(hipGetDevice(&current));
    if (current != device) LR_HIP_TRY(hipSetDevice(device));
    void* found = nullptr;
    const hipError_t status = hipGetSymbolAddress(&found, HIP_SYMBOL(scratch));
    if (current != device) LR_HIP_TRY(hipSetDevice(current));
    if (status != hipSuccess || found == nullptr) {
      (void)hipGetLastError();
      set_error(std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(status));
      return LR_ERR_HIP;
    }
    g_scratch_address[device] = found;
  }
  *address = g_scratch_address[device];
  return LR_OK;
}

}  // namespace
}  // namespace lr

extern "C" int lr_packed_attention(const void* queries, int64_t q_batch_stride,
                                   int64_t q_head_stride, int64_t q_query_stride,
                                   const void* keys, const void* values, int64_t key_rows,
                                   const int32_t* cu_seqlens_k, int64_t batch, int64_t kv_heads,
                                   int64_t groups, int64_t length, int64_t dim, int dtype,
                                   int64_t max_keys, float scale, void* out, void* workspace,
                                   size_t workspace_size, void* stream) {
  clear_error();
  return packed_attention(queries, q_batch_stride, q_head_stride, q_query_stride, keys, values,
                          key_rows, cu_seqlens_k, batch, kv_heads, groups, length, dim, dtype,
                          max_keys, scale, out, workspace, workspace_size, stream);
}

extern "C" size_t lr_packed_attention_pending_workspace_bytes(int64_t segments, int64_t groups,
                                                              int64_t max_keys, int64_t dim) {
  return lr_packed_attention_workspace_bytes(segments, groups, 1, max_keys + 1, dim);
}

extern "C" int lr_packed_attention_pending(const void* queries, int64_t q_batch_stride,
                                           int64_t q_head_stride, int64_t q_query_stride,
                                           const void* keys, const void* values,
                                           int64_t key_rows, const int32_t* cu_seqlens_k,
                                           int64_t batch, int64_t kv_heads, int64_t groups,
                                           int64_t dim, int dtype, int64_t max_keys, float scale,
                                           const void* pending_keys, const void* pending_values,
                                           void* out, void* workspace, size_t workspace_size,
                                           void* stream) {
  clear_error();
  LR_REQUIRE(pending_keys != nullptr && pending_values != nullptr, "Invalid attention buffers");
  return packed_attention(queries, q_batch_stride, q_head_stride, q_query_stride, keys, values,
                          key_rows, cu_seqlens_k, batch, kv_heads, groups, 1, dim, dtype,
                          max_keys, scale, out, workspace, workspace_size, stream, pending_keys, pending_values);
}

extern "C" size_t lr_packed_attention_scratch_bytes(void) { return kAttentionScratchBytes; }

extern "C" int lr_packed_attention_noalloc(const void* queries, int64_t q_batch_stride,
                                           int64_t q_head_stride, int64_t q_query_stride,
                                           const void* keys, const void* values,
                                           int64_t key_rows, const int32_t* cu_seqlens_k,
                                           int64_t batch, int64_t kv_heads, int64_t groups,
                                           int64_t length, int64_t dim, int dtype,
                                           int64_t max_keys, float scale, void* out,
                                           void* stream) {
  clear_error();
  // The size check comes first and needs no HIP call; a call that needs no partial states
  // (every segment within one block of keys, whichever kernel runs) does not touch the scratch array.
  const int64_t segments =
      batch > 0 && kv_heads > 0 && batch <= (int64_t{1} << 31) / kv_heads ? batch * kv_heads : 0;
  // The limit is stated in the split-key plan's bytes whichever kernels run (plan_tiles keeps the
  // prefill kernel's partial states of an accepted call within the array).
  const bool sized = segments > 0 && groups > 0 && length > 0 && max_keys >= 0 && dim > 0;
  const size_t blocks =
      sized ? workspace_bytes(plan_attention(segments, groups, length, max_keys, dim), dim) : 0;
  LR_REQUIRE(blocks <= kAttentionScratchBytes,
             "Attention needs " + std::to_string(blocks) +
                 " bytes of scratch; the allocation-free entry point holds at most " +
                 std::to_string(kAttentionScratchBytes) + " bytes per device");
  const size_t needed = lr_packed_attention_workspace_bytes(segments, groups, length, max_keys, dim);
  void* workspace = nullptr;
  if (needed) {
    if (int status = scratch_address(as_stream(stream), &workspace)) return status;
  }
  return packed_attention(queries, q_batch_stride, q_head_stride, q_query_stride, keys, values,
                          key_rows, cu_seqlens_k, batch, kv_heads, groups, length, dim, dtype,
                          max_keys, scale, out, workspace, needed ? kAttentionScratchBytes : 0,
                          stream);
}
