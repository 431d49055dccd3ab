// Prefill attention: packed attention (attention.hip states the layout and the causal rule) for
// calls with many query rows, where both products are matrix work.
//
// A workgroup of four waves owns 128 query rows (row = i*G + g) of one segment, 32 per wave, or one
// of a single wave 32 rows (short calls, where 128-row tiles would leave CUs idle). It streams the
// segment's keys in stages of 32 rows of K and V, copied straight to LDS and double-buffered. In a
// stage a wave forms S^T = K Q^T on v_mfma_f32_32x32x16 (a lane holds one query's scores of 16
// keys), takes the exponentials against a running reference, and accumulates O^T += V^T P^T. The
// contraction's key order is free, so the probabilities stay where S^T left them: a lane's
// accumulators 8k .. 8k+7 are the B operand of 16 keys, and the A operand reads the same keys' V
// columns with the transposing LDS load (ds_read_b64_tr_b16: 4 keys of one column per lane).
//
// Precision. P is f32 and stays f32: it enters the 16-bit MFMA as a sum of 16-bit pieces whose
// products with V are exact in f32. bf16: three pieces by truncation, 3 x 8 bits = the whole
// 24-bit significand. f16: pieces by rounding. With P scaled by 2^11 two of them hold 11 + 11 bits
// and a sign, but nothing below 2^-25 (f16's subnormals), which is 2^-12 of P = 2^-24. So what they
// leave goes, 2^24 times larger, into two more pieces (the tails), whose products are summed in
// accumulators of their own, or, where those would cost occupancy, a stage at a time. The four are
// within 2^-60 of P (all of its bits down to 2^-36 of the reference): n keys are within 2^-44 n of
// the sum with f32 P, for any f16 V, against output steps of 2^-24 and more.
//
// The reference of a row's exponentials only moves when the row's maximum has outgrown it by
// 2^kSlack (the accumulators are rescaled then, seldom after the first stages); sums and products
// are f32 throughout, so a reference below the maximum loses nothing.
//
// What bounds it: the matrix cores, at 8 MFMAs of scores and 24 of products (bf16; f16 32) per 32
// keys and wave at d128, with about 170 vector instructions beside them. Measured (us, against the
// split-key kernel of attention.hip, whose 8-row tiles read every K and V row once each and
// multiply P*V on the VALU): 8192 queries of the 8B shape 868 against 10,878 (1.25 PFLOP/s of
// MFMA work), 1000 queries on 4,000 cached keys at d256, G6, 233 against 2,115. f16: 333 queries
// at d64 13.4 against 24.3, 8192 at d128 1,120 against 10,768 (two pieces without the tails, which
// lose the small P, 10.6 and 772; V as two bf16 pieces and six products 15.3 and 1,717; every
// tail a stage at a time 14.6 and 1,139). Three waves per SIMD (168 VGPRs, a few spills outside the
// loop) beat two without spills at d <= 128: 890 against 928; f16 at d128 holds two. d256 holds one
// wave per SIMD (its accumulators alone take 128 VGPRs), so its stream is laid out by hand: 233
// against 285. Stages of 64 keys, a third stage buffer, 32-row tiles for long prompts: no faster or
// slower.
//
// A masked key never contributes: scores past a query's limit become -inf. Their P is 0, and as
// 0 * V is NaN for a non-finite V, a wave that ends with a non-finite accumulator recomputes its
// rows key by key over the visible keys only.

#include <algorithm>
#include <cmath>

#include "attention_tile.hpp"
#include "lds_copy.hpp"

namespace lr {
namespace {

typedef float tile_f32x16 __attribute__((ext_vector_type(16)));
typedef short tile_s16x4 __attribute__((ext_vector_type(4)));
typedef short tile_s16x8 __attribute__((ext_vector_type(8)));
typedef unsigned tile_u32x2 __attribute__((ext_vector_type(2)));

constexpr int kTileWaves = 4;
constexpr int kWaveRows = 32;
constexpr float kSlack = 4.0f;  // exponents of two a row maximum may exceed its reference by

constexpr int kStageKeys = 32;
constexpr int kBuffers = 2;     // K and V stages in LDS

template <typename T> struct TileVec;
template <> struct TileVec<__bf16> {
  static constexpr int kPieces = 3, kTails = 0;
  static constexpr float kTailScale = 1.0f;
  static constexpr float kRaise = 0.0f;
  static __device__ __forceinline__ tile_f32x16 mfma(attn_u32x4 a, attn_u32x4 b, tile_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(attn_bf16x8, a),
                                                   __builtin_bit_cast(attn_bf16x8, b), c, 0, 0, 0);
  }
  // Two f32 values as sums of three bf16 pieces each, word `w` of the piece vectors: the top
  // halves of x, of x minus that, and of what is left (each difference is exact and the last one
  // has at most 8 significant bits).
  static __device__ __forceinline__ void split(float x, float y, attn_u32x4 (&piece)[3], int w) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const unsigned a = __builtin_bit_cast(unsigned, x), b = __builtin_bit_cast(unsigned, y);
      piece[i][w] = __builtin_amdgcn_perm(b, a, 0x07060302u);
      if (i == 2) break;
      x -= __builtin_bit_cast(float, a & 0xffff0000u);
      y -= __builtin_bit_cast(float, b & 0xffff0000u);
    }
  }
};
template <> struct TileVec<_Float16> {
  static constexpr int kPieces = 2, kTails = 2;
  static constexpr float kRaise = 11.0f;  // P <= 2^(kSlack + 11), half of f16's range
  static constexpr float kTailScale = 0x1p24f;
  static __device__ __forceinline__ tile_f32x16 mfma(attn_u32x4 a, attn_u32x4 b, tile_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(attn_f16x8, a),
                                                  __builtin_bit_cast(attn_f16x8, b), c, 0, 0, 0);
  }
  // Each piece rounds what the ones before have left (exact differences); the tails are pieces of
  // 2^24 times the rest, which is at most 2^-24 of x or 2^-25.
  static __device__ __forceinline__ void split(float x, float y, attn_u32x4 (&piece)[4], int w) {
    typedef _Float16 half2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i == kPieces) x *= kTailScale, y *= kTailScale;
      half2 part = {static_cast<_Float16>(x), static_cast<_Float16>(y)};
      // Hidden from the compiler, which would round each half once more for the differences, and not
      // take them in one instruction of mixed types each.
      float minus = -1.0f;
      asm("" : "+v"(part), "+s"(minus));
      piece[i][w] = __builtin_bit_cast(unsigned, part);
      if (i == 3) break;
      x = __builtin_fmaf(static_cast<float>(part[0]), minus, x);
      y = __builtin_fmaf(static_cast<float>(part[1]), minus, y);
    }
  }
};

// Key of accumulator element r in a 32-key tile (lane half h): the MFMA's row order.
__device__ __forceinline__ int tile_key(int r, int half) { return 8 * (r >> 2) + 4 * half + (r & 3); }

// Four rows' elements of one column: lanes 4k .. 4k+3 of each 16 address row k (8 bytes each),
// lane i receives column i of the 16. `p` is the lane's LDS byte address.
__device__ __forceinline__ tile_u32x2 read_transposed(uint32_t p) {
  return __builtin_bit_cast(tile_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) tile_s16x4*)(uintptr_t)p));
}

// The larger of a value's copies in lanes l and l + 32, in both lanes.
__device__ __forceinline__ float both_halves_max(float x) {
  const LanePair pair = lane_pair<32>(x);
  return fmaxf(pair.first, pair.second);
}

// The tile's place in its segment: bounds clamped into the key buffer as in attention.hip.
struct TileBounds {
  int64_t key0;
  int keys, shift, key_end;  // query i sees keys j <= i + shift; key_end: past the tile's last one
};
__device__ __forceinline__ TileBounds tile_bounds(const AttnArgs& a, int64_t seg, int last_query) {
  TileBounds t;
  int64_t key0 = a.cu[seg], n = static_cast<int64_t>(a.cu[seg + 1]) - key0;
  key0 = key0 < 0 ? 0 : (key0 > a.key_rows ? a.key_rows : key0);
  n = n < 0 ? 0 : (n > a.key_rows - key0 ? a.key_rows - key0 : n);
  t.key0 = key0;
  t.keys = static_cast<int>(n);
  t.shift = static_cast<int>(n - a.length);
  const int end = last_query + t.shift + 1;
  t.key_end = end < 0 ? 0 : (end > t.keys ? t.keys : end);
  return t;
}

// Key chunks a tile has visible keys in (its partial states), as both launches count them.
__device__ __forceinline__ int chunks_needed(int key_end, int chunk, int splits) {
  return key_end == 0 ? 0 : min((key_end - 1) / chunk + 1, splits);
}

template <typename T, int D, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(
    D == 256 || WAVES == 1 ? 1 : D == 128 && TileVec<T>::kTails > 0 ? 2 : 3))) void prefill_attention_kernel(
    AttnArgs a, unsigned segments, int chunk) {
  using Vec = TileVec<T>;
  constexpr int KEYS = kStageKeys;
  constexpr int KS = D / 16;  // MFMA k-steps over the head dimension
  constexpr int DT = D / 32;  // 32-column tiles of the output
  constexpr bool kLaidOut = D == 256 || WAVES == 1;
  // Accumulators of the tails' products, or (0) none kept: at d128 they would leave a four-wave
  // tile one wave a SIMD and at d256 spill, so each stage's go into the output at once there.
  constexpr int kKept = Vec::kTails == 0 || D == 256 || (D == 128 && !kLaidOut) ? 0 : DT;
  constexpr int kThreads = 64 * WAVES, kRows = kWaveRows * WAVES;
  __shared__ __align__(16) uint16_t k_lds[kBuffers][KEYS * D];
  __shared__ __align__(16) uint16_t v_lds[kBuffers][KEYS * D];

  const int lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
  const int wave = WAVES == 1 ? 0 : static_cast<int>(wave_index());
  // Consecutive blocks take consecutive segments, so with 8 segments (or a divisor or multiple of
  // it) each XCD's L2 serves its own segments' K and V; within a segment the tiles with the most
  // visible keys come first, so that the launch's tail is short.
  const unsigned splits = static_cast<unsigned>(a.splits), tiles = static_cast<unsigned>(a.tiles);
  const unsigned seg = blockIdx.x % segments, rest = blockIdx.x / segments;
  const unsigned split = rest % splits, tile = tiles - 1 - rest / splits;
  const int groups = static_cast<int>(a.groups);
  const int rows = static_cast<int>(a.length) * groups;
  const int row0 = static_cast<int>(tile) * kRows;
  const int last_row = min(row0 + kRows, rows) - 1;
  const TileBounds bounds = tile_bounds(a, seg, last_row / groups);
  const int wave_row0 = row0 + wave * kWaveRows;
  const int row = wave_row0 + col;
  const bool row_valid = row < rows;

  const int needed = chunks_needed(bounds.key_end, chunk, static_cast<int>(splits));
  if (needed == 0) {  // no visible key for any row of the tile: zeros
    if (split != 0) return;
    for (int item = threadIdx.x; item < kRows * (D / 8); item += kThreads) {
      const int r = item / (D / 8), c = item - r * (D / 8);
      if (row0 + r < rows)
        *reinterpret_cast<attn_u32x4*>(output_row<T, D>(a, seg, row0 + r) + 8 * c) =
            attn_u32x4{0u, 0u, 0u, 0u};
    }
    return;
  }
  if (static_cast<int>(split) >= needed) return;  // uniform across the workgroup
  const int begin = static_cast<int>(split) * chunk;
  const int end = bounds.key_end - begin > chunk ? begin + chunk : bounds.key_end;

  // Visible keys: this lane's row sees keys <= limit; the wave's rows see keys < wave_end, and
  // those <= wave_limit are seen by all of them (with a zero scale no key counts as such).
  const int query = row_valid ? row / groups : 0;
  const int limit = row_valid ? query + bounds.shift : -1;
  const int wave_last = min(wave_row0 + kWaveRows, rows) - 1;
  const int wave_end = wave_row0 < rows ? min(end, wave_last / groups + bounds.shift + 1) : 0;
  const int wave_limit =
      wave_row0 < rows && a.scale != 0.0f ? wave_row0 / groups + bounds.shift : -1;

  const T* q_row = nullptr;
  {
    const int64_t b = seg / static_cast<unsigned>(a.kv_heads), h = seg - b * a.kv_heads;
    q_row = static_cast<const T*>(a.queries) + b * a.q_batch +
            (h * groups + (row_valid ? row - query * groups : 0)) * a.q_head +
            static_cast<int64_t>(query) * a.q_query;
  }
  // B operand: k = half * D/2 + 8 * ks + [0, 8). The kernel works with a positive scale: a
  // negative one goes into the queries' sign bits, and a zero one is multiplied into the scores as
  // they are masked (then every stage's are), so that an infinite or NaN score becomes NaN.
  attn_u32x4 qop[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qop[ks] = load16(q_row + half * (D / 2) + 8 * ks);
    if (a.scale < 0.0f) qop[ks] ^= 0x80008000u;
  }

  const __bf16* keys = static_cast<const __bf16*>(a.keys) + bounds.key0 * D;
  const __bf16* values = static_cast<const __bf16*>(a.values) + bounds.key0 * D;
  const uint32_t k_base = lds_address(&k_lds[0][0]), v_base = lds_address(&v_lds[0][0]);
  // d256 keeps 8 chunk slots: with 16 the copies' offsets differ from row group to row group, and
  // the bank conflicts they would save are hidden here (1000 queries onto 4000 cached keys, 4 heads
  // x 6 groups: 234.5 us with 8, 237.7 with 16).
  using KeySwizzle = RowSwizzle<D, D == 128 ? 16 : 8>;
  const uint32_t k_offset = dma_row_offset<D, KeySwizzle, kThreads>();
  const uint32_t v_offset = dma_row_offset<D, ColumnSwizzle<D>, kThreads>();
  constexpr uint32_t kStageBytes = KEYS * D * 2;
  // Rows past the last visible key re-read it (masked). K runs one stage ahead of V; `at` is the
  // byte offset of the stage's buffer.
  auto fetch_k = [&](int key, uint32_t at) {
    dma_rows<D, KEYS, KeySwizzle, kThreads>(keys, key, bounds.key_end - 1,
                                            k_base + at, k_offset);
  };
  auto fetch_v = [&](int key, uint32_t at) {
    dma_rows<D, KEYS, ColumnSwizzle<D>, kThreads>(values, key, bounds.key_end - 1,
                                                  v_base + at, v_offset);
  };

  const float unit = a.scale == 0.0f ? 0.0f : 1.0f;
  const float scale = a.scale == 0.0f ? 1.0f : __builtin_fabsf(a.scale);
  const float to_log2 = scale * kAttnLog2e;  // scores -> exponents of two
  float reference = kNegInf, sum = 0.0f;       // in exponents of two; the same in both halves
  tile_f32x16 out[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) out[dt][r] = 0.0f;
  tile_f32x16 tail[kKept > 0 ? kKept : 1];
#pragma unroll
  for (int dt = 0; dt < kKept; ++dt) tail[dt] = out[dt];

  // The lane's transposed reads: row 4 * half + (lane % 16) / 4 of an 8-row group, columns
  // 16 * (lane / 16 % 2) + 4 * (lane % 4) .. + 3 of a 32-column tile (chunk dt * 4 + v_chunk).
  const int v_row = 4 * half + ((lane & 15) >> 2);
  const int v_chunk = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  uint32_t v_lane[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
    v_lane[dt] = v_base + v_row * (D * 2) + 16 * ColumnSwizzle<D>::slot(v_row, 4 * dt + v_chunk) +
                 8 * (lane & 1);

  // S^T of the stage whose K rows start `at` bytes into the buffers.
  auto scores = [&](uint32_t at) {
    const char* k_row = reinterpret_cast<const char*>(&k_lds[0][0]) + at + col * (D * 2);
    tile_f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      acc = Vec::mfma(*reinterpret_cast<const attn_u32x4*>(
                          k_row + 16 * KeySwizzle::slot(col, half * KS + ks)),
                      qop[ks], acc);
    return acc;
  };
  // Masks a stage's scores and moves the rows' references where a maximum has outgrown them;
  // `top` is the lane's largest score before the mask.
  auto refer = [&](tile_f32x16& s, float top, int key) {
    if (key > wave_limit - (KEYS - 1)) {
      top = kNegInf;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = key + tile_key(r, half) <= limit ? s[r] * unit : kNegInf;
        top = fmaxf(top, s[r]);
      }
    }
    top = both_halves_max(top) * to_log2;
    if (__any(top > reference + kSlack)) {
      const float raised = fmaxf(reference, top);
      const float factor = reference == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(reference - raised);
      sum *= factor;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          out[dt][r] *= factor;
          if constexpr (kKept > 0) tail[dt][r] *= factor;
        }
      reference = raised;
    }
  };

  fetch_k(begin, 0);
  fetch_v(begin, 0);
  if (end - begin > KEYS) fetch_k(begin + KEYS, kStageBytes);
  dma_wait();
  __syncthreads();
  tile_f32x16 s;
  if (begin < wave_end) {
    s = scores(0);
    float top = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) top = fmaxf(top, s[r]);
    refer(s, top, begin);
  }
  __syncthreads();  // every wave has read the first stage's K: its buffer takes the third's
  // Stage j: its probabilities from s, the next stage's scores, and O^T += V^T P^T. A wave's own
  // matrix and vector work only overlap as far as they alternate in its instruction stream, so
  // the stream is laid out by hand: each MFMA is followed by its share of the vector work that is
  // not waiting for it. The scores' MFMAs carry the first 16 keys' exponentials and pieces, the
  // first 16 keys' MFMAs those of the second 16, and the second 16 keys' MFMAs the next stage's
  // maximum; LDS reads go out a few MFMAs ahead of their use.
  uint32_t here = 0, ahead = kStageBytes;  // buffers of stages j and j + 1
  for (int key = begin;; key += KEYS) {
    const int after = end - key;  // keys from this stage on
    if (after > 2 * KEYS) fetch_k(key + 2 * KEYS, here);  // stage j's K was read in the last pass
    if (after > KEYS) fetch_v(key + KEYS, ahead);
    if (key < wave_end) {
      const float base = reference == kNegInf ? 0.0f : reference - Vec::kRaise;
      tile_f32x16 next;  // past the last stage: not used
#pragma unroll
      for (int r = 0; r < 16; ++r) next[r] = 0.0f;
      const char* k_row = reinterpret_cast<const char*>(&k_lds[0][0]) + ahead + col * (D * 2);
      attn_u32x4 k_op[KS], v_op[2][DT], piece[2][Vec::kPieces + Vec::kTails];
      float p[16], part = 0.0f;
      auto load_k = [&](int ks) {
        k_op[ks] = *reinterpret_cast<const attn_u32x4*>(
            k_row + 16 * KeySwizzle::slot(col, half * KS + ks));
      };
      auto load_v = [&](int k, int dt) {  // 16 keys: accumulators 8k .. 8k + 7
        const uint32_t at = v_lane[dt] + here + 16 * k * (D * 2);
        const tile_u32x2 lo = read_transposed(at), hi = read_transposed(at + 8 * (D * 2));
        v_op[k][dt] = attn_u32x4{lo[0], lo[1], hi[0], hi[1]};
      };
      // Vector work in sixteen shares: exponentials and sums of two keys, then their pieces.
      auto share = [&](int n) {
        const int e = n & ~1;
        if (n % 2 == 0) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            p[e + i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e + i], to_log2, -base));
            part += p[e + i];
          }
        } else {
          Vec::split(p[e], p[e + 1], piece[e / 8], (e / 2) % 4);
        }
      };
      constexpr int kProducts = Vec::kPieces * DT + Vec::kTails * kKept;
      float top = kNegInf;
      auto product = [&](int k, int i) {
        tile_f32x16& sums = i < Vec::kPieces * DT ? out[i % DT] : tail[kKept > 0 ? i % DT : 0];
        sums = Vec::mfma(v_op[k][i % DT], piece[k][i / DT], sums);
      };
      // The tails' products with all 32 keys where no accumulators are kept, by column tiles.
      auto add_tails = [&]() {
        if constexpr (Vec::kTails > 0 && kKept == 0) {
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            tile_f32x16 rest;
#pragma unroll
            for (int r = 0; r < 16; ++r) rest[r] = 0.0f;
#pragma unroll
            for (int i = 0; i < 2 * Vec::kTails; ++i)
              rest = Vec::mfma(v_op[i / Vec::kTails][dt],
                               piece[i / Vec::kTails][Vec::kPieces + i % Vec::kTails], rest);
#pragma unroll
            for (int r = 0; r < 16; ++r)
              out[dt][r] = __builtin_fmaf(rest[r], 1.0f / Vec::kTailScale, out[dt][r]);
          }
        }
      };
      if constexpr (kLaidOut) {
        constexpr int kLead = KS < 4 ? KS : 4;
#pragma unroll
        for (int ks = 0; ks < kLead; ++ks) load_k(ks);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          next = Vec::mfma(k_op[ks], qop[ks], next);
          if (ks + kLead < KS) load_k(ks + kLead);
#pragma unroll
          for (int dt = ks * DT / KS; dt < (ks + 1) * DT / KS; ++dt) load_v(0, dt);
#pragma unroll
          for (int n = ks * 8 / KS; n < (ks + 1) * 8 / KS; ++n) share(n);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < kProducts; ++i) {
          product(0, i);
          if (i < DT) load_v(1, i);
#pragma unroll
          for (int n = 8 + i * 8 / kProducts; n < 8 + (i + 1) * 8 / kProducts; ++n) share(n);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < kProducts; ++i) {
          product(1, i);
#pragma unroll
          for (int r = i * 8 / kProducts; r < (i + 1) * 8 / kProducts; ++r)
            top = fmaxf(fmaxf(top, next[2 * r]), next[2 * r + 1]);
          __builtin_amdgcn_sched_barrier(0);
        }
        add_tails();
      } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          load_k(ks);
          next = Vec::mfma(k_op[ks], qop[ks], next);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
#pragma unroll
          for (int n = 0; n < 8; ++n) share(8 * k + n);
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) load_v(k, dt);
#pragma unroll
          for (int i = 0; i < kProducts; ++i) product(k, i);
        }
        add_tails();
#pragma unroll
        for (int r = 0; r < 8; ++r) top = fmaxf(fmaxf(top, next[2 * r]), next[2 * r + 1]);
      }
      sum += part;
      s = next;
      if (after > KEYS) refer(s, top, key + KEYS);
    }
    if (after <= KEYS) break;
    dma_wait();
    __syncthreads();
    const uint32_t done = here;
    here = ahead, ahead = done;
  }
  sum += __shfl_xor(sum, 32);
#pragma unroll
  for (int dt = 0; dt < kKept; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      out[dt][r] = __builtin_fmaf(tail[dt][r], 1.0f / Vec::kTailScale, out[dt][r]);

  float poison = 0.0f;  // NaN if any accumulator is not finite
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) poison = __builtin_fmaf(out[dt][r], 0.0f, poison);
  if (__any(row_valid && poison != poison)) {
    // Non-finite inputs (or sums past f32): this wave's rows again over their visible keys only.
    const int stop = min(end, limit + 1);
    auto score = [&](int key) {
      const T* k_row = reinterpret_cast<const T*>(keys) + static_cast<int64_t>(key) * D;
      float dot = 0.0f;
#pragma unroll 1
      for (int d = 0; d < D; d += 8) {
        float x[8], y[8];
        unpack8<T>(load16(q_row + d), x);
        unpack8<T>(load16(k_row + d), y);
#pragma unroll
        for (int e = 0; e < 8; ++e) dot = __builtin_fmaf(x[e], y[e], dot);
      }
      return a.scale < 0.0f ? -dot : a.scale == 0.0f ? dot * 0.0f : dot;
    };
    float top = kNegInf;
#pragma unroll 1
    for (int key = begin; key < stop; ++key) top = fmaxf(top, score(key));
    reference = top * to_log2;
    const float base = reference == kNegInf ? 0.0f : reference - Vec::kRaise;
    sum = 0.0f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) out[dt][r] = 0.0f;
#pragma unroll 1
    for (int key = begin; key < stop; ++key) {
      const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(score(key), to_log2, -base));
      sum += p;
      const T* v = reinterpret_cast<const T*>(values) + static_cast<int64_t>(key) * D + 4 * half;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          out[dt][r] = __builtin_fmaf(p, static_cast<float>(v[32 * dt + 8 * (r >> 2) + (r & 3)]),
                                      out[dt][r]);
    }
  }

  // Lane (row, half) holds columns 32 * dt + 8 * c + 4 * half + [0, 4).
  if (needed == 1) {
    if (!row_valid) return;
    const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
    T* o = output_row<T, D>(a, seg, row) + 4 * half;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        typedef T T4 __attribute__((ext_vector_type(4)));
        T4 packed;
#pragma unroll
        for (int e = 0; e < 4; ++e) packed[e] = static_cast<T>(out[dt][4 * c + e] * inv);
        *reinterpret_cast<T4*>(o + 32 * dt + 8 * c) = packed;
      }
    return;
  }
  const int64_t slot = (static_cast<int64_t>(seg) * tiles + tile) * splits + split;
  const int64_t at = slot * kRows + wave * kWaveRows + col;
  float* o = a.part_o + at * D + 4 * half;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      *reinterpret_cast<attn_f32x4*>(o + 32 * dt + 8 * c) =
          attn_f32x4{out[dt][4 * c], out[dt][4 * c + 1], out[dt][4 * c + 2], out[dt][4 * c + 3]};
  if (half == 0) {
    // the reference the exponentials were taken against, so that the merge's weights are exact
    a.part_ml[at * 2] = reference == kNegInf ? kNegInf : reference - Vec::kRaise;
    a.part_ml[at * 2 + 1] = sum;
  }
}

// Second launch of a split call: a thread folds one (row, 8 columns) slice of a tile over the
// key chunks, in chunk order, a round of chunks' states loaded together: a memory round trip a
// round. (One a chunk: 16 queries on 4,000 keys, 8 segments, G4, d64 28.7 us against 15.) References
// are exponents of two.
constexpr int kMergeRound = 8;

template <typename T, int D, int ROWS>
__global__ __launch_bounds__(kAttnThreads) void prefill_merge_kernel(AttnArgs a, int chunk) {
  constexpr int LPR = D / 8, kBlocks = ROWS * LPR / kAttnThreads;
  const unsigned unit = blockIdx.x / kBlocks, tiles = static_cast<unsigned>(a.tiles);
  const unsigned seg = unit / tiles, tile = unit - seg * tiles;
  const int groups = static_cast<int>(a.groups);
  const int rows = static_cast<int>(a.length) * groups;
  const int row0 = static_cast<int>(tile) * ROWS;
  const int last_row = min(row0 + ROWS, rows) - 1;
  const TileBounds bounds = tile_bounds(a, seg, last_row / groups);
  const int needed = chunks_needed(bounds.key_end, chunk, static_cast<int>(a.splits));
  const int item = static_cast<int>(blockIdx.x % kBlocks) * kAttnThreads + threadIdx.x;
  const int r = item / LPR, c = item - r * LPR;
  if (needed <= 1 || row0 + r >= rows) return;
  float top = kNegInf, sum = 0.0f, o[8] = {};
  const int64_t first = static_cast<int64_t>(unit) * a.splits * ROWS + r;
  for (int k0 = 0; k0 < needed; k0 += kMergeRound) {
    float m[kMergeRound], l[kMergeRound];
    attn_f32x4 x[kMergeRound], y[kMergeRound];
#pragma unroll
    for (int i = 0; i < kMergeRound; ++i) {
      const int64_t at = first + static_cast<int64_t>(min(k0 + i, needed - 1)) * ROWS;
      m[i] = k0 + i < needed ? a.part_ml[at * 2] : kNegInf;
      l[i] = a.part_ml[at * 2 + 1];
      x[i] = *reinterpret_cast<const attn_f32x4*>(a.part_o + at * D + 8 * c);
      y[i] = *reinterpret_cast<const attn_f32x4*>(a.part_o + at * D + 8 * c + 4);
    }
#pragma unroll
    for (int i = 0; i < kMergeRound; ++i) {
      if (m[i] == kNegInf) continue;
      const float higher = fmaxf(top, m[i]);
      const float ws = top == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(top - higher);
      const float wo = __builtin_amdgcn_exp2f(m[i] - higher);
      sum = __builtin_fmaf(wo, l[i], sum * ws);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[e] = __builtin_fmaf(wo, x[i][e], o[e] * ws);
        o[4 + e] = __builtin_fmaf(wo, y[i][e], o[4 + e] * ws);
      }
      top = higher;
    }
  }
  const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] *= inv;
  *reinterpret_cast<attn_u32x4*>(output_row<T, D>(a, seg, row0 + r) + 8 * c) = pack8<T>(o);
}

template <typename T, int D, int WAVES>
int launch_waves(const AttnArgs& args, const AttnTilePlan& plan, hipStream_t stream) {
  const unsigned segments = static_cast<unsigned>(plan.segments);
  const int chunk = static_cast<int>(plan.chunk);
  const int64_t units = plan.segments * plan.tiles;
  hipLaunchKernelGGL((prefill_attention_kernel<T, D, WAVES>),
                     dim3(static_cast<unsigned>(units * plan.splits)), dim3(64 * WAVES), 0,
                     stream, args, segments, chunk);
  if (int status = check_launch("packed_attention")) return status;
  if (plan.splits == 1) return LR_OK;
  constexpr int kRows = kWaveRows * WAVES;
  hipLaunchKernelGGL((prefill_merge_kernel<T, D, kRows>),
                     dim3(static_cast<unsigned>(units * (kRows * (D / 8) / kAttnThreads))),
                     dim3(kAttnThreads), 0, stream, args, chunk);
  return check_launch("packed_attention merge");
}

template <typename T, int D>
int launch_tiles(const AttnArgs& args, const AttnTilePlan& plan, hipStream_t stream) {
  return plan.rows == kWaveRows ? launch_waves<T, D, 1>(args, plan, stream)
                                : launch_waves<T, D, kTileWaves>(args, plan, stream);
}

template <typename T>
int launch_tile_dim(const AttnArgs& args, const AttnTilePlan& plan, int64_t dim,
                    hipStream_t stream) {
  switch (dim) {
    case 64: return launch_tiles<T, 64>(args, plan, stream);
    case 128: return launch_tiles<T, 128>(args, plan, stream);
    default: return launch_tiles<T, 256>(args, plan, stream);
  }
}

}  // namespace

// Which tile and how many key chunks a call gets: the candidate with the least estimated time, in
// us. A stage of 32 keys takes a lone wave `alone` (a chain of MFMAs, exponentials and LDS reads
// that one wave cannot overlap); 128-row workgroups add up on a CU once it holds more than
// alone / tile of them, and single-wave workgroups, which share no K or V tile, on the chip's L2
// once there are more than 1024 * alone / wave. Splitting the keys costs the merge launch and its
// partial states. Fitted to 129 shapes (every head dimension, 2 to 2048 queries on 0 to 4096
// cached keys, 1 to 8 groups, each at up to 20 tile and chunk choices): the choice is 2.6% above
// the best one on average. One tile and no chunks, by contrast: 8192 new queries the same 850 us,
// 32 queries on 4000 keys 126 us instead of 22 (8B shape).
struct StageTimes {
  double alone, tile, wave;
};

AttnTilePlan plan_attention_tiles(int64_t segments, int64_t groups, int64_t length,
                                  int64_t max_keys, int64_t dim, int64_t scratch_bytes) {
  constexpr int64_t kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32};
  constexpr int64_t kMinStages = 4;  // of a chunk
  const StageTimes us = dim == 64    ? StageTimes{0.7, 0.25, 0.5}
                        : dim == 128 ? StageTimes{1.0, 0.75, 1.2}
                                     : StageTimes{1.6, 1.6, 3.5};
  const int64_t stages =
      std::max<int64_t>(1, ceil_div(std::min<int64_t>(max_keys, INT32_MAX), kStageKeys));
  AttnTilePlan best{};
  double least = 0.0;
  for (const int64_t rows : {int64_t{kWaveRows}, int64_t{kWaveRows * kTileWaves}}) {
    const int64_t tiles = ceil_div(length * groups, rows);
    for (const int64_t wanted : kSplits) {
      const int64_t per = ceil_div(stages, wanted), splits = ceil_div(stages, per);
      const int64_t blocks = segments * tiles * splits;
      const double bytes = static_cast<double>(blocks) * rows * (dim + 2) * 4;
      if (splits > 1 && (per < kMinStages || bytes > static_cast<double>(scratch_bytes))) continue;
      const double load = rows == kWaveRows ? us.wave * static_cast<double>(blocks) / 1024.0
                                            : us.tile * static_cast<double>(ceil_div(blocks, 256));
      const double time = static_cast<double>(per) * std::max(us.alone, load) +
                          (splits > 1 ? 2.0 + 0.4e-6 * bytes : 0.0);
      if (best.splits == 0 || time < least) {
        least = time;
        best = {segments, rows, tiles, splits, std::min<int64_t>(per * kStageKeys, INT32_MAX), time};
      }
    }
  }
  return best;
}

size_t attention_tiles_bytes(const AttnTilePlan& plan, int64_t dim) {
  if (plan.splits == 1) return 0;
  return static_cast<size_t>(plan.segments * plan.tiles * plan.splits * plan.rows) *
         static_cast<size_t>(dim + 2) * 4;
}

int launch_attention_tiles(const AttnArgs& args, const AttnTilePlan& plan, int64_t dim, int dtype,
                           hipStream_t stream) {
  return dtype == LR_DTYPE_BF16 ? launch_tile_dim<__bf16>(args, plan, dim, stream)
                                : launch_tile_dim<_Float16>(args, plan, dim, stream);
}

}  // namespace lr
