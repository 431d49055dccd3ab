// The margin helpers' products with a bf16 weight W [vocab, dim] for several f32 rows at once, on
// v_mfma_f32_32x32x16_bf16 (the definitions are in vjp.hip):
//   head_products_kernel    Y[r, v] = X[r] . W[v]
//   column_products_kernel  Z[r, d] = sum_v c[r, v] * W[v, d]
// The f32 operand (X or c) enters as three bf16 pieces by truncation, 3 x 8 bits = its whole 24-bit
// significand, so every product is exact in f32; piece p of row r is row 8p + r of the MFMA's A
// operand (24 of 32 rows used), W is the B operand, and a lane's result registers hold the three
// pieces of four rows, which it adds.
//
// Both are bound by reading W once. On the VALU, eight rows cost eight FMAs and an LDS operand
// each per weight element; here one MFMA covers 512 weight elements and all rows. Every wave
// copies its own W tiles straight to LDS, ahead of use, and waits only for its own copies. Measured
// (128,256 x 4096, eight rows, us): logits 207 (5.1 TB/s) against 1,299 for two VALU passes of four
// rows each; gradient products 215 against 511. Deeper copy queues (64-column stages, three in
// flight) changed nothing. The error against 64 bits is that of shorter chains of f32 sums: 1.1e-7
// of the logits against 1.6e-7.

#include <algorithm>

#include "lds_copy.hpp"
#include "vjp_products.hpp"

namespace lr {
namespace {

typedef __bf16 prod_bf16x8 __attribute__((ext_vector_type(8)));
typedef float prod_f32x16 __attribute__((ext_vector_type(16)));
typedef float prod_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned prod_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned prod_u32x2 __attribute__((ext_vector_type(2)));
typedef short prod_s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ prod_f32x16 product(prod_u32x4 a, prod_u32x4 b, prod_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(prod_bf16x8, a),
                                                 __builtin_bit_cast(prod_bf16x8, b), c, 0, 0, 0);
}

// Piece `p` of x as bf16 bits: x's top half, that of what is left, and the rest (both differences
// are exact). An infinity or NaN is piece 0 alone (0 in the others), quieted.
__device__ __forceinline__ unsigned piece_of(float x, int p) {
  const unsigned bits = __builtin_bit_cast(unsigned, x);
  if ((bits & 0x7f800000u) == 0x7f800000u)
    return p ? 0u : (bits >> 16) | ((bits & 0x7fffffu) ? 0x40u : 0u);
  const float rest = x - __builtin_bit_cast(float, bits & 0xffff0000u);
  const unsigned rest_bits = __builtin_bit_cast(unsigned, rest);
  const float last = rest - __builtin_bit_cast(float, rest_bits & 0xffff0000u);
  return (p == 0 ? bits : p == 1 ? rest_bits : __builtin_bit_cast(unsigned, last)) >> 16;
}

// Rows 4 * half + j, j = 0..3, of a product tile: the three pieces' sums added. A non-finite sum
// of the first piece is the result: against an infinite weight the other pieces may be 0 * inf.
__device__ __forceinline__ prod_f32x4 row_sums(const prod_f32x16& acc) {
  prod_f32x4 y;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    y[j] = __builtin_isfinite(acc[j]) ? acc[j] + (acc[4 + j] + acc[8 + j]) : acc[j];
  return y;
}

constexpr int kHeadWaves = 8;
constexpr int kHeadThreads = 64 * kHeadWaves;
constexpr int kHeadTile = 32;     // weight rows of a tile
constexpr int kStageColumns = 128;  // hidden elements of a stage (256 B of each weight row)
constexpr int kHeadStageBytes = kHeadTile * kStageColumns * 2;
constexpr int kMaxHeadStages = 5;  // hidden size / 1024: the pieces of X take 32 VGPRs each

// Persistent workgroups of eight waves. Wave w owns hidden elements [w, w + 1) * dim / 8 and
// keeps X's pieces for them in registers for the whole launch; it streams those columns of the
// workgroup's weight tiles (32 rows each) through two private LDS buffers, the next stage's copy
// in flight while the current one is multiplied. The waves' partial dots meet in LDS once a tile.
template <int STAGES>
__global__ __launch_bounds__(kHeadThreads, 2) void head_products_kernel(
    const float* __restrict__ hidden, int rows, int dim, const __bf16* __restrict__ weight,
    const __bf16* __restrict__ bias, int vocab, float* __restrict__ out, int64_t out_stride) {
  __shared__ __align__(16) char tiles[kHeadWaves][2][kHeadStageBytes];
  __shared__ __align__(16) float partial[2][kHeadWaves][kProductRows][kHeadTile];
  const int wave = static_cast<int>(wave_index()), lane = threadIdx.x & 63;
  const int half = lane >> 5, col = lane & 31;
  const int first = wave * (STAGES * kStageColumns);  // this wave's first hidden element

  // A operand: row m = lane & 31 = 8 * piece + r; in k-step ks of stage s, hidden elements
  // first + 128 * s + 64 * half + 8 * ks + [0, 8).
  prod_u32x4 x[STAGES][8];
  {
    const int r = col & 7, piece = col >> 3;
    const bool live = piece < 3 && r < rows;
    const float* row = hidden + static_cast<int64_t>(live ? r : 0) * dim + first + 64 * half;
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        const prod_f32x4 lo = *reinterpret_cast<const prod_f32x4*>(row + 128 * s + 8 * ks);
        const prod_f32x4 hi = *reinterpret_cast<const prod_f32x4*>(row + 128 * s + 8 * ks + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = e < 2 ? lo[2 * e] : hi[2 * e - 4], b = e < 2 ? lo[2 * e + 1] : hi[2 * e - 3];
          x[s][ks][e] = live ? piece_of(a, piece) | (piece_of(b, piece) << 16) : 0u;
        }
      }
  }

  const int tile_count = (vocab + kHeadTile - 1) / kHeadTile;
  const uint32_t lds = lds_address(&tiles[wave][0][0]);
  const uint32_t row_offset = dma_row_offset<kStageColumns, RowSwizzle<kStageColumns>, 64>(lane, dim);
  constexpr int kCopies = kHeadStageBytes / (64 * 16);
  // the last tile reaches back over rows of the one before (vocab >= 32): they come out the same
  auto first_row = [&](int tile) { return min(tile * kHeadTile, vocab - kHeadTile); };
  auto fetch = [&](int tile, int s, int buf) {
    dma_rows<kStageColumns, kHeadTile, RowSwizzle<kStageColumns>, 64, false>(
        weight + first + s * kStageColumns, first_row(tile), 0,
        lds + buf * kHeadStageBytes, row_offset, dim);
  };
  int buf = 0, parity = 0;
  int tile = static_cast<int>(blockIdx.x);
  dma_wait();  // the loads above: from here on the copies are the only loads
  if (tile < tile_count) fetch(tile, 0, 0);
  for (; tile < tile_count; tile += static_cast<int>(gridDim.x)) {
    const int next_tile = tile + static_cast<int>(gridDim.x);
    prod_f32x16 acc[2];  // two chains: a product does not wait for the one before it
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
#pragma unroll
    for (int s = 0; s < STAGES; ++s) {
      // the other buffer was read a stage ago, and those reads have returned
      const bool more = s + 1 < STAGES || next_tile < tile_count;
      if (more) fetch(s + 1 < STAGES ? tile : next_tile, s + 1 < STAGES ? s + 1 : 0, buf ^ 1);
      if (more) dma_wait_but<kCopies>();
      else dma_wait();
      const char* w_row = &tiles[wave][0][0] + buf * kHeadStageBytes + col * (kStageColumns * 2);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks)
        acc[ks & 1] = product(x[s][ks],
                              *reinterpret_cast<const prod_u32x4*>(
                                  w_row + 16 * swizzled_chunk<kStageColumns>(col, 8 * half + ks)),
                              acc[ks & 1]);
      buf ^= 1;
      // every read of this stage's buffer is done before a copy into it can be issued
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      asm volatile("" ::: "memory");
    }
    const prod_f32x4 y = row_sums(acc[0]) + row_sums(acc[1]);
#pragma unroll
    for (int j = 0; j < 4; ++j) partial[parity][wave][4 * half + j][col] = y[j];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    // The sums of the eight waves, in wave order. The next tile's partials go to the other half,
    // whose last readers passed this barrier.
    const int r = static_cast<int>(threadIdx.x) >> 5, v = first_row(tile) + col;
    if (r < rows) {
      float sum = partial[parity][0][r][col];
#pragma unroll
      for (int w = 1; w < kHeadWaves; ++w) sum += partial[parity][w][r][col];
      if (bias) sum += static_cast<float>(bias[v]);
      out[r * out_stride + v] = sum;
    }
    parity ^= 1;
  }
}

constexpr int kColumnWaves = 4;
constexpr int kColumnThreads = 64 * kColumnWaves;
constexpr int kColumnTile = 128;    // columns of a wave (256 B of each weight row)
constexpr int kColumnStage = 16;    // weight rows of a stage: one k-step
constexpr int kColumnStageBytes = kColumnStage * kColumnTile * 2;
constexpr int kColumnBuffers = 3;  // with the pieces 80 KB: two workgroups a CU
constexpr int kMaxBlockRows = 512;  // weight rows of a workgroup: their pieces take 32 KB of LDS

// grid: (ceil(dim / 512), row blocks). The workgroup forms the pieces of its block's coefficients
// in LDS once; then each wave streams its 128 columns of the block's weight rows through private
// LDS buffers (two stages in flight) and reads them transposed (a lane: 4 rows of one column).
__global__ __launch_bounds__(kColumnThreads) void column_products_kernel(
    const __bf16* __restrict__ weight, int64_t vocab, int dim, int block_rows, int rows,
    const float* __restrict__ logits, const float* __restrict__ stats,
    const int64_t* __restrict__ targets, float* __restrict__ partial) {
  __shared__ __align__(16) uint16_t pieces[kMaxBlockRows * 32];
  __shared__ __align__(16) char tiles[kColumnWaves][kColumnBuffers][kColumnStageBytes];
  const int wave = static_cast<int>(wave_index()), lane = threadIdx.x & 63;
  const int half = lane >> 5, col = lane & 31;
  const int64_t v0 = static_cast<int64_t>(blockIdx.y) * block_rows;
  const int count = static_cast<int>(min(vocab - v0, static_cast<int64_t>(block_rows)));
  const int stages = (count + kColumnStage - 1) / kColumnStage;
  const int column0 = (static_cast<int>(blockIdx.x) * kColumnWaves + wave) * kColumnTile;
  const bool live = column0 < dim;  // dim is a multiple of a wave's columns

  const uint32_t buffers = lds_address(&tiles[wave][0][0]);
  using Swizzle = ColumnSwizzle<kColumnTile>;
  const uint32_t row_offset = dma_row_offset<kColumnTile, Swizzle, 64>(lane, dim);
  constexpr int kCopies = kColumnStageBytes / (64 * 16);
  const __bf16* source = weight + v0 * dim + column0;
  auto fetch = [&](int stage, uint32_t offset) {  // rows past the block re-read its last one
    dma_rows<kColumnTile, kColumnStage, Swizzle, 64>(source, stage * kColumnStage, count - 1,
                                                     buffers + offset, row_offset, dim);
  };

  // Coefficient k of row r: piece p goes to A row m = 8p + r of 16-row group k / 16, in the
  // k-order of the transposed reads (rows 4 * half + 0..3, then 8 + 4 * half + 0..3). Rows past
  // the block and A rows past the last row are zero.
  for (int i = threadIdx.x; i < stages * kColumnStage * kProductRows; i += kColumnThreads) {
    const int k = i % (stages * kColumnStage), r = i / (stages * kColumnStage);
    float c = 0.0f;
    if (k < count && r < rows) {
      const int64_t v = v0 + k;
      if (v != targets[r]) c = expf(logits[r * vocab + v] - stats[2 * r]) / stats[2 * r + 1];
    }
    const int w = k & 15, at = (((k >> 4) * 2 + ((w >> 2) & 1)) * 32 + r) * 8 + (w & 3) + 4 * (w >> 3);
#pragma unroll
    for (int p = 0; p < 4; ++p)
      pieces[at + p * 64] = p < 3 ? static_cast<uint16_t>(piece_of(c, p)) : uint16_t{0};
  }
  __syncthreads();
  dma_wait();  // from here on the copies are the only loads
  if (!live) return;  // no barrier follows

  // Transposed reads: row 4 * half + lane % 16 / 4 of eight, columns 16 * (lane / 16 % 2) +
  // 4 * (lane % 4) .. + 3 of a 32-column tile.
  constexpr int kTiles = kColumnTile / 32;
  const int w_row = 4 * half + ((lane & 15) >> 2);
  const int w_chunk = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  uint32_t w_lane[kTiles];
#pragma unroll
  for (int t = 0; t < kTiles; ++t)
    w_lane[t] = buffers + w_row * (kColumnTile * 2) + 16 * Swizzle::slot(w_row, 4 * t + w_chunk) +
                8 * (lane & 1);
  auto transposed = [&](uint32_t at) {
    return __builtin_bit_cast(prod_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) prod_s16x4*)(uintptr_t)at));
  };
  prod_f32x16 acc[kTiles];
#pragma unroll
  for (int t = 0; t < kTiles; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[t][e] = 0.0f;
  uint32_t offset = 0, free = 2 * kColumnStageBytes;  // buffers of stage s and of stage s + 2
  fetch(0, 0);
  if (stages > 1) fetch(1, kColumnStageBytes);
  for (int s = 0; s < stages; ++s) {
    if (s + 2 < stages) {
      fetch(s + 2, free);  // its buffer was read a stage ago
      dma_wait_but<2 * kCopies>();
    } else {
      dma_wait();
    }
    const prod_u32x4 c = *reinterpret_cast<const prod_u32x4*>(pieces + ((s * 2 + half) * 32 + col) * 8);
    prod_u32x4 w[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      const prod_u32x2 lo = transposed(w_lane[t] + offset);
      const prod_u32x2 hi = transposed(w_lane[t] + offset + 8 * (kColumnTile * 2));
      w[t] = prod_u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
    // The copies of the last row stand for no row: their coefficients are zero, and as 0 * W is NaN
    // for an infinite W they are cleared.
    if (const int left = count - s * kColumnStage; left < kColumnStage) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = 4 * half + 8 * (i >> 1) + 2 * (i & 1);
        const unsigned live_rows = k + 1 < left ? ~0u : k < left ? 0xffffu : 0u;
#pragma unroll
        for (int t = 0; t < kTiles; ++t) w[t][i] &= live_rows;
      }
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t) acc[t] = product(c, w[t], acc[t]);
    free = offset;
    offset = offset == 2 * kColumnStageBytes ? 0 : offset + kColumnStageBytes;
    // every read of this stage's buffer is done before a copy into it can be issued
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
  }
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    const prod_f32x4 z = row_sums(acc[t]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (4 * half + j < rows)
        partial[(static_cast<int64_t>(blockIdx.y) * rows + 4 * half + j) * dim + column0 + 32 * t + col] = z[j];
  }
}

template <int STAGES>
void start_head(const float* hidden, int64_t rows, const void* weight, const void* bias,
                int64_t vocab, int64_t dim, float* out, hipStream_t stream) {
  const int64_t tiles = ceil_div(vocab, kHeadTile);
  // one workgroup a CU: its 128 KB of buffers leave no room for a second
  const unsigned blocks = static_cast<unsigned>(std::min<int64_t>(tiles, 256));
  hipLaunchKernelGGL((head_products_kernel<STAGES>), dim3(blocks), dim3(kHeadThreads), 0, stream,
                     hidden, static_cast<int>(rows), static_cast<int>(dim),
                     static_cast<const __bf16*>(weight), static_cast<const __bf16*>(bias),
                     static_cast<int>(vocab), out, vocab);
}

}  // namespace

// One row stays on the VALU, which already streams W at the card's rate (128,256 x 4096: 188 us
// against 197 here; 8,001 x 2048: 12.5 against 15.4). Few rows need many weight rows to be worth
// eight waves' start (us, VALU and here): two rows of 1,000 x 4096 11.4 and 22.3, of 8,001 x 3072
// 18.2 and 22.0, of 32,000 x 1024 18.4 and 15.6, of 128,256 x 4096 261 and 205; three rows of 1,000 x
// 5120 20.0 and 27.5, of 8,001 x 2048 18.0 and 13.6. Weight rows a multiple of 8 KB apart put the
// 256 bytes a stage takes of each on the same memory channels, so two such rows change sides later
// (32,000 x 4096 57 and 68). Hidden sizes: eight waves with whole 128-column stages, X's pieces in
// registers.
bool takes_head_products(int dtype, int64_t rows, int64_t vocab, int64_t dim) {
  const int64_t least = rows <= 1   ? INT64_MAX
                        : rows == 2 ? (dim % 4096 == 0 ? 65536 : 16384)
                        : rows <= 4 ? 2048
                                    : kHeadTile;
  return dtype == LR_DTYPE_BF16 && dim % 1024 == 0 && dim / 1024 <= kMaxHeadStages &&
         vocab >= least && vocab < (int64_t{1} << 30);
}

int launch_head_products(const float* hidden, int64_t rows, const void* weight, const void* bias,
                         int64_t vocab, int64_t dim, float* out, hipStream_t stream) {
  switch (dim / 1024) {
    case 1: start_head<1>(hidden, rows, weight, bias, vocab, dim, out, stream); break;
    case 2: start_head<2>(hidden, rows, weight, bias, vocab, dim, out, stream); break;
    case 3: start_head<3>(hidden, rows, weight, bias, vocab, dim, out, stream); break;
    case 4: start_head<4>(hidden, rows, weight, bias, vocab, dim, out, stream); break;
    default: start_head<5>(hidden, rows, weight, bias, vocab, dim, out, stream); break;
  }
  return check_launch("head_logits");
}

// Up to two rows stay on the VALU (128,256 x 4096, two rows, with the statistics: 218 us against
// 238), and three or four against many weights (us, VALU and here: three rows of 32,000 x 2048 29.6 and
// 37.2, of 128,256 x 4096 189 and 205, but of 8,001 x 2048 24.5 and 13.6; more rows of few weights
// gain more than of many lose: five of 32,000 x 3072 60 and 42, of 128,256 x 4096 202 and 216).
bool takes_column_products(int dtype, int64_t rows, int64_t vocab, int64_t dim) {
  return dtype == LR_DTYPE_BF16 && dim % kColumnTile == 0 &&
         (rows > 4 || (rows > 2 && vocab * dim < 60'000'000));
}

int64_t column_product_block_rows(int64_t vocab, int64_t dim) {
  const int64_t column_blocks = ceil_div(dim, kColumnTile * kColumnWaves);
  const int64_t per = ceil_div(vocab, std::max<int64_t>(1, 2048 / column_blocks));
  return std::min<int64_t>(kMaxBlockRows, std::max<int64_t>(64, ceil_div(per, kColumnStage) * kColumnStage));
}

int launch_column_products(const void* weight, int64_t vocab, int64_t dim, int64_t rows,
                           const float* logits, const float* stats, const int64_t* targets,
                           float* partial, hipStream_t stream) {
  const int64_t block_rows = column_product_block_rows(vocab, dim);
  const dim3 grid(static_cast<unsigned>(ceil_div(dim, kColumnTile * kColumnWaves)),
                  static_cast<unsigned>(ceil_div(vocab, block_rows)));
  hipLaunchKernelGGL(column_products_kernel, grid, dim3(kColumnThreads), 0, stream,
                     static_cast<const __bf16*>(weight), vocab, static_cast<int>(dim),
                     static_cast<int>(block_rows), static_cast<int>(rows), logits, stats, targets,
                     partial);
  return check_launch("row_sum");
}

}  // namespace lr
