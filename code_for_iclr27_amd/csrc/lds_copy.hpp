// Direct global -> LDS copies and swizzled LDS tiles of 16-bit rows, shared by the kernels that
// stage K, V, Q or weight tiles (scorer.hip, attention_tile.hip, vjp_products.hip), by whole
// workgroups or by single waves.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace lr {
namespace {

// Direct global -> LDS copies (global_load_lds_dword / _dwordx4): lane L of a wave writes its
// granule at LDS `wave_base` + L * granule; `wave_base` must be the same for the whole wave.
// Nothing passes through VGPRs. Completion is awaited with dma_wait() before the barrier that
// publishes the data.
// The copies are issued by inline assembly, not by the compiler's builtin: for the builtin the
// compiler makes every later LDS read that it cannot prove disjoint from the copy wait for it
// (s_waitcnt vmcnt(0)), and a buffer picked at run time is never provably disjoint, so the
// copy of the next stage would be waited for at the first read of the current one. Copies the
// compiler does not see only lengthen its own vmcnt waits (counts drain in order), never
// shorten them. M0 (the wave's LDS base for the copy) is set inside the same statement; no
// compiler-generated code in these kernels keeps a value in M0.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // M0 is a reserved register; clobbered on purpose
// Copy from a per-lane address to the (wave-uniform) LDS byte address `lds`.
__device__ __forceinline__ void dma16_to(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :: "v"(src), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void dma4_to(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
               :: "v"(src), "s"(lds) : "memory", "m0");
}
// The same copies addressed as a wave-uniform base (an SGPR pair) plus a per-lane 32-bit byte
// offset: the per-copy address arithmetic is then scalar, and a lane's offset can be computed
// once.
__device__ __forceinline__ void dma16_at(const void* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(offset), "s"(base), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void dma4_at(const void* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
               :: "v"(offset), "s"(base), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

// LDS byte address of a __shared__ object.
template <typename T>
__device__ __forceinline__ uint32_t lds_address(T* object) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) T*)object));
}

__device__ __forceinline__ uint32_t wave_index() {
  return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

// A wave-uniform address in scalar registers, also where the compiler formed it in vector ones.
__device__ __forceinline__ const char* uniform_address(const void* p) {
  const uint64_t bits = reinterpret_cast<uint64_t>(p);
  const uint32_t low = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bits));
  const uint32_t high = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bits >> 32));
  return reinterpret_cast<const char*>(static_cast<uint64_t>(high) << 32 | low);
}

// vmcnt(0) through the builtin, so that the compiler knows every vector-memory load has landed
// here (loads issued before a loop, such as the resident MFMA operands, are then not waited for
// again inside it); the empty statement keeps LDS accesses from moving across the wait.
__device__ __forceinline__ void dma_wait() {
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0) expcnt(7) lgkmcnt(15)
  asm volatile("" ::: "memory");
}

// The same, leaving the `N` newest of the wave's vector-memory operations in flight.
template <int N>
__device__ __forceinline__ void dma_wait_but() {
  static_assert(N >= 0 && N <= 63, "vmcnt holds six bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));  // vmcnt(N)
  asm volatile("" ::: "memory");
}

// Swizzled LDS rows: D 16-bit elements per row, no padding; 16-byte chunk c of row r is stored in
// chunk slot c ^ (r % P), so the lanes that read chunk c of consecutive rows (an MFMA operand)
// touch P different 16-byte bank groups per P rows. P = 16 where a row has the chunks for it
// (d64 has 8): then 16 rows' chunks touch all 64 banks once. With P = 8 at d256 four of every
// twelve LDS cycles of the audit were conflicts, with 16 there are none (row pass over 9216 keys,
// 16 layers x 4 heads x 6 groups, window 512: 945 -> 914 us).
template <int D>
constexpr int swizzle_period() { return D == 64 ? 8 : 16; }

template <int D, int P = swizzle_period<D>()>
__device__ __forceinline__ int swizzled_chunk(int row, int chunk) {
  return chunk ^ (row & (P - 1));
}

// The swizzles a copy can apply: rows read as MFMA operand rows (above), or read transposed
// (ds_read_b64_tr_b16: 16 lanes take 4 consecutive rows x 16 columns, 4 x 32 bytes). For the
// latter, 64-byte blocks of four consecutive rows go to the four 64-byte quarters of the 64
// banks, so that 32 lanes' reads (4 rows x 64 bytes) touch every bank once.
template <int D, int P = swizzle_period<D>()>
struct RowSwizzle {
  static __device__ __forceinline__ int slot(int row, int chunk) { return swizzled_chunk<D, P>(row, chunk); }
};
template <int D>
struct ColumnSwizzle {
  // which 64-byte block of a row (4 chunks) is exchanged: d64 rows are half a bank cycle long
  static __device__ __forceinline__ int block(int row) { return D == 64 ? (row >> 1) & 1 : row & 3; }
  static __device__ __forceinline__ int slot(int row, int chunk) { return chunk ^ (block(row) << 2); }
};

// DMA of `ROWS` consecutive rows (row0..) of a 16-bit matrix, D elements of each (`stride` elements
// from row to row: D, or a multiple of 128), into swizzled LDS rows at LDS byte address `lds`; rows
// at or past `last_row` re-read row `last_row` (callers mask them; no CLAMP: there are none). All
// THREADS threads of the workgroup call it, or, with 64, one wave (with its lane as `thread`).
// Copy i moves rows [i * RPI, (i + 1) * RPI), RPI = THREADS / (D / 8): while every row lies before
// `last_row` the addresses are a scalar base plus the thread's byte offset within copy 0
// (`dma_row_offset`), its chunk exchanged with what the swizzle does to row i * RPI (nothing where
// RPI is a multiple of the swizzle's period; the swizzle is an exclusive or of row bits, so the
// two parts of the row combine).
template <int D, typename Swizzle = RowSwizzle<D>, int THREADS = 256>
__device__ __forceinline__ uint32_t dma_row_offset(int thread = threadIdx.x, int stride = D) {
  constexpr int CH = D / 8;
  const int row = thread / CH, chunk = thread % CH;
  return static_cast<uint32_t>((row * stride + 8 * Swizzle::slot(row, chunk)) * 2);
}

template <int D, int ROWS, typename Swizzle = RowSwizzle<D>, int THREADS = 256, bool CLAMP = true>
__device__ __forceinline__ void dma_rows(const __bf16* matrix, int row0, int last_row,
                                         uint32_t lds, uint32_t row_offset, int stride = D) {
  constexpr int CH = D / 8, CHUNKS = ROWS * CH, RPI = THREADS / CH;
  static_assert(CHUNKS % THREADS == 0 && THREADS % CH == 0, "whole copies of whole rows");
  const uint32_t wave_lds = lds + (THREADS == 64 ? 0 : wave_index() * 64 * 16);
  if (!CLAMP || row0 + ROWS - 1 <= last_row) {
    const char* base = uniform_address(matrix + static_cast<int64_t>(row0) * stride);
#pragma unroll
    for (int i = 0; i < CHUNKS / THREADS; ++i)
      dma16_at(base + static_cast<int64_t>(i) * RPI * stride * 2,
               row_offset ^ (16 * static_cast<uint32_t>(Swizzle::slot(i * RPI, 0))),
               wave_lds + THREADS * 16 * i);
  } else {
#pragma unroll
    for (int i = 0; i < CHUNKS / THREADS; ++i) {
      const int slot = THREADS * i + (THREADS == 64 ? threadIdx.x & 63 : threadIdx.x);
      const int row = slot / CH, chunk = slot % CH;
      const int source = min(row0 + row, last_row);
      dma16_to(matrix + static_cast<int64_t>(source) * stride + 8 * Swizzle::slot(row, chunk),
               wave_lds + THREADS * 16 * i);
    }
  }
}

}  // namespace
}  // namespace lr
