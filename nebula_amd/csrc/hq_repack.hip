// hq_repack.hip — device repack of linear int4 / ternary weights into the gfx950 tile
// layout (hq_layout.hpp). Int4: one thread per packed output word; the host variants in
// hq_api.cpp (hq_repack_int4, hq_repack_ternary2, hq_convert_tq1_0) produce the same words.
#include <hip/hip_runtime.h>

#include "hq_internal.hpp"
#include "hq_layout.hpp"
#include "hq_plan.hpp"

namespace hq {
namespace {

__global__ void __launch_bounds__(256) repack_int4_kernel(const uint32_t* __restrict__ src,
                                                          uint32_t* __restrict__ dst, uint32_t N,
                                                          uint32_t nkb, size_t total) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const uint32_t w = (uint32_t)(idx & 3u);
  const uint32_t lane = (uint32_t)((idx >> 2) & 63u);
  const size_t blk = idx >> 8;
  const uint32_t kb = (uint32_t)(blk % nkb);
  const uint32_t ct = (uint32_t)(blk / nkb);
  const uint32_t n = ct * 16u + (lane & 15u);
  const uint32_t lin = n < N ? src[(size_t)int4_linear_kw(kb, lane, w) * N + n] : 0x88888888u;
  dst[idx] = int4_linear_to_tile(lin);
}

// Ternary words. Both repacks form a word's 16 fields in descending order (element i at bits
// 31 - 2i, 30 - 2i: two runs of 8 elements, k-slices 2p and 2p + 1 of a chunk) and shuffle whole
// words: tern_split gathers each run's even and odd elements into bytes (evens of run 0, odds of
// run 0, evens of run 1, odds of run 1, from the top), and one byte permutation of a chunk pair's
// words gives a packed word. Placing the fields one by one took 64 shifts and masks per packed word
// and left the kernels bound by the VALU, and 4-byte stores half filled each row: MI355X, ternary
// 17408 x 5120 25.7 -> 8.7 us, 5120 x 10240 16.5 -> 7.1, TQ1_0 17408 x 5120 14.1 -> 9.1 (4.7 TB/s read and
// written, a large copy's rate).
__device__ __forceinline__ uint32_t tern_split(uint32_t x) {
  uint32_t t = (x ^ (x >> 2)) & 0x0C0C0C0Cu;  // e0 e1 e2 e3 -> e0 e2 e1 e3
  x ^= t ^ (t << 2);
  t = (x ^ (x >> 4)) & 0x00F000F0u;  // e0e2 e1e3 e4e6 e5e7 -> e0e2 e4e6 e1e3 e5e7
  return x ^ t ^ (t << 4);
}
// A column's 128 elements of one k-block (split words f[0..7], 16 elements each) -> its eight packed
// words, both words of k-slice g4 in one 8-byte store (16 columns: 128 bytes); o: lane 0's words.
__device__ __forceinline__ void tern_store_block(const uint32_t* f, uint32_t* o, uint32_t c16) {
  typedef uint32_t w2 __attribute__((ext_vector_type(2), aligned(4)));  // packed is 4-byte aligned
#pragma unroll
  for (uint32_t g4 = 0; g4 < 4; ++g4) {
    const uint32_t p = g4 >> 1, sel = g4 & 1u ? 0x04000501u : 0x06020703u;
    const w2 v = {__builtin_amdgcn_perm(f[p], f[2 + p], sel), __builtin_amdgcn_perm(f[4 + p], f[6 + p], sel)};
    *reinterpret_cast<w2*>(o + (16u * g4 + c16) * 2u) = v;
  }
}

// One thread per (column, k-block), columns fastest: eight loads of one row of words each.
__global__ void __launch_bounds__(256) repack_tern_kernel(const uint32_t* __restrict__ src,
                                                          uint32_t* __restrict__ dst, uint32_t N, uint32_t N16,
                                                          uint32_t n16_m, uint32_t nkb, uint32_t total,
                                                          uint32_t* __restrict__ bad_flag) {
  const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const uint32_t kb = plan_div(idx, N16, n16_m), n = idx - kb * N16;
  uint32_t f[8];
  uint32_t bad = 0;
#pragma unroll
  for (uint32_t j = 0; j < 8; ++j) {
    // Code c = t + 1: nonzero where its low bit is clear, negative where both are; 3 is invalid.
    const uint32_t x = n < N ? src[(size_t)(8u * kb + j) * N + n] : 0x55555555u;
    const uint32_t lo = x & 0x55555555u, hi = (x >> 1) & 0x55555555u, nz = lo ^ 0x55555555u;
    bad |= lo & hi;
    f[j] = tern_split(__builtin_bitreverse32((nz & ~hi) | (nz << 1)));
  }
  tern_store_block(f, dst + ((size_t)(n / 16u) * nkb + kb) * 128u, n % 16u);
  if (bad && bad_flag) *bad_flag = 1u;
}

// GGUF TQ1_0 blocks straight into the ternary tile layout: one thread per (column n, block b), 16
// columns of a tile in consecutive threads and then the tile's blocks, so that a wavefront reads
// four neighbouring blocks of each column and stores whole 128-byte rows of the tile. A thread reads
// its 56-byte block with seven 8-byte loads, expands the 52 trit bytes through a 256-entry table
// (byte -> the (sign, nonzero) fields of its five digits, the first on top, 10 bits) into the
// block's 256 fields, then writes the 16 packed words of column n in k-blocks 2b and 2b + 1, and
// the block's d as the scale of group b. Columns past N up to the next multiple of 16 write zero
// words (padding decodes to zero).
__global__ void __launch_bounds__(256) repack_tq1_0_kernel(const uint8_t* __restrict__ blocks,
                                                           uint32_t* __restrict__ dst,
                                                           uint16_t* __restrict__ scales, uint32_t N,
                                                           uint32_t nb, uint32_t nb_m, uint32_t total) {
  __shared__ uint32_t tab[256];
  {
    uint32_t v = threadIdx.x, f = 0;
#pragma unroll
    for (uint32_t d = 0; d < 5; ++d) {
      f |= tern_c_to_field(v % 3u) << (8u - 2u * d);
      v /= 3u;
    }
    tab[threadIdx.x] = f;
  }
  __syncthreads();
  const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const uint32_t c16 = idx % 16u;
  const uint32_t ct = plan_div(idx / 16u, nb, nb_m), b = idx / 16u - ct * nb;
  const uint32_t n = 16u * ct + c16;
  // F: the fields of elements 0..255, element i at bits 31 - 2 (i % 16) and below of F[i / 16].
  uint32_t F[16];
#pragma unroll
  for (int w = 0; w < 16; ++w) F[w] = 0u;
  if (n < N) {
    const uint64_t* p = reinterpret_cast<const uint64_t*>(blocks + ((size_t)n * nb + b) * kTq1Bytes);
    uint64_t q[7];
#pragma unroll
    for (int i = 0; i < 7; ++i) q[i] = p[i];
    auto byte_at = [&](uint32_t o) { return (uint32_t)(q[o / 8u] >> (8u * (o % 8u))) & 0xFFu; };
    scales[(size_t)b * N + n] = (uint16_t)(q[0] & 0xFFFFu);
#pragma unroll
    for (uint32_t j = 0; j < 52; ++j) {
      // Trit byte j holds elements 5 j .. 5 j + 4 (j < 50) or 250 + 3 (j - 50) .. + 2.
      const uint32_t bits = j < 50u ? 10u : 6u, at = j < 50u ? 10u * j : 500u + 6u * (j - 50u);
      const uint32_t t = tab[byte_at(2u + j)] >> (10u - bits), end = at % 32u + bits;
      if (end <= 32u) {
        F[at / 32u] |= t << (32u - end);
      } else {
        F[at / 32u] |= t >> (end - 32u);
        F[at / 32u + 1u] |= t << (64u - end);
      }
    }
  }
#pragma unroll
  for (int w = 0; w < 16; ++w) F[w] = tern_split(F[w]);
#pragma unroll
  for (uint32_t h = 0; h < 2; ++h)  // k-block 2 b + h
    tern_store_block(F + 8u * h, dst + ((size_t)ct * 2u * nb + 2u * b + h) * 128u, c16);
}

}  // namespace

hipError_t launch_repack_tq1_0(const uint8_t* blocks, uint32_t* dst, uint16_t* scales, uint32_t K, uint32_t N,
                               hipStream_t stream) {
  const uint32_t nb = K / kTq1K, N16 = col_tiles(N) * 16u;
  const size_t total = (size_t)N16 * nb;
  if (total > 0xFFFFFF00u) return hipErrorInvalidValue;  // 32-bit thread numbers
  const size_t grid = (total + 255) / 256;
  hipLaunchKernelGGL(repack_tq1_0_kernel, dim3((uint32_t)grid), dim3(256), 0, stream, blocks, dst, scales, N, nb,
                     plan_div_magic(nb), (uint32_t)total);
  return hipGetLastError();
}

hipError_t launch_repack_int4(const uint32_t* src, uint32_t* dst, uint32_t K, uint32_t N,
                              hipStream_t stream) {
  const uint32_t nkb = K / kBlockK;
  const size_t total = (size_t)col_tiles(N) * nkb * 64u * 4u;
  const size_t grid = (total + 255) / 256;
  hipLaunchKernelGGL(repack_int4_kernel, dim3((uint32_t)grid), dim3(256), 0, stream, src, dst, N, nkb, total);
  return hipGetLastError();
}

hipError_t launch_repack_ternary2(const uint32_t* src, uint32_t* dst, uint32_t K, uint32_t N,
                                  uint32_t* bad_flag, hipStream_t stream) {
  const uint32_t nkb = K / kBlockK;
  const uint32_t N16 = col_tiles(N) * 16u;
  const size_t total = (size_t)N16 * nkb;
  if (total > 0xFFFFFF00u) return hipErrorInvalidValue;  // 32-bit thread numbers
  const size_t grid = (total + 255) / 256;
  hipLaunchKernelGGL(repack_tern_kernel, dim3((uint32_t)grid), dim3(256), 0, stream, src, dst, N, N16,
                     plan_div_magic(N16), nkb, (uint32_t)total, bad_flag);
  return hipGetLastError();
}

}  // namespace hq
