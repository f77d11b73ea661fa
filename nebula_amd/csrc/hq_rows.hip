// hq_rows.hip — memory-bound qGEMM for 17 <= M <= 80 on grids of at most one slab per CU (split-fuse
// steps, small prompt chunks), gfx950: shared row tiles.
//
// A workgroup owns a slab of four column tiles (64 columns) and one piece of its k-blocks (S pieces
// per slab when the slabs alone leave CUs idle). Its eight wavefronts are four k-groups of two: at
// step q k-group kg takes k-block 4 q + kg of the piece, and its two wavefronts stream two tiles each
// into a register ring. The k-block's activation rows (MT tiles of 16) go from L2 to the k-group's
// LDS stage by LDS-DMA (16-byte units XOR-swizzled by row: conflict-free fragment reads), one step
// ahead, two stages; one workgroup barrier a step publishes them.
//
// What bounds it is latency and issue slots, not bytes: a step's loads are therefore issued one by
// one between the fragments' MFMAs (all at the step's start they queue in the address unit and
// hold the MFMAs back), fragments are read from LDS four ahead with explicit counts (the compiler
// waits for each right after its read), the next chunk's dequantisation follows each fragment's
// MFMAs, and the k-block's sums are scaled in fp32 row tile by row tile behind the last chunk's.
// The k-groups' sums meet in LDS in k-group order; pieces through the workspace, summed in piece
// order by the last to arrive.
//
// Against the lockstep kernel (hq_decode_ls.hip), whose k-groups meet by polling and stage the
// rows through registers, MI355X (lockstep -> this one): ternary 4096 x 4096 M = 33 / 64 / 80 13.1 /
// 16.6 / 19.2 -> 8.5 / 9.6 / 10.5 us, 6144 x 5120 M = 80 20.7 -> 13.1, 5120 x 16384 M = 80 26.7 -> 20.0,
// 17408 x 5120 M = 80 30.4 -> 24.5; int4 bf16 4096 x 11008 M = 33 / 80 17.9 / 28.9 -> 13.4 / 18.0; int4
// fp16 5120 x 16384 M = 80 28.5 -> 22.6 (scales in fp32, where lockstep folds them into fp16 weights).
// Slabs of eight tiles (four per wavefront) were slower, three stages of half a k-block too.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "hq_device.hpp"
#include "hq_internal.hpp"
#include "hq_plan.hpp"

namespace hq {
namespace {

struct RowsPlan {
  uint32_t S, kq, kr;  // pieces per slab; piece p holds kq (+1 if p < kr) k-blocks
  uint32_t gmul;       // plan_gmul(gkb)
  uint32_t* cnt;       // [slabs] arrival counters, zero between launches (S > 1)
  float* part;         // [slabs][S][16 x 16 tiles][64 lanes] f4 partial tiles (S > 1)
};

constexpr uint32_t kXTile = 4096;  // 16 rows x 128 elements
constexpr int T = 2;               // column tiles per wavefront
constexpr uint32_t kGC = 2;        // wavefronts of a k-group (column halves of a slab)
constexpr uint32_t KG = 4;         // k-groups
constexpr int R = 3;               // weight ring slots (two steps ahead)

// 16 bytes from row tile r of a stage (addr: the lane's offset in row tile 0).
__device__ __forceinline__ u4 rw_lds_read(uint32_t addr, int r) {
  u4 v;
  if (r == 0) asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr));
  else if (r == 1) asm volatile("ds_read_b128 %0, %1 offset:4096" : "=v"(v) : "v"(addr));
  else if (r == 2) asm volatile("ds_read_b128 %0, %1 offset:8192" : "=v"(v) : "v"(addr));
  else if (r == 3) asm volatile("ds_read_b128 %0, %1 offset:12288" : "=v"(v) : "v"(addr));
  else asm volatile("ds_read_b128 %0, %1 offset:16384" : "=v"(v) : "v"(addr));
  return v;
}
__device__ __forceinline__ uint32_t rw_bpermute(uint32_t byte_lane, uint32_t v) {
  uint32_t r;
  asm volatile("ds_bpermute_b32 %0, %1, %2" : "=v"(r) : "v"(byte_lane), "v"(v));
  return r;
}
template <int N>
__device__ __forceinline__ void rw_wait_lgkm() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(N));
}
__device__ __forceinline__ void rw_tie(u4& a) { asm volatile("" : "+v"(a)); }
__device__ __forceinline__ void rw_tie(uint32_t& a) { asm volatile("" : "+v"(a)); }

template <int FMT, int DT, int MT, bool FUSED>
__global__ void __launch_bounds__(512, 2) hq_rows_kernel(const GemmDesc d, const RowsPlan pl) {
  constexpr bool kInt4 = FMT == HQ_FORMAT_INT4;
  constexpr uint32_t kLaneBytes = kInt4 ? 16u : 8u;
  constexpr uint32_t kBlockBytes = 64u * kLaneBytes;
  constexpr bool kSeed = kInt4 && DT == HQ_DTYPE_BF16;
  constexpr uint32_t kStage = MT * kXTile;  // a k-block of one k-group
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t kg = wave / kGC, wi = wave % kGC;
  const uint32_t c16 = lane & 15u, g4 = lane >> 4;
  const uint32_t nkb = d.nkb, M = d.M;
  const uint32_t g = blockIdx.x, piece = blockIdx.y;

  uint32_t si = 0;
  if constexpr (FUSED) {
    for (uint32_t i = 1; i < d.nseg; ++i)
      if (g >= d.seg[i].blk_begin) si = i;
    si = __builtin_amdgcn_readfirstlane(si);
  }
  const SegDesc& sg = d.seg[si];
  const uint32_t sN = sg.N, sLdy = (uint32_t)sg.ldy;
  const uint32_t l = g - sg.blk_begin;
  const uint32_t ct0 = l * sg.slab_w + min(l, sg.slab_r) + wi * T;  // this wavefront's first tile
  const uint32_t sw = sg.slab_w + (l < sg.slab_r ? 1u : 0u);
  const uint32_t ntw = sw > wi * T ? min((uint32_t)T, sw - wi * T) : 0u;
  const uint32_t tile_bytes = nkb * kBlockBytes;
  const uint32_t ctb = min(ct0, sg.ntiles - 1u);
  const char* const wbase = reinterpret_cast<const char*>(sg.Wp) + (size_t)ctb * tile_bytes;
  const uint32_t wbytes = ntw * tile_bytes;
  const uint32_t srow = sg.lds * 2u;
  const uint16_t* const sbase = sg.S;
  const uint32_t sbytes = ((nkb / d.gkb - 1u) * sg.lds + sN) * 2u;
  const uint32_t xbytes = M * (uint32_t)d.ldx * 2u, xtile = 16u * (uint32_t)d.ldx * 2u;

  const uint32_t ka = piece * pl.kq + min(piece, pl.kr);
  const uint32_t kz = ka + pl.kq + (piece < pl.kr ? 1u : 0u);
  const uint32_t nst = (kz - ka + KG - 1u) / KG;
  // k-block of step q (kz or more: none).
  auto kb_of = [&](uint32_t q) { return ka + q * KG + kg; };

  char* const stages = smem + kg * (2u * kStage);
  const uint32_t lds0 = (uint32_t)(uintptr_t)stages;
  uint32_t aoff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t row = 4u * (2u * wi + i) + g4;
    aoff[i] = row * (uint32_t)d.ldx * 2u + ((c16 ^ row) * 16u);
  }
  uint32_t ldsoff[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) ldsoff[c] = lds0 + c16 * 256u + (((4u * c + g4) ^ c16) * 16u);
  // Scales: lane l loads column 16 (ct0 + l / 16) + l % 16 (clamped to N - 1).
  const uint32_t svo = min((ct0 + min(g4, (uint32_t)T - 1u)) * 16u + c16, sN - 1u) * 2u;
  const uint32_t wvo = lane * kLaneBytes;
  uint32_t wso[T];  // missing tiles re-read the last one (their columns are not stored)
#pragma unroll
  for (int t = 0; t < T; ++t) wso[t] = min((uint32_t)t, max(ntw, 1u) - 1u) * tile_bytes;

  typedef typename std::conditional<kInt4, u4, u2>::type WV;
  WV wr[R][T];
  uint32_t sr[R];
  // Load n of step q's activations (2 MT of them), and load n of its weights (T and a scale).
  auto load_x1 = [&](uint32_t q, int n) {
    const uint32_t kb = kb_of(q);
    const uint32_t lm = 0u - (uint32_t)(kb < kz);
    const int r = n / 2;
    const __amdgpu_buffer_rsrc_t xr =
        make_rsrc(reinterpret_cast<const char*>(d.X) + (size_t)r * xtile, (r == MT - 1 ? xbytes - (MT - 1) * xtile : xtile) & lm);
    buffer_to_lds16(xr, stages + (q & 1u) * kStage + wi * 2048u + r * kXTile + (n & 1) * 1024u, aoff[n & 1], (kb * 256u) & lm);
  };
  auto load_w1 = [&](int slot, uint32_t q, int n) {
    const uint32_t kb = kb_of(q);
    const uint32_t lm = 0u - (uint32_t)(kb < kz);
    if (n < T) {
      const __amdgpu_buffer_rsrc_t r = make_rsrc(wbase, wbytes & lm);
      const uint32_t so = (kb * kBlockBytes + wso[n]) & lm;
      if constexpr (kInt4) wr[slot][n] = __builtin_amdgcn_raw_buffer_load_b128(r, wvo, so, kStreamAux);
      else wr[slot][n] = __builtin_amdgcn_raw_buffer_load_b64(r, wvo, so, kStreamAux);
    } else {
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(sbase, sbytes & lm);
      sr[slot] = __builtin_amdgcn_raw_buffer_load_b16(rs, svo, (plan_group_of_kb(kb, pl.gmul) * srow) & lm, 0);
    }
  };

  f4 acc[MT][T];
#pragma unroll
  for (int r = 0; r < MT; ++r)
#pragma unroll
    for (int t = 0; t < T; ++t) acc[r][t] = f4{0.f, 0.f, 0.f, 0.f};
  const DqConst dqk = dq_const_f16();
  const DqBiasConst dqb = dq_bias_const_bf16();
  const u4 corr_b = int4_corr_fragment<DT>();

  constexpr int NF = 4 * MT;               // A fragments of a k-block: fragment c * MT + r
  constexpr int NL = 2 * MT + T + 1;       // loads of a step
  auto step = [&](int slot, uint32_t q) {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((R - 2) * (T + 1)));  // X(q), W(q) have landed for this wavefront
    __builtin_amdgcn_s_barrier();  // ... for all; the other stage is free
    __builtin_amdgcn_sched_barrier(0);
    if (kb_of(q) < kz) {  // uniform
      const uint32_t so = (q & 1u) * kStage;
      constexpr int NA = 4;  // A fragments in flight
      uint32_t sc[T];
#pragma unroll
      for (int t = 0; t < T; ++t) sc[t] = rw_bpermute((16u * t + c16) * 4u, sr[slot]);
      u4 a[NA];
#pragma unroll
      for (int i = 0; i < NA; ++i) a[i] = rw_lds_read(ldsoff[i / MT] + so, i % MT);
      u4 b[2][T];
      auto dq = [&](int c, int t) {
        if constexpr (kInt4) {
          if constexpr (DT == HQ_DTYPE_F16) b[c & 1][t] = dq_int4_f16(wr[slot][t][c], dqk);
          else b[c & 1][t] = dq_int4_biased<DT>(wr[slot][t][c], dqb);
        } else {
          const uint32_t word = wr[slot][t][c >> 1];
          b[c & 1][t] = (c & 1) ? dq_tern2<1>(word) : dq_tern2<0>(word);
        }
      };
#pragma unroll
      for (int t = 0; t < T; ++t) dq(0, t);
      f4 gs[MT][T], corr[MT];
#pragma unroll
      for (int r = 0; r < MT; ++r) {
        corr[r] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < T; ++t) gs[r][t] = f4{0.f, 0.f, 0.f, 0.f};
      }
      float scf[T];
      auto scale_row = [&](int r) {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            acc[r][t][v] = __builtin_fmaf(kSeed ? gs[r][t][v] + corr[r][v] : gs[r][t][v], scf[t], acc[r][t][v]);
      };
#pragma unroll
      for (int i = 0; i < NF; ++i) {
        const int c = i / MT, r = i % MT;
        __builtin_amdgcn_sched_barrier(0);
        if (NF - 1 - i >= NA - 1) rw_wait_lgkm<NA - 1>();
        else if (NF - 1 - i == 2) rw_wait_lgkm<2>();
        else if (NF - 1 - i == 1) rw_wait_lgkm<1>();
        else rw_wait_lgkm<0>();
        rw_tie(a[i % NA]);
        if (i == 0) {
#pragma unroll
          for (int t = 0; t < T; ++t) rw_tie(sc[t]);
#pragma unroll
          for (int t = 0; t < T; ++t) {
            scf[t] = f16_to_f32((uint16_t)sc[t]);
            if constexpr (!kInt4) scf[t] = __builtin_isfinite(scf[t]) ? 0.5f * scf[t] : 0.0f;  // fields hold 2t
          }
        }
        if constexpr (kSeed) corr[r] = mfma16x16x32<DT>(a[i % NA], corr_b, corr[r]);
#pragma unroll
        for (int t = 0; t < T; ++t) gs[r][t] = mfma16x16x32<DT>(a[i % NA], b[c & 1][t], gs[r][t]);
        if (c < 3) {
          // The next chunk's fragments, T tiles spread over the MT rows.
#pragma unroll
          for (int t = 0; t < T; ++t)
            if (t * MT / T == r) dq(c + 1, t);
        } else if (r > 0) {
          scale_row(r - 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (i + NA < NF) a[i % NA] = rw_lds_read(ldsoff[(i + NA) / MT] + so, (i + NA) % MT);
        // The next step's loads, spread over the fragments.
#pragma unroll
        for (int n = i * NL / NF; n < (i + 1) * NL / NF; ++n) {
          if (n < 2 * MT) load_x1(q + 1u, n);
          else load_w1((slot + R - 1) % R, q + R - 1u, n - 2 * MT);
        }
      }
      scale_row(MT - 1);
    }
  };

  auto load_all_w = [&](int slot, uint32_t q) {
#pragma unroll
    for (int n = 0; n <= T; ++n) load_w1(slot, q, n);
    __builtin_amdgcn_sched_barrier(0);
  };
  load_all_w(0, 0);
#pragma unroll
  for (int n = 0; n < 2 * MT; ++n) load_x1(0, n);
  __builtin_amdgcn_sched_barrier(0);
  load_all_w(1, 1);
  for (uint32_t q = 0; q < nst; q += R) {
#pragma unroll
    for (int s = 0; s < R; ++s) step(s, q + s);
  }
  __builtin_amdgcn_s_waitcnt(0);

  // Sum over the k-groups through the stages' LDS.
  const __amdgpu_buffer_rsrc_t yr = make_rsrc(sg.Y, M * sLdy * 2u);
  const uint32_t ct_slab = l * sg.slab_w + min(l, sg.slab_r);
  auto store_out = [&](uint32_t r, uint32_t tile, const f4& v) {
    const uint32_t col = (ct_slab + tile) * 16u + c16;
    const bool mine = tile < sw && col < sN;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t row = 16u * r + 4u * g4 + e;
      const uint32_t o = row < M && mine ? (row * sLdy + col) * 2u : kOutOfRange;
      __builtin_amdgcn_raw_buffer_store_b16(f32_to_out<DT>(v[e]), yr, o, 0, 0);
    }
  };
  constexpr int kCoherent = 16;
  const uint32_t pieces = pl.S;
  constexpr uint32_t kUnits = kGC * T * MT;
  const __amdgpu_buffer_rsrc_t partr = make_rsrc(pl.part, pl.part ? gridDim.x * pieces * kUnits * 1024u : 0u);
  f4* const red = reinterpret_cast<f4*>(smem);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int r = 0; r < MT; ++r) red[(wave * (T * MT) + t * MT + r) * 64u + lane] = acc[r][t];
  __syncthreads();
  for (uint32_t u = wave; u < kUnits; u += kGC * KG) {  // uniform: unit = (column half, tile, row tile)
    f4 v = red[u * 64u + lane];
    for (uint32_t k = 1; k < KG; ++k) v += red[(k * kUnits + u) * 64u + lane];
    if (pieces == 1u) {
      const uint32_t tile = u / MT;
      store_out(u - tile * MT, tile, v);
    } else {
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), partr,
                                             (((g * pieces + piece) * kUnits + u) * 64u + lane) * 16u, 0, kCoherent);
    }
  }
  if (pieces == 1u) return;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  uint32_t* const sh_last = reinterpret_cast<uint32_t*>(smem);
  if (threadIdx.x == 0) {
    const uint32_t old = __hip_atomic_fetch_add(pl.cnt + g, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t last = old == pieces - 1u;
    if (last) __hip_atomic_store(pl.cnt + g, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *sh_last = last;
  }
  __syncthreads();
  if (!*sh_last) return;
  for (uint32_t u = wave; u < kUnits; u += kGC * KG) {
    f4 v = f4{0.f, 0.f, 0.f, 0.f};
    for (uint32_t p0 = 0; p0 < pieces; p0 += 8u) {
      u4 part[8];
#pragma unroll
      for (uint32_t p = 0; p < 8u; ++p) {
        const uint32_t o = p0 + p < pieces ? (((g * pieces + p0 + p) * kUnits + u) * 64u + lane) * 16u : kOutOfRange;
        part[p] = __builtin_amdgcn_raw_buffer_load_b128(partr, o, 0, kCoherent);
      }
#pragma unroll
      for (uint32_t p = 0; p < 8u; ++p) v += __builtin_bit_cast(f4, part[p]);
    }
    const uint32_t tile = u / MT;
    store_out(u - tile * MT, tile, v);
  }
}

uint32_t rows_assign(GemmDesc& d) {
  uint32_t g = 0;
  for (uint32_t i = 0; i < d.nseg; ++i) {
    const uint32_t nt = d.seg[i].ntiles, ns = (nt + kGC * T - 1) / (kGC * T);
    d.seg[i].blk_begin = g;
    d.seg[i].blk_count = ns;
    d.seg[i].slab_w = nt / ns;
    d.seg[i].slab_r = nt % ns;
    g += ns;
  }
  return g;
}

template <int FMT, int DT, int MT>
hipError_t rows_launch(GemmDesc d, const RowsConfig& c, void* ws, hipStream_t stream) {
  RowsPlan pl{};
  const uint32_t G = rows_assign(d);
  if (d.M > 16u * MT || d.M <= 16u * (MT - 1) || c.S < 1 || (uint32_t)c.S > d.nkb || G > 65535u) return hipErrorInvalidValue;
  pl.S = (uint32_t)c.S;
  pl.kq = d.nkb / pl.S;
  pl.kr = d.nkb % pl.S;
  pl.gmul = plan_gmul(d.gkb);
  if (c.S > 1) {
    if (!ws || G > kMaxCounters || (uint64_t)G * pl.S * kGC * T * MT * 1024u >= (1ull << 31)) return hipErrorInvalidValue;
    pl.cnt = static_cast<uint32_t*>(ws);
    pl.part = reinterpret_cast<float*>(static_cast<char*>(ws) + kCounterBytes);
  }
  constexpr size_t lds = (size_t)KG * 2 * MT * kXTile;
  static_assert(lds >= (size_t)KG * kGC * T * MT * 1024u, "the k-groups' sums reuse the stages");
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&hq_rows_kernel<FMT, DT, MT, false>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess
          ? hipErrorInvalidConfiguration
          : hipFuncSetAttribute(reinterpret_cast<const void*>(&hq_rows_kernel<FMT, DT, MT, true>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return attr;
  const dim3 grid(G, pl.S), block(64u * kGC * KG);
  if (d.nseg > 1) hipLaunchKernelGGL((hq_rows_kernel<FMT, DT, MT, true>), grid, block, lds, stream, d, pl);
  else hipLaunchKernelGGL((hq_rows_kernel<FMT, DT, MT, false>), grid, block, lds, stream, d, pl);
  return hipGetLastError();
}

template <int FMT, int DT>
hipError_t rows_mt(const GemmDesc& d, const RowsConfig& c, void* ws, hipStream_t stream) {
  switch ((d.M + 15u) / 16u) {
    case 2: return rows_launch<FMT, DT, 2>(d, c, ws, stream);
    case 3: return rows_launch<FMT, DT, 3>(d, c, ws, stream);
    case 4: return rows_launch<FMT, DT, 4>(d, c, ws, stream);
    case 5: return rows_launch<FMT, DT, 5>(d, c, ws, stream);
    default: return hipErrorInvalidConfiguration;
  }
}

}  // namespace

// The longest piece, in k-blocks, at which slabs of four tiles in S pieces still beat the lockstep
// kernel, by the type and the row tiles (2 .. 5): what they save is spent once a launch, and over a long
// piece its slabs of eight tiles, cut finer, keep more of the chip busy. Four kinds of grids: lockstep's
// past one workgroup per CU (171-184 slabs here); its workgroups with under 6/7 of the work of ours (81-102 and
// 129-170 slabs, which leave CUs idle here); as much work, whole slabs; in pieces. Fitted to 22,000 pairs on
// MI355X (80 slab counts of 16..256, 8..216 k-blocks, weights from memory), each within 5% of the faster
// kernel, nearly all within 2%; int4 fp16 at 65 to 80 rows is held against lockstep with fp32 scales (with them
// in the fp16 weights it is up to 9% faster than this kernel past 140 k-blocks). Lockstep -> this kernel, us,
// by k-blocks: 172 slabs int4 bf16 M = 80 176 110.5 -> 76.4; 130 slabs ternary fp16 M = 56 32 15.7 -> 14.0, 48
// 18.6 -> 19.4, 152 37.9 -> 51.9, M = 80 48 22.5 -> 21.2, 96 33.1 -> 37.0; 256 slabs ternary M = 33 96 29.1 ->
// 30.9, M = 80 44.8 -> 38.7, int4 bf16 M = 80 152 86.5 -> 76.5.
constexpr uint16_t kAny = 0xFFFF;
constexpr uint16_t kMaxPiece[4][3][4] = {
    // int4 fp16, int4 bf16, ternary
    {{kAny, kAny, kAny, kAny}, {kAny, kAny, kAny, kAny}, {36, 96, kAny, kAny}},
    {{20, 32, 46, 52}, {20, 40, 46, 64}, {20, 32, 46, 64}},
    {{36, 64, 96, 216}, {36, 96, 152, kAny}, {36, 64, 96, 176}},
    {{24, 48, 80, kAny}, {24, kAny, kAny, kAny}, {24, 46, 80, kAny}},
};
bool rows_piece_too_long(int fmt, int dtype, const GemmDesc& d, uint32_t S, size_t ws_cap) {
  uint32_t slabs = 0;
  for (uint32_t i = 0; i < d.nseg; ++i) slabs += (d.seg[i].ntiles + 7u) / 8u;
  const uint32_t pieces = (uint32_t)choose_decode_ls(fmt, d, ws_cap, false).S;
  const int grid = slabs * pieces > (uint32_t)cu_count() ? 0 : 7u * S < 3u * pieces ? 1 : S == 1u ? 2 : 3;
  const int type = fmt != HQ_FORMAT_INT4 ? 2 : dtype == HQ_DTYPE_F16 ? 0 : 1;
  uint32_t most = kMaxPiece[grid][type][(d.M + 15u) / 16u - 2u];
  // Pieces just short of lockstep's (69-72 slabs in three): 72 k-blocks each ternary M = 56 27.9 -> 30.2 us.
  if (grid == 3 && 2u * S < pieces && d.M <= 64u) most = std::min(most, 64u);
  return most != kAny && (d.nkb + S - 1u) / S > most;
}

// Taken when the slabs number at most the CUs, cut into as many pieces (at most eight, each at
// least one step per k-group) as stay within one workgroup per CU and fill half of them. Measured on
// MI355X at G x S workgroups, M = 20..80, ternary and int4, fp16 and bf16: 2-113% faster than the
// lockstep kernel (most at few slabs: 1024 x 4096 M = 80 18.1 -> 8.6 us), except, kept there: pieces too
// long for their grid (kMaxPiece), grids
// under two thirds of the CUs at few rows (5120 x 9000, 141 slabs: M = 20 11.8 against 13.2, M = 33 14.4
// against 15.0; M = 64 18.0 -> 17.0), a long K at few rows (17408 x 5120: M = 20 16.0 against 17.1, M = 33
// 19.9 -> 19.4), and int4 up to 32 rows, where lockstep's balanced grids run the wide shapes (5120 x
// 34816) and one kernel serves the range. More slabs than CUs: two rounds lose (ternary 5120 x 34816 M
// = 80 50.7 against 53.4).
// HQ_ROWS = 0 keeps the lockstep kernel, a number forces that many pieces (tuning and tests); any
// lockstep override keeps it too.
RowsConfig choose_rows(int fmt, const GemmDesc& d, size_t ws_cap, int dtype) {
  RowsConfig c{1, false};
  if (d.M <= 16u || d.M > 80u || d.gen) return c;
  const char* e = std::getenv("HQ_ROWS");
  const int force = e && *e ? std::atoi(e) : -1;
  if (force == 0) return c;
  for (const char* n : {"HQ_DECODE_KERNEL", "HQ_DECODE_LS_BAL", "HQ_DECODE_LS_GW", "HQ_DECODE_LS_KG", "HQ_DECODE_LS_S",
                        "HQ_DECODE_LS_SPIN", "HQ_DECODE_LS_SW", "HQ_DECODE_LS_T", "HQ_DECODE_LS_U"}) {
    const char* v = std::getenv(n);
    if (force < 0 && v && *v) return c;
  }
  GemmDesc t = d;
  const uint32_t G = rows_assign(t), cus = (uint32_t)cu_count();
  if (force > 0) {
    c.S = std::min(force, (int)d.nkb);
  } else {
    if (G > cus || (fmt == HQ_FORMAT_INT4 && d.M <= 32u)) return c;
    c.S = (int)std::min(std::min(cus / G, 8u), std::max(1u, d.nkb / KG));
    const uint32_t wgs = G * (uint32_t)c.S;
    if (2u * wgs < cus || (3u * wgs < 2u * cus && d.M <= 48u && G > cus / 2u)) return c;
    if (d.nkb > (d.M <= 32u ? 64u : d.M <= 48u ? 144u : ~0u)) return c;
    c.long_k = rows_piece_too_long(fmt, dtype, d, (uint32_t)c.S, ws_cap);
    if (c.long_k) return c;
  }
  c.ok = rows_workspace_bytes(d, c) <= ws_cap;
  return c;
}
size_t rows_workspace_bytes(const GemmDesc& d, const RowsConfig& c) {
  if (c.S <= 1) return 0;
  GemmDesc t = d;
  return kCounterBytes + (size_t)rows_assign(t) * c.S * ((d.M + 15u) / 16u) * kGC * T * 1024u;
}
hipError_t launch_rows(int fmt, int dtype, const GemmDesc& d, const RowsConfig& c, void* ws, hipStream_t stream) {
  if (fmt == HQ_FORMAT_INT4)
    return dtype == HQ_DTYPE_F16 ? rows_mt<HQ_FORMAT_INT4, HQ_DTYPE_F16>(d, c, ws, stream)
                                 : rows_mt<HQ_FORMAT_INT4, HQ_DTYPE_BF16>(d, c, ws, stream);
  return dtype == HQ_DTYPE_F16 ? rows_mt<HQ_FORMAT_TERNARY2, HQ_DTYPE_F16>(d, c, ws, stream)
                               : rows_mt<HQ_FORMAT_TERNARY2, HQ_DTYPE_BF16>(d, c, ws, stream);
}

}  // namespace hq
