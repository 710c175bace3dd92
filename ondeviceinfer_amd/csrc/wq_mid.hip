// Batches of 5 to 64 rows: W4A16 and W8A16 linears whose activations are
// staged once per workgroup in LDS and shared by its tile waves.
//
// Bound: a weight stream (HBM) as long as the activations stay cheap.  The
// skinny kernels give every wave its own copy of the activation fragments, so
// at M = 49..64 a wave moves 16 KiB of x from L2 for every 2 KiB of W4
// weights; here a workgroup moves M * 256 B of x per 128-k block once for its
// 2 P 16-row tiles (P = 4 or 5).  Workgroup (g, s) = 2 P waves owns tile group
// g over the k range s of S (both from mid_split):
//  * wave (p, h) takes the tile pair p (two tiles, so that an x fragment read
//    from LDS feeds two MFMAs) and the 128-k blocks of parity h, which halves
//    the number of barriers per block; the two parities meet in LDS at the end;
//  * a stage is two blocks: its x goes buffer -> LDS (rows past M read as
//    zero, chunks at the slots of frag_slot), its weights straight
//    into registers, D - 1 stages ahead (D = 3, and 2 where 48 or 64 rows fill
//    the LDS and the registers: a deeper ring measured no faster there, nor
//    did x staged through registers with the LDS reads one k-step ahead);
//  * per block the skinny kernels' arithmetic: W4 the exact fp16 (q - z) on
//    MFMA 16x16x32, then the group scale times the block sum added in fp32;
//    INT8 the exact fp16 q, the row scale applied to the final sum.
// Each split stores its fp32 partials with device-coherent stores (0.1-0.8 us
// ahead of plain and non-temporal ones) and a second small launch adds them
// in split order.  Against a last-arriver sum inside this kernel (arrival
// counters, as the deep-ring GEMM) that is 0.3-0.8 us slower at some W4 shapes
// and 0.4-4 us faster at N = 1024 and on INT8, and it needs no zeroed counters,
// so any scratch of the call's own will do.  The short W4 shapes of 12 to 32
// rows keep the last arriver (mid_counts): they finish before the host has
// queued a second launch (fused QKV M = 24 called from Python 11.5 us against
// 13.3).
// MI355X, graphs of distinct weights, us, the skinny kernels (W4 12..32 rows up
// to 1152 tiles: wq_batch.hip, 17..64 rows from 2048 tiles on: the deep-ring
// GEMM) -> this one:
//   W4 17408->5120    M = 8 / 24 / 40 / 56   20.1 / 35.9 / 49.3 / 64.8 -> 15.9 / 18.7 / 21.6 / 24.9
//   W4 5120->7168     M = 24 / 40 / 56       12.4 / 17.5 / 23.5 -> 11.7 / 14.0 / 16.2
//   W4 5120->17408    M = 8 / 24 / 40 / 56   21.6 / 27.3 / 39.1 / 55.2 -> 17.4 / 21.0 / 23.9 / 27.2
//   W4 5120->34816    M = 8 / 24 / 40 / 56   28.7 / 37.5 / 49.9 / 51.2 -> 27.5 / 31.4 / 35.6 / 40.4
//   INT8 17408->5120  M = 8 / 24 / 56        31.4 / 37.8 / 66.7 -> 20.6 / 21.9 / 29.2
//   INT8 5120->17408  M = 8 / 24 / 56        25.0 / 37.7 / 71.2 -> 21.7 / 24.4 / 28.3
//   INT8 5120->34816  M = 8 / 24 / 56        46.6 / 62.4 / 120 -> 35.0 / 37.5 / 48.4
// i.e. 93 MB of W4 weights at M = 8 in 27.5 us (3.4 TB/s) and 178 MB of INT8
// in 35.0 us (5.1 TB/s); what remains is about 6 us of launch, first load and
// partial sum, then 16 B per cycle and compute unit of weights and x.
#include "wq_common.h"
#include "wq_mid_plan.h"
#include "wq_status.h"

namespace wq {
namespace {

enum class MFmt { W4, W8 };

// Largest k: 64 rows of x stay inside the 31-bit buffer range.
constexpr int64_t kMidMaxK = 1 << 23;
static_assert(1152 / (4 * kMidTilesPerWave) <= kSplitMaxCounters, "one counter per tile group");

template <int N>
__device__ __forceinline__ void mid_wait_vm() {
  static_assert(N >= 0 && N <= 63, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// The MC fragments of one k-step (16 rows apart inside a stage), read and
// waited for in one asm block.
template <int MC>
__device__ __forceinline__ void mid_read(uint4_t (&f)[MC], uint32_t a) {
  if constexpr (MC == 1)
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(f[0]) : "v"(a));
  else if constexpr (MC == 2)
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:4096\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(f[0]), "=&v"(f[1]) : "v"(a));
  else if constexpr (MC == 3)
    asm volatile("ds_read_b128 %0, %3\n\tds_read_b128 %1, %3 offset:4096\n\tds_read_b128 %2, %3 offset:8192\n\t"
                 "s_waitcnt lgkmcnt(0)" : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]) : "v"(a));
  else
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:4096\n\tds_read_b128 %2, %4 offset:8192\n\t"
                 "ds_read_b128 %3, %4 offset:12288\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]) : "v"(a));
}

// Columns n0 .. n0 + 3 of row m (N % 8 == 0 for W4; INT8 takes any N and
// stores the quad at once when row m keeps 8-byte alignment).
template <MFmt F>
__device__ __forceinline__ void mid_store(float4_t s, int m, int n0, int M, int N, const void* __restrict__ wmeta,
                                          const half_t* __restrict__ bias, half_t* __restrict__ y) {
  if (m >= M || n0 >= N) return;
  half4_t o;
  if constexpr (F == MFmt::W4) {
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = (half_t)s[v];
    *reinterpret_cast<half4_t*>(y + (size_t)m * N + n0) = o;
  } else {
    const half_t* scale = reinterpret_cast<const half_t*>(wmeta);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int n = min(n0 + v, N - 1);
      float r = s[v] * (float)scale[n];
      if (bias) r += (float)bias[n];
      o[v] = (half_t)r;
    }
    if ((N & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 7) == 0) {
      *reinterpret_cast<half4_t*>(y + (size_t)m * N + n0) = o;
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (n0 + v < N) y[(size_t)m * N + n0 + v] = o[v];
    }
  }
}

// One wave's weights of one 128-k block.
template <MFmt F>
struct MidRegs;
template <>
struct MidRegs<MFmt::W4> {
  uint4_t w[kMidTilesPerWave];
  uint2_t s[kMidTilesPerWave];
  uint32_t z[kMidTilesPerWave];
};
template <>
struct MidRegs<MFmt::W8> {
  uint4_t a[kMidTilesPerWave], b[kMidTilesPerWave];
};

template <MFmt F, int P, int MC, int D, int MINW>
__global__ __launch_bounds__(128 * P, MINW) void mid_kernel(
    const half_t* __restrict__ x, int M, int K, const void* __restrict__ wsrc, const void* __restrict__ wmeta, int N,
    int bpg, const half_t* __restrict__ bias, half_t* __restrict__ y, float4_t* ws_part, uint32_t* ws_cnt, int tiled) {
  constexpr int NT = kMidTilesPerWave;
  constexpr int kSubBytes = MC * 16 * 256;      // one 128-k block of x
  constexpr int kStageBytes = 2 * kSubBytes;
  constexpr int kWLoads = (F == MFmt::W4 ? 3 : 2) * NT;   // weight loads per wave and stage
  constexpr int kUnits = P * NT * MC;           // 1 KiB accumulator units of the workgroup
  static_assert(D >= 2 && (D - 2) * (MC + kWLoads) <= 63, "ring depth");
  static_assert(kUnits * 1024 <= D * kStageBytes, "the parity sum reuses the ring");
  __shared__ __attribute__((aligned(1024))) uint8_t xs[D * kStageBytes];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = wave >= P ? 1 : 0, p = wave - h * P;
  const int i = lane & 15, kb = lane >> 4;
  const int ntile = (N + 15) >> 4;
  const int nblk = K / kW4BlockK, nst = (nblk + 1) >> 1;
  const int group = blockIdx.x, split = blockIdx.y, S = gridDim.y;
  const int st_lo = (split * nst) / S, nloc = ((split + 1) * nst) / S - st_lo;
  const int tile0 = (group * P + p) * NT;
  constexpr uint32_t kPastEnd = 0x80000000u;

  uint32_t xvo[MC];
#pragma unroll
  for (int j = 0; j < MC; ++j) {
    const int rr = 4 * (p * MC + j) + (lane >> 4);
    xvo[j] = (uint32_t)(rr * K * 2 + slot_chunk<F == MFmt::W4>(rr, lane & 15) * 16);
  }
  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(x, (int64_t)M * K * 2);

  const int ngrp = F == MFmt::W4 ? nblk / bpg : 0;
  __amdgpu_buffer_rsrc_t rw, rm;
  if constexpr (F == MFmt::W4) {
    rw = buf_rsrc(reinterpret_cast<const uint8_t*>(wsrc) + (size_t)tile0 * nblk * 1024,
                  (int64_t)(ntile - tile0) * nblk * 1024);
    rm = buf_rsrc(reinterpret_cast<const uint8_t*>(wmeta) + (size_t)tile0 * ngrp * kW4MetaBytes,
                  (int64_t)(ntile - tile0) * ngrp * kW4MetaBytes);
  } else {
    rw = tiled ? buf_rsrc(reinterpret_cast<const int8_t*>(wsrc) + (size_t)tile0 * nblk * kW8TileBlockBytes,
                          (int64_t)(ntile - tile0) * nblk * kW8TileBlockBytes)
               : buf_rsrc(reinterpret_cast<const int8_t*>(wsrc) + (size_t)tile0 * 16 * K, (int64_t)(N - tile0 * 16) * K);
    rm = rw;
  }
  // Stages are requested in order, so the next block, its group and the
  // group's remainder advance by two blocks a stage (no division per stage).
  int nx = 2 * st_lo + h;
  const int nx_end = min(2 * (st_lo + nloc), nblk);
  int gq = F == MFmt::W4 ? nx / bpg : 0, gr = F == MFmt::W4 ? nx - gq * bpg : 0;
  const int gq2 = F == MFmt::W4 ? 2 / bpg : 0, gr2 = F == MFmt::W4 ? 2 - gq2 * bpg : 0;
  const uint32_t wvo = F == MFmt::W4 || tiled ? (uint32_t)lane * 16 : (uint32_t)(i * K + 16 * kb);
  const uint32_t wstep = F == MFmt::W4 ? 1024 : tiled ? kW8TileBlockBytes : kW8BlockK;
  const uint32_t wtile = F == MFmt::W4 ? (uint32_t)nblk * 1024 : tiled ? (uint32_t)nblk * kW8TileBlockBytes : (uint32_t)(16 * K);
  auto fetch = [&](int st, MidRegs<F>& r) {
    const bool live = nx < nx_end;
    const uint32_t xo = live ? (uint32_t)nx * 256 : kPastEnd;
    if (P == 4 || p < 4) {   // four of the P waves of a parity copy its x
#pragma unroll
      for (int j = 0; j < MC; ++j)
        lds_load16(rx, xvo[j], xo, xs + st * kStageBytes + h * kSubBytes + (p * MC + j) * 1024);
    }
    const uint32_t wo = live ? (uint32_t)nx * wstep : kPastEnd;
    if constexpr (F == MFmt::W4) {
      const uint32_t mo = live ? (uint32_t)(gq * kW4MetaBytes) : kPastEnd;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        r.w[t] = __builtin_amdgcn_raw_buffer_load_b128(rw, wvo, wo + t * wtile, kNtPolicy);
        r.s[t] = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(rm, (uint32_t)kb * 8, mo + t * ngrp * kW4MetaBytes, 0));
        r.z[t] = __builtin_amdgcn_raw_buffer_load_b32(rm, 32 + (uint32_t)(i >> 3) * 4, mo + t * ngrp * kW4MetaBytes, 0);
      }
      gq += gq2;
      gr += gr2;
      if (gr >= bpg) {
        gr -= bpg;
        ++gq;
      }
    } else {
      const uint32_t p1 = tiled ? kW8TileBlockBytes / 2 : 64;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        r.a[t] = __builtin_amdgcn_raw_buffer_load_b128(rw, wvo, wo + t * wtile, kNtPolicy);
        r.b[t] = __builtin_amdgcn_raw_buffer_load_b128(rw, wvo + p1, wo + t * wtile, kNtPolicy);
      }
    }
    nx += 2;
  };

  float4_t acc[NT][MC];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mc = 0; mc < MC; ++mc) acc[t][mc] = float4_t{0.f, 0.f, 0.f, 0.f};
  const uint32_t xs_base = (uint32_t)(size_t)((const __attribute__((address_space(3))) uint8_t*)xs) +
                           (uint32_t)(h * kSubBytes + i * 256);

  auto block = [&](int st, const MidRegs<F>& r) {
    float4_t cg[NT][MC];
    uint32_t c_lo[NT], c_hi[NT];
    if constexpr (F == MFmt::W4) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        w4_zero_consts((r.z[t] >> (4 * (i & 7))) & 0xFu, c_lo[t], c_hi[t]);
#pragma unroll
        for (int mc = 0; mc < MC; ++mc) cg[t][mc] = float4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
    const uint32_t base = xs_base + (uint32_t)(st * kStageBytes);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      uint4_t f[MC];
      mid_read<MC>(f, base + (uint32_t)(frag_slot(i, kb, w) * 16));
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        half8_t a;
        if constexpr (F == MFmt::W4) {
          const uint32_t word = w == 0 ? r.w[t].x : w == 1 ? r.w[t].y : w == 2 ? r.w[t].z : r.w[t].w;
          a = w4_word_to_h8(word, c_lo[t], c_hi[t]);
        } else {
          const uint4_t& v = w < 2 ? r.a[t] : r.b[t];
          a = (w & 1) == 0 ? i8x8_to_h8(v.x, v.y) : i8x8_to_h8(v.z, v.w);
        }
#pragma unroll
        for (int mc = 0; mc < MC; ++mc) {
          if constexpr (F == MFmt::W4) cg[t][mc] = mfma16(a, __builtin_bit_cast(half8_t, f[mc]), cg[t][mc]);
          else acc[t][mc] = mfma16(a, __builtin_bit_cast(half8_t, f[mc]), acc[t][mc]);
        }
      }
    }
    if constexpr (F == MFmt::W4) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const half4_t s4 = __builtin_bit_cast(half4_t, r.s[t]);
#pragma unroll
        for (int mc = 0; mc < MC; ++mc)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[t][mc][v] += (float)s4[v] * cg[t][mc][v];
      }
    }
  };

  MidRegs<F> wr[D];
#pragma unroll
  for (int j = 0; j < D - 1; ++j) {
    fetch(j, wr[j]);
    __builtin_amdgcn_sched_barrier(0);   // loads stay in stage order: the waits below count them
  }
  auto wait = [&]() {   // the next stage has landed: this wave's part, then everyone's
    if (P == 4 || p < 4) mid_wait_vm<(D - 2) * (MC + kWLoads)>();
    else mid_wait_vm<(D - 2) * kWLoads>();
    __builtin_amdgcn_s_barrier();
  };
  wait();
  int base = 0;
  do {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      fetch((u + D - 1) % D, wr[(u + D - 1) % D]);
      __builtin_amdgcn_sched_barrier(0);
      if (base + u < nloc) block(u, wr[u]);
      wait();
    }
    base += D;
  } while (base < nloc);
  mid_wait_vm<0>();            // the run-out's empty copies have landed ...
  __builtin_amdgcn_s_barrier();   // ... everyone's: the ring is dead

  // Unit (p, t, mc) at 1 KiB granules: the odd-block waves hand theirs over.
  float4_t* red = reinterpret_cast<float4_t*>(xs);
  if (h == 1) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int mc = 0; mc < MC; ++mc) red[((p * NT + t) * MC + mc) * 64 + lane] = acc[t][mc];
  }
  __syncthreads();
  if (h == 0) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int mc = 0; mc < MC; ++mc) {
        const int unit = (p * NT + t) * MC + mc;
        const float4_t s = acc[t][mc] + red[unit * 64 + lane];
        if (S == 1) mid_store<F>(s, mc * 16 + i, (tile0 + t) * 16 + 4 * kb, M, N, wmeta, bias, y);
        else coherent_store16(ws_part, (uint32_t)(((group * S + split) * kUnits + unit) * 1024 + lane * 16),
                              __builtin_bit_cast(uint4_t, s));
      }
  }
  if constexpr (F == MFmt::W4 && MC <= 2) {
    if (ws_cnt == nullptr) return;   // uniform: S == 1, or mid_sum_kernel adds the partials
    // The last of the group's S workgroups to arrive adds the partials, in
    // split order, and stores y.
    __builtin_amdgcn_s_waitcnt(0);   // this wave's partials are acknowledged
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();                 // ... and every wave's; the sums above are read
    uint32_t* arrival = reinterpret_cast<uint32_t*>(xs);
    if (threadIdx.x == 0)
      *arrival = __hip_atomic_fetch_add(&ws_cnt[group], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrival != (uint32_t)(S - 1)) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    static_assert(kUnits == MC * 2 * P, "MC units per wave");
    constexpr int Q = 8 / MC;        // splits of each unit requested at once
    float4_t sum[MC];
    for (int s0 = 0; s0 < S; s0 += Q) {
      float4_t v[MC][Q];
#pragma unroll
      for (int q = 0; q < Q; ++q)   // past the last split: that split again, not added
#pragma unroll
        for (int u = 0; u < MC; ++u)
          v[u][q] = __builtin_bit_cast(
              float4_t, coherent_load16(ws_part, (uint32_t)(((group * S + min(s0 + q, S - 1)) * kUnits + wave +
                                                             u * 2 * P) * 1024 + lane * 16)));
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (s0 + q < S)
#pragma unroll
          for (int u = 0; u < MC; ++u) sum[u] = s0 + q == 0 ? v[u][q] : sum[u] + v[u][q];
    }
#pragma unroll
    for (int u = 0; u < MC; ++u) {
      const int unit = wave + u * 2 * P;
      mid_store<F>(sum[u], (unit % MC) * 16 + i, (group * P * NT + unit / MC) * 16 + 4 * kb, M, N, wmeta, bias, y);
    }
    if (threadIdx.x == 0) __hip_atomic_store(&ws_cnt[group], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The S partials of every unit, in split order.  One wave per unit, all of a
// lane's loads (up to six) in flight at once.
template <MFmt F, int P, int MC>
__global__ __launch_bounds__(256) void mid_sum_kernel(const float4_t* __restrict__ part, int S, int groups, int M, int N,
                                                      const void* __restrict__ wmeta, const half_t* __restrict__ bias,
                                                      half_t* __restrict__ y) {
  constexpr int kUnits = P * kMidTilesPerWave * MC;
  constexpr int Q = 5;   // partials after the first requested at once
  const int lane = threadIdx.x & 63, i = lane & 15, kb = lane >> 4;
  const int gu = blockIdx.x * 4 + (threadIdx.x >> 6);   // group * kUnits + unit
  if (gu >= groups * kUnits) return;   // the last workgroup's spare waves
  const int group = gu / kUnits, unit = gu % kUnits;
  const int m = (unit % MC) * 16 + i, n0 = (group * P * kMidTilesPerWave + unit / MC) * 16 + 4 * kb;
  if (m >= M || n0 >= N) return;
  const float4_t* q = part + ((size_t)group * S * kUnits + unit) * 64 + lane;
  float4_t s = q[0];
  for (int s0 = 1; s0 < S; s0 += Q) {
    float4_t v[Q];
#pragma unroll
    for (int j = 0; j < Q; ++j) v[j] = q[(size_t)min(s0 + j, S - 1) * kUnits * 64];   // past the last: not added
#pragma unroll
    for (int j = 0; j < Q; ++j)
      if (s0 + j < S) s += v[j];
  }
  mid_store<F>(s, m, n0, M, N, wmeta, bias, y);
}

// Tile groups and k splits (two-block stages) of a shape.
MidSplit mid_plan(bool w4, int64_t M, int64_t N, int64_t K) {
  const int mc = (int)((M + 15) / 16);
  return mid_split((N + 15) / 16, (K / kW4BlockK + 1) / 2, w4 ? 2 * (1024 + kW4MetaBytes) : 2 * kW8TileBlockBytes,
                   2 * mc * 16 * 256, 1, mc);
}

// Whether the last arriver sums (W4, mid_kernel's ws_cnt): 12 to 32 rows on up
// to 1152 tiles and k chains of 4 to 64 blocks (a multiple of four), the
// shapes whose workspace carried zeroed counters before this kernel.
bool mid_counts(bool w4, int64_t M, int64_t N, int64_t K) {
  const int64_t nblk = K / kW4BlockK;
  return w4 && M >= 12 && M <= 32 && (N + 15) / 16 <= 1152 && nblk <= 64 && nblk % 4 == 0;
}

// The shapes this file takes: those whose plan is estimated below the other
// kernels' time.  W4: the skinny kernels take rounds of 256 workgroups (two
// tiles a wave, four from 1024 tiles on) whose time is a chain of k blocks,
//   rounds x blocks x (0.034 + 0.108 per 16-row chunk + 0.006 per row) us
// and about twice that at four tiles; the constants are fitted so that the
// measured faster side wins, over k = 512..17408, N = 512..34816, M = 5..64
// (2700 points: the chosen side is 0.2 % off the faster one on average, 18 %
// at most; one threshold per row range was 7.9 % off, and 1.3 to 2 times on
// short narrow chains and at 33 to 35 rows).  Both sides, skinny against this
// file, us: 512->512 M = 16 3.3 / 4.9, 1024->2048 M = 36 5.8 / 8.0, 2048->6144
// M = 33 8.4 / 9.7; 2048->12288 M = 33 14.7 / 11.9, 5120->1024 M = 33 15.2 /
// 8.9, 5120->7168 M = 8 / 12 / 24 9.4 / 10.3 / 14.5 against 10.0 / 10.1 / 11.3,
// 5120->17408 M = 34 36.5 / 23.9, 17408->5120 M = 8 20.4 / 15.8.
// From 2048 tiles on and 17 rows the other side is the deep-ring GEMM: only
// chains of at least 32 blocks leave it (5120->34816 M = 24 / 56 37 / 50 ->
// 31 / 41 us).  Shorter ones would gain as well (2048->34816 M = 24 / 48 17.0 /
// 23.1 against 15.0 / 16.5) but keep the deep ring, whose rows equal those of a
// longer call bit for bit; the long chains' rows no longer do.
// INT8: the same with the INT8 skinny kernels' chain, one tile a wave up to 16
// rows and two above:
//   rounds x blocks x (0.124 + 0.0129 per row, from 17 rows 0.407 + 0.0094) us
// (0.07 % off the faster side on average, 10 % at most; the line on the weight's
// size and the chain before was 2.5 % off).  Skinny against this file, us:
// 5120->1024 M = 8 / 24 / 33 6.7 / 12.8 / 18.1 against 8.1 / 9.2 / 10.2, 512->2048
// M = 33 6.1 / 8.6, 1024->6144 M = 36 7.5 / 9.9, 5120->4040 M = 8 8.1 / 10.1,
// 2048->17408 M = 5 11.8 / 13.6, 5120->17408 M = 8 26.9 / 22.
// wq_batch.hip's shapes come off both (w4_batch_plan).
// Returns the plan, or one without groups for the other shapes; W4 only:
// best_us the estimated time of the faster of the two sides.
MidSplit mid_route(bool w4, int64_t M, int64_t N, int64_t K, double* best_us = nullptr) {
  constexpr MidSplit kNone{0, 0, 0};
  if (M <= 4 || M > 64 || K % kW4BlockK != 0 || K < kW4BlockK || K > kMidMaxK) return kNone;
  const int64_t ntile = (N + 15) / 16, nblk = K / kW4BlockK;
  if (!w4) {
    const int64_t rounds = ((M <= 16 ? ntile : (ntile + 1) / 2) + 255) / 256;
    const double chain = (double)(rounds * nblk) * (M <= 16 ? 0.124 + 0.0129 * (double)M : 0.407 + 0.0094 * (double)M);
    const double skinny = chain + 1.94 * (double)((M + 15) / 16) + (M <= 16 ? 0.86 : 0.0) - 9.4;
    if (skinny <= 0.0) return kNone;
    const MidSplit p = mid_plan(w4, M, N, K);
    return p.us + (p.s > 1 ? 1.0 : 0.0) < skinny ? p : kNone;
  }
  if (ntile >= 2048 && M > 16) return nblk >= 32 ? mid_plan(w4, M, N, K) : kNone;
  const double mc = (double)((M + 15) / 16);
  const bool four = ntile >= 1024;   // tiles per wave of the skinny kernels (pick_skinny)
  const int64_t rounds = ((ntile + (four ? 3 : 1)) / (four ? 4 : 2) + 255) / 256;
  const double skinny = (double)(rounds * nblk) * (0.034 + 0.108 * mc + 0.006 * (double)M + (four ? 0.038 + 0.098 * mc : 0.0)) - 2.4;
  if (best_us) *best_us = 4.2 + skinny;
  if (skinny <= -0.3) return kNone;   // whatever the plan
  const MidSplit p = mid_plan(w4, M, N, K);
  const double split = p.s <= 1 ? 0.0 : mid_counts(w4, M, N, K) ? -0.3 : 1.3;   // partial sums, in the same launch or a second
  if (best_us) {
    const double mid = p.us + (p.s > 1 ? 0.9 : 0.0);
    *best_us = 4.2 + (mid < skinny ? mid : skinny);
  }
  return p.us < skinny - split && (best_us || w4_batch_route(M, N, K).r == 0) ? p : kNone;
}

}  // namespace

W4BatchPlan w4_batch_route(int64_t m, int64_t n, int64_t k) {
  const W4BatchPlan p = w4_batch_plan(m, n, k);
  if (p.r == 0) return {};
  double other = 0;
  mid_route(true, m, n, k, &other);
  return p.us < other + 0.7 ? p : W4BatchPlan{};   // 0.7: where the fitted estimates cross on measured times
}

namespace {

size_t mid_route_bytes(const MidSplit& p, int64_t M) {
  return p.groups == 0 ? 0 : mid_partial_bytes(p, 1, (int)((M + 15) / 16));
}

template <MFmt F, int P, int MC, int D, int MINW>
int launch_mid(const half_t* x, int M, int K, const void* w, const void* meta, int N, int bpg, const half_t* bias,
               half_t* y, void* ws, const MidSplit& m, int tiled, hipStream_t st) {
  float4_t* part = m.s > 1 ? reinterpret_cast<float4_t*>(reinterpret_cast<uint8_t*>(ws) + kSplitCounterBytes) : nullptr;
  uint32_t* cnt = m.s > 1 && mid_counts(F == MFmt::W4, M, N, K) ? reinterpret_cast<uint32_t*>(ws) : nullptr;
  hipLaunchKernelGGL((mid_kernel<F, P, MC, D, MINW>), dim3((unsigned)m.groups, (unsigned)m.s), dim3(128 * P), 0, st, x,
                     M, K, w, meta, N, bpg, bias, y, part, cnt, tiled);
  if (m.s > 1 && cnt == nullptr)
    hipLaunchKernelGGL((mid_sum_kernel<F, P, MC>), dim3((unsigned)((m.groups * P * kMidTilesPerWave * MC + 3) / 4)),
                       dim3(256), 0, st, part, m.s, (int)m.groups, M, N, meta, bias, y);
  return check_launch(F == MFmt::W4 ? "w4_mid" : "w8_mid");
}

template <MFmt F, int P>
int launch_mid_p(const half_t* x, int M, int K, const void* w, const void* meta, int N, int bpg, const half_t* bias,
                 half_t* y, void* ws, const MidSplit& m, int tiled, hipStream_t st) {
  constexpr int kMin = P == 4 ? 4 : 3;   // waves per SIMD: two workgroups of eight waves, or one of ten
  switch ((M + 15) / 16) {
    case 1: return launch_mid<F, P, 1, 3, kMin>(x, M, K, w, meta, N, bpg, bias, y, ws, m, tiled, st);
    case 2: return launch_mid<F, P, 2, 3, kMin>(x, M, K, w, meta, N, bpg, bias, y, ws, m, tiled, st);
    case 3: return launch_mid<F, P, 3, F == MFmt::W4 ? 2 : 3, kMin>(x, M, K, w, meta, N, bpg, bias, y, ws, m, tiled, st);
    default: return launch_mid<F, P, 4, 2, P == 4 ? 2 : 3>(x, M, K, w, meta, N, bpg, bias, y, ws, m, tiled, st);
  }
}

// Returns -1 (not taken) when the shape is not this file's or its splits need
// more workspace than given; the caller then runs the skinny kernels.
template <MFmt F>
int launch_mid_auto(const half_t* x, int M, int K, const void* w, const void* meta, int N, int bpg, const half_t* bias,
                    half_t* y, void* ws, size_t ws_bytes, int tiled, hipStream_t st) {
  const MidSplit m = mid_route(F == MFmt::W4, M, N, K);
  if (m.groups == 0) return -1;
  const size_t need = mid_route_bytes(m, M);
  if (need > 0 && (ws == nullptr || ws_bytes < need)) return -1;
  return m.p == 4 ? launch_mid_p<F, 4>(x, M, K, w, meta, N, bpg, bias, y, ws, m, tiled, st)
                  : launch_mid_p<F, 5>(x, M, K, w, meta, N, bpg, bias, y, ws, m, tiled, st);
}

}  // namespace

// Writes the plan of a shape this file takes; false otherwise.
bool mid_plan_text(bool w4, int64_t m, int64_t n, int64_t k, char* text, size_t bytes) {
  const MidSplit p = mid_route(w4, m, n, k);
  if (p.groups > 0) snprintf(text, bytes, "mid %dx%d", p.p, p.s);
  return p.groups > 0;
}

// Whether a W4 shape's workspace carries arrival counters.
bool w4_mid_has_counters(int64_t m, int64_t n, int64_t k) {
  return mid_route(true, m, n, k).s > 1 && mid_counts(true, m, n, k);
}

size_t w4_mid_workspace_bytes(int64_t m, int64_t n, int64_t k) { return mid_route_bytes(mid_route(true, m, n, k), m); }
size_t w8_mid_workspace_bytes(int64_t m, int64_t n, int64_t k) { return mid_route_bytes(mid_route(false, m, n, k), m); }

int launch_w4_mid(const half_t* x, int M, int K, const uint4_t* tiles, const uint8_t* meta, int N, int G, half_t* y,
                  void* ws, size_t ws_bytes, hipStream_t st) {
  return launch_mid_auto<MFmt::W4>(x, M, K, tiles, meta, N, G / kW4BlockK, nullptr, y, ws, ws_bytes, 0, st);
}

int launch_w8_mid(const half_t* x, int M, int K, const int8_t* q, const half_t* scale, const half_t* bias, int N,
                  half_t* y, void* ws, size_t ws_bytes, hipStream_t st, int tiled) {
  return launch_mid_auto<MFmt::W8>(x, M, K, q, scale, N, 1, bias, y, ws, ws_bytes, tiled, st);
}

}  // namespace wq
