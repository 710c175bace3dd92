// W8A8: dynamic per-token symmetric INT8 activations times per-output-channel
// INT8 weights, accumulated exactly in int32 on the int8 matrix cores
// (v_mfma_i32_16x16x64_i8) and scaled once per output in fp32.
//
// Fragment convention of v_mfma_i32_16x16x64_i8: lane l supplies 16 bytes of
// A row l%16 and 16 bytes of B column l%16 taken from k-slot l/16; A and B
// use the same (lane, byte) -> k map, which is all the dot product needs, so
// both are loaded as 16 consecutive bytes at k = 64s + 16(l/16).  The
// accumulator lane l holds D[row = 4(l/16) + v][column = l%16].  Weights are
// the A operand (rows n), activations the B operand (columns m).
#include "ondeviceinfer_wq.h"
#include "wq_common.h"
#include "wq_mid_plan.h"
#include "wq_status.h"

#include <math.h>
#include <type_traits>

namespace wq {
namespace {

typedef int32_t int4v_t __attribute__((ext_vector_type(4)));

constexpr int kI8Step = 64;   // k per int8 MFMA

__device__ __forceinline__ int4v_t mfma_i8(uint4_t a, uint4_t b, int4v_t c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(int4v_t, a), __builtin_bit_cast(int4v_t, b), c, 0,
                                               0, 0);
}

__device__ __forceinline__ float wave_max_abs(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}

// clamp(rint(v / s), -127, 127) of eight values, packed; rs = RN(1 / s).  The
// quotient of one row's values by one s: Markstein's correction of v * rs
// (IBM J. Res. Dev. 34, 1990), a remainder by fma and a corrected quotient,
// applied twice, which rounds like the IEEE divide (the first leaves a
// faithful quotient, the second the nearest) in five operations a value
// instead of the divide's dozen.  v and s are normal or v is zero, |v| <= 127 s,
// so no step over- or underflows.  MARKSTEIN = false is the plain divide.
template <bool MARKSTEIN>
__device__ __forceinline__ uint2_t w8a8_codes8(half8_t v, float s, float rs) {
  uint32_t w[2] = {0u, 0u};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float a = (float)v[e];
    float d;
    if constexpr (MARKSTEIN) {
      d = a * rs;
      d = __builtin_fmaf(__builtin_fmaf(-d, s, a), rs, d);
      d = __builtin_fmaf(__builtin_fmaf(-d, s, a), rs, d);
    } else {
      d = a / s;
    }
    const float r = fminf(fmaxf(rintf(d), -127.0f), 127.0f);
    w[e >> 2] |= (uint32_t)(uint8_t)(int8_t)(int)r << (8 * (e & 3));
  }
  return uint2_t{w[0], w[1]};
}

// One workgroup of T threads per row of x [M, K] (K % 8 == 0): absmax in
// fp32, scale = max(absmax, 1e-12) / 127, q = clamp(rint(x / scale), -127, 127)
// with the IEEE quotient and round-half-even, as the reference's W8A8 oracle
// (backend.py:258-261).  With C > 0 the row (at most C chunks of 8 per thread)
// stays in registers between the two steps; C == 0 reads it again (longer
// rows).  Bound: at 2048 rows of 5120 by issue (the divide), at few rows by
// the chain load -> reduce -> store, hence 1024 threads per row there.
template <int T, int C>
__global__ __launch_bounds__(T) void w8a8_quantize_kernel(const half_t* __restrict__ x, int K, int8_t* __restrict__ q,
                                                          float* __restrict__ scale) {
  __shared__ float part[T / 64];
  const size_t base = (size_t)blockIdx.x * K;
  const int nc = K >> 3;
  half8_t v[C > 0 ? C : 1];
  float mx = 0.f;
  auto absmax = [&](half8_t h) {
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf((float)h[e]));
  };
  if constexpr (C > 0) {
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int c = threadIdx.x + j * T;
      v[j] = c < nc ? ld_h8(x + base + 8 * c) : half8_t{};
    }
#pragma unroll
    for (int j = 0; j < C; ++j) absmax(v[j]);
  } else {
    for (int c = threadIdx.x; c < nc; c += T) absmax(ld_h8(x + base + 8 * c));
  }
  mx = wave_max_abs(mx);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < T / 64; ++w) mx = fmaxf(mx, part[w]);
  const float s = fmaxf(mx, 1e-12f) / 127.0f;
  if (threadIdx.x == 0) scale[blockIdx.x] = s;
  const float rs = 1.0f / s;
  const bool finite = s < __builtin_inff();   // an infinite row: the plain divide's 0 and NaN
  auto put = [&](int c, half8_t h) {
    *reinterpret_cast<uint2_t*>(q + base + 8 * c) = finite ? w8a8_codes8<true>(h, s, rs) : w8a8_codes8<false>(h, s, rs);
  };
  if constexpr (C > 0) {
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int c = threadIdx.x + j * T;
      if (c < nc) put(c, v[j]);
    }
  } else {
    for (int c = threadIdx.x; c < nc; c += T) put(c, ld_h8(x + base + 8 * c));
  }
}

// y = fp16(float(acc) * sx[m] * sw[n] (+ bias[n])), the scaling of the
// int32 sum in that order, each operation rounded on its own (no fma).
__device__ __forceinline__ void w8a8_store(int32_t acc, int m, int n, const float* __restrict__ sx,
                                           const float* __restrict__ sw, const half_t* __restrict__ bias, int N,
                                           half_t* __restrict__ y) {
#pragma clang fp contract(off)
  float r = (float)acc * sx[m] * sw[n];
  if (bias) r += (float)bias[n];
  y[(size_t)m * N + n] = (half_t)r;
}

// Decode (M <= 16): grid = 16-row tiles of the weight, 64*ksw threads.  The
// tile's K/64 steps are split evenly over the ksw waves; a wave requests
// eight steps' weight fragments (non-temporal, 16 B per lane) and x
// fragments (row min(l%16, M-1)) at once, then issues eight MFMAs (a step
// past its range repeats the last one and is skipped).  The waves' int32
// sums meet in LDS (exact, order-free); wave 0 scales and stores.
__global__ __launch_bounds__(1024) void w8a8_gemv_kernel(const int8_t* __restrict__ qx, const float* __restrict__ sx,
                                                         int M, int K, const int8_t* __restrict__ qw,
                                                         const float* __restrict__ sw, const half_t* __restrict__ bias,
                                                         int N, half_t* __restrict__ y, W8Layout wl8) {
  __shared__ int4v_t red[16][64];
  const int ksw = blockDim.x >> 6, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int i = lane & 15, kb = lane >> 4;
  const int tile = blockIdx.x;
  const int nsteps = K / kI8Step;
  const int s_lo = (wave * nsteps) / ksw, s_hi = ((wave + 1) * nsteps) / ksw;
  const int8_t* wp = qw + wl8.lane_base(tile, lane, N, K);
  const int8_t* xp = qx + (size_t)min(i, M - 1) * K + 16 * kb;
  const int blk_bytes = wl8.block_bytes(), p1 = wl8.piece1();
  int4v_t acc = {0, 0, 0, 0};
  for (int s0 = s_lo; s0 < s_hi; s0 += 8) {
    uint4_t a[8], b[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int st = min(s0 + j, s_hi - 1);   // 64-k step: block st / 2, piece st % 2
      a[j] = __builtin_nontemporal_load(
          reinterpret_cast<const uint4_t*>(wp + (size_t)(st >> 1) * blk_bytes + (st & 1) * p1));
      b[j] = *reinterpret_cast<const uint4_t*>(xp + (size_t)kI8Step * st);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s0 + j < s_hi) acc = mfma_i8(a[j], b[j], acc);
  }
  red[wave][lane] = acc;
  __syncthreads();
  if (wave != 0) return;
  int4v_t sum = red[0][lane];
  for (int w2 = 1; w2 < ksw; ++w2) sum += red[w2][lane];
  if (i < M) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int n = tile * 16 + 4 * kb + v;
      if (n < N) w8a8_store(sum[v], i, n, sx, sw, bias, N, y);
    }
  }
}

// LDS slot of 16-byte chunk c (0..7) in row r of a 128-byte stage row: rows
// 2 apart share banks, so the slot is permuted by r / 2; the sixteen rows a
// B-fragment read touches then hit sixteen distinct 16-byte bank groups.
__device__ __forceinline__ int i8_swz(int r, int c) { return c ^ ((r >> 1) & 7); }

constexpr int kI8Blk = 128;              // k per GEMM stage (two int8 MFMA steps)
constexpr int kI8RowBytes = kI8Blk;      // one int8 x row per stage

// The MT B-fragments of one 64-k step, fragment mt from row mt*16 + i of the
// stage: a per-lane address plus the immediate mt * 16 rows.  Inline asm,
// as in the W4 GEMM: a read the compiler can see makes it wait for every
// outstanding buffer -> LDS copy (vmcnt(0)) first, the next stage's included,
// which serializes the copies with the math; these reads are completed by
// lds_wait_frags.
template <int OFF>
__device__ __forceinline__ uint4_t i8_lds_read_off(uint32_t a) {
  uint4_t v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "i"(OFF));
  return v;
}
template <int MT, int MTI = 0>
__device__ __forceinline__ void i8_read_frags(uint4_t (&b)[MT], uint32_t a) {
  if constexpr (MTI < MT) {
    b[MTI] = i8_lds_read_off<MTI * 16 * kI8RowBytes>(a);
    i8_read_frags<MT, MTI + 1>(b, a);
  }
}

// M > 16: grid = (ceil(tiles / (4 NT)), ceil(M / BM)), 256 threads, BM = 16 MT.
// Wave w owns the NT 16-row weight tiles (4 bx + w) NT .. +NT-1 (disjoint
// between waves); all four share the BM x rows of the workgroup.  Per 128-k
// stage the x tile goes global -> LDS with global_load_lds_dwordx4 into a
// two-stage ring (row r's chunk c at slot i8_swz(r, c)); each wave's weight
// fragments come straight from memory into registers one stage ahead.  Per
// 64-k step a wave reads MT x fragments from LDS and issues NT x MT int8
// MFMAs.  Two workgroups per CU (the accumulators then live in VGPRs, not
// AGPRs: 236 registers, no scratch), so one workgroup's load wait overlaps
// the other's math: 1.4-1.8x the throughput of one per CU.  K % 128 == 0.
template <int NT, int MT>
__global__ __launch_bounds__(256, 2) void w8a8_gemm_kernel(const int8_t* __restrict__ qx,
                                                           const float* __restrict__ sx, int M, int K,
                                                           const int8_t* __restrict__ qw,
                                                           const float* __restrict__ sw,
                                                           const half_t* __restrict__ bias, int N,
                                                           half_t* __restrict__ y, W8Layout wl8) {
  constexpr int BM = MT * 16;
  constexpr int kStageBytes = BM * kI8RowBytes;
  constexpr int kInstrPerWave = kStageBytes / 1024 / 4;   // 1 KiB per wave-wide DMA instruction
  static_assert(kInstrPerWave >= 1, "stage too small for four waves");
  __shared__ __attribute__((aligned(1024))) uint8_t xs[2 * kStageBytes];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, kb = lane >> 4;
  const int ntile = (N + 15) >> 4;
  const int nblk = K / kI8Blk;
  const int m0 = blockIdx.y * BM;
  const int tile0 = ((int)blockIdx.x * 4 + wave) * NT;
  // Every load goes through a buffer resource with a wave-uniform base and
  // 32-bit offsets (K <= 2^23, checked by the host): rows past M and tiles
  // past N fall outside the buffers and read as zero (never stored).  With
  // plain global loads of the weights the compiler put a vmcnt(0) before
  // each block's first MFMA, waiting for the next block's loads as well.
  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(qx + (size_t)m0 * K, (int64_t)(M - m0) * K);
  const __amdgpu_buffer_rsrc_t rw =
      wl8.tiled ? buf_rsrc(qw + (size_t)tile0 * nblk * kW8TileBlockBytes, (int64_t)(ntile - tile0) * nblk * kW8TileBlockBytes)
                : buf_rsrc(qw + (size_t)tile0 * 16 * K, (int64_t)(N - tile0 * 16) * K);
  const uint32_t w_voff = wl8.tiled ? (uint32_t)lane * 16 : (uint32_t)(i * K + 16 * kb);
  const uint32_t w_p1 = (uint32_t)wl8.piece1();

  // Stage `st` <- x rows m0 .. m0+BM-1, k block `blk`: instruction J of the
  // workgroup fills bytes [1024 J, 1024 J + 1024), i.e. rows 8J .. 8J+7;
  // lane L lands in row 8J + L/8, slot L%8, so it fetches chunk
  // i8_swz(row, L%8) of that row.
  auto copy_x = [&](int blk, int st) {
#pragma unroll
    for (int j = 0; j < kInstrPerWave; ++j) {
      const int J = wave * kInstrPerWave + j;
      const int r = 8 * J + (lane >> 3);
      const int c = i8_swz(r, lane & 7);
      lds_load16(rx, (uint32_t)(r * K + 16 * c), (uint32_t)(blk * kI8Blk), xs + st * kStageBytes + J * 1024);
    }
  };
  auto fetch_w = [&](int blk, uint4_t (&r)[NT][2]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const uint32_t so = wl8.tiled ? (uint32_t)((t * nblk + blk) * kW8TileBlockBytes)
                                    : (uint32_t)(t * 16 * K + blk * kI8Blk);
      r[t][0] = __builtin_amdgcn_raw_buffer_load_b128(rw, w_voff, so, 0);          // k + 16 kb .. +15
      r[t][1] = __builtin_amdgcn_raw_buffer_load_b128(rw, w_voff + w_p1, so, 0);   // k + 64 + 16 kb .. +15
    }
  };

  int4v_t acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = int4v_t{0, 0, 0, 0};

  const uint32_t xs_lds = (uint32_t)(size_t)((const __attribute__((address_space(3))) uint8_t*)xs);
  // The one-tile path's block math: two 64-k MFMA steps of stage `st` with
  // the weight registers w (the same steps as the loop of the wider grids).
  auto block_math = [&](int st, const uint4_t (&w)[NT][2]) {
    // Row r = mt*16 + i of the stage holds chunk c at slot i8_swz(r, c) =
    // c ^ ((i >> 1) & 7): one lane address per step, mt in the offset.
    const uint32_t stage = xs_lds + (uint32_t)(st * kStageBytes + i * kI8RowBytes);
#pragma unroll
    for (int step = 0; step < 2; ++step) {
      const int c = 4 * step + kb;   // 16-byte chunk of this lane's k range
      uint4_t b[MT];
      i8_read_frags<MT>(b, stage + (uint32_t)(i8_swz(i, c) * 16));
      lds_wait_frags<MT, 0, MT / 2, MT - MT / 2>(b);
#pragma unroll
      for (int mt = 0; mt < MT / 2; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t][mt] = mfma_i8(w[t][step], b[mt], acc[t][mt]);
      lds_wait_frags<MT, MT / 2, MT, 0>(b);
#pragma unroll
      for (int mt = MT / 2; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t][mt] = mfma_i8(w[t][step], b[mt], acc[t][mt]);
    }
  };
  if constexpr (NT == 1) {
    // One weight tile per wave (grids of at most one round of workgroups):
    // the loop is unrolled by two over two fixed register sets, every step
    // issues its loads (the block after the last reads nothing: a
    // past-the-end offset), and the per-block wait covers only the x copy,
    // issued before the weights, so the next block's weights may still be in
    // flight across the barrier (M = 512, same box, same bits: 17408->5120
    // 116.7 -> 84.1 us, 5120^2 38.8 -> 33.7 us; M = 4096 k_proj 43.0 ->
    // 40.2 us).  The larger grids keep the loop below: this form cost them
    // 1-2 %.
    constexpr uint32_t kPastEnd = 0x80000000u;
    constexpr int kWLoads = 2 * NT;   // weight loads per block per wave
    uint4_t wr[2][NT][2];
    copy_x(0, 0);
    fetch_w(0, wr[0]);
    __builtin_amdgcn_s_waitcnt(0);   // stage 0 landed
    __syncthreads();
    int base = 0;
    do {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int blk = base + u;
#pragma unroll
        for (int j = 0; j < kInstrPerWave; ++j) {   // copy_x(blk + 1, u ^ 1), empty past the end
          const int J = wave * kInstrPerWave + j;
          const int r = 8 * J + (lane >> 3);
          lds_load16(rx, (uint32_t)(r * K + 16 * i8_swz(r, lane & 7)),
                     blk + 1 < nblk ? (uint32_t)((blk + 1) * kI8Blk) : kPastEnd, xs + (u ^ 1) * kStageBytes + J * 1024);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {               // fetch_w(blk + 1, wr[u ^ 1]), empty past the end
          const uint32_t so = blk + 1 >= nblk ? kPastEnd
                              : wl8.tiled ? (uint32_t)((t * nblk + blk + 1) * kW8TileBlockBytes)
                                          : (uint32_t)(t * 16 * K + (blk + 1) * kI8Blk);
          wr[u ^ 1][t][0] = __builtin_amdgcn_raw_buffer_load_b128(rw, w_voff, so, 0);
          wr[u ^ 1][t][1] = __builtin_amdgcn_raw_buffer_load_b128(rw, w_voff + w_p1, so, 0);
        }
        __builtin_amdgcn_sched_barrier(0);   // keep the loads in this order: the wait below counts them
        if (blk < nblk) block_math(u, wr[u]);
        __builtin_amdgcn_s_waitcnt((kWLoads & 0xF) | ((kWLoads >> 4) << 14) | (0x7 << 4) | (0xF << 8));
        __builtin_amdgcn_s_barrier();   // every wave's part of stage u ^ 1 landed
      }
      base += 2;
    } while (base < nblk);
    __builtin_amdgcn_s_waitcnt(0);   // the run-out block's empty loads, before the stores
  } else {
    uint4_t cur[NT][2], nxt[NT][2];
    copy_x(0, 0);
    fetch_w(0, cur);
    __builtin_amdgcn_s_waitcnt(0);   // stage 0 landed
    __syncthreads();
    for (int blk = 0; blk < nblk; ++blk) {
      const int st = blk & 1;
      const bool more = blk + 1 < nblk;
      if (more) {
        copy_x(blk + 1, st ^ 1);
        fetch_w(blk + 1, nxt);
      }
      // Row r = mt*16 + i of the stage holds chunk c at slot i8_swz(r, c) =
      // c ^ ((i >> 1) & 7): one lane address per step, mt in the offset.
      const uint32_t stage = xs_lds + (uint32_t)(st * kStageBytes + i * kI8RowBytes);
#pragma unroll
      for (int step = 0; step < 2; ++step) {
        const int c = 4 * step + kb;   // 16-byte chunk of this lane's k range
        uint4_t b[MT];
        i8_read_frags<MT>(b, stage + (uint32_t)(i8_swz(i, c) * 16));
        lds_wait_frags<MT, 0, MT / 2, MT - MT / 2>(b);
#pragma unroll
        for (int mt = 0; mt < MT / 2; ++mt)
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[t][mt] = mfma_i8(cur[t][step], b[mt], acc[t][mt]);
        lds_wait_frags<MT, MT / 2, MT, 0>(b);
#pragma unroll
        for (int mt = MT / 2; mt < MT; ++mt)
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[t][mt] = mfma_i8(cur[t][step], b[mt], acc[t][mt]);
      }
      if (more) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          cur[t][0] = nxt[t][0];
          cur[t][1] = nxt[t][1];
        }
      }
      __builtin_amdgcn_s_waitcnt(0);   // this wave's part of the next stage landed
      __syncthreads();                  // ... and everyone's; stage st may be overwritten next
    }
  }

#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (tile0 + t >= ntile) continue;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = m0 + mt * 16 + i;
      if (m >= M) continue;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int n = (tile0 + t) * 16 + 4 * kb + v;
        if (n < N) w8a8_store(acc[t][mt][v], m, n, sx, sw, bias, N, y);
      }
    }
  }
}

// Batches of 5 to 255 rows: the activation tile of a workgroup shared in LDS
// and the k range split over workgroups, as the fp16 kernel of 5 to 64 rows
// (wq_mid.hip), on the int8 matrix cores.
//
// Bound: the weight stream, at the rate a compute unit takes bytes in
// (wq_mid_plan.h).  The GEMM below takes 32-row tiles at these M, so it reads
// the weights once per 32 rows with one 128-k block in flight; here a workgroup
// covers up to 128 rows (MC chunks of 16) of its 2 P 16-row weight tiles.  Its
// 2 P waves (p, h) take the tile pair p and two of the four 128-k blocks of a
// stage (h), weights straight into registers and x buffer -> LDS D - 1 stages
// ahead; the two halves meet in LDS, S > 1 k ranges through int32 partials that
// a second launch adds and scales.  The sums are exact integers, so every plan
// gives the same bits.
// MI355X, graphs of distinct weights, us without the quantizer, GEMV or 32-row
// GEMM -> this kernel:
//   17408->5120  M = 8 / 24 / 56 / 96 / 200   31.3 / 52.9 / 53.2 / 53.8 / 60.7 -> 20.5 / 21.5 / 24.3 / 28.3 / 42.0
//   5120->17408  M = 8 / 24 / 56              23.6 / 26.8 / 31.7 -> 21.6 / 22.4 / 27.3
//   5120->34816  M = 8 / 24 / 56              42.9 / 41.5 / 63.6 -> 35.0 / 36.8 / 41.3
//   5120->5120   M = 16 / 56 / 96             12.7 / 18.5 / 18.5 -> 11.1 / 15.9 / 16.1
// i.e. 178 MB of weights at M = 8 in 35 us (5.1 TB/s).
constexpr int kM8Tiles = kMidTilesPerWave;
constexpr int kM8MaxM = 255;   // from 256 rows the GEMM takes 128-row tiles
constexpr int kM8GemvMaxM = 16;

// The MC fragments of one k-step (16 rows apart in a stage), read and waited
// for in one asm block (see i8_lds_read_off for why asm).
template <int MC>
__device__ __forceinline__ void m8_read(uint4_t (&f)[MC], uint32_t a) {
  if constexpr (MC == 1)
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(f[0]) : "v"(a));
  else if constexpr (MC == 2)
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:2048\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(f[0]), "=&v"(f[1]) : "v"(a));
  else if constexpr (MC == 3)
    asm volatile("ds_read_b128 %0, %3\n\tds_read_b128 %1, %3 offset:2048\n\tds_read_b128 %2, %3 offset:4096\n\t"
                 "s_waitcnt lgkmcnt(0)" : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]) : "v"(a));
  else if constexpr (MC == 4)
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:2048\n\tds_read_b128 %2, %4 offset:4096\n\t"
                 "ds_read_b128 %3, %4 offset:6144\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]) : "v"(a));
  else if constexpr (MC == 6)
    asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %6 offset:2048\n\tds_read_b128 %2, %6 offset:4096\n\t"
                 "ds_read_b128 %3, %6 offset:6144\n\tds_read_b128 %4, %6 offset:8192\n\tds_read_b128 %5, %6 offset:10240\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(f[4]), "=&v"(f[5]) : "v"(a));
  else
    asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:2048\n\tds_read_b128 %2, %8 offset:4096\n\t"
                 "ds_read_b128 %3, %8 offset:6144\n\tds_read_b128 %4, %8 offset:8192\n\tds_read_b128 %5, %8 offset:10240\n\t"
                 "ds_read_b128 %6, %8 offset:12288\n\tds_read_b128 %7, %8 offset:14336\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(f[4]), "=&v"(f[5]), "=&v"(f[6]), "=&v"(f[7])
                 : "v"(a));
}

// As w8a8_store, the four columns n0 .. n0 + 3 at once where row m keeps
// 8-byte alignment.
__device__ __forceinline__ void m8_store(int4v_t s, int m, int n0, int M, int N, const float* __restrict__ sx,
                                         const float* __restrict__ sw, const half_t* __restrict__ bias,
                                         half_t* __restrict__ y) {
#pragma clang fp contract(off)
  if (m >= M || n0 >= N) return;
  half4_t o;
  const float xs = sx[m];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int n = min(n0 + v, N - 1);
    float r = (float)s[v] * xs * sw[n];
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

template <int P, int MC, int D>
__global__ __launch_bounds__(128 * P, P == 4 ? 2 : 3) void w8a8_mid_kernel(
    const int8_t* __restrict__ qx, const float* __restrict__ sx, int M, int K, const int8_t* __restrict__ qw,
    const float* __restrict__ sw, const half_t* __restrict__ bias, int N, half_t* __restrict__ y, int4v_t* ws_part,
    W8Layout wl8) {
  constexpr int NT = kM8Tiles;
  constexpr int kSubBytes = MC * 16 * kI8RowBytes;   // x of one 128-k block
  constexpr int kStageBytes = 4 * kSubBytes;
  constexpr int kUnits = P * NT * MC;
  static_assert(kUnits * 1024 <= D * kStageBytes && (D - 2) * (MC + 4 * NT) <= 63, "ring");
  __shared__ __attribute__((aligned(1024))) uint8_t xs[D * kStageBytes];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = wave >= P ? 1 : 0, p = wave - h * P;
  const int i = lane & 15, kb = lane >> 4;
  const int ntile = (N + 15) >> 4, nblk = K / kI8Blk, nst = (nblk + 3) >> 2;
  const int group = blockIdx.x, split = blockIdx.y, S = gridDim.y;
  const int st_lo = (split * nst) / S, nloc = ((split + 1) * nst) / S - st_lo;
  const int tile0 = (group * P + p) * NT;
  const int m0 = blockIdx.z * (MC * 16);
  constexpr uint32_t kPastEnd = 0x80000000u;

  // A stage is four 128-k blocks, 2h and 2h + 1 this wave's.  x instruction
  // J = p MC + j of the parity's 4 MC: block J / (2 MC), rows 8 (J % (2 MC)) ..
  uint32_t xvo[MC];
#pragma unroll
  for (int j = 0; j < MC; ++j) {
    const int J = p * MC + j, sub = J / (2 * MC), rr = 8 * (J % (2 * MC)) + (lane >> 3);
    xvo[j] = (uint32_t)(rr * K + 16 * i8_swz(rr, lane & 7) + sub * kI8Blk);
  }
  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(qx + (size_t)m0 * K, (int64_t)(M - m0) * K);
  const __amdgpu_buffer_rsrc_t rw =
      wl8.tiled ? buf_rsrc(qw + (size_t)tile0 * nblk * kW8TileBlockBytes, (int64_t)(ntile - tile0) * nblk * kW8TileBlockBytes)
                : buf_rsrc(qw + (size_t)tile0 * 16 * K, (int64_t)(N - tile0 * 16) * K);
  const uint32_t wvo = wl8.tiled ? (uint32_t)lane * 16 : (uint32_t)(i * K + 16 * kb);
  const uint32_t wstep = (uint32_t)wl8.block_bytes(), p1 = (uint32_t)wl8.piece1();
  const uint32_t wtile = wl8.tiled ? (uint32_t)nblk * kW8TileBlockBytes : (uint32_t)(16 * K);
  int nx = 4 * st_lo + 2 * h;
  const int nx_end = min(4 * (st_lo + nloc), nblk);
  struct Regs { uint4_t w[2][NT][2]; };
  auto fetch = [&](int st, Regs& r) {
    // x of a block past the range: the second block of an odd tail reads the
    // next row's bytes (or past the buffer) and meets zero weights.
    const uint32_t xo = nx < nx_end ? (uint32_t)nx * kI8Blk : kPastEnd;
    if (P == 4 || p < 4) {   // four of the P waves of a half copy its x
#pragma unroll
      for (int j = 0; j < MC; ++j)
        lds_load16(rx, xvo[j], xo, xs + st * kStageBytes + h * 2 * kSubBytes + (p * MC + j) * 1024);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint32_t wo = nx + b < nx_end ? (uint32_t)(nx + b) * wstep : kPastEnd;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        r.w[b][t][0] = __builtin_amdgcn_raw_buffer_load_b128(rw, wvo, wo + t * wtile, kNtPolicy);
        r.w[b][t][1] = __builtin_amdgcn_raw_buffer_load_b128(rw, wvo + p1, wo + t * wtile, kNtPolicy);
      }
    }
    nx += 4;
  };
  int4v_t acc[NT][MC];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mc = 0; mc < MC; ++mc) acc[t][mc] = int4v_t{0, 0, 0, 0};
  const uint32_t xs_base = (uint32_t)(size_t)((const __attribute__((address_space(3))) uint8_t*)xs) +
                           (uint32_t)(h * 2 * kSubBytes + i * kI8RowBytes);
  auto stage_math = [&](int st, const Regs& r) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int step = 0; step < 2; ++step) {
        uint4_t f[MC];
        m8_read<MC>(f, xs_base + (uint32_t)(st * kStageBytes + b * kSubBytes + i8_swz(i, 4 * step + kb) * 16));
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int mc = 0; mc < MC; ++mc) acc[t][mc] = mfma_i8(r.w[b][t][step], f[mc], acc[t][mc]);
      }
  };
  Regs wr[D];
#pragma unroll
  for (int j = 0; j < D - 1; ++j) {
    fetch(j, wr[j]);
    __builtin_amdgcn_sched_barrier(0);
  }
  auto wait = [&]() {
    constexpr int W = (D - 2) * (MC + 4 * NT), W2 = (D - 2) * 4 * NT;
    if (P == 4 || p < 4) __builtin_amdgcn_s_waitcnt((W & 0xF) | ((W >> 4) << 14) | (0x7 << 4) | (0xF << 8));
    else __builtin_amdgcn_s_waitcnt((W2 & 0xF) | ((W2 >> 4) << 14) | (0x7 << 4) | (0xF << 8));
    __builtin_amdgcn_s_barrier();
  };
  wait();   // stage 0 landed (this wave's part, then everyone's)
  int base = 0;
  do {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      fetch((u + D - 1) % D, wr[(u + D - 1) % D]);
      __builtin_amdgcn_sched_barrier(0);
      if (base + u < nloc) stage_math(u, wr[u]);
      wait();
    }
    base += D;
  } while (base < nloc);
  __builtin_amdgcn_s_waitcnt(0);   // the run-out's empty copies
  __builtin_amdgcn_s_barrier();    // ... everyone's: the ring is dead
  int4v_t* red = reinterpret_cast<int4v_t*>(xs);
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
        const int4v_t s = acc[t][mc] + red[unit * 64 + lane];
        if (S == 1) m8_store(s, m0 + mc * 16 + i, (tile0 + t) * 16 + 4 * kb, M, N, sx, sw, bias, y);
        else coherent_store16(ws_part, (uint32_t)((((blockIdx.z * gridDim.x + group) * S + split) * kUnits + unit) * 1024 + lane * 16),
                              __builtin_bit_cast(uint4_t, s));
      }
  }
}

// The S partials of every unit, one wave per unit, then the scaling.
template <int P, int MC>
__global__ __launch_bounds__(256) void w8a8_mid_sum_kernel(const int4v_t* __restrict__ part, int S, int groups, int nz, int M, int N,
                                                           const float* __restrict__ sx, const float* __restrict__ sw,
                                                           const half_t* __restrict__ bias, half_t* __restrict__ y) {
  constexpr int kUnits = P * kM8Tiles * MC, Q = 5;
  const int lane = threadIdx.x & 63, i = lane & 15, kb = lane >> 4;
  const int gu = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (gu >= nz * groups * kUnits) return;   // the last workgroup's spare waves
  const int zg = gu / kUnits, unit = gu % kUnits, group = zg % groups;
  const int m = (zg / groups) * (MC * 16) + (unit % MC) * 16 + i, n0 = (group * P * kM8Tiles + unit / MC) * 16 + 4 * kb;
  if (m >= M || n0 >= N) return;
  const int4v_t* q = part + ((size_t)zg * S * kUnits + unit) * 64 + lane;
  int4v_t s = q[0];
  for (int s0 = 1; s0 < S; s0 += Q) {
    int4v_t v[Q];
#pragma unroll
    for (int j = 0; j < Q; ++j) v[j] = q[(size_t)min(s0 + j, S - 1) * kUnits * 64];
#pragma unroll
    for (int j = 0; j < Q; ++j)
      if (s0 + j < S) s += v[j];
  }
  m8_store(s, m, n0, M, N, sx, sw, bias, y);
}

struct M8Plan {
  int mc, nz, d;   // 16-row chunks, row blocks, ring depth; mc == 0: not taken
  MidSplit m;
  size_t bytes() const { return mid_partial_bytes(m, nz, mc); }
};

// What the GEMV (up to 16 rows) or the GEMM on 32-row tiles below would take
// beside this kernel, us above this kernel's constant part.  GEMV: one round of
// loads per chain, rounds of 256 workgroups (one per tile), and x read by every
// tile; GEMM: a chain of k blocks whose cost grows with the workgroups, at one
// or four tiles a wave (w8a8_route).  Constants fitted so that the measured
// faster side wins, over k = 512..17408, N = 512..34816, M = 5..255 (4000
// points: 0.35 % off the faster side on average, 10 % at most on the projection
// shapes of 5120 and 17408; five thresholds on M, the chain and the tiles were
// 1.4 % off).
double m8_other_us(int64_t M, int64_t ntile, int64_t nblk, int mc) {
  const double b = (double)nblk;
  if (M <= kM8GemvMaxM)
    return b * (0.048 + 0.087 * (double)((ntile + 255) / 256) + 0.114 * (double)(ntile * M) / (320.0 * 16)) - 4.3;
  const int64_t mblocks = (M + 31) / 32, wide = (ntile + 15) / 16 * mblocks;
  const double x = 0.31 * mc / 8;   // this kernel's row chunks
  if (wide >= 256) return b * (1.024 + 0.576 * (double)((wide + 255) / 256) - x) - 4.3;
  return b * (0.544 + 0.224 * (double)((ntile + 3) / 4 * mblocks) / 256 - x) - 4.3;
}

// Taken where the plan is estimated below the others (with the quantizer left
// out, us, others against this kernel: N = 1024 M = 8 5.9 / 8.8; 5120^2 M = 8 / 16
// 10.5 / 11.1, 13.1 / 11.2; 2048->4040 M = 16 5.2 / 9.1; 3328->13000 M = 96 / 200
// 20.2 / 22.4, 52 / 31; 2048->17408 M = 65 16.9 / 19.9; 5120->17408 M = 128 / 200
// 53 / 39, 54.6 / 59; 5120->34816 M = 129 / 255 90 / 98, 148 / 116).
// Row blocks: one up to 128 rows (the weights are read once), except two on
// narrow N with short k chains, where the rows give the parallelism that more
// splits would (5120^2 M = 96: 15.2 us for two blocks in three splits, 16.9
// for one in six).  Depth: three stages while a compute unit holds one
// workgroup, two (two workgroups fit) beyond.
M8Plan m8_plan(int64_t M, int64_t N, int64_t K) {
  M8Plan p{0, 1, 2, {4, 1, 0}};
  const int64_t ntile = (N + 15) / 16, nblk = K / kI8Blk, g8 = (ntile + 7) / 8;
  if (M <= 4 || M > kM8MaxM || K % kI8Blk != 0 || K > (1 << 23)) return p;
  if (M > 128 && nblk < 64 && ntile < 320) return p;   // two row blocks of few tiles: 5120->2048 M = 192 16.2 against 13.2
  if (M > 128 || (nblk < 64 && g8 <= 64 && M > (g8 <= 16 ? 32 : 48))) p.nz = 2;
  const int chunks = (int)((M + 16 * p.nz - 1) / (16 * p.nz));
  const int mc = chunks <= 4 ? chunks : chunks <= 6 ? 6 : 8;
  double other = m8_other_us(M, ntile, nblk, mc);
  if (other + 0.38 * (double)nblk <= 0.0) return p;
  p.m = mid_split(ntile, (nblk + 3) / 4, 4 * kW8TileBlockBytes, 4.0 * mc * 16 * kI8RowBytes, p.nz, mc);
  if (M > kM8GemvMaxM && p.m.p == 5) other += 0.38 * (double)nblk;   // ten-tile groups: estimated high by that
  if (p.m.us + (p.m.s > 1 ? 0.4 : 0.0) >= other) return p;
  p.mc = mc;
  p.d = p.m.groups * p.nz * p.m.s <= 256 && mc < 8 ? 3 : 2;
  return p;
}

template <int P, int MC, int D>
int launch_m8(const int8_t* qx, const float* sx, int M, int K, const int8_t* qw, const float* sw, const half_t* bias,
              int N, half_t* y, const M8Plan& p, void* ws, W8Layout wl8, hipStream_t st) {
  int4v_t* part = p.m.s > 1 ? reinterpret_cast<int4v_t*>(reinterpret_cast<uint8_t*>(ws) + kSplitCounterBytes) : nullptr;
  hipLaunchKernelGGL((w8a8_mid_kernel<P, MC, D>), dim3((unsigned)p.m.groups, (unsigned)p.m.s, (unsigned)p.nz),
                     dim3(128 * P), 0, st, qx, sx, M, K, qw, sw, bias, N, y, part, wl8);
  if (p.m.s > 1)
    hipLaunchKernelGGL((w8a8_mid_sum_kernel<P, MC>), dim3((unsigned)((p.nz * p.m.groups * P * kM8Tiles * MC + 3) / 4)),
                       dim3(256), 0, st, part, p.m.s, (int)p.m.groups, p.nz, M, N, sx, sw, bias, y);
  return check_launch("w8a8_mid");
}

template <int P>
int launch_m8_plan(const int8_t* qx, const float* sx, int M, int K, const int8_t* qw, const float* sw,
                   const half_t* bias, int N, half_t* y, const M8Plan& p, void* ws, W8Layout wl8, hipStream_t st) {
  switch (p.mc * 10 + p.d) {
    case 12: return launch_m8<P, 1, 2>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);
    case 13: return launch_m8<P, 1, 3>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);
    case 22: return launch_m8<P, 2, 2>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);
    case 23: return launch_m8<P, 2, 3>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);
    case 32: return launch_m8<P, 3, 2>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);
    case 33: return launch_m8<P, 3, 3>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);
    case 42: return launch_m8<P, 4, 2>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);
    case 43: return launch_m8<P, 4, 3>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);
    case 62: return launch_m8<4, 6, 2>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);   // P = 4 beyond mc = 4
    case 63: return launch_m8<4, 6, 3>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);
    default: return launch_m8<4, 8, 2>(qx, sx, M, K, qw, sw, bias, N, y, p, ws, wl8, st);
  }
}

// Long batches over INT8 tiles: 256 x 256 output tiles, both operands in LDS.
//
// The 128 x 128 tiles of the kernel above stop at every 128-k block for its
// copies (vmcnt(0), barrier, first fragment reads) and read each x fragment for
// two MFMAs.  Here eight waves (wm, wn) of 128 rows x 64 columns share stages of
// x (32 KiB, rows as above) and weights (32 KiB; the tile layout already is the
// order fragments are read in) in a two-stage ring, copied buffer -> LDS a whole
// block ahead; the 4 + 8 fragments of a 64-k step are read while the 32 MFMAs of
// the step before run, across the block's barrier too.  A block takes 1.7-2.0 us
// whether 4 or 256 workgroups run and however the reads are placed or the slots
// ordered, i.e. about 32 cycles per MFMA: bound by issue to the matrix cores.
// Workgroups resident on one XCD take neighbouring row blocks of one column
// slice.  One workgroup per compute unit (128 KiB of LDS).
// MI355X, us before -> now (without the quantizer): 5120->7168 M = 2048 / 4096
// 112.9 / 181.9 -> 80.8 / 161.7, 5120^2 M = 3000 114 -> 81, 5120->17408 M = 1500 /
// 4096 184 / 463 -> 158 / 399, 5120->34816 M = 4096 968 -> 777 (1.88 POP/s),
// 17408->5120 M = 3000 291 -> 228.
constexpr int kBigTiles = 16, kBigRows = 256;            // of a workgroup
constexpr int kBigXBytes = kBigRows * kI8RowBytes;       // x of a stage
constexpr int kBigStageBytes = kBigXBytes + kBigTiles * (int)kW8TileBlockBytes;

template <int LO, int N>
__device__ __forceinline__ void big_read_x(uint4_t (&b)[8], uint32_t a) {
  if constexpr (N > 0) {
    b[LO] = i8_lds_read_off<LO * 16 * kI8RowBytes>(a);
    big_read_x<LO + 1, N - 1>(b, a);
  }
}
// All LDS reads done, tied to the fragments so that no use moves above it.
__device__ __forceinline__ void big_wait(uint4_t (&a)[4], uint4_t (&b)[8]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]),
                 "+v"(b[4]), "+v"(b[5]), "+v"(b[6]), "+v"(b[7]));
}

__global__ __launch_bounds__(512, 2) void w8a8_gemm256_kernel(const int8_t* __restrict__ qx, const float* __restrict__ sx,
                                                              int M, int K, const int8_t* __restrict__ qw,
                                                              const float* __restrict__ sw,
                                                              const half_t* __restrict__ bias, int N,
                                                              half_t* __restrict__ y) {
  __shared__ __attribute__((aligned(1024))) uint8_t xs[2 * kBigStageBytes];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 3, wm = wave >> 2, i = lane & 15, kb = lane >> 4;
  const int ntile = (N + 15) >> 4, nblk = K / kI8Blk, mblk = (M + kBigRows - 1) / kBigRows;
  // XCD x (flat id mod 8) takes the x-th run of workgroups, row block fastest.
  const int g = (int)gridDim.x, q8 = g >> 3, r8 = g & 7, xcd = (int)blockIdx.x & 7;
  const int id = xcd * q8 + min(xcd, r8) + ((int)blockIdx.x >> 3);
  const int tile0 = id / mblk * kBigTiles, m0 = id % mblk * kBigRows;

  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(qx + (size_t)m0 * K, (int64_t)(M - m0) * K);
  const __amdgpu_buffer_rsrc_t rw = buf_rsrc(qw + (size_t)tile0 * nblk * kW8TileBlockBytes,
                                             (int64_t)(ntile - tile0) * nblk * kW8TileBlockBytes);
  // x instruction J = 4 wave + j: rows 8 J .. 8 J + 7, lane L chunk
  // i8_swz(row, L % 8) of row 8 J + L / 8; weight instruction: piece j & 1 of
  // tile 2 wave + j / 2.
  uint32_t xvo[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) xvo[j] = (uint32_t)((lane >> 3) * K + 16 * i8_swz(8 * j + (lane >> 3), lane & 7));
  constexpr uint32_t kPastEnd = 0x80000000u;
  auto fetch = [&](int blk, int st) {   // past the last block: zeros
    uint8_t* stage = xs + st * kBigStageBytes;
    const bool live = blk < nblk;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int J = 4 * wave + j;
      lds_load16(rx, xvo[j & 1], live ? (uint32_t)(8 * J) * (uint32_t)K + (uint32_t)(blk * kI8Blk) : kPastEnd,
                 stage + J * 1024);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = 2 * wave + (j >> 1);
      lds_load16(rw, (uint32_t)lane * 16,
                 live ? (uint32_t)(t * nblk + blk) * (uint32_t)kW8TileBlockBytes + (uint32_t)(j & 1) * 1024 : kPastEnd,
                 stage + kBigXBytes + t * kW8TileBlockBytes + (j & 1) * 1024);
    }
  };

  int4v_t acc[4][8];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) acc[t][mt] = int4v_t{0, 0, 0, 0};
  const uint32_t lds = (uint32_t)(size_t)((const __attribute__((address_space(3))) uint8_t*)xs);
  const uint32_t xa = lds + (uint32_t)((wm * 128 + i) * kI8RowBytes);
  const uint32_t wa = lds + (uint32_t)(kBigXBytes + wn * 4 * kW8TileBlockBytes + lane * 16);

  uint4_t a0[4], b0[8], a1[4], b1[8];   // fragments of the two 64-k steps
  auto read = [&](auto step, uint32_t so, uint4_t (&a)[4], uint4_t (&b)[8]) {
    constexpr int s = decltype(step)::value;
    a[0] = i8_lds_read_off<s * 1024>(wa + so);
    a[1] = i8_lds_read_off<s * 1024 + 2048>(wa + so);
    a[2] = i8_lds_read_off<s * 1024 + 4096>(wa + so);
    a[3] = i8_lds_read_off<s * 1024 + 6144>(wa + so);
    big_read_x<0, 8>(b, xa + so + (uint32_t)(i8_swz(i, 4 * s + kb) * 16));
  };
  auto math = [&](const uint4_t (&a)[4], const uint4_t (&b)[8]) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < 8; ++mt)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t][mt] = mfma_i8(a[t], b[mt], acc[t][mt]);
    __builtin_amdgcn_sched_barrier(0);
  };
  fetch(0, 0);
  fetch(1, 1);
  __builtin_amdgcn_s_waitcnt(8 | (0x7 << 4) | (0xF << 8));   // stage 0 landed, stage 1's eight copies may be in flight
  __builtin_amdgcn_s_barrier();
  read(std::integral_constant<int, 0>{}, 0, a0, b0);
  for (int blk = 0; blk < nblk; ++blk) {
    const uint32_t so = (uint32_t)((blk & 1) * kBigStageBytes);
    big_wait(a0, b0);
    read(std::integral_constant<int, 1>{}, so, a1, b1);
    math(a0, b0);
    big_wait(a1, b1);
    __builtin_amdgcn_s_waitcnt(0);    // this wave's part of the next stage landed ...
    __builtin_amdgcn_s_barrier();     // ... everyone's, and everyone has read this stage
    __builtin_amdgcn_sched_barrier(0);
    fetch(blk + 2, blk & 1);
    __builtin_amdgcn_sched_barrier(0);
    read(std::integral_constant<int, 0>{}, (uint32_t)kBigStageBytes - so, a0, b0);
    math(a1, b1);
  }
  big_wait(a0, b0);                 // the run-out's reads and copies
  __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int mt = 0; mt < 8; ++mt)
      m8_store(acc[t][mt], m0 + wm * 128 + mt * 16 + i, (tile0 + wn * 4 + t) * 16 + 4 * kb, M, N, sx, sw, bias, y);
}

constexpr int kW8A8GemvMaxM = kM8GemvMaxM;
// Largest k of the W8A8 GEMM: a workgroup reads its 128 x rows and up to 64
// weight rows of k bytes each through one buffer apiece, whose record count is
// capped at 2^31 - 1 bytes; longer rows run the GEMV kernel 16 rows at a time.
constexpr int64_t kW8A8GemmMaxK = 1 << 23;
static_assert(128 * kW8A8GemmMaxK <= 0x7fffffff, "GEMM x and weight offsets must fit the 31-bit buffer range");
// The 256 x 256 tiles read 256 rows of each, so their last block at k = 2^23
// would end past that cap and come back as zeros: one 128-k block less.
constexpr int64_t kBigMaxK = kW8A8GemmMaxK - kI8Blk;
static_assert(kBigRows * kBigMaxK <= 0x7fffffff && kBigTiles * 16 * kBigMaxK <= 0x7fffffff,
              "256 x 256 tile offsets must fit the 31-bit buffer range");

// The kernel and grid of a shape.
struct W8A8Route {
  enum Kernel { kGemv, kGemm, kGemm256, kMid } kernel;
  M8Plan plan;             // kMid
  int nt, mt;              // kGemm: weight tiles per wave, 16-row chunks of x
  int64_t mblocks, wgs256; // row blocks of kGemm, workgroups of kGemm256
};

W8A8Route w8a8_route(int64_t m, int64_t n, int64_t k, bool tiled, size_t ws_bytes) {
  W8A8Route r{W8A8Route::kGemv, m8_plan(m, n, k), 0, 0, 0, 0};
  if (r.plan.mc > 0 && (r.plan.m.s == 1 || ws_bytes >= r.plan.bytes())) {
    r.kernel = W8A8Route::kMid;
    return r;
  }
  if (m <= kW8A8GemvMaxM || k % kI8Blk != 0 || k > kW8A8GemmMaxK) return r;
  // GEMM: 128-row x tiles for long batches, 32-row ones otherwise; four
  // weight tiles per wave while that still leaves a full machine of
  // workgroups, else one.  Over INT8 tiles, long batches take two tiles
  // per wave while that gives 512 workgroups (M = 4096: 5120^2 197 ->
  // 159 us, 5120->17408 513 -> 454 us, 17408->5120 466 -> 410 us).
  const int64_t ntile = (n + 15) / 16;
  const bool big_m = m >= 256;
  r.kernel = W8A8Route::kGemm;
  r.mblocks = big_m ? (m + 127) / 128 : (m + 31) / 32;
  r.mt = big_m ? 8 : 2;
  const bool two_tiles = tiled && big_m && (ntile + 7) / 8 * r.mblocks >= 512;
  r.nt = two_tiles ? 2 : (ntile + 15) / 16 * r.mblocks >= 256 ? 4 : 1;
  // 256 x 256 tiles where their rounds of 256 workgroups cost less: one costs
  // 3.0 to 3.15 rounds of the 128 x 128 tiles (72-86 against 26-28 us at
  // K = 5120, 63-67 against 20-22 us per 5120 of K = 17408).  Just past the
  // line the other way: 5120^2 M = 4096 (2 against 5 rounds) 152 against 128 us,
  // 5120->17408 M = 777 (2 against 4) 148 against 118.
  r.wgs256 = (ntile + kBigTiles - 1) / kBigTiles * ((m + kBigRows - 1) / kBigRows);
  if (two_tiles && k <= kBigMaxK && 31 * ((r.wgs256 + 255) / 256) < 10 * (((ntile + 7) / 8 * r.mblocks + 255) / 256))
    r.kernel = W8A8Route::kGemm256;
  return r;
}

}  // namespace
}  // namespace wq

using namespace wq;

extern "C" int wq_w8a8_quantize(const uint16_t* x, int64_t m, int64_t k, int8_t* qx, float* x_scale, void* stream) {
  if (m == 0) return WQ_OK;
  WQ_REQUIRE(x && qx && x_scale, WQ_ERR_INVALID_ARGUMENT, "null pointer argument");
  WQ_REQUIRE(m > 0 && m <= 0x7fffffff && k > 0 && k % 8 == 0 && k <= (1 << 26), WQ_ERR_INVALID_ARGUMENT,
             "need m >= 0 and 0 < k, k %% 8 == 0 (k = %lld)", (long long)k);
  WQ_REQUIRE(((uintptr_t)x | (uintptr_t)qx) % 16 == 0, WQ_ERR_INVALID_ARGUMENT, "x and qx must be 16-byte aligned");
  auto launch = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)m), dim3(threads), 0, as_stream(stream),
                       reinterpret_cast<const half_t*>(x), (int)k, qx, x_scale);
  };
  const int64_t nc = k / 8;
  if (m <= 512 && nc > 256 && nc <= 3 * 1024) {   // few rows: one round of loads over 16 waves
    if (nc <= 1024) launch(w8a8_quantize_kernel<1024, 1>, 1024);
    else launch(w8a8_quantize_kernel<1024, 3>, 1024);
  } else if (nc <= 256) launch(w8a8_quantize_kernel<256, 1>, 256);
  else if (nc <= 3 * 256) launch(w8a8_quantize_kernel<256, 3>, 256);
  else if (nc <= 9 * 256) launch(w8a8_quantize_kernel<256, 9>, 256);
  else launch(w8a8_quantize_kernel<256, 0>, 256);
  return check_launch("w8a8_quantize");
}

namespace {

int w8a8_linear_impl(const int8_t* qx, const float* x_scale, int64_t m, int64_t k, const int8_t* qweight,
                     const float* w_scale, int64_t n, const uint16_t* bias, uint16_t* y, void* ws, size_t ws_bytes,
                     void* stream, int tiled) {
  if (m == 0 || n == 0) return WQ_OK;
  WQ_REQUIRE(qx && x_scale && qweight && w_scale && y, WQ_ERR_INVALID_ARGUMENT, "null pointer argument");
  WQ_REQUIRE(m > 0 && n > 0 && k > 0 && m <= 0x7fffffff && n <= 0x7fffffff && k <= (1 << 26),
             WQ_ERR_INVALID_ARGUMENT, "m, n, k out of range");
  WQ_REQUIRE(k % (tiled ? kI8Blk : kI8Step) == 0, WQ_ERR_UNSUPPORTED, "W8A8 linear needs k %% %d == 0 (got %lld)",
             tiled ? kI8Blk : kI8Step, (long long)k);
  const W8Layout wl8{tiled};
  WQ_REQUIRE(((uintptr_t)qx | (uintptr_t)qweight) % 16 == 0, WQ_ERR_INVALID_ARGUMENT,
             "qx and qweight must be 16-byte aligned");
  const half_t* b = reinterpret_cast<const half_t*>(bias);
  half_t* yy = reinterpret_cast<half_t*>(y);
  const int64_t nsteps = k / kI8Step, ntile = (n + 15) / 16;
  const W8A8Route r = w8a8_route(m, n, k, tiled, ws != nullptr ? ws_bytes : 0);
  if (r.kernel == W8A8Route::kMid)
    return (r.plan.m.p == 4 ? launch_m8_plan<4> : launch_m8_plan<5>)(qx, x_scale, (int)m, (int)k, qweight, w_scale, b,
                                                                    (int)n, yy, r.plan, ws, wl8, as_stream(stream));
  if (r.kernel == W8A8Route::kGemm || r.kernel == W8A8Route::kGemm256)
    WQ_REQUIRE(r.mblocks <= 65535, WQ_ERR_UNSUPPORTED, "too many rows for the W8A8 GEMM grid");
  if (r.kernel == W8A8Route::kGemm256) {
    hipLaunchKernelGGL(w8a8_gemm256_kernel, dim3((unsigned)r.wgs256), dim3(512), 0, as_stream(stream), qx, x_scale,
                       (int)m, (int)k, qweight, w_scale, b, (int)n, yy);
    return check_launch("w8a8_gemm256");
  }
  if (r.kernel == W8A8Route::kGemm) {
    const dim3 grid((unsigned)((ntile + 4 * r.nt - 1) / (4 * r.nt)), (unsigned)r.mblocks);
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, as_stream(stream), qx, x_scale, (int)m, (int)k, qweight,
                         w_scale, b, (int)n, yy, wl8);
    };
    if (r.mt == 8) {
      if (r.nt == 4) launch(w8a8_gemm_kernel<4, 8>);
      else if (r.nt == 2) launch(w8a8_gemm_kernel<2, 8>);
      else launch(w8a8_gemm_kernel<1, 8>);
    } else {
      if (r.nt == 4) launch(w8a8_gemm_kernel<4, 2>); else launch(w8a8_gemm_kernel<1, 2>);
    }
    return check_launch("w8a8_gemm");
  }
  // Decode kernel: about eight 64-k steps per wave (one round of loads).
  int ksw = (int)((nsteps + 7) / 8);
  ksw = ksw < 1 ? 1 : (ksw > 16 ? 16 : ksw);
  for (int64_t m0 = 0; m0 < m; m0 += kW8A8GemvMaxM) {   // batches beyond 16 rows only when k % 128 != 0 or k > 2^23
    const int64_t mr = m - m0 < kW8A8GemvMaxM ? m - m0 : kW8A8GemvMaxM;
    hipLaunchKernelGGL(w8a8_gemv_kernel, dim3((unsigned)ntile), dim3(64 * ksw), 0, as_stream(stream), qx + m0 * k,
                       x_scale + m0, (int)mr, (int)k, qweight, w_scale, b, (int)n, yy + m0 * n, wl8);
    const int rc = check_launch("w8a8_gemv");
    if (rc != WQ_OK) return rc;
  }
  return WQ_OK;
}

}  // namespace

namespace wq {
void w8a8_plan_text(int64_t m, int64_t n, int64_t k, char* text, size_t bytes) {
  const W8A8Route r = w8a8_route(m, n, k, true, SIZE_MAX);
  switch (r.kernel) {
    case W8A8Route::kMid: snprintf(text, bytes, "mid %dx%d", r.plan.m.p, r.plan.m.s); break;
    case W8A8Route::kGemm256: snprintf(text, bytes, "gemm 256x256"); break;
    case W8A8Route::kGemm: snprintf(text, bytes, "gemm %dx%d", r.nt, r.mt); break;
    default: snprintf(text, bytes, "gemv"); break;
  }
}
}  // namespace wq

extern "C" int wq_w8a8_workspace_size(int64_t m, int64_t n, int64_t k, size_t* bytes) {
  WQ_REQUIRE(bytes, WQ_ERR_INVALID_ARGUMENT, "null size output");
  WQ_REQUIRE(m >= 0 && n > 0 && k > 0 && m <= 0x7fffffff && n <= 0x7fffffff && k <= (1 << 26), WQ_ERR_INVALID_ARGUMENT,
             "m, n, k out of range");
  const M8Plan p = m8_plan(m, n, k);
  *bytes = p.mc > 0 ? p.bytes() : 0;
  return WQ_OK;
}

extern "C" int wq_w8a8_linear(const int8_t* qx, const float* x_scale, int64_t m, int64_t k, const int8_t* qweight,
                              const float* w_scale, int64_t n, const uint16_t* bias, uint16_t* y, void* stream) {
  return w8a8_linear_impl(qx, x_scale, m, k, qweight, w_scale, n, bias, y, nullptr, 0, stream, 0);
}

extern "C" int wq_w8a8_linear_tiled(const int8_t* qx, const float* x_scale, int64_t m, int64_t k, const void* tiles,
                                    const float* w_scale, int64_t n, const uint16_t* bias, uint16_t* y, void* stream) {
  return w8a8_linear_impl(qx, x_scale, m, k, reinterpret_cast<const int8_t*>(tiles), w_scale, n, bias, y, nullptr, 0,
                          stream, 1);
}

extern "C" int wq_w8a8_linear_ws(const int8_t* qx, const float* x_scale, int64_t m, int64_t k, const void* weight,
                                 int32_t tiled, const float* w_scale, int64_t n, const uint16_t* bias, uint16_t* y,
                                 void* workspace, size_t workspace_bytes, void* stream) {
  return w8a8_linear_impl(qx, x_scale, m, k, reinterpret_cast<const int8_t*>(weight), w_scale, n, bias, y, workspace,
                          workspace_bytes, stream, tiled ? 1 : 0);
}
