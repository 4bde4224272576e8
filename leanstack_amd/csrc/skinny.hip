// Projections of 17..128 rows (9..16 for a wide SiLU*up) on gfx950: y[M][N] = epilogue(x[M][K] . W[N][K]^T).
//
// At these row counts a projection is still bound by the bytes that each CU
// pulls: the weights from HBM once (the arithmetic intensity is M FLOP per
// weight byte, under 128) and, per workgroup, the activations from L2.  A
// workgroup owns RBW row-blocks (16 output rows each) and all tokens over one
// K range, which its 4 wavefronts take in 64-K steps in turn.  Each wave DMAs
// the weight tiles and activation rows of its steps into a ring of its own in
// LDS, 1-4 steps deep (up to 160 KB in flight per CU, no registers), and
// multiplies a step on v_mfma_f32_16x16x32_bf16 as it lands: no barrier and no
// shared stage until the waves' partial tiles are summed through LDS, in wave
// order.
//
// Activations are read 8 lanes per row, whole 128-byte lines: read as B
// fragments straight from global memory (16 rows of 64 bytes per load, each
// 16 bytes of it another cache access), they cost four times the accesses and
// the weights waited behind them.  17.5 / 14.0 / 45.0 / 24.5 -> 12.9 / 10.8 /
// 24.8 / 17.6 us for QKV / o / gate_up + SiLU*up / down at 64 rows, 32 / 24 /
// 56 / 42 -> 18.5 / 15.4 / 32.6 / 25 at 128; per CU about 33 bytes/ns of weights
// and activations together, against 27 of weights alone in the decode kernels.
//
// When the row-blocks alone would leave CUs idle (kv/o/down-sized N), the call's
// workspace lets the K range of every row-block be split over S workgroups:
// each publishes its fp32 partial with device-coherent stores and counts its
// arrival, and the workgroup that arrives last adds the S partials in split
// order, applies the epilogue and stores the rows.  Nothing waits on another
// workgroup, and every sum has a fixed order, so results are bitwise
// reproducible; the split form and the unsplit one add in different orders
// and agree to fp32 rounding.
//
// Reference arithmetic replaced: F.linear at
// src/leanstack/runtime/qwen_explicit.py:748, :819, :828-830, :1202-1208 for
// the verify and short prefill batches, and the hot-kernel GEMM cases of
// src/leanstack/hot_kernels.py:81-194 (M = 64).

#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>
#include <vector>

#include "lsk_internal.h"

namespace lsk {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kNW = kSkinnyWaves;  // wavefronts per workgroup
constexpr int kCoherent = 16;      // buffer cache policy: device-coherent (sc1)
constexpr unsigned kRawBufferDword3 = 0x00020000u;
constexpr int kLdsBytes = 160 * 1024;  // of one CU

__device__ __forceinline__ f32x4_t mfma16(bf16x8_t a, bf16x8_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ u32x4_t buffer_words(const void* base, size_t bytes) {
  const unsigned long long p = reinterpret_cast<unsigned long long>(base);
  return u32x4_t{(unsigned)p, (unsigned)(p >> 32) & 0xffffu, (unsigned)(bytes < 0x7fffffffu ? bytes : 0x7fffffffu),
                 kRawBufferDword3};
}

// 1 KB of global memory straight into LDS: lane l's 16 bytes at voff + soff
// land at lds + 16 l.  In assembly, with no result register, so that the
// compiler neither counts it nor waits for it before unrelated LDS reads (one
// ring in one LDS array would otherwise be drained before every read); each
// use waits for its own data (wait_steps).  m0, the LDS address of such a load,
// is written here and named as clobbered.
template <bool STREAM>
__device__ __forceinline__ void dma_1k(u32x4_t rsrc, unsigned voff, unsigned soff, unsigned lds) {
  soff = __builtin_amdgcn_readfirstlane(soff);  // wave-uniform; says so to the compiler
  lds = __builtin_amdgcn_readfirstlane(lds);
  if constexpr (STREAM)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"s"(lds), "v"(voff),
                 "s"(rsrc), "s"(soff)
                 : "m0", "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff),
                 "s"(rsrc), "s"(soff)
                 : "m0", "memory");
}

// Wait until at most `steps` (0..D-1, wave-uniform) steps of NL loads are in
// flight.
template <int NL, int D>
__device__ __forceinline__ void wait_steps(int steps) {
  if constexpr (D >= 4) {
    if (steps >= 3) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * NL < 63 ? 3 * NL : 63) : "memory");
      return;
    }
  }
  if constexpr (D >= 3) {
    if (steps == 2) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NL < 63 ? 2 * NL : 63) : "memory");
      return;
    }
  }
  if constexpr (D >= 2) {
    if (steps == 1) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL < 63 ? NL : 63) : "memory");
      return;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// RBW row-blocks x MG token groups per workgroup; 64-K steps of (2 RBW + 2 MG)
// KB, each loaded and multiplied by one wave.
template <int RBW, int MG>
struct Shape {
  static constexpr int kLoads = 2 * RBW + 2 * MG;  // 1 KB loads per step
  static constexpr int kSlot = kLoads * 1024;
  // Workgroups of two row-blocks are what wide N runs in several rounds: half
  // of the LDS each, so that a CU holds two and the first loads and last sums of
  // one hide behind the other's stream (SiLU*up 22016 x 1024 at 17 rows 15.0 ->
  // 11.3 us, plain 24576 x 2560 at 32 rows 11 % less; calls of one round lose
  // nothing).
  static constexpr int kWgLds = RBW == 2 && MG <= 4 ? kLdsBytes / 2 : kLdsBytes;
  static constexpr int kFit = kWgLds / (kNW * kSlot);
  static constexpr int kDepth = kFit < 1 ? 1 : kFit > 4 ? 4 : kFit;  // steps in flight per wave
  // Where only one step fits (RBW 5 from 6 token groups, RBW 2 at 4), the weights
  // of the step after it still fit beside it, and they are what comes from HBM: a
  // wave then waits for activations from L2 alone (19456 x 2560 with SiLU*up:
  // 36.0 -> 32.6 us at 128 rows, 29.5 -> 28.8 at 96).
  static constexpr bool kAhead = kDepth == 1 && kNW * (kSlot + 2 * RBW * 1024) <= kWgLds;
  static constexpr int kWaveRing = kDepth * kSlot + (kAhead ? 2 * RBW * 1024 : 0);
  static constexpr int kRing = kNW * kWaveRing;
  // Row-blocks whose partial tiles of all waves fit the ring at once.
  static constexpr int kSumRows = kRing / (kNW * MG * 1024) < RBW ? kRing / (kNW * MG * 1024) : RBW;
  static_assert(kFit >= 1 && kSumRows >= 1, "one step per wave fits the LDS");
};

// EPI SiLU*up: a "row-block" is a unit of 8 gate rows and the 8 up rows of the
// same outputs (half a gate/up pair of the packed layout), so units, not
// pairs, are what the workgroups share out.
template <int RBW, int MG, int EPI>
__global__ __launch_bounds__(kNW * 64) void skinny_kernel(
    const bf16x8_t* __restrict__ w, const __bf16* __restrict__ x, int ldx, __bf16* __restrict__ y, int ldy,
    const __bf16* __restrict__ residual, int ldr, int M, int NB, int KT, int S, unsigned* __restrict__ counters,
    unsigned char* __restrict__ partials, unsigned partial_bytes) {
  using Sh = Shape<RBW, MG>;
  constexpr bool kSilu = EPI == static_cast<int>(Epilogue::kSiluMul);
  constexpr int D = Sh::kDepth;
  __shared__ __attribute__((aligned(1024))) unsigned char ring[Sh::kRing];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 15;  // B-operand column = token within its group
  const int g = lane >> 4;  // K group inside a tile / output row quad
  const int grp = blockIdx.x / S;
  const int split = blockIdx.x - grp * S;
  const int rb0 = grp * RBW;

  // Steps of 64 K: this split's are [ub, ue), dealt to the waves in turn, so
  // that the four waves read neighbouring 128-byte pieces of the same rows.
  const int units = (KT + 1) / 2;
  const int ub = (int)((long long)units * split / S), ue = (int)((long long)units * (split + 1) / S);
  const int n = ue - ub > wave ? (ue - ub - wave + kNW - 1) / kNW : 0;

  // Weight loads: one packed tile (or the 8 + 8 rows of a unit) in A-operand
  // order per KB.  Blocks past the last repeat it; they are never stored.
  const int first = kSilu ? (rb0 >> 1) * 2 : rb0;  // packed row-block the buffer starts at
  const u32x4_t wrsrc = buffer_words(w + (size_t)first * KT * 64, (size_t)(NB - first) * KT * 1024);
  unsigned wvoff[RBW];
#pragma unroll
  for (int r = 0; r < RBW; ++r) {
    const int rb = min(rb0 + r, NB - 1);
    if constexpr (kSilu)
      wvoff[r] = (unsigned)((rb & ~1) - first + (m >> 3)) * KT * 1024u + (g * 16 + 8 * (rb & 1) + (m & 7)) * 16u;
    else
      wvoff[r] = (unsigned)(rb - first) * KT * 1024u + lane * 16u;
  }
  // Activation loads: 8 token rows x 128 bytes (whole lines) per KB.  Row t's
  // 16-byte chunk c is stored at position c ^ ((t >> 1) & 7) of its 128
  // bytes, which puts the 16 lanes of a fragment read on distinct banks.
  // Rows past M repeat row M - 1; their columns are never stored.
  const u32x4_t xrsrc = buffer_words(x, ((size_t)(M - 1) * ldx + (size_t)KT * kTileK) * 2);
  unsigned xrow[2 * MG];
  const int xr = lane >> 3;
#pragma unroll
  for (int i = 0; i < 2 * MG; ++i) xrow[i] = (unsigned)min(8 * i + xr, M - 1) * ldx * 2u;
  const unsigned ring0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)ring +
                         wave * Sh::kWaveRing;

  // A wave's ring: D slots of weights, then activations; kAhead: one slot of
  // activations between two of weights.
  constexpr unsigned kXSlot = Sh::kAhead ? 0 : Sh::kSlot;
  auto issue_w = [&](int step, int slot) {
    const int u = ub + wave + kNW * step;
    const bool half = 2 * u + 1 >= KT;  // odd KT: the last step has one k-tile
    const unsigned lds = ring0 + slot * Sh::kSlot;
#pragma unroll
    for (int r = 0; r < RBW; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        dma_1k<true>(wrsrc, wvoff[r], (unsigned)(2 * u + (half ? 0 : h)) * 1024u, lds + (2 * r + h) * 1024);
  };
  auto issue_x = [&](int step, int slot) {
    const int u = ub + wave + kNW * step;
    const bool half = 2 * u + 1 >= KT;
    const unsigned lds = ring0 + 2 * RBW * 1024 + slot * kXSlot;
#pragma unroll
    for (int i = 0; i < 2 * MG; ++i) {
      int c = (lane & 7) ^ (((i & 1) << 2) | (xr >> 1));
      if (half) c &= 3;
      dma_1k<false>(xrsrc, xrow[i] + c * 16u, (unsigned)u * 128u, lds + i * 1024);
    }
  };

  f32x4_t acc[RBW][MG];
#pragma unroll
  for (int r = 0; r < RBW; ++r)
#pragma unroll
    for (int q = 0; q < MG; ++q) acc[r][q] = f32x4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < n) {
      issue_w(d, d);
      issue_x(d, d);
    }
  if (Sh::kAhead && n > 1) issue_w(1, 1);
  int slot = 0;
  for (int i = 0; i < n; ++i) {
    if constexpr (Sh::kAhead)
      wait_steps<2 * RBW, 2>(min(1, n - 1 - i));  // all but the next step's weights
    else
      wait_steps<Sh::kLoads, D>(min(D - 1, n - 1 - i));
    const unsigned char* buf = ring + wave * Sh::kWaveRing + slot * Sh::kSlot;
    const unsigned char* xbuf = ring + wave * Sh::kWaveRing + 2 * RBW * 1024 + slot * kXSlot;
    bf16x8_t wv[2][RBW], xv[2][MG];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int r = 0; r < RBW; ++r) wv[h][r] = *reinterpret_cast<const bf16x8_t*>(buf + (2 * r + h) * 1024 + lane * 16);
#pragma unroll
      for (int q = 0; q < MG; ++q)
        xv[h][q] = *reinterpret_cast<const bf16x8_t*>(xbuf + (16 * q + m) * 128 + (((4 * h + g) ^ (m >> 1)) << 4));
    }
    // The slot's values are in registers before its next loads may land.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if constexpr (Sh::kAhead) {
      if (i + 1 < n) issue_x(i + 1, 0);
      if (i + 2 < n) issue_w(i + 2, slot);
    } else if (i + D < n) {
      issue_w(i + D, slot);
      issue_x(i + D, slot);
    }
    const bool half = 2 * (ub + wave + kNW * i) + 1 >= KT;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h == 1 && half) break;
#pragma unroll
      for (int r = 0; r < RBW; ++r)
#pragma unroll
        for (int q = 0; q < MG; ++q) acc[r][q] = mfma16(wv[h][r], xv[h][q], acc[r][q]);
    }
    slot = slot + 1 == (Sh::kAhead ? 2 : D) ? 0 : slot + 1;
  }

  // Cross-wave sum in wave order through the drained ring, kSumRows row-blocks
  // at a time: tile t = r MG + q is summed (and stored) by wave t % 4.
  constexpr int kTiles = RBW * MG;
  constexpr int kMine = (kTiles + kNW - 1) / kNW;
  f32x4_t sum[kMine];
#pragma unroll
  for (int r0 = 0; r0 < RBW; r0 += Sh::kSumRows) {
    __syncthreads();
#pragma unroll
    for (int r = r0; r < RBW && r < r0 + Sh::kSumRows; ++r)
#pragma unroll
      for (int q = 0; q < MG; ++q)
        *reinterpret_cast<f32x4_t*>(ring + ((wave * Sh::kSumRows + r - r0) * MG + q) * 1024 + lane * 16) = acc[r][q];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      const int t = j * kNW + wave;
      if (t < r0 * MG || t >= (r0 + Sh::kSumRows) * MG || t >= kTiles) continue;
      const unsigned char* src = ring + (t - r0 * MG) * 1024 + lane * 16;
      f32x4_t v = *reinterpret_cast<const f32x4_t*>(src);
#pragma unroll
      for (int o = 1; o < kNW; ++o) v += *reinterpret_cast<const f32x4_t*>(src + o * Sh::kSumRows * MG * 1024);
      sum[j] = v;
    }
  }

  if (S > 1) {
    // Publish this split's sums, count the arrival; the last of the S splits
    // of the row-blocks adds them in split order.  Partials cross XCDs, whose
    // L2s are not coherent with each other: device-coherent buffer stores and
    // loads, and the arrival only after every wave's stores are acknowledged.
    const __amdgpu_buffer_rsrc_t parts =
        __builtin_amdgcn_make_buffer_rsrc(partials, (short)0, (int)partial_bytes, (int)kRawBufferDword3);
    constexpr unsigned kPart = kTiles * 1024;
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      const int t = j * kNW + wave;
      if (t < kTiles)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, sum[j]), parts, lane * 16,
                                               (unsigned)blockIdx.x * kPart + t * 1024u, kCoherent);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* last = reinterpret_cast<int*>(ring);
    if (threadIdx.x == 0)
      *last = __hip_atomic_fetch_add(counters + grp, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
              (unsigned)S - 1;
    __syncthreads();
    if (!*last) return;
    // Re-arm the counter for the next call, then add the S partials, this
    // split's own from its registers, the others PB splits at a time (every load
    // of a round goes out before the first add: a branch around an add would
    // let the compiler sink the load into it); slots past the last split are
    // read at an offset beyond the buffer's range, which returns zeros without
    // a memory access.
    if (threadIdx.x == 0) __hip_atomic_store(counters + grp, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    constexpr int PB = kMine >= 8 ? 2 : 4;
    f32x4_t total[kMine];
#pragma unroll
    for (int j = 0; j < kMine; ++j) total[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < S; s0 += PB) {
      f32x4_t v[PB][kMine];
#pragma unroll
      for (int b = 0; b < PB; ++b) {
        // Out of range goes in the vector offset: the range check covers the
        // vector and instruction offsets, not the scalar one.
        const bool real = s0 + b < S && s0 + b != split;
        const unsigned voff = (real ? 0u : 0x80000000u) + (unsigned)lane * 16u;
        const unsigned base = real ? (unsigned)(grp * S + s0 + b) * kPart : 0u;
#pragma unroll
        for (int j = 0; j < kMine; ++j) {
          const int t = min(j * kNW + wave, kTiles - 1);
          v[b][j] = __builtin_bit_cast(
              f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(parts, voff, base + t * 1024u, kCoherent));
        }
      }
#pragma unroll
      for (int b = 0; b < PB; ++b) {
#pragma unroll
        for (int j = 0; j < kMine; ++j) total[j] += s0 + b == split ? sum[j] : v[b][j];
      }
    }
#pragma unroll
    for (int j = 0; j < kMine; ++j) sum[j] = total[j];
  }

  // Lane (g, m) holds output rows 4g..4g+3 of a tile's row-block for token
  // 16q + m; of a SiLU*up unit, g = 0, 1 gate rows and g = 2, 3 the up rows of
  // lanes 32 below.
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    const int t = j * kNW + wave;
    if (t >= kTiles) break;
    const int rb = rb0 + t / MG;
    const int tok = 16 * (t % MG) + m;
    if constexpr (kSilu) {
      float up[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) up[i] = __shfl_xor(sum[j][i], 32);
      if (rb >= NB || tok >= M || g >= 2) continue;
      unsigned short o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = bf16_bits(silu_mul_bf16(sum[j][i], up[i]));
      *reinterpret_cast<u32x2_t*>(y + (size_t)tok * ldy + rb * 8 + 4 * g) =
          u32x2_t{o[0] | ((unsigned)o[1] << 16), o[2] | ((unsigned)o[3] << 16)};
    } else {
      if (rb >= NB || tok >= M) continue;
      const int col = rb * 16 + 4 * g;
      unsigned short o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v = bf16_round(sum[j][i]);
        if constexpr (EPI == static_cast<int>(Epilogue::kResidualAdd))
          v = static_cast<float>(residual[(size_t)tok * ldr + col + i]) + v;
        o[i] = bf16_bits(v);
      }
      *reinterpret_cast<u32x2_t*>(y + (size_t)tok * ldy + col) =
          u32x2_t{o[0] | ((unsigned)o[1] << 16), o[2] | ((unsigned)o[3] << 16)};
    }
  }
}

template <int RBW, int MG, int EPI>
hipError_t launch_cfg(const SkinnyPlan& p, const void* w, const void* x, int ldx, void* y, int ldy,
                      const void* residual, int ldr, int M, int NB, int KT, void* workspace, hipStream_t stream) {
  auto* ws = static_cast<unsigned char*>(workspace);
  unsigned* counters = p.S > 1 ? reinterpret_cast<unsigned*>(ws + kSkFlagsOffset) : nullptr;
  unsigned char* partials = p.S > 1 ? ws + kSkPartialsOffset : nullptr;
  const unsigned partial_bytes = p.S > 1 ? (unsigned)(p.groups * p.S * RBW * MG * 1024) : 0u;
  launch_kernel(skinny_kernel<RBW, MG, EPI>, dim3(p.groups * p.S), dim3(kNW * 64), 0, stream,
                static_cast<const bf16x8_t*>(w), static_cast<const __bf16*>(x), ldx, static_cast<__bf16*>(y), ldy,
                static_cast<const __bf16*>(residual), ldr, M, NB, KT, p.S, counters, partials, partial_bytes);
  return hipGetLastError();
}

template <int RBW, int EPI>
hipError_t launch_rbw(const SkinnyPlan& p, const void* w, const void* x, int ldx, void* y, int ldy,
                      const void* residual, int ldr, int M, int NB, int KT, void* workspace, hipStream_t stream) {
  switch (skinny_groups(M)) {
    case 1:  // 9..16 rows: SiLU*up only, in twos or fives (skinny_route, skinny_plan)
      if constexpr (EPI == static_cast<int>(Epilogue::kSiluMul) && RBW != 4)
        return launch_cfg<RBW, 1, EPI>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
      break;
    case 2:
      return launch_cfg<RBW, 2, EPI>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
    case 3:
      return launch_cfg<RBW, 3, EPI>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
    case 4:
      return launch_cfg<RBW, 4, EPI>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
    case 6:
      if constexpr (RBW != 4) return launch_cfg<RBW, 6, EPI>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
      break;
    case 8:
      if constexpr (RBW != 4) return launch_cfg<RBW, 8, EPI>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
      break;
    default:
      break;
  }
  return hipErrorInvalidValue;
}

template <int EPI>
hipError_t launch_epi(const SkinnyPlan& p, const void* w, const void* x, int ldx, void* y, int ldy,
                      const void* residual, int ldr, int M, int NB, int KT, void* workspace, hipStream_t stream) {
  switch (p.rows / kTileRows) {
    case 1:
      if constexpr (EPI != static_cast<int>(Epilogue::kSiluMul))
        return launch_rbw<1, EPI>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
      break;
    case 2:
      return launch_rbw<2, EPI>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
    case 4:
      return launch_rbw<4, EPI>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
    case 5:
      if constexpr (EPI == static_cast<int>(Epilogue::kSiluMul))
        return launch_rbw<5, EPI>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
      break;
    default:
      break;
  }
  return hipErrorInvalidValue;
}

}  // namespace

// CUs of the current device (cached per device): the skinny split covers them.
hipError_t current_device_cus(int* cus_out) {
  static std::mutex mu;
  static std::vector<int> cache;
  int device = 0;
  hipError_t err = hipGetDevice(&device);
  if (err != hipSuccess) return err;
  std::lock_guard<std::mutex> lock(mu);
  if (device >= (int)cache.size()) cache.resize(device + 1, 0);
  if (cache[device] == 0) {
    int cus = 0;
    err = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    if (err != hipSuccess) return err;
    cache[device] = cus > 0 ? cus : 1;
  }
  *cus_out = cache[device];
  return hipSuccess;
}

// Token groups a call of M rows computes (5 and 7 run as 6 and 8: the LDS
// sum takes whole chunks).
int skinny_groups(int M) {
  const int mg = (M + kTileRows - 1) / kTileRows;
  return mg == 5 ? 6 : mg == 7 ? 8 : mg;
}

// Whether lsk_linear_bf16 runs M rows of an [N, K] projection on the skinny
// kernel: 17..64 rows always; 65..128 rows unless N is wide (>= 8192) and on
// the 128 x 128 GEMM's grid, whose blocks then fill the chip and read each
// activation fragment once per 128 weight rows instead of once per 32 --
// except with SiLU*up, where units of 8 outputs give every CU 80 weight rows
// in one round (19456 x 2560 at 128 rows: 32.6 us, the GEMM 56 us) and the
// GEMM catches up as N needs more rounds and K leaves fewer steps in each (at
// 128 rows 22016 x 1024 29 us, the GEMM 25; 28672 x 2048 50 and 46, x 3072 65
// and 68; 57344 x 2560 95 and 73; at 96 rows 28672 x 2048 41 and 44, 22016 x 1024
// 24.4 and 23.5, 19456 x 512 12.0 and 13.3).
//
// 9..16 rows with SiLU*up too when every CU gets four units or more (N >=
// 16384; 19.7 us at 12 rows of 19456 x 2560, the decode kernel 22.0) and K
// streams for a while (22016 x 512 7.5 us, the decode kernel 6.5; x 1024 11.0 and
// 11.4); there a call has no workspace.
bool skinny_route(int M, int N, int K, bool silu) {
  if (M <= 8 || M > kSkinnyMaxM || N % kTileRows != 0 || K % kTileK != 0) return false;
  if (M <= kDecodeMaxM) return silu && N >= 16384 && K >= 1024;
  const bool gemm_grid = N % kGemmBN == 0 && K % kGemmBK == 0;
  if (M <= 64 || !gemm_grid || N < 8192) return true;
  if (!silu) return false;
  if (N <= 20480) return N <= 8192 || K >= 768 || (K >= 512 && (M <= 96 || N < 12288));
  if (N <= 24576) return K >= 2048;
  return N <= 40960 && K >= (M <= 96 ? 2048 : 3072);
}

// Row-blocks per workgroup and the K split, from sweeps of (rows, S) over the
// Qwen3-4B projections at 17, 32, 64 and 128 rows on 256 CUs.  Two row-blocks
// per workgroup by default, since the activations are read once for all of
// them (QKV at 32 rows: 10.0 us with two, 13.2 with one, 10.9 with four in two
// splits; o_proj at 64 rows 10.8 with two in three splits, 17.9 with one in
// two, 13.4 with four in six); one for narrow N (fewer than 64 pairs of
// row-blocks) and for up to 32 rows when the row-blocks are one round of the
// CUs by themselves; four (up to 64 rows) when two would take more than one
// round of the CUs and four still cover half of them.  SiLU*up takes as many
// units per workgroup as bring them to one round: five for the 1216 units of
// 19456 rows (21.3 us at 32 rows; four, in two rounds, 28.6).  Past one round of
// fives: two, which overlap (above), up to 32 rows and up to three rounds of
// them (22016 x 2560: 22.3 us at 17 rows, fives 32.2, fours 28.4; 33 at 64 rows,
// 42 and 37), else four or five by the rounds they take (28672 x 2560 at 64 rows
// 38 us in fours, 43 in twos and fives; 40960 48 in fives, 55 in twos).  Two also
// for 16384 rows at up to 16 tokens (x 2560 at 12 15.9 us, fours 17.0).  With a
// workspace the K range is split so that the grid comes to about one
// workgroup per CU, each split keeping at least 16 k-tiles; a second split
// that leaves the CUs two rounds costs more than it balances (QKV at 64 rows
// 12.8 -> 17.9 us).
SkinnyPlan skinny_plan(int M, int N, int K, bool silu, int cus, bool has_workspace) {
  const int NB = N / kTileRows;
  const int KT = K / kTileK;
  const int mg = skinny_groups(M);
  int rbw = 2;
  if (silu) {  // NB units of 8 outputs
    auto rounds = [&](int r) { return ((NB + r - 1) / r + cus - 1) / cus; };
    if (rounds(5) == 1) {
      if (NB > 2 * cus && (mg > 1 || NB > 4 * cus)) rbw = mg <= 4 && NB <= 4 * cus ? 4 : 5;
    } else if (mg > 2 && NB > 6 * cus) {
      rbw = mg <= 4 && 7 * rounds(4) <= 8 * rounds(5) ? 4 : 5;
    }
  } else if ((mg <= 2 && NB >= cus && NB <= cus + cus / 8) || NB / 2 < 64 || NB % 2 != 0) {
    rbw = 1;
  } else if (mg <= 4 && NB % 4 == 0 && NB / 2 > cus && NB / 4 <= cus && 2 * (NB / 4) >= cus) {
    rbw = 4;
  }
  const int groups = (NB + rbw - 1) / rbw;
  int S = 1;
  const int max_s = KT / 16;
  if (has_workspace && skinny_route(M, N, K, false) && groups <= kSkinnyMaxGroups && max_s >= 2) {
    S = (4 * cus + groups) / (4 * groups);  // floor(cus / groups + 1/4)
    if (S > max_s) S = max_s;
    if (S < 1) S = 1;
  }
  SkinnyPlan p;
  p.rows = kTileRows * rbw;
  p.groups = groups;
  p.S = S;
  p.bytes = p.S > 1 ? kSkPartialsOffset + (size_t)p.groups * p.S * rbw * mg * 1024 : 0;
  return p;
}

hipError_t launch_skinny_linear(const void* w, int N, int K, const void* x, int M, int ldx, void* y, int ldy,
                                Epilogue epi, const void* residual, int ldr, void* workspace, size_t ws_bytes,
                                int cus, hipStream_t stream) {
  const bool silu = epi == Epilogue::kSiluMul;
  SkinnyPlan p = skinny_plan(M, N, K, silu, cus, workspace != nullptr);
  if (p.S > 1 && ws_bytes < p.bytes) return hipErrorInvalidValue;  // checked by the caller
  const int NB = N / kTileRows;
  const int KT = K / kTileK;
  switch (epi) {
    case Epilogue::kSiluMul:
      return launch_epi<1>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
    case Epilogue::kResidualAdd:
      return launch_epi<2>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
    case Epilogue::kNone:
    default:
      return launch_epi<0>(p, w, x, ldx, y, ldy, residual, ldr, M, NB, KT, workspace, stream);
  }
}

}  // namespace lsk
