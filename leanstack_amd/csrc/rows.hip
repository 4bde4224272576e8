// Row kernels between the projections of verify and prefill rows (M > 1) on
// gfx950, both HBM-bound streams with a little arithmetic per value:
//
//  * rms_rows_kernel: the RMSNorm of [M][K] rows that no projection computes in
//    its own prologue (src/leanstack/runtime/qwen_explicit.py:621-628).
//  * qk_rope_kernel: the q and k heads of the raw QKV rows -- per-head
//    RMSNorm, rotate-half RoPE and the [T, heads] -> [heads, T] reorder in one
//    pass (qwen_explicit.py:748-770, RoPE :690-716; :788-806 for one row).
//
// Rounding chain of both: bf16((x * r) * w) with r = 1/sqrt(mean + eps) in
// fp32, and for RoPE a bf16 rounding after every product and after the sum,
// as the reference's separate bf16 tensor ops round.

#include <hip/hip_runtime.h>

#include "lsk_internal.h"

namespace lsk {
namespace {

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kRowsThreads = 256;
constexpr int kRowsWaves = kRowsThreads / 64;

__device__ __forceinline__ float chunk_squares(bf16x8_t v) {
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float f = static_cast<float>(v[e]);
    s += f * f;
  }
  return s;
}

// bf16((x * r) * w) of 8 values.
__device__ __forceinline__ bf16x8_t norm_chunk(bf16x8_t x, bf16x8_t w, float r) {
  bf16x8_t o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = static_cast<__bf16>((static_cast<float>(x[e]) * r) * static_cast<float>(w[e]));
  return o;
}

// One wave per row, the row in registers (NC chunks of 8 values per lane,
// K = 512 NC), so x is read once and y written once: the bytes are the bound.
// Four rows per workgroup keep enough waves in flight at any M; a row per
// wave needs no LDS and no barrier.  K = 2560: 16.2 us at 8192 rows (84 MB,
// 5.2 TB/s, a large copy's rate; F.rms_norm 25.5 us), 3.2 us at 64 rows, where
// the launch is what is left.
template <int NC>
__global__ __launch_bounds__(kRowsThreads) void rms_rows_kernel(const __bf16* __restrict__ x, size_t ldx,
                                                                const __bf16* __restrict__ w,
                                                                __bf16* __restrict__ y, int M, float eps) {
  constexpr int K = NC * 512;
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kRowsWaves + (threadIdx.x >> 6);
  if (row >= M) return;
  const bf16x8_t* xr = reinterpret_cast<const bf16x8_t*>(x + (size_t)row * ldx) + lane;
  const bf16x8_t* wr = reinterpret_cast<const bf16x8_t*>(w) + lane;
  bf16x8_t xv[NC], wv[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) xv[i] = xr[i * 64];
#pragma unroll
  for (int i = 0; i < NC; ++i) wv[i] = wr[i * 64];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) ss += chunk_squares(xv[i]);
  const float r = inv_rms(wave_sum(ss), K, eps);
  bf16x8_t* yr = reinterpret_cast<bf16x8_t*>(y + (size_t)row * K) + lane;
#pragma unroll
  for (int i = 0; i < NC; ++i) yr[i * 64] = norm_chunk(xv[i], wv[i], r);
}

// 8 lanes per head: lane c holds dims 8c..8c+7 and 64+8c..64+8c+7, so both
// halves of a rotation pair are in one lane and the head's sum of squares is
// three DPP steps over the 8 lanes.  A wave takes 8 heads of one token (2 KB
// of the QKV row); the 4 waves of a workgroup take 4 consecutive tokens of
// the same heads, so a head's 4 output rows are 1 KB contiguous.  Bound by
// its bytes: 32 + 8 heads at 8192 rows (168 MB) 36 us, 4.7 TB/s, against
// 580 us of torch's norms, products, sums and concatenations; 3-5 us at
// 1..64 rows, against 60-80 us.
// Grid: (ceil(M / 4), ceil((n_q + n_kv) / 8)).
__global__ __launch_bounds__(kRowsThreads) void qk_rope_kernel(QkRopeArgs a) {
  const int lane = threadIdx.x & 63;
  const int c = lane & 7;
  const int row = blockIdx.x * kRowsWaves + (threadIdx.x >> 6);
  const int head = blockIdx.y * 8 + (lane >> 3);
  if (row >= a.M || head >= a.n_q + a.n_kv) return;
  const int b = row / a.T;
  const int t = row - b * a.T;
  const __bf16* src = a.qkv + (size_t)row * a.ld + (size_t)head * kAttnHeadDim + 8 * c;
  const bool is_q = head < a.n_q;
  const __bf16* nw = (is_q ? a.q_norm_w : a.k_norm_w) + 8 * c;
  const size_t pos = (size_t)b * a.rope_batch + (size_t)t * a.rope_row + 8 * c;
  const bf16x8_t x0 = *reinterpret_cast<const bf16x8_t*>(src);
  const bf16x8_t x1 = *reinterpret_cast<const bf16x8_t*>(src + 64);
  const bf16x8_t w0 = *reinterpret_cast<const bf16x8_t*>(nw);
  const bf16x8_t w1 = *reinterpret_cast<const bf16x8_t*>(nw + 64);
  const bf16x8_t cs = *reinterpret_cast<const bf16x8_t*>(a.cos + pos);
  const bf16x8_t sn = *reinterpret_cast<const bf16x8_t*>(a.sin + pos);
  float ss = chunk_squares(x0) + chunk_squares(x1);
  ss += dpp<0xb1>(ss);   // quad_perm [1,0,3,2]
  ss += dpp<0x4e>(ss);   // quad_perm [2,3,0,1]
  ss += dpp<0x141>(ss);  // row_half_mirror: the other quad of the 8 lanes
  const float r = inv_rms(ss, kAttnHeadDim, a.eps);
  const bf16x8_t n0 = norm_chunk(x0, w0, r);
  const bf16x8_t n1 = norm_chunk(x1, w1, r);
  bf16x8_t o0, o1;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float p = static_cast<float>(n0[e]), q = static_cast<float>(n1[e]);
    const float cc = static_cast<float>(cs[e]), s = static_cast<float>(sn[e]);
    o0[e] = rope_half(p, q, cc, s, -1.f);
    o1[e] = rope_half(q, p, cc, s, 1.f);
  }
  __bf16* dst = is_q ? a.q_out + (((size_t)b * a.n_q + head) * a.T + t) * kAttnHeadDim
                     : a.k_out + (((size_t)b * a.n_kv + (head - a.n_q)) * a.T + t) * kAttnHeadDim;
  *reinterpret_cast<bf16x8_t*>(dst + 8 * c) = o0;
  *reinterpret_cast<bf16x8_t*>(dst + 64 + 8 * c) = o1;
}

}  // namespace

hipError_t launch_rms_rows(const void* x, int M, int K, size_t ldx, const void* w, float eps, void* y,
                           hipStream_t stream) {
  const dim3 grid((M - 1) / kRowsWaves + 1);
  auto go = [&](auto* kernel) {
    launch_kernel(kernel, grid, dim3(kRowsThreads), 0, stream, static_cast<const __bf16*>(x), ldx,
                  static_cast<const __bf16*>(w), static_cast<__bf16*>(y), M, eps);
    return hipGetLastError();
  };
  switch (K / 512) {
    case 1: return go(rms_rows_kernel<1>);
    case 2: return go(rms_rows_kernel<2>);
    case 3: return go(rms_rows_kernel<3>);
    case 4: return go(rms_rows_kernel<4>);
    case 5: return go(rms_rows_kernel<5>);
    case 6: return go(rms_rows_kernel<6>);
    case 7: return go(rms_rows_kernel<7>);
    case 8: return go(rms_rows_kernel<8>);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_qk_rope(const QkRopeArgs& a, hipStream_t stream) {
  const dim3 grid((a.M - 1) / kRowsWaves + 1, (a.n_q + a.n_kv + 7) / 8);
  launch_kernel(qk_rope_kernel, grid, dim3(kRowsThreads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace lsk
