// Decode attention (one new token) for gfx950: the work between the QKV and
// o_proj projections of a Qwen3 decode layer, in one launch.
//
// Per (kv head j, chunk of the rows attended) one workgroup of 8 waves, from
// the raw QKV projection row (attention_rows_per_chunk: one chunk up to 128
// rows, 64-row chunks up to 512 rows, then at most 32 chunks of 128, 256,
// 384 or 512 rows):
//   1. q heads jG..jG+G-1 and k head j: RMSNorm over head_dim with the q / k
//      norm weights, then rotate-half RoPE with this position's cos / sin
//      (src/leanstack/runtime/qwen_explicit.py:796-806, :690-716), in the
//      reference's bf16 rounding chain: bf16(x*r*w) for the norm (torch's
//      fused F.rms_norm order (x*r)*w), and a bf16 rounding after every
//      multiply and every add / subtract of the rotation;
//   2. k and v of the token appended to the static cache at row `pos`
//      (src/leanstack/runtime/kv_cache.py:222-245, batch 1);
//   3. softmax(q K^T * scale) V over rows 0..pos of kv head j for its G q
//      heads (F.scaled_dot_product_attention with enable_gqa, no mask:
//      qwen_explicit.py:894-912), scores and softmax in fp32, output bf16.
//
// Scores run on MFMA: 16 cache rows x 32 dims of K form the A operand
// (one 16-byte load per lane, straight from the row-major cache) and the G
// bf16 q heads, padded to 16 columns, the B operand.  Softmax weights and P.V
// are fp32 on the VALU, each wave over its 16-row groups, weights through the
// wave's own LDS; the waves' partial sums are added in wave order.  A context
// longer than one chunk leaves each chunk's (max, sum, unnormalised P.V) in
// the workspace; the workgroup that arrives last for kv head j combines the
// chunks in chunk order and re-arms the head's counter.  Every sum has a fixed
// order, so results are bitwise reproducible.  The new row is read from LDS,
// not back from the cache it was just written to.
//
// Bound: latency up to some 4096 rows, then the cache bytes (67 MB at 16384
// rows of 8 kv heads, 9.9 us at the chip's streaming rate) and the steps after
// the last of them.  Cache rows by counted buffer loads, half of V
// after the scores, one barrier around the softmax instead of three, and the
// combine in 16-byte loads and unrolled LDS reads: 5.9 -> 5.7 us at 128 rows,
// 9.2 -> 9.15 at 1088, 14.1 -> 12.6 at 4001, 24.1 -> 20.85 at 16384 (position
// read from the device, 36 launches per graph).

#include <hip/hip_runtime.h>

#include "lsk_internal.h"

namespace lsk {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kHeadDim = kAttnHeadDim;
constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;

struct AttnArgs {
  const __bf16* qkv;       // [n_q*d | n_kv*d | n_kv*d]; kGiven: the q heads, [n_q*d]
  const __bf16* q_norm_w;  // [d]
  const __bf16* k_norm_w;  // [d]
  const __bf16* cos;       // [d/2], this position
  const __bf16* sin;       // [d/2]
  __bf16* k_cache;         // [n_kv][s_max][d], this layer; kGiven: [n_kv] blocks of rows, kv_stride apart
  __bf16* v_cache;
  size_t kv_stride;        // elements from one kv head's rows to the next one's
  __bf16* out;             // [n_q*d]
  unsigned* counters;      // workspace: one arrival counter per kv head
  unsigned char* partials; // workspace: one AttnPartial slot per (kv head, chunk)
  unsigned partial_bytes;  // bytes of all slots of this launch
  int n_q, n_kv, s_max, pos, chunks;  // chunks of attention_rows_per_chunk(pos + 1) rows
  float eps, scale;
  int grid_chunks;                    // workgroups per kv head in the grid (>= chunks)
  const int* pos_ptr;                 // device-resident pos (then cos / sin are whole tables)
};

constexpr int kCoherent = 16;  // device-coherent buffer access (partials cross XCDs)
// A buffer offset past every partial slot (num_records is at most 2^31 - 1):
// the load returns zero without a memory access.
constexpr unsigned kOutOfRange = 0x80000000u;
constexpr unsigned kRawBufferDword3 = 0x00020000u;
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// One chunk's softmax state for its G heads: running max m, sum l, and the
// unnormalised P.V rows, in floats at slot offset: m[G], l[G], then acc[G][d].
__host__ __device__ constexpr unsigned partial_slot_bytes(int G) {
  return (unsigned)(G * 2 + G * kAttnHeadDim) * 4u + 12u & ~15u;
}

// The last workgroup of kv head j: M_h = max_c m_c and
// out = sum_c e^(m_c - M) acc_c / sum_c e^(m_c - M) l_c.  The workgroup's
// threads are up to 8 groups of 32 G; a group takes its share of up to MAX
// chunks in chunk order, four values of them per thread (16-byte loads: the 66 KB of 32 chunks come
// through one CU, and as single values they were four times the requests),
// and the groups' sums are added in order.  Every partial is requested in one
// round with the (m, l) pairs, those past the last chunk from outside the
// buffer's range, which returns zero and moves no data; their weight is 0.
template <int G, int MAX>
__device__ __forceinline__ void combine_chunks(const AttnArgs& a, __amdgpu_buffer_rsrc_t parts, unsigned first,
                                               unsigned slot_bytes, int j, float (*mx)[G], float (*lsum)[G],
                                               float (*wts)[G], float* sums) {
  constexpr int kQuads = G * kHeadDim / 4;
  // As many groups as `sums`, the memory of the waves' sums, has rows.
  constexpr int kGroups = kThreads / kQuads < kWaves ? kThreads / kQuads : kWaves;
  constexpr int kSlots = MAX / kGroups;
  const int quad = threadIdx.x % kQuads;
  const int grp = threadIdx.x / kQuads;
  // (m, l) of chunk k, head h, to thread kG + h.
  const int wk = threadIdx.x / G;
  const int wh = threadIdx.x - wk * G;
  const unsigned wbase = wk < a.chunks ? first + wk * slot_bytes : 0u;
  const unsigned wout = wk < a.chunks ? 0u : kOutOfRange;
  const float cm = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(parts, wout + (unsigned)wh * 4u,
                                                                                  wbase, kCoherent));
  const float cl = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                 parts, wout + (unsigned)(G + wh) * 4u, wbase, kCoherent));
  f32x4_t v[kSlots];
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    // Out of range goes in the vector offset: the range check covers the
    // vector and instruction offsets, not the scalar one.
    const int k = grp * kSlots + i;
    const unsigned off = (k < a.chunks && grp < kGroups ? first + (unsigned)k * slot_bytes : kOutOfRange) + (unsigned)(2 * G + 4 * quad) * 4u;
    v[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(parts, off, 0, kCoherent));
  }
  if (wk < MAX) {
    mx[wk][wh] = wk < a.chunks ? cm : -__builtin_huge_valf();
  }
  __syncthreads();
  // (Over all chunk slots, so that the LDS reads are issued together: a loop
  // over a.chunks pays an LDS access per chunk, 1.5 us of 32.)
  if (wk < MAX) {
    float m = -__builtin_huge_valf();
#pragma unroll
    for (int k = 0; k < MAX; ++k) m = fmaxf(m, mx[k][wh]);
    const float w = mx[wk][wh] != -__builtin_huge_valf() ? expf(mx[wk][wh] - m) : 0.f;
    wts[wk][wh] = w;
    lsum[wk][wh] = wk < a.chunks ? w * cl : 0.f;
  }
  __syncthreads();
  f32x4_t num = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < kSlots; ++i)
    num += wts[min(grp * kSlots + i, MAX - 1)][quad / (kHeadDim / 4)] * v[i];
  if (grp < kGroups) *reinterpret_cast<f32x4_t*>(sums + grp * G * kHeadDim + 4 * quad) = num;
  __syncthreads();
  for (int e = threadIdx.x; e < G * kHeadDim; e += kThreads) {
    const int h = e / kHeadDim;
    float s = sums[e], den = 0.f;
#pragma unroll
    for (int q = 1; q < kGroups; ++q) s += sums[q * G * kHeadDim + e];
#pragma unroll
    for (int k = 0; k < MAX; ++k) den += lsum[k][h];
    a.out[(size_t)(j * G) * kHeadDim + e] = static_cast<__bf16>(s / den);
  }
}

// Where the rows attended come from: a decode token at a position the host
// gives, one at a position read from device memory, or q heads and cached
// rows given as they are (no norms, no RoPE, no append: pos is the last row).
// kGiven takes the place of an fp32 softmax(q K^T) V in torch ops, which
// expanded and converted the caches on every call: 9.0 us against 95 us of
// kernels (and 13 launches) at 700 rows.
enum AttnMode { kHostPos, kDevicePos, kGiven };

// One chunk, rows row0 .. row0 + n - 1 of kv head j, of a chunk size that NU
// 16-row groups per wave cover: prologue items, scores, softmax weights and
// P.V.  Leaves each wave's P.V and weight sums in part and stat[1] (behind a
// barrier) and returns the chunk's maximum of head c (lanes c < G).
template <int G, int NU, AttnMode MODE>
__device__ __forceinline__ float attend_chunk(const AttnArgs& a, int j, int row0, int rows, int n,
                                              __bf16 (&qs)[16][kHeadDim], __bf16 (&kv_new)[2][kHeadDim],
                                              float (&pw)[kWaves][NU][4][4][G], float (&part)[kWaves][G][kHeadDim],
                                              float (&stat)[2][kWaves][G]) {
  constexpr int kGroups = NU;  // 16-row groups per wave
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int g = lane >> 4;
  const int c = lane & 15;
  // Wave w owns the chunk's 16-row groups w, w + 8, w + 16, ...: group u of
  // the wave starts at chunk row lb(u) = 16 (w + 8u).  Groups past the last
  // row are skipped, so short contexts cost little and the waves share the
  // rows evenly.
  auto lb = [&](int u) { return 16 * (wave + kWaves * u); };
  const bool has_new = MODE != kGiven && a.pos >= row0 && a.pos < row0 + rows;
  const int cached = MODE == kGiven ? a.pos + 1 : a.pos;  // rows read from the caches
  // ---- inputs of this wave's prologue items, loaded before the cache rows
  // so that the norms and rotations run while the rows stream in.  Item
  // i = wave + 8u: i < G is q head jG+i, i == G the k head j (only in the
  // chunk holding row pos).  Loads are unconditional (items past the last
  // read a q head again and store nothing): a load used only under a branch
  // may be sunk into it, behind the cache-row loads.  Lane l: dims l, l + 64.
  constexpr int kItems = (G + kWaves) / kWaves;  // ceil((G + 1) / kWaves)
  __bf16 px0[kItems], px1[kItems], pw0[kItems], pw1[kItems];
#pragma unroll
  for (int u = 0; u < kItems; ++u) {
    const int i = wave + kWaves * u;
    if constexpr (MODE == kGiven) {
      const __bf16* src = a.qkv + (size_t)(j * G + (i < G ? i : G - 1)) * kHeadDim;
      px0[u] = src[lane];
      px1[u] = src[lane + 64];
      continue;
    }
    const bool is_k = i == G;
    const int src_head = is_k ? a.n_q + j : j * G + (i < G ? i : G - 1);
    const __bf16* src = a.qkv + (size_t)src_head * kHeadDim;
    const __bf16* nw = is_k ? a.k_norm_w : a.q_norm_w;
    px0[u] = src[lane];
    px1[u] = src[lane + 64];
    pw0[u] = nw[lane];
    pw1[u] = nw[lane + 64];
  }
  __bf16 cs = __bf16(0.f), sn = __bf16(0.f);
  __bf16 v_new0 = __bf16(0.f), v_new1 = __bf16(0.f);
  if constexpr (MODE != kGiven) {
    cs = a.cos[lane];
    sn = a.sin[lane];
    const __bf16* vsrc = a.qkv + ((size_t)a.n_q + a.n_kv + j) * kHeadDim;
    v_new0 = vsrc[lane];
    v_new1 = vsrc[lane + 64];
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- cache rows of this wave (they do not depend on q).  K as MFMA A
  // fragments: group u, lane (g, c) = row lb(u) + c, dims 32kt + 8g .. +7.
  // V: lane (g, c) = dims 8c .. 8c+7 of rows lb(u) + 4i + g.  Row pos is this
  // token's (from LDS below); rows past it are not read.
  // Buffer loads over the cached rows: a row past them, or past the chunk,
  // lies beyond the buffer's range and reads as zero without a branch (with
  // one, the compiler cannot count the loads in flight and the prologue waits
  // for every row).  All K first, then V of the first half of the groups: a CU
  // takes only some 60 KB of loads at a time, so a wave with more than that to
  // issue gets to its prologue when the last one is accepted; the other half
  // goes out after the scores, while the first is multiplied.
  constexpr int kEarly = kGroups > 1 ? kGroups / 2 : 1;
  const unsigned cached_bytes = (unsigned)cached * (kHeadDim * 2);
  const __amdgpu_buffer_rsrc_t kbuf = __builtin_amdgcn_make_buffer_rsrc(
      a.k_cache + (size_t)j * a.kv_stride, (short)0, (int)cached_bytes, (int)kRawBufferDword3);
  const __amdgpu_buffer_rsrc_t vbuf = __builtin_amdgcn_make_buffer_rsrc(
      a.v_cache + (size_t)j * a.kv_stride, (short)0, (int)cached_bytes, (int)kRawBufferDword3);
  auto row_at = [&](int u, int r) {  // byte offset of row r of the wave's group u
    return (lb(u) < rows ? 0u : kOutOfRange) + (unsigned)(row0 + lb(u) + r) * (kHeadDim * 2);
  };
  bf16x8_t kf[kGroups][4];
  bf16x8_t vf[kGroups][4];
  auto load_v = [&](int u) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      vf[u][i] = __builtin_bit_cast(
          bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(vbuf, row_at(u, 4 * i + g) + 16 * c, 0, 0));
  };
  // A wave without rows loads none: its loads beyond the range move no data,
  // but go through the CU's address path in front of other waves' inputs.  The
  // inputs are waited for first: past the branch the compiler could not tell
  // them from the rows in flight and would wait for all.  The other side
  // defines the row registers in place (they are not used there), or each would
  // be copied, behind a wait, at the join.  Without / with the branch: 4.54 /
  // 4.35 us at 11 rows of a 576-row cache, 7.40 / 7.22 at 300, 9.05 / 9.15 at
  // 1088, 12.5 / 12.6 at 4001, 20.65 / 20.85 at 16384.  A second copy of the
  // prologue, or of the kernel, for waves with rows instead: as fast on its
  // own, 0.2 us slower between other kernels (instruction fetch).
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  if (16 * __builtin_amdgcn_readfirstlane(wave) < n) {
#pragma unroll
    for (int u = 0; u < kGroups; ++u)
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
        kf[u][kt] = __builtin_bit_cast(
            bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(kbuf, row_at(u, c) + 64 * kt + 16 * g, 0, 0));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kEarly; ++u) load_v(u);
  } else {
#pragma unroll
    for (int u = 0; u < kGroups; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        asm volatile("" : "=v"(kf[u][i]));
        if (u < kEarly) asm volatile("" : "=v"(vf[u][i]));
      }
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- the prologue items: RMSNorm, RoPE; k and v appended to the caches.
#pragma unroll
  for (int u = 0; u < kItems; ++u) {
    const int i = wave + kWaves * u;
    if constexpr (MODE == kGiven) {
      if (i < G) {
        qs[i][lane] = px0[u];
        qs[i][lane + 64] = px1[u];
      }
      continue;
    }
    const float x0 = static_cast<float>(px0[u]), x1 = static_cast<float>(px1[u]);
    const float cf = static_cast<float>(cs), sf = static_cast<float>(sn);
    const float r = inv_rms(wave_sum(x0 * x0 + x1 * x1), kHeadDim, a.eps);
    const float n0 = bf16_round((x0 * r) * static_cast<float>(pw0[u]));
    const float n1 = bf16_round((x1 * r) * static_cast<float>(pw1[u]));
    const __bf16 o0 = rope_half(n0, n1, cf, sf, -1.f);
    const __bf16 o1 = rope_half(n1, n0, cf, sf, 1.f);
    if (i < G) {
      qs[i][lane] = o0;
      qs[i][lane + 64] = o1;
    } else if (i == G && has_new) {
      kv_new[0][lane] = o0;
      kv_new[0][lane + 64] = o1;
      kv_new[1][lane] = v_new0;
      kv_new[1][lane + 64] = v_new1;
      __bf16* kc = a.k_cache + (size_t)j * a.kv_stride + (size_t)a.pos * kHeadDim;
      __bf16* vc = a.v_cache + (size_t)j * a.kv_stride + (size_t)a.pos * kHeadDim;
      kc[lane] = o0;
      kc[lane + 64] = o1;
      vc[lane] = v_new0;
      vc[lane + 64] = v_new1;
    }
  }
  for (int e = threadIdx.x; e < (16 - G) * kHeadDim; e += kThreads) qs[G + e / kHeadDim][e % kHeadDim] = __bf16(0.f);
  __syncthreads();

  // ---- scores: output lane (g, c) holds rows lb(u) + 4g .. +3 of head c.
  // This token's row pos, if it falls in one of the wave's groups, comes from
  // LDS.  (Unrolled selects: a runtime index would put kf / vf in scratch
  // memory.)
  const float kNegInf = -__builtin_huge_valf();
  bf16x8_t qf[4];
#pragma unroll
  for (int kt = 0; kt < 4; ++kt) qf[kt] = *reinterpret_cast<const bf16x8_t*>(&qs[c][32 * kt + 8 * g]);
  f32x4_t sv[kGroups];
  float mx = kNegInf;
#pragma unroll
  for (int u = 0; u < kGroups; ++u) {
    sv[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (lb(u) >= n) continue;
    if (has_new && c == a.pos - row0 - lb(u)) {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) kf[u][kt] = *reinterpret_cast<const bf16x8_t*>(&kv_new[0][32 * kt + 8 * g]);
    }
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) sv[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[u][kt], qf[kt], sv[u], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sv[u][i] *= a.scale;
      if (lb(u) + 4 * g + i < n) mx = fmaxf(mx, sv[u][i]);
    }
  }

  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = kEarly; u < kGroups; ++u) load_v(u);
  __builtin_amdgcn_sched_barrier(0);

  // ---- the chunk's maximum m per head, the weights e^(s - m) (to the wave's
  // own LDS, no barrier) and each wave's sum of them.  Rows that score -inf
  // weigh nothing, also in a chunk without others (m = -inf; a NaN beside them
  // stays NaN); a context of such rows alone gives 0 / 0 in the end, as
  // torch's softmax.
  mx = fmaxf(mx, __shfl_xor(mx, 16));
  mx = fmaxf(mx, __shfl_xor(mx, 32));
  if (g == 0 && c < G) stat[0][wave][c] = mx;
  __syncthreads();
  float m = kNegInf;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) m = fmaxf(m, stat[0][w][c < G ? c : 0]);
  float sum = 0.f;
#pragma unroll
  for (int u = 0; u < kGroups; ++u) {
    if (lb(u) >= n) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool live = lb(u) + 4 * g + i < n && sv[u][i] != kNegInf;
      const float e = live ? expf(sv[u][i] - m) : 0.f;
      sum += e;
      // P.V lane (g', c') takes rows 4i' + g' of every head: row 4g + i is
      // i' = g, g' = i.
      if (c < G) pw[wave][u][i][g][c] = e;
    }
  }
  sum += __shfl_xor(sum, 16);
  sum += __shfl_xor(sum, 32);
  if (g == 0 && c < G) stat[1][wave][c] = sum;
  wave_lds_order();

  // ---- P.V over this wave's groups: lane (g, c) sums rows lb(u) + 4i + g
  // for dims 8c .. 8c+7, then the four row phases g are added as
  // (g0 + g1) + (g2 + g3) by a reduce-scatter (each exchange sends half of
  // what a lane holds, so lane (g, c) ends with a quarter of the 8G sums),
  // and the waves' sums in wave order.
  float acc8[G][8];
#pragma unroll
  for (int h = 0; h < G; ++h)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc8[h][e] = 0.f;
#pragma unroll
  for (int u = 0; u < kGroups; ++u) {
    if (lb(u) >= n) continue;
    float pr[4][G];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int h = 0; h < G; ++h) pr[i][h] = pw[wave][u][g][i][h];
    if (has_new) {
      const int d = a.pos - row0 - lb(u);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (d == 4 * i + g) vf[u][i] = *reinterpret_cast<const bf16x8_t*>(&kv_new[1][8 * c]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int h = 0; h < G; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc8[h][e] += pr[i][h] * static_cast<float>(vf[u][i][e]);
  }
  constexpr int kHalf = 4 * G;  // of the 8G values (flat index q = 8h + e)
  const bool odd = g & 1, high = g >> 1;
  float half[kHalf];
#pragma unroll
  for (int q = 0; q < kHalf; ++q) {
    const float lo = acc8[q / 8][q % 8], hi = acc8[(q + kHalf) / 8][(q + kHalf) % 8];
    half[q] = (odd ? hi : lo) + __shfl_xor(odd ? lo : hi, 16);
  }
  // lane (g, c) now holds flat indices kHalf * odd + q, q < kHalf
  float quarter[kHalf / 2];
#pragma unroll
  for (int q = 0; q < kHalf / 2; ++q) {
    const float lo = half[q], hi = half[q + kHalf / 2];
    quarter[q] = (high ? hi : lo) + __shfl_xor(high ? lo : hi, 32);
  }
  const int q0 = kHalf * odd + (kHalf / 2) * high;
#pragma unroll
  for (int q = 0; q < kHalf / 2; ++q) part[wave][(q0 + q) / 8][8 * c + (q0 + q) % 8] = quarter[q];
  __syncthreads();
  return m;
}

// attend_chunk for the groups per wave that chunks of `rows` rows take, LO..NU.
template <int G, int U, int LO, int NU, AttnMode MODE>
__device__ __forceinline__ float attend_chunk_of(const AttnArgs& a, int j, int row0, int rows, int n,
                                                 __bf16 (&qs)[16][kHeadDim], __bf16 (&kv_new)[2][kHeadDim],
                                                 float (&pw)[kWaves][NU][4][4][G], float (&part)[kWaves][G][kHeadDim],
                                                 float (&stat)[2][kWaves][G]) {
  if constexpr (U > LO) {
    if (rows <= 16 * kWaves * (U - 1))
      return attend_chunk_of<G, U - 1, LO, NU, MODE>(a, j, row0, rows, n, qs, kv_new, pw, part, stat);
  }
  return attend_chunk<G, U, MODE>(a, j, row0, rows, n, qs, kv_new,
                                  reinterpret_cast<float (&)[kWaves][U][4][4][G]>(pw), part, stat);
}

// kDevicePos: pos is read from device memory (a.pos_ptr), cos / sin are the whole
// position tables ([s_max][d/2]), and the chunk size and count follow from
// pos here; the grid holds the most chunks max_seq_len can need and the
// workgroups past this pos's count leave at once.  A pos outside
// [0, s_max) leaves every buffer untouched.
//
// NU: groups per wave of the largest chunk that the launch can meet.  With the
// position on the device the chunk may be smaller, and the code for its own
// size runs (every workgroup of the launch the same; the largest, nearest in
// memory, first): the code for the largest would issue a load for every row that the chunk does not have, which moves
// no data but goes through the CU's address path (a 16384-row cache of 8 kv
// heads of 4 q heads, NU = 4: 7.5 -> 6.4 us at 128 rows, 9.9 -> 8.8 at 700, 10.8
// -> 9.6 at 1088, 12.1 -> 10.8 at 2000, 13.8 -> 12.7 at 4001).
template <int G, int NU, AttnMode MODE>
__global__ __launch_bounds__(kThreads) void decode_attention_kernel(AttnArgs args) {
  static_assert(G >= 1 && G <= 16, "q heads per kv head are the MFMA B columns");
  constexpr int kMaxChunks = kAttnMaxChunks;
  AttnArgs a = args;
  if constexpr (MODE == kDevicePos) {
    const int pos = *args.pos_ptr;
    if (pos < 0 || pos >= a.s_max) return;
    a.pos = pos;
    a.cos += (size_t)pos * (kHeadDim / 2);
    a.sin += (size_t)pos * (kHeadDim / 2);
  }
  // Rows per chunk (at most 16 kWaves NU: the launch picks NU for the largest chunk
  // it can meet) and the chunk count, as the host computes them.
  const int rows = attention_rows_per_chunk(a.pos + 1);
  a.chunks = (a.pos + rows) / rows;  // ceil((pos + 1) / rows)
  const int j = blockIdx.x / a.grid_chunks;
  const int ci = blockIdx.x - j * a.grid_chunks;
  if (ci >= a.chunks) return;
  const int L = a.pos + 1;
  const int row0 = ci * rows;
  const int n = min(rows, L - row0);  // filled rows of the chunk

  __shared__ __align__(16) __bf16 qs[16][kHeadDim];     // rotated q heads; rows >= G are zero
  __shared__ __align__(16) __bf16 kv_new[2][kHeadDim];  // this token's rotated k and its v
  // A wave's softmax weights e^(s - m) of its group u, row 4i + g: [g][i][head]
  __shared__ __align__(16) float pw[kWaves][NU][4][4][G];
  __shared__ __align__(16) float part[kWaves][G][kHeadDim];
  __shared__ float stat[2][kWaves][G];                  // each wave's max and sum
  __shared__ float cmax[kMaxChunks][G];                 // combine: chunk maxima m_c
  __shared__ float lsum[kMaxChunks][G];                 // combine: e^(m_c - M) l_c
  __shared__ float wts[kMaxChunks][G];                  // combine: e^(m_c - M)
  __shared__ int last;

  const float m = attend_chunk_of<G, NU, MODE == kDevicePos ? 1 : NU, NU, MODE>(a, j, row0, rows, n, qs, kv_new, pw,
                                                                           part, stat);

  // Sums over the waves, in wave order: the chunk's P.V of head h, dim d, and
  // its sum of weights.
  auto chunk_sum = [&](int h, int d) {
    float s = part[0][h][d];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) s += part[w][h][d];
    return s;
  };
  auto weight_sum = [&](int h) {
    float l = stat[1][0][h];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) l += stat[1][w][h];
    return l;
  };

  if (a.chunks == 1) {
    for (int e = threadIdx.x; e < G * kHeadDim; e += kThreads) {
      const int h = e / kHeadDim;
      const int d = e - h * kHeadDim;
      a.out[(size_t)(j * G + h) * kHeadDim + d] = static_cast<__bf16>(chunk_sum(h, d) / weight_sum(h));
    }
    return;
  }

  // ---- several chunks: publish (m, l, acc) to slot (j, ci) with
  // device-coherent stores; the last chunk of kv head j to arrive combines
  // all of them in chunk order (so the result does not depend on which
  // one), writes the output and re-arms the counter.  Nothing waits.
  const __amdgpu_buffer_rsrc_t parts =
      __builtin_amdgcn_make_buffer_rsrc(a.partials, (short)0, (int)a.partial_bytes, (int)kRawBufferDword3);
  const unsigned slot_bytes = partial_slot_bytes(G);
  const unsigned slot = (unsigned)(j * a.chunks + ci) * slot_bytes;
  for (int e = threadIdx.x; e < G * kHeadDim; e += kThreads) {
    const int h = e / kHeadDim;
    const int d = e - h * kHeadDim;
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, chunk_sum(h, d)), parts,
                                          (unsigned)(2 * G + e) * 4u, slot, kCoherent);
  }
  // Lanes c < G of every wave hold the chunk's maximum of head c.
  if (threadIdx.x < G) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, m), parts, threadIdx.x * 4u, slot, kCoherent);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, weight_sum(threadIdx.x)), parts,
                                          (unsigned)(G + threadIdx.x) * 4u, slot, kCoherent);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    last = __hip_atomic_fetch_add(a.counters + j, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           (unsigned)a.chunks - 1;
  }
  __syncthreads();
  if (!last) return;

  const unsigned first = (unsigned)(j * a.chunks) * slot_bytes;
  // (The waves' sums in `part` have been published: its memory takes the
  // groups' sums.)
  if (a.chunks <= 8)
    combine_chunks<G, 8>(a, parts, first, slot_bytes, j, cmax, lsum, wts, &part[0][0][0]);
  else
    combine_chunks<G, kMaxChunks>(a, parts, first, slot_bytes, j, cmax, lsum, wts, &part[0][0][0]);
  if (threadIdx.x == 0) __hip_atomic_store(a.counters + j, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int G, int NU, AttnMode MODE>
hipError_t launch_gu(const AttnArgs& a, hipStream_t stream) {
  launch_kernel(decode_attention_kernel<G, NU, MODE>, dim3(a.n_kv * a.grid_chunks), dim3(kThreads), 0, stream, a);
  return hipGetLastError();
}

template <int G, AttnMode MODE>
hipError_t launch_g(const AttnArgs& a, int nu, hipStream_t stream) {
  switch (nu) {
    case 1:
      return launch_gu<G, 1, MODE>(a, stream);
    case 2:
      return launch_gu<G, 2, MODE>(a, stream);
    case 3:
      return launch_gu<G, 3, MODE>(a, stream);
    case 4:
      return launch_gu<G, 4, MODE>(a, stream);
    default:
      return hipErrorInvalidValue;
  }
}

template <AttnMode MODE>
hipError_t launch_mode(const AttnArgs& a, int nu, hipStream_t stream) {
  switch (a.n_q / a.n_kv) {
    case 1:
      return launch_g<1, MODE>(a, nu, stream);
    case 2:
      return launch_g<2, MODE>(a, nu, stream);
    case 4:
      return launch_g<4, MODE>(a, nu, stream);
    case 8:
      return launch_g<8, MODE>(a, nu, stream);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace

int attention_chunk_rows(int rows) { return attention_rows_per_chunk(rows); }

size_t attention_workspace_bytes(int n_q, int n_kv, int max_seq_len) {
  const int group = n_q / n_kv;
  return kAttnPartialsOffset + (size_t)n_kv * attention_most_chunks(max_seq_len) * partial_slot_bytes(group);
}

namespace {

AttnArgs common_args(const void* qkv, int n_q, int n_kv, const void* q_norm_w, const void* k_norm_w, float eps,
                     const void* cos, const void* sin, void* k_cache, void* v_cache, int s_max, float scale,
                     void* out, void* workspace, size_t ws_bytes) {
  AttnArgs a;
  a.qkv = static_cast<const __bf16*>(qkv);
  a.q_norm_w = static_cast<const __bf16*>(q_norm_w);
  a.k_norm_w = static_cast<const __bf16*>(k_norm_w);
  a.cos = static_cast<const __bf16*>(cos);
  a.sin = static_cast<const __bf16*>(sin);
  a.k_cache = static_cast<__bf16*>(k_cache);
  a.v_cache = static_cast<__bf16*>(v_cache);
  a.out = static_cast<__bf16*>(out);
  a.n_q = n_q;
  a.n_kv = n_kv;
  a.s_max = s_max;
  a.kv_stride = (size_t)s_max * kHeadDim;
  a.pos = 0;
  a.chunks = 1;
  a.grid_chunks = 1;
  a.pos_ptr = nullptr;
  a.eps = eps;
  a.scale = scale;
  auto* ws = static_cast<unsigned char*>(workspace);
  a.counters = reinterpret_cast<unsigned*>(ws);
  a.partials = ws != nullptr ? ws + kAttnPartialsOffset : nullptr;
  const size_t pb = ws_bytes > kAttnPartialsOffset ? ws_bytes - kAttnPartialsOffset : 0;
  a.partial_bytes = (unsigned)(pb < 0x7fffffffu ? pb : 0x7fffffffu);
  return a;
}

}  // namespace

hipError_t launch_decode_attention(const void* qkv, int n_q, int n_kv, const void* q_norm_w, const void* k_norm_w,
                                   float eps, const void* cos, const void* sin, void* k_cache, void* v_cache,
                                   int s_max, int pos, float scale, void* out, void* workspace, size_t ws_bytes,
                                   hipStream_t stream) {
  AttnArgs a = common_args(qkv, n_q, n_kv, q_norm_w, k_norm_w, eps, cos, sin, k_cache, v_cache, s_max, scale, out,
                           workspace, ws_bytes);
  a.pos = pos;
  const int rows = attention_chunk_rows(pos + 1);
  const int nu = (rows + 127) / 128;  // 16-row groups per wave: 8 waves x 16 rows x nu cover the chunk
  a.chunks = (pos + 1 + rows - 1) / rows;
  a.grid_chunks = a.chunks;
  return launch_mode<kHostPos>(a, nu, stream);
}

hipError_t launch_gqa_attention(const void* q, int n_q, int n_kv, const void* k, const void* v, size_t kv_stride,
                                int rows, float scale, void* out, void* workspace, size_t ws_bytes,
                                hipStream_t stream) {
  AttnArgs a = common_args(q, n_q, n_kv, nullptr, nullptr, 0.f, nullptr, nullptr, const_cast<void*>(k),
                           const_cast<void*>(v), rows, scale, out, workspace, ws_bytes);
  a.kv_stride = kv_stride;
  a.pos = rows - 1;
  const int per_chunk = attention_chunk_rows(rows);
  a.chunks = (rows + per_chunk - 1) / per_chunk;
  a.grid_chunks = a.chunks;
  return launch_mode<kGiven>(a, (per_chunk + 127) / 128, stream);
}

int attention_grid_chunks(int max_seq_len) { return attention_most_chunks(max_seq_len); }

hipError_t launch_decode_attention_at(const void* qkv, int n_q, int n_kv, const void* q_norm_w, const void* k_norm_w,
                                      float eps, const void* cos_table, const void* sin_table, void* k_cache,
                                      void* v_cache, int s_max, const int* pos_device, float scale, void* out,
                                      void* workspace, size_t ws_bytes, hipStream_t stream) {
  AttnArgs a = common_args(qkv, n_q, n_kv, q_norm_w, k_norm_w, eps, cos_table, sin_table, k_cache, v_cache, s_max,
                           scale, out, workspace, ws_bytes);
  a.pos_ptr = pos_device;
  a.grid_chunks = attention_grid_chunks(s_max);
  // Chunks never exceed the size max_seq_len rows need (the rule grows with
  // the rows attended), so that size fixes the kernel's groups per wave.
  const int nu = (attention_chunk_rows(s_max) + 127) / 128;
  return launch_mode<kDevicePos>(a, nu, stream);
}

}  // namespace lsk
