// Single-token GQA decode attention (fp16/bf16 KV) for gfx950, split over the KV
// sequence.  Semantics follow the reference kernel (triton_kernels.py:15-109):
// softmax(q.k * head_dim^-0.5) v in binary32 with an optional per-head sink that
// joins the softmax denominator but carries no value.
//
// Order of evaluation (restated in oracle/tt_oracle.c):
//   * the KV sequence is cut into chunks of 64 tokens; one wave handles one
//     (kv_head, chunk) for all query heads of that KV head;
//   * score_t = (fma chain over d ascending of q_d k_td) * scale;
//   * chunk max m_c (order free), p_t = exp(score_t - m_c), l_c = butterfly sum of p
//     over the 64 token lanes, o_c[d] = fma chain over the chunk's tokens ascending;
//   * combine in chunk order: M = max(sink, m_c...), den starts at exp(sink - M)
//     (or 0), den = fma(l_c, e_c, den), acc_d = fma(o_c[d], e_c, acc_d) with
//     e_c = exp(m_c - M); out_d = acc_d / den.
// The active token count may be read from device memory (count = tokens_dev[0] +
// tokens, so a decode step can pass its position and 1) so graph replays follow the
// growing cache; chunks past the count exit without work.  The count is clamped to
// max_tokens so a runaway device counter can never read past the cache.
//
// Four forms, all with these bits: for contiguous head_dim-64 caches one launch of small
// grids (attn_kvchunk_kernel), and its partials with a fold (attn_fold_kernel) of middling
// ones; matrix-core partials (attn_mfma_kernel) and the fold for everything else of head_dim
// 64 or 128; scalar loads for the rest (attn_partial_kernel, attn_combine_kernel).  Where the
// host knows the count only its chunks are launched.
#include "tt_abi_internal.h"
#include "tt_common.h"

#include <type_traits>

namespace tt {

constexpr int kChunk = 64;

struct AttnParams {
  const void* q;          // [heads, D]
  const void* keys;       // [kv_heads, tokens, D] with strides
  const void* values;
  int64_t k_head, k_tok, v_head, v_tok;
  const void* sinks;      // [heads] or null
  const int32_t* tokens_dev;
  int tokens;
  float* part_m;          // [heads, max_chunks]
  float* part_l;
  float* part_o;          // [heads, max_chunks, D]
  int heads, kv_heads, head_dim, max_chunks, max_tokens;
  int grid_chunks;        // chunks launched: those of the count where the host knows it
  float scale;
  void* out;              // [heads, D]
};

// Any head_dim up to 256, strides and alignment: scalar loads.
template <typename T, int G>
__device__ void attn_chunk(const AttnParams& P, int kvh, int c, int T_act) {
  const int D = P.head_dim;
  const int lane = threadIdx.x;
  __shared__ float q_s[G * 256];
  __shared__ float p_s[G * kChunk];
  const int h0 = kvh * G;
  for (int i = lane; i < G * D; i += 64) q_s[i] = to_f32(reinterpret_cast<const T*>(P.q)[(int64_t)h0 * D + i]);
  __syncthreads();
  // phase 1: lane = token
  const int t = c * kChunk + lane;
  const bool valid = t < T_act;
  const int nt = min(kChunk, T_act - c * kChunk);
  float sc[G];
#pragma unroll
  for (int g = 0; g < G; g++) sc[g] = 0.0f;
  const T* krow = reinterpret_cast<const T*>(P.keys) + kvh * P.k_head + (int64_t)(valid ? t : 0) * P.k_tok;
  for (int d = 0; d < D; d++) {
    const float kv = to_f32(krow[d]);
#pragma unroll
    for (int g = 0; g < G; g++) sc[g] = __builtin_fmaf(q_s[g * D + d], kv, sc[g]);
  }
  const float ninf = __builtin_bit_cast(float, 0xff800000u);
#pragma unroll
  for (int g = 0; g < G; g++) {
    float s = valid ? sc[g] * P.scale : ninf;
    float m = s;
    // chunk max (order-independent)
    m = fmaxf(m, xor_partner<1>(m));
    m = fmaxf(m, xor_partner<2>(m));
    m = fmaxf(m, xor_partner<4>(m));
    m = fmaxf(m, xor_partner<8>(m));
    m = fmaxf(m, xor_partner<16>(m));
    m = fmaxf(m, xor_partner<32>(m));
    const float p = valid ? exp_f32(s - m) : 0.0f;
    const float l = xor_sum(p, 1, 64);
    p_s[g * kChunk + lane] = p;
    if (lane == 0) {
      P.part_m[(int64_t)(h0 + g) * P.max_chunks + c] = m;
      P.part_l[(int64_t)(h0 + g) * P.max_chunks + c] = l;
    }
  }
  __syncthreads();
  // phase 2: lane = dimension, o = fma chain over the chunk's tokens ascending
  for (int d = lane; d < D; d += 64) {
    float o[G];
#pragma unroll
    for (int g = 0; g < G; g++) o[g] = 0.0f;
    const T* vcol = reinterpret_cast<const T*>(P.values) + kvh * P.v_head + (int64_t)(c * kChunk) * P.v_tok + d;
    for (int tt = 0; tt < nt; tt++) {
      const float vv = to_f32(vcol[(int64_t)tt * P.v_tok]);
#pragma unroll
      for (int g = 0; g < G; g++) o[g] = __builtin_fmaf(p_s[g * kChunk + tt], vv, o[g]);
    }
#pragma unroll
    for (int g = 0; g < G; g++) P.part_o[((int64_t)(h0 + g) * P.max_chunks + c) * D + d] = o[g];
  }
}

template <typename T, int G>
__global__ __launch_bounds__(64) void attn_partial_kernel(AttnParams P) {
  const int kvh = blockIdx.y;
  const int c = blockIdx.x;
  const int T_act = min(P.tokens_dev ? P.tokens_dev[0] + P.tokens : P.tokens, P.max_tokens);
  if (c * kChunk < T_act) attn_chunk<T, G>(P, kvh, c, T_act);
}

// Combine of one head, same arithmetic as the sequential description above: the
// chunk metadata is loaded one chunk per lane, exp(m_c - M) is evaluated per lane and
// the chunk-order folds read it back lane by lane.  One wave.
template <typename T, typename SKT>
__device__ void combine_head(const AttnParams& P, int h, int lane) {
  const int T_act = min(P.tokens_dev ? P.tokens_dev[0] + P.tokens : P.tokens, P.max_tokens);
  const int nc = T_act > 0 ? (T_act + kChunk - 1) / kChunk : 0;
  const float* pm = P.part_m + (int64_t)h * P.max_chunks;
  const float* pl = P.part_l + (int64_t)h * P.max_chunks;
  const float ninf = __builtin_bit_cast(float, 0xff800000u);
  float M = ninf;
  const bool has_sink = P.sinks != nullptr;
  float sink = 0.0f;
  if (has_sink) {
    sink = to_f32(reinterpret_cast<const SKT*>(P.sinks)[h]);
    M = sink;
  }
  // the maximum ignores NaN and does not depend on the order
  for (int c0 = 0; c0 < nc; c0 += 64) {
    float m = c0 + lane < nc ? pm[c0 + lane] : ninf;
    m = fmaxf(m, xor_partner<1>(m));
    m = fmaxf(m, xor_partner<2>(m));
    m = fmaxf(m, xor_partner<4>(m));
    m = fmaxf(m, xor_partner<8>(m));
    m = fmaxf(m, xor_partner<16>(m));
    m = fmaxf(m, xor_partner<32>(m));
    M = fmaxf(M, m);
  }
  float den = has_sink ? exp_f32(sink - M) : 0.0f;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const int D = P.head_dim;
  for (int c0 = 0; c0 < nc; c0 += 64) {
    const int n = min(64, nc - c0);
    const float e = c0 + lane < nc ? exp_f32(pm[c0 + lane] - M) : 0.0f;
    const float l = c0 + lane < nc ? pl[c0 + lane] : 0.0f;
    for (int c1 = 0; c1 < n; c1 += 8) {
      // partials of eight chunks are loaded before they are folded in chunk order
      float po[8][4];
#pragma unroll
      for (int u = 0; u < 8; u++) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int d = lane + 64 * q;
          po[u][q] = (c1 + u < n && d < D) ? P.part_o[((int64_t)h * P.max_chunks + c0 + c1 + u) * D + d] : 0.0f;
        }
      }
#pragma unroll
      for (int u = 0; u < 8; u++) {
        if (c1 + u < n) {
          const int c = c1 + u;
          const float ec = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, e), c));
          const float lc = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, l), c));
          den = __builtin_fmaf(lc, ec, den);
#pragma unroll
          for (int q = 0; q < 4; q++) acc[q] = __builtin_fmaf(po[u][q], ec, acc[q]);
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int d = lane + 64 * q;
    if (d < D) store<T>(reinterpret_cast<T*>(P.out) + (int64_t)h * D + d, acc[q] / den);
  }
}

template <typename T, typename SKT>
__global__ __launch_bounds__(64) void attn_combine_kernel(AttnParams P) {
  combine_head<T, SKT>(P, blockIdx.x, threadIdx.x);
}

// One workgroup per (KV head, chunk) with one wave per query head of that KV head
// (contiguous head_dim-64 caches, whole-chunk capacity): the chunk's K and V blocks are
// read once per KV head -- each CU moves 16 KB instead of a whole sequence -- staged in
// LDS (K row r's piece d at slot 8r + (d xor r mod 8), V rows of tokens past the count zeroed), and
// wave g computes the chunk partial of query head G kvh + g with the arithmetic of
// attn_chunk.  The partials go to the scratch with device-scope atomic stores;
// the workgroup counts itself in its KV head's arrival counter once its stores have
// completed, and the last of the head's active chunks combines every query head of the
// KV head in chunk order (the arithmetic of combine_head, partials read with
// device-scope atomic loads) and resets the counter to zero.  No workgroup waits for
// another.
__device__ __forceinline__ void st_dev(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float ld_dev(const float* p) {
  return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Grids of at most kOneLaunchChunks chunks combine.  Without COMBINE the partials are the
// result; there a grid of many chunks may lie mostly past the count, which is then read first
// (COUNT_FIRST, above kCountFirstChunks: 100 tokens of 256 chunks, 32 / 8 heads with the o_proj
// GEMV: 15.5 -> 10.9 us, full 112 -> 111).
constexpr int kOneLaunchChunks = 32;
constexpr int kCountFirstChunks = 64;

template <typename T, typename SKT, int G, bool COMBINE = true, bool COUNT_FIRST = false>
__global__ __launch_bounds__(64 * G) void attn_kvchunk_kernel(AttnParams P, int* counters) {
  constexpr int D = 64;
  const int c = blockIdx.x, kvh = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int h = kvh * G + wave;
  constexpr int nthr = 64 * G;
  __shared__ uint4 ks[kChunk * D / 8], vs_s[kChunk * D / 8];
  __shared__ float q_s[G][D];
  __shared__ float p_s[G][kChunk];
  __shared__ int last;
  const float ninf = __builtin_bit_cast(float, 0xff800000u);
  if (COUNT_FIRST && c * kChunk >= (P.tokens_dev ? P.tokens_dev[0] + P.tokens : P.tokens)) return;
  // every load before the active count is known (chunks below max_chunks are inside the
  // capacity): K and V pieces of the chunk, this wave's query row
  constexpr int kPer = kChunk * D / 8 / nthr;   // 16-byte pieces per thread
  // (native 4-vectors: arrays of the uint4 struct type are kept in scratch memory here)
  typedef uint32_t piece_t __attribute__((ext_vector_type(4)));
  piece_t kr[kPer], vr[kPer];
  {
    const piece_t* kblk = reinterpret_cast<const piece_t*>(reinterpret_cast<const T*>(P.keys) + kvh * P.k_head) +
                          (int64_t)c * (kChunk * D / 8);
    const piece_t* vblk = reinterpret_cast<const piece_t*>(reinterpret_cast<const T*>(P.values) + kvh * P.v_head) +
                          (int64_t)c * (kChunk * D / 8);
#pragma unroll
    for (int j = 0; j < kPer; j++) {
      kr[j] = kblk[(int)threadIdx.x + nthr * j];
      vr[j] = vblk[(int)threadIdx.x + nthr * j];
    }
  }
  const T qraw = reinterpret_cast<const T*>(P.q)[(int64_t)h * D + lane];
  const int T_act = min(P.tokens_dev ? P.tokens_dev[0] + P.tokens : P.tokens, P.max_tokens);
  const int nc = T_act > 0 ? (T_act + kChunk - 1) / kChunk : 0;
  if (c >= nc) return;
  q_s[wave][lane] = to_f32(qraw);
  {
    const int nt = min(kChunk, T_act - c * kChunk);
#pragma unroll
    for (int j = 0; j < kPer; j++) {
      const int pidx = (int)threadIdx.x + nthr * j;
      const int r = pidx >> 3, col = pidx & 7;
      reinterpret_cast<piece_t*>(ks)[r * 8 + (col ^ (r & 7))] = kr[j];
      const uint32_t keep = r < nt ? ~0u : 0u;
      reinterpret_cast<piece_t*>(vs_s)[pidx] = vr[j] & keep;
    }
    __syncthreads();

    // ---- chunk partial of query head h (lane = token, then lane = dimension)
    const int t = c * kChunk + lane;
    const bool valid = t < T_act;
    uint32_t krow[8][4];
#pragma unroll
    for (int d = 0; d < 8; d++) {
      const uint4 k = ks[lane * 8 + (d ^ (lane & 7))];
      krow[d][0] = k.x; krow[d][1] = k.y; krow[d][2] = k.z; krow[d][3] = k.w;
    }
    const float* qw = q_s[wave];
    float sc = 0.0f;
#pragma unroll
    for (int i = 0; i < D / 8; i++) {
      if ((i & 3) == 0) asm volatile("" : "+v"(sc)::"memory");
      const uint32_t* kw = krow[i];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float kv = (e & 1) ? hi_f32<T>(kw[e >> 1]) : lo_f32<T>(kw[e >> 1]);
        sc = __builtin_fmaf(qw[8 * i + e], kv, sc);
      }
    }
    const float s = valid ? sc * P.scale : ninf;
    float m = s;
    m = fmaxf(m, xor_partner<1>(m));
    m = fmaxf(m, xor_partner<2>(m));
    m = fmaxf(m, xor_partner<4>(m));
    m = fmaxf(m, xor_partner<8>(m));
    m = fmaxf(m, xor_partner<16>(m));
    m = fmaxf(m, xor_partner<32>(m));
    const float p = valid ? exp_f32(s - m) : 0.0f;
    const float l = xor_sum(p, 1, 64);
    float* p_w = p_s[wave];
    p_w[lane] = p;
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave's p stores done
    __builtin_amdgcn_wave_barrier();
    const T* vsp = reinterpret_cast<const T*>(vs_s);
    float o = 0.0f;
#pragma unroll
    for (int tt = 0; tt < kChunk; tt++) {
      if ((tt & 31) == 0) asm volatile("" : "+v"(o)::"memory");
      o = __builtin_fmaf(p_w[tt], to_f32(vsp[tt * D + lane]), o);
    }
    const int64_t slot = (int64_t)h * P.max_chunks + c;
    if (lane == 0) {
      st_dev(P.part_m + slot, m);
      st_dev(P.part_l + slot, l);
    }
    st_dev(P.part_o + slot * D + lane, o);
  }
  // without COMBINE the partials are the result: the kernel that consumes them runs after
  // this one on the stream
  if constexpr (!COMBINE) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(counters + kvh, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nc - 1;
  __syncthreads();
  if (!last) return;

  // ---- combine of query head h in chunk order (combine_head's arithmetic); (m, l) and the
  // partial rows of every chunk are requested together with the sink, one round trip, before
  // the maximum is formed
  const float* pm = P.part_m + (int64_t)h * P.max_chunks;
  const float* pl = P.part_l + (int64_t)h * P.max_chunks;
  const float* po = P.part_o + (int64_t)h * P.max_chunks * D + lane;
  const bool has_sink = P.sinks != nullptr;
  const float mc = lane < nc ? ld_dev(pm + lane) : ninf;
  const float lv = lane < nc ? ld_dev(pl + lane) : 0.0f;
  float ov[kOneLaunchChunks];
#pragma unroll
  for (int u = 0; u < kOneLaunchChunks; u++) ov[u] = u < nc ? ld_dev(po + (int64_t)u * D) : 0.0f;
  const float sink = has_sink ? to_f32(reinterpret_cast<const SKT*>(P.sinks)[h]) : 0.0f;
  float M = mc;
  M = fmaxf(M, xor_partner<1>(M));
  M = fmaxf(M, xor_partner<2>(M));
  M = fmaxf(M, xor_partner<4>(M));
  M = fmaxf(M, xor_partner<8>(M));
  M = fmaxf(M, xor_partner<16>(M));
  M = fmaxf(M, xor_partner<32>(M));
  if (has_sink) M = fmaxf(sink, M);
  float den = has_sink ? exp_f32(sink - M) : 0.0f;
  float acc = 0.0f;
  const float e = lane < nc ? exp_f32(mc - M) : 0.0f;
#pragma unroll
  for (int u = 0; u < kOneLaunchChunks; u++) {
    if (u < nc) {
      const float ec = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, e), u));
      const float lc = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, lv), u));
      den = __builtin_fmaf(lc, ec, den);
      acc = __builtin_fmaf(ov[u], ec, acc);
    }
  }
  store<T>(reinterpret_cast<T*>(P.out) + (int64_t)h * D + lane, acc / den);
  if (threadIdx.x == 0) __hip_atomic_store(counters + kvh, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------- matrix-core partials
// Chunk partials of head_dim 64 or 128 on the binary32 matrix cores: v_mfma_f32_4x4x1
// multiplies, in sixteen blocks, a column of four rows by a row of four columns and adds the
// products with one rounding each (a fused multiply-add, subnormals included; checked
// against fmaf chains), so instruction k of a sequence is step k of sixty-four fma chains
// for each of four query heads:
//   * scores: lane = token, operand B its K row's element k, operand A the four heads' q_k;
//     accumulator register g is head g's chain over d ascending;
//   * values: lane = dimension (head_dim 128: two per lane), B the token's V element, A the
//     four heads' p of the token.
// One wave computes four query heads of one (KV head, chunk) -- K and V elements are
// converted once for the four -- and a workgroup all heads of the KV head: it reads the active
// count, then requests K, V and query rows together, K staged in LDS (rows xor-swizzled) for
// the scores while V arrives.  Only rows below the count are read (a caller's cache need not
// hold max_tokens rows); rows past it repeat the last one and are staged as zeros for V (p is
// 0 there, and fma(0, 0, o) == o).  Any token stride: caches of a whole number of chunks or
// not.
//
// Partials and fold against what ran before (microseconds a call, graph-timed, caches in
// rotation): heads / KV heads x head_dim, tokens -- 64 / 8 x 64, 32768: 77 -> 31 (one wave
// per query head and one workgroup per KV head folding 512 chunks); 512 / 64 x 64, 4096: 46 ->
// 27; 40 / 10 x 128, 4001: 30.8 -> 14.7; 64 / 8 x 128, 32768: 148 -> 49.5 (2.7 TB/s; both
// scalar loads before; they are faster only for 20 tokens or fewer, 8 / 8 x 128, 16 tokens:
// 8.0 against 8.8).  Past a few thousand tokens the partials bound it:
// 64 / 8 x 64, 16385 tokens: 17 us of partials and 6 of the fold under the profiler; 4112 waves
// of about 595 vector, 128 matrix and 118 LDS instructions, the matrix cores busy 15% of the
// time, and the latency of 2 x 64 dependent MFMAs rather than memory.
typedef float acc4_t __attribute__((ext_vector_type(4)));

template <typename T, int G, int D>
__global__ __launch_bounds__(64 * ((G + 3) / 4)) void attn_mfma_kernel(AttnParams P) {
  static_assert(D == 64 || D == 128, "one or two dimensions per lane");
  constexpr int W = (G + 3) / 4;                // waves, four query heads each
  constexpr int HW = G < 4 ? G : 4;
  constexpr int NV = D / 64;                    // dimensions per lane
  constexpr int kRow = D / 8;                   // 16-byte pieces per row
  constexpr int kPer = kChunk * kRow / (64 * W);   // pieces per thread
  typedef uint32_t quad_t __attribute__((ext_vector_type(4)));
  __shared__ quad_t kvs[kChunk * kRow];         // the K block, then the V block
  __shared__ __attribute__((aligned(16))) float q_s[W][HW][D];
  __shared__ __attribute__((aligned(16))) float p_s[W][HW][kChunk];
  const int c = blockIdx.x, kvh = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int h0 = kvh * G + 4 * wave;
  const int row = (lane & 3) < HW ? (lane & 3) : HW - 1;   // head of this lane's A operand
  const T* kbase = reinterpret_cast<const T*>(P.keys) + kvh * P.k_head;
  const T* vbase = reinterpret_cast<const T*>(P.values) + kvh * P.v_head;
  const int T_act = min(P.tokens_dev ? P.tokens_dev[0] + P.tokens : P.tokens, P.max_tokens);
  if (c * kChunk >= T_act) return;
  quad_t kr[kPer], vr[kPer];
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    const int f = (int)threadIdx.x + 64 * W * j;
    const int64_t t = min(c * kChunk + f / kRow, T_act - 1);
    kr[j] = *reinterpret_cast<const quad_t*>(kbase + t * P.k_tok + 8 * (f % kRow));
  }
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    const int f = (int)threadIdx.x + 64 * W * j;
    const int64_t t = min(c * kChunk + f / kRow, T_act - 1);
    vr[j] = *reinterpret_cast<const quad_t*>(vbase + t * P.v_tok + 8 * (f % kRow));
  }
  T qraw[HW][NV];
#pragma unroll
  for (int g = 0; g < HW; g++)
#pragma unroll
    for (int n = 0; n < NV; n++) qraw[g][n] = reinterpret_cast<const T*>(P.q)[(int64_t)(h0 + g) * D + 64 * n + lane];
  __builtin_amdgcn_sched_barrier(0);   // every load above is requested first
  const int t = c * kChunk + lane;
  const bool valid = t < T_act;
  const int nt = min(kChunk, T_act - c * kChunk);
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    const int f = (int)threadIdx.x + 64 * W * j;
    const int r = f / kRow, col = f % kRow;
    kvs[r * kRow + (col ^ (r & (kRow - 1)))] = kr[j];
  }
#pragma unroll
  for (int g = 0; g < HW; g++)
#pragma unroll
    for (int n = 0; n < NV; n++) q_s[wave][g][64 * n + lane] = to_f32(qraw[g][n]);
  lds_barrier();

  acc4_t sc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < kRow; i++) {
    const quad_t k8 = kvs[lane * kRow + (i ^ (lane & (kRow - 1)))];
    const acc4_t qa = *reinterpret_cast<const acc4_t*>(&q_s[wave][row][8 * i]);
    const acc4_t qb = *reinterpret_cast<const acc4_t*>(&q_s[wave][row][8 * i + 4]);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint32_t kw = k8[e >> 1];
      const float kv = (e & 1) ? hi_f32<T>(kw) : lo_f32<T>(kw);
      sc = __builtin_amdgcn_mfma_f32_4x4x1f32(e < 4 ? qa[e & 3] : qb[e & 3], kv, sc, 0, 0, 0);
    }
  }
  if constexpr (W > 1) lds_barrier();   // every wave has read its K rows
  // V pieces of tokens past the count as zeros
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    const int f = (int)threadIdx.x + 64 * W * j;
    const uint32_t keep = f / kRow < nt ? ~0u : 0u;
    kvs[f] = vr[j] & keep;
  }
  const float ninf = __builtin_bit_cast(float, 0xff800000u);
  float sv[HW], m[HW], l[HW];
#pragma unroll
  for (int g = 0; g < HW; g++) m[g] = sv[g] = valid ? sc[g] * P.scale : ninf;
#pragma unroll
  for (int g = 0; g < HW; g++) m[g] = fmaxf(m[g], xor_partner<1>(m[g]));
#pragma unroll
  for (int g = 0; g < HW; g++) m[g] = fmaxf(m[g], xor_partner<2>(m[g]));
#pragma unroll
  for (int g = 0; g < HW; g++) m[g] = fmaxf(m[g], xor_partner<4>(m[g]));
#pragma unroll
  for (int g = 0; g < HW; g++) m[g] = fmaxf(m[g], xor_partner<8>(m[g]));
#pragma unroll
  for (int g = 0; g < HW; g++) m[g] = fmaxf(m[g], xor_partner<16>(m[g]));
#pragma unroll
  for (int g = 0; g < HW; g++) m[g] = fmaxf(m[g], xor_partner<32>(m[g]));
#pragma unroll
  for (int g = 0; g < HW; g++) {
    l[g] = valid ? exp_f32(sv[g] - m[g]) : 0.0f;
    p_s[wave][g][lane] = l[g];
  }
  lds_barrier();   // p and V are staged
  acc4_t o[NV];
#pragma unroll
  for (int n = 0; n < NV; n++) o[n] = (acc4_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int t4 = 0; t4 < kChunk / 4; t4++) {
    const acc4_t pa = *reinterpret_cast<const acc4_t*>(&p_s[wave][row][4 * t4]);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int tt = 4 * t4 + e;
      if constexpr (D == 64) {
        const T v = reinterpret_cast<const T*>(kvs)[tt * D + lane];
        o[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(pa[e], to_f32(v), o[0], 0, 0, 0);
      } else {
        const uint32_t w = reinterpret_cast<const uint32_t*>(kvs)[tt * 64 + lane];
        o[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(pa[e], lo_f32<T>(w), o[0], 0, 0, 0);
        o[NV - 1] = __builtin_amdgcn_mfma_f32_4x4x1f32(pa[e], hi_f32<T>(w), o[NV - 1], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int g = 0; g < HW; g++) l[g] = xor_sum(l[g], 1, 64);
#pragma unroll
  for (int g = 0; g < HW; g++) {
    const int64_t slot = (int64_t)(h0 + g) * P.max_chunks + c;
    if (lane == 0) {
      P.part_m[slot] = m[g];
      P.part_l[slot] = l[g];
    }
    if constexpr (D == 64) {
      P.part_o[slot * D + lane] = o[0][g];
    } else {
      typedef float f2_t __attribute__((ext_vector_type(2), aligned(4)));
      *reinterpret_cast<f2_t*>(P.part_o + slot * D + 2 * lane) = (f2_t){o[0][g], o[NV - 1][g]};
    }
  }
}

// Fold of the chunk partials in chunk order (the arithmetic of combine_head), one workgroup
// per (head, 64 dimensions).  Blocks of kFoldBlk chunks: the four waves request the block's
// rows together (16 bytes a thread and load), leave them with e_c = exp(m_c - M) and l_c in
// LDS, wave 0 runs the chains of the 64 dimensions and wave 1 the denominator's.
constexpr int kFoldBlk = 128;

// acc = fma(v[u STEP], e[u], acc) for u = 0 .. n - 1 in order, the next sixteen operands read
// from LDS while sixteen are consumed (reads past n stay inside the kFoldBlk entries).
template <int STEP>
__device__ __forceinline__ void chain_step(const float* v, const float* e, int n, float& acc) {
  float ov[2][16];
  acc4_t ev[2][4];
  auto load = [&](auto bc, int u) __attribute__((always_inline)) {
    constexpr int b = decltype(bc)::value;
#pragma unroll
    for (int k = 0; k < 4; k++) ev[b][k] = *reinterpret_cast<const acc4_t*>(e + u + 4 * k);
#pragma unroll
    for (int k = 0; k < 16; k++) ov[b][k] = v[(u + k) * STEP];
  };
  auto use = [&](auto bc) __attribute__((always_inline)) {
    constexpr int b = decltype(bc)::value;
#pragma unroll
    for (int k = 0; k < 16; k++) acc = __builtin_fmaf(ov[b][k], ev[b][k >> 2][k & 3], acc);
  };
  const std::integral_constant<int, 0> b0{};
  const std::integral_constant<int, 1> b1{};
  int u = 0;
  load(b0, 0);
  for (; u + 32 <= n; u += 32) {
    load(b1, u + 16);
    use(b0);
    load(b0, u + 32 < kFoldBlk ? u + 32 : 0);
    use(b1);
  }
  if (u + 16 <= n) {
    use(b0);
    u += 16;
  }
  for (; u < n; u++) acc = __builtin_fmaf(v[u * STEP], e[u], acc);
}

template <typename T, typename SKT>
__global__ __launch_bounds__(256) void attn_fold_kernel(AttnParams P) {
  const int h = blockIdx.x, d0 = 64 * blockIdx.y, D = P.head_dim;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  __shared__ __attribute__((aligned(16))) float rows[2][kFoldBlk][64];
  __shared__ __attribute__((aligned(16))) float e_s[2][kFoldBlk], l_s[2][kFoldBlk];
  __shared__ float red[4], den;
  const float* pm = P.part_m + (int64_t)h * P.max_chunks;
  const float* pl = P.part_l + (int64_t)h * P.max_chunks;
  const float* po = P.part_o + (int64_t)h * P.max_chunks * D + d0;
  // the scratch's rows start at any multiple of eight bytes (2 heads max_chunks floats precede them)
  typedef acc4_t row4_t __attribute__((aligned(4)));
  acc4_t rr[kFoldBlk / 16];
  float mr = 0.0f, lr = 0.0f;
  auto request = [&](int c0, int last) __attribute__((always_inline)) {
    const int cm = min(c0 + (tid & (kFoldBlk - 1)), last);
    mr = pm[cm];
    lr = pl[cm];
#pragma unroll
    for (int u = 0; u < kFoldBlk / 16; u++) {
      const int cc = min(c0 + 16 * u + (tid >> 4), last);
      rr[u] = *reinterpret_cast<const row4_t*>(po + (int64_t)cc * D + 4 * (tid & 15));
    }
  };
  const float ninf = __builtin_bit_cast(float, 0xff800000u);
  const bool has_sink = P.sinks != nullptr;
  const float sink = has_sink ? to_f32(reinterpret_cast<const SKT*>(P.sinks)[h]) : 0.0f;
  const int T_act = min(P.tokens_dev ? P.tokens_dev[0] + P.tokens : P.tokens, P.max_tokens);
  const int nc = T_act > 0 ? (T_act + kChunk - 1) / kChunk : 0;
  const int last = nc > 0 ? nc - 1 : 0;
  request(0, last);
  float mm = ninf;   // the maximum ignores NaN and does not depend on the order
  for (int c = tid; c < nc; c += 256) mm = fmaxf(mm, pm[c]);
  mm = fmaxf(mm, xor_partner<1>(mm));
  mm = fmaxf(mm, xor_partner<2>(mm));
  mm = fmaxf(mm, xor_partner<4>(mm));
  mm = fmaxf(mm, xor_partner<8>(mm));
  mm = fmaxf(mm, xor_partner<16>(mm));
  mm = fmaxf(mm, xor_partner<32>(mm));
  if (lane == 0) red[wave] = mm;
  lds_barrier();
  float M = has_sink ? sink : ninf;
  M = fmaxf(fmaxf(M, fmaxf(red[0], red[1])), fmaxf(red[2], red[3]));
  float acc = wave == 1 && has_sink ? exp_f32(sink - M) : 0.0f;   // wave 1: the denominator
  int buf = 0;
  for (int c0 = 0; c0 < nc; c0 += kFoldBlk, buf ^= 1) {
    if (tid < kFoldBlk) {
      e_s[buf][tid] = exp_f32(mr - M);
      l_s[buf][tid] = lr;
    }
#pragma unroll
    for (int u = 0; u < kFoldBlk / 16; u++)
      *reinterpret_cast<acc4_t*>(&rows[buf][16 * u + (tid >> 4)][4 * (tid & 15)]) = rr[u];
    if (c0 + kFoldBlk < nc) request(c0 + kFoldBlk, last);
    lds_barrier();   // alternating buffers: one barrier per block
    const int n = min(kFoldBlk, nc - c0);
    if (wave == 0) chain_step<64>(&rows[buf][0][lane], &e_s[buf][0], n, acc);
    else if (wave == 1) chain_step<1>(&l_s[buf][0], &e_s[buf][0], n, acc);
  }
  if (tid == 64) den = acc;
  __syncthreads();
  if (wave == 0) store<T>(reinterpret_cast<T*>(P.out) + (int64_t)h * D + d0 + lane, acc / den);
}

template <typename T>
static int launch_fold(const AttnParams& P, int sink_dtype, hipStream_t st) {
  const dim3 grid(P.heads, P.head_dim / 64);
  switch (sink_dtype) {
    case TT_BF16: hipLaunchKernelGGL((attn_fold_kernel<T, bf16_t>), grid, dim3(256), 0, st, P); break;
    case TT_F32: hipLaunchKernelGGL((attn_fold_kernel<T, float>), grid, dim3(256), 0, st, P); break;
    default: hipLaunchKernelGGL((attn_fold_kernel<T, f16_t>), grid, dim3(256), 0, st, P); break;
  }
  return check_launch("gqa_attention");
}

// Operands that attn_mfma_kernel reads as they are: 16-byte pieces of K and V rows.
static bool mfma_operands(const AttnParams& P) {
  return (P.head_dim == 64 || P.head_dim == 128) && aligned(P.keys, 16) && P.k_tok % 8 == 0 &&
         P.k_head % 8 == 0 && aligned(P.values, 16) && P.v_tok % 8 == 0 && P.v_head % 8 == 0;
}

// Chunk partials of contiguous head_dim-64 caches of whole chunks: attn_kvchunk_kernel without
// its arrival count and combine, for the fold or for a consumer that combines the partials
// itself (tt_attention_combine_int4_matvec; matrix-core partials were slower there below the
// largest grids: 32 / 8 heads with the GEMV, 33 chunks 8.0 - 18.5 us against 10.0 - 20.0, 256
// chunks, full, 112 against 111).
template <typename T, int G>
static int launch_kvchunk_partials(const AttnParams& P, hipStream_t st) {
  const dim3 grid((unsigned)P.grid_chunks, (unsigned)P.kv_heads), block(64 * G);
  if (P.grid_chunks > kCountFirstChunks)
    hipLaunchKernelGGL((attn_kvchunk_kernel<T, f16_t, G, false, true>), grid, block, 0, st, P, nullptr);
  else
    hipLaunchKernelGGL((attn_kvchunk_kernel<T, f16_t, G, false, false>), grid, block, 0, st, P, nullptr);
  return check_launch("gqa_attention_partials");
}

template <typename T, int G>
static int launch_mfma_partials(const AttnParams& P, hipStream_t st) {
  const dim3 grid((unsigned)P.grid_chunks, (unsigned)P.kv_heads), block(64 * ((G + 3) / 4));
  if (P.head_dim == 64) hipLaunchKernelGGL((attn_mfma_kernel<T, G, 64>), grid, block, 0, st, P);
  else hipLaunchKernelGGL((attn_mfma_kernel<T, G, 128>), grid, block, 0, st, P);
  return check_launch("gqa_attention");
}

// Grids that one launch serves better than partials and fold, where the second launch costs
// more than the last workgroup's fold: one workgroup per CU and, of a count the host knows, 20
// chunks (64 / 8 heads: 16 chunks 7.7 us in one launch against 7.8 in two, 32 chunks 10.0
// against 8.7); a count that only the device knows is taken to be half the capacity or more
// (33 chunks: 64 tokens 6.2 against 7.3 us, 1000 tokens 8.0 against 7.8, all 11.9 against
// 8.9).  Several workgroups per CU while their fold is short (512 / 64 heads: 9 chunks, 288
// tokens, 8.4 against 9.8 us, full 11.3 against 11.0; 16 chunks 17.9 against 12.5).
static bool one_launch_grid(const AttnParams& P) {
  const int64_t groups = (int64_t)P.grid_chunks * P.kv_heads;
  if (P.grid_chunks <= 10) return 2 * groups <= 5 * device_cus();
  return P.grid_chunks <= (P.tokens_dev ? kOneLaunchChunks : 20) && groups <= device_cus();
}

// Partials of one wave per query head: where the chip holds most of the waves at once they
// end sooner than the matrix-core partials, whose two chains of 64 dependent MFMAs take about
// 1.5 us more than fused multiply-adds (with the fold, 64 / 8 heads: 33 chunks 10.4 -> 8.9
// us, 192 chunks 18.3 -> 17.3, 256 chunks 19.5 -> 20.4; 512 / 64 heads: 24 chunks 17.1 ->
// 15.6, 32 chunks 17.1 -> 17.8; 100 tokens of 64 chunks, 64 / 8 heads, 10.5 -> 8.6).
static bool head_wave_grid(const AttnParams& P) { return (int64_t)P.grid_chunks * P.heads <= 48 * device_cus(); }

template <typename T, int G>
static int launch_attn(const AttnParams& P, int sink_dtype, bool contiguous64, int* counters, hipStream_t st) {
  if constexpr (G <= 8) {
    if (contiguous64 && counters != nullptr && one_launch_grid(P)) {
      const dim3 block(64 * G), grid((unsigned)P.grid_chunks, (unsigned)P.kv_heads);
      switch (sink_dtype) {
        case TT_BF16: hipLaunchKernelGGL((attn_kvchunk_kernel<T, bf16_t, G>), grid, block, 0, st, P, counters); break;
        case TT_F32: hipLaunchKernelGGL((attn_kvchunk_kernel<T, float, G>), grid, block, 0, st, P, counters); break;
        default: hipLaunchKernelGGL((attn_kvchunk_kernel<T, f16_t, G>), grid, block, 0, st, P, counters); break;
      }
      return check_launch("gqa_attention");
    }
    if (contiguous64 && head_wave_grid(P)) {
      const int rc = launch_kvchunk_partials<T, G>(P, st);
      return rc ? rc : launch_fold<T>(P, sink_dtype, st);
    }
  }
  if (mfma_operands(P)) {
    const int rc = launch_mfma_partials<T, G>(P, st);
    return rc ? rc : launch_fold<T>(P, sink_dtype, st);
  }
  hipLaunchKernelGGL((attn_partial_kernel<T, G>), dim3(P.grid_chunks, P.kv_heads), dim3(64), 0, st, P);
  int rc = check_launch("gqa_attention");
  if (rc) return rc;
  switch (sink_dtype) {
    case TT_BF16: hipLaunchKernelGGL((attn_combine_kernel<T, bf16_t>), dim3(P.heads), dim3(64), 0, st, P); break;
    case TT_F32: hipLaunchKernelGGL((attn_combine_kernel<T, float>), dim3(P.heads), dim3(64), 0, st, P); break;
    default: hipLaunchKernelGGL((attn_combine_kernel<T, f16_t>), dim3(P.heads), dim3(64), 0, st, P); break;
  }
  return check_launch("gqa_attention");
}

}  // namespace tt

using namespace tt;


extern "C" int tt_attention_scratch_floats(int64_t heads, int64_t max_tokens, int64_t head_dim) {
  const int64_t chunks = (max_tokens + kChunk - 1) / kChunk;
  return (int)(kAttnCounters + heads * chunks * (2 + head_dim));
}

extern "C" int tt_single_token_gqa_attention_partials(const void* q, const void* keys, const void* values, int dtype,
                                                      int64_t k_head, int64_t k_tok, int64_t v_head, int64_t v_tok,
                                                      const int32_t* tokens_dev, int64_t tokens, int64_t max_tokens,
                                                      int64_t heads, int64_t kv_heads, int64_t head_dim, float* scratch,
                                                      int64_t scratch_floats, void* stream) {
  const char* what = "single_token_gqa_attention_partials";
  TT_REQUIRE(q && keys && values && scratch, "%s: null pointer", what);
  TT_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "%s: heads must be a multiple of kv_heads", what);
  TT_REQUIRE(tokens_dev != nullptr || (tokens > 0 && tokens <= max_tokens), "%s: attention requires at least one KV token", what);
  TT_REQUIRE(tokens_dev == nullptr || (tokens >= 0 && tokens <= 1), "%s: device token count offset must be 0 or 1", what);
  TT_REQUIRE(max_tokens > 0 && kv_heads <= 65535, "%s: bad max_tokens / kv_heads", what);
  const int64_t chunks = (max_tokens + kChunk - 1) / kChunk;
  TT_REQUIRE(chunks <= 65535, "%s: sequence too long", what);
  TT_REQUIRE(scratch_floats >= kAttnCounters + heads * chunks * (2 + head_dim), "%s: scratch too small", what);
  const int64_t G = heads / kv_heads;
  TT_UNSUPPORTED(head_dim == 64 && k_tok == 64 && v_tok == 64 && max_tokens % kChunk == 0 && aligned(keys, 16) &&
                     aligned(values, 16) && k_head % 8 == 0 && v_head % 8 == 0 && (G == 1 || G == 2 || G == 4 || G == 8),
                 "%s: needs contiguous head_dim-64 caches whose capacity is a multiple of %d tokens and 1, 2, 4 or 8 "
                 "query heads per KV head", what, kChunk);
  AttnParams P{};
  P.q = q; P.keys = keys; P.values = values;
  P.k_head = k_head; P.k_tok = k_tok; P.v_head = v_head; P.v_tok = v_tok;
  P.sinks = nullptr; P.tokens_dev = tokens_dev; P.tokens = (int)tokens;
  scratch += kAttnCounters;
  P.part_m = scratch;
  P.part_l = scratch + heads * chunks;
  P.part_o = scratch + 2 * heads * chunks;
  P.heads = (int)heads; P.kv_heads = (int)kv_heads; P.head_dim = (int)head_dim; P.max_chunks = (int)chunks;
  P.max_tokens = (int)max_tokens;
  P.grid_chunks = (int)(tokens_dev ? chunks : (tokens + kChunk - 1) / kChunk);
  P.scale = (float)(1.0 / __builtin_sqrt((double)head_dim));
  P.out = nullptr;
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto by_g = [&](auto t) -> int {
    using T = decltype(t);
    switch (G) {
      case 1: return launch_kvchunk_partials<T, 1>(P, st);
      case 2: return launch_kvchunk_partials<T, 2>(P, st);
      case 4: return launch_kvchunk_partials<T, 4>(P, st);
      default: return launch_kvchunk_partials<T, 8>(P, st);
    }
  };
  if (dtype == TT_F16) return by_g(f16_t{});
  if (dtype == TT_BF16) return by_g(bf16_t{});
  set_error("%s: KV dtype must be fp16 or bf16", what);
  return TT_ERR_INVALID;
}

extern "C" int tt_single_token_gqa_attention(const void* q, const void* keys, const void* values, int dtype,
                                             int64_t k_head, int64_t k_tok, int64_t v_head, int64_t v_tok,
                                             const void* sinks, int sink_dtype, const int32_t* tokens_dev,
                                             int64_t tokens, int64_t max_tokens, int64_t heads, int64_t kv_heads,
                                             int64_t head_dim, float* scratch, int64_t scratch_floats, void* out,
                                             void* stream) {
  const char* what = "single_token_gqa_attention";
  TT_REQUIRE(q && keys && values && out && scratch, "%s: null pointer", what);
  TT_REQUIRE(head_dim > 0 && head_dim <= 256, "%s: fused single-token attention supports head_dim <= 256", what);
  TT_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "%s: heads must be a multiple of kv_heads", what);
  TT_REQUIRE(tokens_dev != nullptr || (tokens > 0 && tokens <= max_tokens), "%s: attention requires at least one KV token", what);
  TT_REQUIRE(tokens_dev == nullptr || (tokens >= 0 && tokens <= 1), "%s: device token count offset must be 0 or 1", what);
  TT_REQUIRE(max_tokens > 0, "%s: bad max_tokens", what);
  const int64_t chunks = (max_tokens + kChunk - 1) / kChunk;
  TT_REQUIRE(scratch_floats >= kAttnCounters + heads * chunks * (2 + head_dim), "%s: scratch too small", what);
  int* counters = kv_heads <= kAttnCounters ? reinterpret_cast<int*>(scratch) : nullptr;
  scratch += kAttnCounters;
  TT_REQUIRE(chunks <= 65535 && kv_heads <= 65535, "%s: sequence too long", what);
  AttnParams P{};
  P.q = q; P.keys = keys; P.values = values;
  P.k_head = k_head; P.k_tok = k_tok; P.v_head = v_head; P.v_tok = v_tok;
  P.sinks = sinks; P.tokens_dev = tokens_dev; P.tokens = (int)tokens;
  P.part_m = scratch;
  P.part_l = scratch + heads * chunks;
  P.part_o = scratch + 2 * heads * chunks;
  P.heads = (int)heads; P.kv_heads = (int)kv_heads; P.head_dim = (int)head_dim; P.max_chunks = (int)chunks;
  P.max_tokens = (int)max_tokens;
  P.grid_chunks = (int)(tokens_dev ? chunks : (tokens + kChunk - 1) / kChunk);
  P.scale = (float)(1.0 / __builtin_sqrt((double)head_dim));
  P.out = out;
  const int G = (int)(heads / kv_heads);
  hipStream_t st = static_cast<hipStream_t>(stream);
  // 128-bit K loads and whole-chunk V loads need contiguous 64-wide rows and a
  // capacity that is a whole number of chunks
  const bool c64 = head_dim == 64 && k_tok == 64 && v_tok == 64 && max_tokens % kChunk == 0 && aligned(keys, 16) &&
                   aligned(values, 16) && k_head % 8 == 0 && v_head % 8 == 0 && heads / kv_heads <= 8;
  auto by_g = [&](auto t) -> int {
    using T = decltype(t);
    switch (G) {
      case 1: return launch_attn<T, 1>(P, sink_dtype, c64, counters, st);
      case 2: return launch_attn<T, 2>(P, sink_dtype, c64, counters, st);
      case 4: return launch_attn<T, 4>(P, sink_dtype, c64, counters, st);
      case 8: return launch_attn<T, 8>(P, sink_dtype, c64, counters, st);
      case 16: return launch_attn<T, 16>(P, sink_dtype, c64, counters, st);
    }
    set_error("%s: query heads per KV head must be 1, 2, 4, 8 or 16 (got %d)", what, G);
    return TT_ERR_UNSUPPORTED;
  };
  if (dtype == TT_F16) return by_g(f16_t{});
  if (dtype == TT_BF16) return by_g(bf16_t{});
  set_error("%s: KV dtype must be fp16 or bf16", what);
  return TT_ERR_INVALID;
}
