// y[m] = W x[m] for several fp16 activation rows on the binary32 matrix cores, with the
// bits of the single-row GEMV (the reduction order of tt_gemv.h) for every row.
//
// v_mfma_f32_16x16x1_4b_f32 multiplies one column of A (16 rows) by one row of B (16
// columns) in four independent blocks and adds the products to binary32 accumulators with
// one rounding each: a sequence of them is an ascending fma chain per output (checked
// against fmaf chains on random, zero and subnormal inputs; products of fp16 / fp8 values
// are exact in binary32 anyway).  So the reduction order maps onto it directly:
//   * a wave takes 16-row tiles of W; block b of the instruction holds chunk 4c + b of a
//     group c of four adjacent chunks, so lane (r = l % 16, b = l / 16) feeds the 32
//     columns of that chunk of weight row r and of activation row r, 32 instructions a
//     step, and the accumulators are the chunk partials of 16 x 16 outputs in four blocks;
//   * a lane's rounds (chunks LPR apart) are added in round order, register by register;
//     the butterfly over the LPR lanes of a row is the pairwise tree over adjacent chunks:
//     (b0 + b1) + (b2 + b3) inside a group, then pairs of groups, kept in the wave;
//   * the waves of a workgroup (four, or eight where there are few tiles) each own an equal
//     part of the groups -- a subtree -- and meet once per tile in LDS, again in pairs.
// Chunks past the end of K and rows past the end repeat valid addresses; their partials
// are replaced by +0 (chunks) or not stored (rows).
//
// Memory: both operands are requested coalesced one step ahead (16 pieces of 16 bytes
// cover the 256 bytes of a row's four fp16 chunks) and turned into the operand layout
// through a swizzled LDS buffer of the wave's own, so no barrier is needed for it.  (The form
// that takes four columns, 16x16x4, reads a quarter of the accumulators per instruction
// but wants a lane's columns four apart; regrouping them in LDS cost more than that saved:
// 345 -> 350 us for the 152064 x 5120 head at 16 rows, 43 -> 49 us for an fp8 17920 x 5120
// matrix.)
//
// What bounds it: up to four activation rows the weight stream; up to 16 conversions and
// matrix issue on top of it (matrix cores busy 29% of the time at 8 rows, 59% at 16, waves
// waiting to issue 57% and 67% of theirs); past it the binary32 matrix rate (130 - 140 TFLOP/s
// in a loop of these instructions alone, busy 60% at 32 rows).  152064 x 5120 fp16 head with
// argmax, against one GEMV-engine pass per eight (four, two, one) rows: 4 rows 276 -> 259 us
// (6.0 TB/s), 8 rows 339 -> 307, 16 rows 687 -> 341 (4.6 TB/s), 32 rows 1373 -> 603, 64 rows
// 2765 -> 1213 us (82 TFLOP/s); fp8 17920 x 5120, 8 rows 50.9 -> 34.7 us, 15 rows 110 -> 39
// us; fp16 2880 x 4096 + bias, 8 rows 15.7 -> 11.3 us.  Neither the grid, the interleaving of
// conversions and MFMAs nor a fragment pipeline across steps moved the 60%, all-zero operands
// gain 8% (power).
#include "gemv_impl.h"

#include <type_traits>

using namespace tt;

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16x __attribute__((ext_vector_type(16)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(3))) u4 lds_u4;

struct RowsParams {
  const uint8_t* w;
  int64_t w_row;        // bytes
  const float* scale;   // fp8: per output row
  const uint16_t* bias; // fp16, optional
  const uint16_t* x;    // fp16 [m, x_row]
  int64_t x_row;
  uint16_t* out;        // fp16 [m, out_row], optional with the argmax
  int64_t out_row;
  int m, rows, nchunks, rounds, tiles;
  uint64_t* keys;       // argmax: one key per (workgroup, row tile, activation row)
};

template <Fmt F> struct WTile;   // 16 rows x four chunks
template <> struct WTile<Fmt::kF16W> { static constexpr int kLoads = 4, kRowBytes = 256, kChunkBytes = 64; };
template <> struct WTile<Fmt::kFp8> { static constexpr int kLoads = 2, kRowBytes = 128, kChunkBytes = 32; };

// One column of A times one row of B, added to four blocks of 16 x 16 accumulators or to
// sixteen of 4 x 4: lane l feeds row l % 16 of block l / 16, or row l % 4 of block l / 4.
__device__ __forceinline__ f16x mfma_col(float a, float x, f16x c) {
  return __builtin_amdgcn_mfma_f32_16x16x1f32(a, x, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma_col(float a, float x, f4 c) { return __builtin_amdgcn_mfma_f32_4x4x1f32(a, x, c, 0, 0, 0); }

template <int M> __device__ __forceinline__ uint64_t max_over(uint64_t k) {
  const uint32_t hi = __builtin_bit_cast(uint32_t, xor_partner<M>(__builtin_bit_cast(float, (uint32_t)(k >> 32))));
  const uint32_t lo = __builtin_bit_cast(uint32_t, xor_partner<M>(__builtin_bit_cast(float, (uint32_t)k)));
  const uint64_t o = ((uint64_t)hi << 32) | lo;
  return o > k ? o : k;
}

// WV waves of GPW groups of four chunks (LPR = 4 GPW WV), RT 16-row weight tiles and, of the
// activations, MT tiles of 16 rows (NARROW: of four rows) per wave.
template <Fmt F, int WV, int GPW, int RT, int MT, bool NARROW, bool AM>
__global__ __launch_bounds__(64 * WV) __attribute__((amdgpu_waves_per_eu(2)))
void rows_mfma_kernel(RowsParams P) {
  using WT = WTile<F>;
  constexpr int LPR = 4 * GPW * WV;
  constexpr int kPieces = WT::kRowBytes / 16;      // 16-byte pieces per row and step
  constexpr int kRowsPerLoad = 64 / kPieces;
  constexpr int kWBytes = 16 * WT::kRowBytes;      // LDS bytes of one weight tile
  constexpr int kXRows = (NARROW ? 4 : 16) * MT;
  constexpr int kXLoads = kXRows / 4;
  constexpr int kBuf = RT * kWBytes + kXRows * 256;   // per wave
  typedef typename std::conditional<NARROW, f4, f16x>::type acc_t;
  __shared__ __attribute__((aligned(16))) uint8_t lds[WV * kBuf];
  __shared__ __attribute__((aligned(16))) f4 red[2][WV][RT * MT][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int r = lane & 15, b = lane >> 4;
  lds_u8* const buf = reinterpret_cast<lds_u8*>(reinterpret_cast<uintptr_t>(lds)) + wave * kBuf;

  // ---- sources: piece and row of this lane in load v of a tile
  const int wp = lane % kPieces, wr = lane / kPieces;
  const int wc = wp / (WT::kChunkBytes / 16), wo = (wp % (WT::kChunkBytes / 16)) * 16;   // chunk of the group, bytes inside it
  const int xp = lane & 15, xr = lane >> 4;
  const int xc = xp >> 2, xo = (xp & 3) * 16;
  uint32_t xoff[kXLoads];               // bytes from the first activation row
#pragma unroll
  for (int v = 0; v < kXLoads; v++) {
    const int m = 4 * v + xr;
    xoff[v] = (uint32_t)(m < P.m ? m : P.m - 1) * (uint32_t)(P.x_row * 2) + xo;
  }
  uint32_t woff[RT][WT::kLoads];        // bytes from the tile's first row
  const uint8_t* wbase;
  auto set_tile = [&](int tile) __attribute__((always_inline)) {
    const int64_t row0 = (int64_t)tile * (16 * RT);
    const int last = P.rows - 1 - row0 < 16 * RT - 1 ? (int)(P.rows - 1 - row0) : 16 * RT - 1;
    wbase = P.w + row0 * P.w_row;
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int v = 0; v < WT::kLoads; v++) {
        const int row = 16 * t + kRowsPerLoad * v + wr;
        woff[t][v] = (uint32_t)(row < last ? row : last) * (uint32_t)P.w_row + wo;
      }
  };

  u4 wst[RT][WT::kLoads], xst[kXLoads];
  // chunks 4 g + round * LPR .. + 3 of group g
  auto issue = [&](int g, int round) __attribute__((always_inline)) {
    const int j0 = 4 * g + round * LPR;
    const int jw = j0 + wc < P.nchunks ? j0 + wc : P.nchunks - 1;
    const int jx = j0 + xc < P.nchunks ? j0 + xc : P.nchunks - 1;
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int v = 0; v < WT::kLoads; v++)
        wst[t][v] = *reinterpret_cast<const u4*>(wbase + (woff[t][v] + (uint32_t)(jw * WT::kChunkBytes)));
#pragma unroll
    for (int v = 0; v < kXLoads; v++)
      xst[v] = *reinterpret_cast<const u4*>(reinterpret_cast<const uint8_t*>(P.x) + (xoff[v] + (uint32_t)(jx * 64)));
  };

  // staged pieces into the wave's buffer, xor-swizzled by the row
  auto stage = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int v = 0; v < WT::kLoads; v++) {
        const int row = kRowsPerLoad * v + wr;
        *reinterpret_cast<lds_u4*>(buf + t * kWBytes + row * WT::kRowBytes + 16 * (wp ^ (row & (kPieces - 1)))) = wst[t][v];
      }
#pragma unroll
    for (int v = 0; v < kXLoads; v++) {
      const int row = 4 * v + xr;
      *reinterpret_cast<lds_u4*>(buf + RT * kWBytes + row * 256 + 16 * (xp ^ (row & 15))) = xst[v];
    }
  };
  // fragments of columns 8q .. 8q + 7 of the staged chunks (fp8 weights: of sixteen columns)
  constexpr int kWQ = 4 / WT::kLoads;   // eights per weight piece
  u4 wf[2][RT], xf[2][MT];
  auto frags = [&](auto qc) __attribute__((always_inline)) {
    constexpr int q = decltype(qc)::value;
    if constexpr (q % kWQ == 0) {
#pragma unroll
      for (int t = 0; t < RT; t++)
        wf[(q / kWQ) & 1][t] = *reinterpret_cast<const lds_u4*>(
            buf + t * kWBytes + r * WT::kRowBytes + 16 * ((b * WT::kLoads + q / kWQ) ^ (r & (kPieces - 1))));
    }
#pragma unroll
    for (int t = 0; t < MT; t++) {
      const int row = NARROW ? 4 * t + (r & 3) : 16 * t + r;
      xf[q & 1][t] = *reinterpret_cast<const lds_u4*>(buf + RT * kWBytes + row * 256 + 16 * ((4 * b + q) ^ (row & 15)));
    }
  };
  // Their binary32 operands, those of the next eight columns formed in other registers
  // between this eight's MFMAs.
  float wv[2][RT][8], xv8[2][MT][8];
  auto form = [&](auto qc) __attribute__((always_inline)) {
    constexpr int q = decltype(qc)::value;
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int h = 0; h < 4; h++) {
        if constexpr (F == Fmt::kF16W) {
          const uint32_t w = wf[q & 1][t][h];
          wv[q & 1][t][2 * h] = lo_f32<f16_t>(w);
          wv[q & 1][t][2 * h + 1] = hi_f32<f16_t>(w);
        } else {
          const uint32_t w = wf[(q >> 1) & 1][t][2 * (q & 1) + (h >> 1)];
          const auto d = (h & 1) ? __builtin_amdgcn_cvt_pk_f32_fp8(w, true) : __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
          wv[q & 1][t][2 * h] = d[0];
          wv[q & 1][t][2 * h + 1] = d[1];
        }
      }
#pragma unroll
    for (int u = 0; u < MT; u++)
#pragma unroll
      for (int h = 0; h < 4; h++) {
        xv8[q & 1][u][2 * h] = lo_f32<f16_t>(xf[q & 1][u][h]);
        xv8[q & 1][u][2 * h + 1] = hi_f32<f16_t>(xf[q & 1][u][h]);
      }
    // formed here, not where they are consumed
#pragma unroll
    for (int e = 0; e < 8; e++) {
#pragma unroll
      for (int t = 0; t < RT; t++) asm volatile("" : "+v"(wv[q & 1][t][e]));
#pragma unroll
      for (int u = 0; u < MT; u++) asm volatile("" : "+v"(xv8[q & 1][u][e]));
    }
  };
  const std::integral_constant<int, 0> q0{};
  const std::integral_constant<int, 1> q1{};
  const std::integral_constant<int, 2> q2{};
  const std::integral_constant<int, 3> q3{};

  // ---- steps (tile, group, round) in order; the request cursor runs two steps ahead of the
  // one computed (past the last tile it repeats it, values unused)
  int tile = blockIdx.x, gi = 0, round = 0;
  const int g0 = wave * GPW;
  int itile = tile, igi = 0, iround = 0;
  set_tile(itile);
  auto request = [&]() __attribute__((always_inline)) {
    issue(g0 + igi, iround);
    if (++iround == P.rounds) {
      iround = 0;
      if (++igi == GPW) {
        igi = 0;
        const int nt = itile + (int)gridDim.x;
        if (nt < P.tiles) {
          itile = nt;
          set_tile(itile);
        }
      }
    }
  };
  request();
  stage();
  request();
  frags(q0);
  frags(q1);
  form(q0);
  frags(q2);
  uint64_t best = 0;
  int parity = 0;
  acc_t acc[RT][MT];        // the lanes' sums over their rounds, from +0
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int u = 0; u < MT; u++) acc[t][u] = (acc_t){};
  f4 node[RT][MT];          // tree value of the wave's groups
  f4 even[RT][MT];          // value of the even group of a pair
  f4 half[RT][MT];          // value of the last whole pair

  while (true) {
    acc_t p[RT][MT];          // chunk partials (four blocks of four rows; NARROW: the lane's block)
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int u = 0; u < MT; u++) p[t][u] = (acc_t){};
    auto eight = [&](auto qc) __attribute__((always_inline)) {
      constexpr int q = decltype(qc)::value;
#pragma unroll
      for (int e = 0; e < 8; e++)
#pragma unroll
        for (int t = 0; t < RT; t++)
#pragma unroll
          for (int u = 0; u < MT; u++)
            p[t][u] = mfma_col(wv[q & 1][t][e], xv8[q & 1][u][e], p[t][u]);
#pragma unroll
      for (int i = 0; i < 8 * RT * MT; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                    // an MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, (RT + MT + RT * MT - 1) / (RT * MT), 0);  // its share of the conversions
      }
    };
    __builtin_amdgcn_sched_barrier(0);
    form(q1);
    frags(q3);
    eight(q0);
    __builtin_amdgcn_sched_barrier(0);
    form(q2);
    eight(q1);
    __builtin_amdgcn_sched_barrier(0);
    // every fragment of the step has been read: the buffer takes the next step
    stage();
    request();
    __builtin_amdgcn_sched_barrier(0);
    form(q3);
    frags(q0);
    frags(q1);
    eight(q2);
    __builtin_amdgcn_sched_barrier(0);
    form(q0);
    frags(q2);
    eight(q3);
    __builtin_amdgcn_sched_barrier(0);

    // chunks past the end of K contribute +0
    const int left = P.nchunks - (4 * (g0 + gi) + round * LPR);   // valid chunks of this step (uniform)
    if (left < 4) {
#pragma unroll
      for (int t = 0; t < RT; t++)
#pragma unroll
        for (int u = 0; u < MT; u++)
#pragma unroll
          for (int i = 0; i < (NARROW ? 4 : 16); i++)
            if ((NARROW ? b : i >> 2) >= left) p[t][u][i] = 0.0f;
    }
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int u = 0; u < MT; u++) acc[t][u] = acc[t][u] + p[t][u];
    if (++round < P.rounds) continue;
    round = 0;
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int u = 0; u < MT; u++) {
        f4 g4;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          if constexpr (NARROW) g4[i] = bfly<32>(bfly<16>(acc[t][u][i]));   // block b is lane bits 4-5
          else g4[i] = (acc[t][u][i] + acc[t][u][4 + i]) + (acc[t][u][8 + i] + acc[t][u][12 + i]);
        }
        if constexpr (GPW == 1) {
          node[t][u] = g4;
        } else if ((gi & 1) == 0) {
          even[t][u] = g4;
        } else {
          const f4 pair = even[t][u] + g4;
          if (gi == GPW - 1) node[t][u] = GPW == 2 ? pair : half[t][u] + pair;
          half[t][u] = pair;
        }
        acc[t][u] = (acc_t){};
      }
    if (++gi < GPW) continue;
    gi = 0;
    // ---- the waves' subtrees meet; subtile s is finished by wave s
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int u = 0; u < MT; u++) red[parity][wave][t * MT + u][lane] = node[t][u];
    lds_barrier();   // alternating buffers: one barrier per tile
    static_assert(RT * MT <= WV, "one subtile per wave");
    if (wave < RT * MT) {
      const int t = wave / MT, u = wave % MT;
      f4 v = (red[parity][0][wave][lane] + red[parity][1][wave][lane]) +
             (red[parity][2][wave][lane] + red[parity][3][wave][lane]);
      if constexpr (WV == 8)
        v = v + ((red[parity][4][wave][lane] + red[parity][5][wave][lane]) +
                 (red[parity][6][wave][lane] + red[parity][7][wave][lane]));
      // NARROW: every block's lanes hold the sum, block 0 stores it
      const int m = NARROW ? 4 * u + (r & 3) : 16 * u + r;
      const int64_t row0 = (int64_t)tile * (16 * RT) + 16 * t + 4 * (NARROW ? r >> 2 : b);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int64_t row = row0 + i;
        if (row >= P.rows || m >= P.m || (NARROW && b != 0)) continue;
        float y = v[i];
        if constexpr (F == Fmt::kFp8) y = y * P.scale[row];
        if (P.bias != nullptr) y = round_f16(y) + to_f32(reinterpret_cast<const f16_t*>(P.bias)[row]);
        if (P.out != nullptr) P.out[(int64_t)m * P.out_row + row] = f32_to_f16_bits(y);
        if constexpr (AM) {
          const uint64_t key = argmax_key(round_f16(y), (uint32_t)row);
          best = key > best ? key : best;
        }
      }
    }
    tile += gridDim.x;
    parity ^= 1;
    if (tile >= P.tiles) break;
  }
  if constexpr (AM) {
    // lanes r, r + 16, r + 32, r + 48 hold the same activation row (NARROW: r, r + 4, r + 8,
    // r + 12 of block 0)
    if (wave < RT * MT) {
      best = max_over<NARROW ? 4 : 16>(max_over<NARROW ? 8 : 32>(best));
      const int m = NARROW ? 4 * (wave % MT) + r : 16 * (wave % MT) + r;
      if (b == 0 && m < P.m && (!NARROW || r < 4)) P.keys[((int64_t)blockIdx.x * RT + wave / MT) * P.m + m] = best;
    }
  }
}

// Token of each activation row from the keys of passes of up to kRowsPass rows: pass p
// wrote the key of (entry e, row r) at keys[p kRowsPass per + e mr + r], mr the rows of
// the pass; a full pass wrote full_count entries, the last one last_count.
__global__ __launch_bounds__(256) void argmax_rows_mfma_kernel(const uint64_t* keys, int64_t per, int full_count,
                                                               int last_count, int m_total, int64_t* out_idx,
                                                               float* out_val) {
  const int m = blockIdx.x;
  const int m0 = m / kRowsPass * kRowsPass;
  const int mr = m_total - m0 < kRowsPass ? m_total - m0 : kRowsPass;
  const int count = m0 + kRowsPass < m_total ? full_count : last_count;
  const uint64_t* base = keys + (int64_t)m0 * per + (m - m0);
  __shared__ uint64_t red[4];
  uint64_t best = 0;
  for (int i0 = 0; i0 < count; i0 += 256 * 8) {
    uint64_t k[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int i = i0 + (int)threadIdx.x + 256 * u;
      k[u] = base[(int64_t)(i < count ? i : count - 1) * mr];   // repeats leave a maximum as it is
    }
#pragma unroll
    for (int u = 0; u < 8; u++) best = k[u] > best ? k[u] : best;
  }
  best = wave_max_u64(best);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t k = red[0];
    for (int i = 1; i < 4; i++) k = red[i] > k ? red[i] : k;
    const uint32_t o = (uint32_t)(k >> 32);
    const uint32_t bits = o == 0xffffffffu ? 0x7fc00000u : ((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
    out_idx[m] = (int64_t)(0xffffffffu - (uint32_t)k);
    if (out_val) out_val[m] = __builtin_bit_cast(float, bits);
  }
}

template <Fmt F, int RT, int MT, bool NARROW, bool AM>
void launch_lpr_rows(int lpr, bool wide, const RowsParams& P, int grid, hipStream_t st) {
  const dim3 g(grid), t(wide ? 512 : 256);
  if constexpr (RT == 1) {
    if (wide) {
      if (lpr == 64) hipLaunchKernelGGL((rows_mfma_kernel<F, 8, 2, 1, MT, NARROW, AM>), g, t, 0, st, P);
      else hipLaunchKernelGGL((rows_mfma_kernel<F, 8, 1, 1, MT, NARROW, AM>), g, t, 0, st, P);
      return;
    }
  }
  if (lpr == 64) hipLaunchKernelGGL((rows_mfma_kernel<F, 4, 4, RT, MT, NARROW, AM>), g, t, 0, st, P);
  else if (lpr == 32) hipLaunchKernelGGL((rows_mfma_kernel<F, 4, 2, RT, MT, NARROW, AM>), g, t, 0, st, P);
  else hipLaunchKernelGGL((rows_mfma_kernel<F, 4, 1, RT, MT, NARROW, AM>), g, t, 0, st, P);
}

// One pass of at most kRowsPass activation rows.
//   * Up to eight rows run on the 4 x 4 form (16 x 16 would multiply padding: 337 against
//     307 us for the 152064 x 5120 head at 8 rows, 335 against 259 at 4, 39 against 35 us for
//     fp8 17920 x 5120 at 8; the 128256 x 2048 head at 8 rows is the exception, 126 against
//     134).
//   * Two weight tiles per wave, their activation operand built once for both, from 128
//     rows per CU on (152064 x 5120: 16 rows 372 us with one, 341 with two, 8 rows 314 and 307;
//     20000 x 5120, 8 rows, 45 with one and 50 with two: the last turn of tiles counts more).
//   * Eight waves per workgroup while there is at most one tile per CU (8 rows: 12.3 -> 11.3
//     us for 2880 x 4096 fp16, 11.1 -> 10.6 us for 4096 x 5120 fp8; with 320 tiles no gain).
//   * The grid is what the chip holds at once: tiles past it are taken in turn.
template <Fmt F, bool AM>
int launch_pass(int lpr, RowsParams P, int64_t keys_per_row, hipStream_t st, int* entries) {
  const int cus = device_cus();
  const int rt = P.m <= 16 && P.rows >= 128 * (int64_t)cus ? 2 : 1;
  P.tiles = (P.rows + 16 * rt - 1) / (16 * rt);
  const bool wide = rt == 1 && P.tiles <= cus && lpr >= 32;
  const int resident = wide ? 1 : (rt == 2 || P.m > 16 ? 2 : 3);
  const int grid = P.tiles < resident * cus ? P.tiles : resident * cus;
  if (entries) {
    *entries = grid * rt;
    TT_REQUIRE(*entries <= keys_per_row, "rows_mfma: argmax scratch too small");
  }
  if (rt == 2) {
    if (P.m <= 4) launch_lpr_rows<F, 2, 1, true, AM>(lpr, wide, P, grid, st);
    else if (P.m <= 8) launch_lpr_rows<F, 2, 2, true, AM>(lpr, wide, P, grid, st);
    else launch_lpr_rows<F, 2, 1, false, AM>(lpr, wide, P, grid, st);
  } else {
    if (P.m <= 4) launch_lpr_rows<F, 1, 1, true, AM>(lpr, wide, P, grid, st);
    else if (P.m <= 8) launch_lpr_rows<F, 1, 2, true, AM>(lpr, wide, P, grid, st);
    else if (P.m <= 16) launch_lpr_rows<F, 1, 1, false, AM>(lpr, wide, P, grid, st);
    else launch_lpr_rows<F, 1, 2, false, AM>(lpr, wide, P, grid, st);
  }
  return TT_OK;
}

template <Fmt F, bool AM>
int run_passes(const RowsArgs& A, hipStream_t st, const char* what, int* entries) {
  const int lpr = tt_gemv_lanes_per_row(A.cols / 32, 1);
  for (int64_t m0 = 0; m0 < A.m; m0 += kRowsPass) {
    RowsParams P{};
    P.w = static_cast<const uint8_t*>(A.weight);
    P.w_row = A.w_row_bytes;
    P.scale = A.scales;
    P.bias = static_cast<const uint16_t*>(A.bias);
    P.x = static_cast<const uint16_t*>(A.x) + m0 * A.x_row;
    P.x_row = A.x_row;
    P.out = A.out ? static_cast<uint16_t*>(A.out) + m0 * A.out_row : nullptr;
    P.out_row = A.out_row;
    P.m = (int)(A.m - m0 < kRowsPass ? A.m - m0 : kRowsPass);
    P.rows = (int)A.rows;
    P.nchunks = (int)(A.cols / 32);
    P.rounds = (P.nchunks + lpr - 1) / lpr;
    P.keys = AM ? A.keys + m0 * A.keys_per_row : nullptr;
    if (entries) entries[0] = entries[1];   // of the passes before the last: all full, all alike
    const int rc = launch_pass<F, AM>(lpr, P, A.keys_per_row, st, entries ? entries + 1 : nullptr);
    if (rc) return rc;
  }
  return check_launch(what);
}

}  // namespace

namespace tt {

int rows_mfma_f16(const RowsArgs& A, hipStream_t st, const char* what) {
  return run_passes<Fmt::kF16W, false>(A, st, what, nullptr);
}

int rows_mfma_fp8(const RowsArgs& A, hipStream_t st, const char* what) {
  return run_passes<Fmt::kFp8, false>(A, st, what, nullptr);
}

int rows_mfma_argmax_f16(const RowsArgs& A, int64_t* out_idx, float* out_val, hipStream_t st, const char* what) {
  int entries[2] = {0, 0};
  const int rc = run_passes<Fmt::kF16W, true>(A, st, what, entries);
  if (rc) return rc;
  hipLaunchKernelGGL(argmax_rows_mfma_kernel, dim3((unsigned)A.m), dim3(256), 0, st, A.keys, A.keys_per_row, entries[0],
                     entries[1], (int)A.m, out_idx, out_val);
  return check_launch(what);
}

}  // namespace tt
