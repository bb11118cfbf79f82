// Internal helpers for the extern "C" entry points: error reporting and checks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdarg.h>
#include <stdio.h>
#include <atomic>
#include <string>

#include "../../include/thintensor_hip.h"

namespace tt {

void set_error(const char* fmt, ...);

#define TT_REQUIRE(cond, ...)                 \
  do {                                        \
    if (!(cond)) {                            \
      ::tt::set_error(__VA_ARGS__);           \
      return TT_ERR_INVALID;                  \
    }                                         \
  } while (0)

#define TT_UNSUPPORTED(cond, ...)             \
  do {                                        \
    if (!(cond)) {                            \
      ::tt::set_error(__VA_ARGS__);           \
      return TT_ERR_UNSUPPORTED;              \
    }                                         \
  } while (0)

inline int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: kernel launch failed: %s", what, hipGetErrorString(e));
    return TT_ERR_HIP;
  }
  return TT_OK;
}

// Compute units of the current device.
inline int device_cus() {
  static std::atomic<int> known[64];
  int dev = 0, c = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  c = known[dev].load(std::memory_order_relaxed);
  if (c == 0) {
    if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c <= 0) c = 256;
    known[dev].store(c, std::memory_order_relaxed);
  }
  return c;
}

inline bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

// y[r] = W x[r] + bias for m fp16 activation rows, several rows per launch sharing every
// weight load; row r has the bits of the single-row GEMV + bias (batched.hip).  Shapes and
// alignment checked by the caller.
int dense_bias_rows_f16(const void* weight, int64_t w_row, const void* bias, const void* x, int64_t x_row, void* out,
                        int64_t out_row, int64_t m, int64_t rows, int64_t cols, hipStream_t st);

// y[r] = (W x[r]) scale for m fp16 activation rows as slots of the single-row fp8 kernel
// (gemv_dense.hip).  Operands checked by the caller, 32-bit offsets (rows w_row_bytes < 2^31).
int scaled_slots_fp8(const void* weight, int64_t w_row_bytes, const float* scales, const void* x, int64_t x_row, void* out,
                     int64_t out_row, int64_t m, int64_t rows, int64_t cols, hipStream_t st, const char* what);

// y[r] = W x[r] for m fp16 activation rows on the binary32 matrix cores, row r with the
// bits of the single-row GEMV (rows_mfma.hip): fp16 weights with an optional fp16 bias, fp8
// weights with fp32 row scales, and the fp16 lm_head with its argmax.  Passes of kRowsPass
// rows.  Shapes (cols a multiple of 32) and 16-byte alignment checked by the caller.
constexpr int kRowsPass = 32;
// Smallest M of the fp16 GEMVs and of the fp8 GEMM that runs there (same bits as the GEMV
// engine).  Three rows take the engine two launches (fp16 152064 x 5120 522 us against 258,
// fp8 17920 x 5120 39 against 24); at two, one launch each, the head takes 268 us on the engine
// and 263 here, the fp8 matrix 18.8 and 21.2.
constexpr int kRowsMfmaMin = 3;
// Whether the activation rows run sooner as slots of the single-row lean kernel (a grid row
// each, the same bits): their time grows with rows x m, that of a matrix-core pass of up to 4,
// 8, 16 or 32 rows hardly does while there are fewer row tiles than CUs.  Break-even of fp16
// matrices of 2048 to 32768 columns; us as slots against matrix cores: 64 x 5120, 64 rows 5.2
// against 36.9; 1024 x 5120, 3 rows 6.3 against 8.5, 8 rows 9.2 against 11.4, 16 rows 14.1
// against 13.3; 1536 x 5120, 4 rows 9.6 against 8.9; 768 x 8192, 32 rows 27 against 28; 2880 x
// 5120, 8 rows 31 against 12; a fifth earlier where the slots' weight reads miss the L2s
// (1280 x 32768, 4 rows 46 against 34).  (fp8 breaks even later: 2048 x 5120, 8 rows 1.2 times
// as fast as slots, 2880 x 5120 0.85 times.)
inline bool row_slots_better(int64_t m, int64_t rows, int64_t cols) {
  const int64_t tail = m % kRowsPass;
  const int64_t even = m / kRowsPass * 25000 + (tail == 0 ? 0 : tail <= 4 ? 5500 : tail <= 8 ? 9000 : tail <= 16 ? 12500 : 25000);
  return rows * m < (cols > 16384 ? even / 5 * 4 : even);
}
struct RowsArgs {
  const void* weight;
  int64_t w_row_bytes;
  const float* scales;
  const void* bias;
  const void* x;
  int64_t x_row;
  void* out;
  int64_t out_row;
  int64_t m, rows, cols;
  uint64_t* keys;         // argmax scratch, keys_per_row entries per activation row
  int64_t keys_per_row;
};
// 32-bit byte offsets inside a weight tile (32 rows) and an activation pass
inline bool rows_mfma_fits(int64_t w_row_bytes, int64_t x_row) {
  return w_row_bytes < (1LL << 26) && x_row < (1LL << 25);
}
int rows_mfma_f16(const RowsArgs& A, hipStream_t st, const char* what);
int rows_mfma_fp8(const RowsArgs& A, hipStream_t st, const char* what);
int rows_mfma_argmax_f16(const RowsArgs& A, int64_t* out_idx, float* out_val, hipStream_t st, const char* what);

// Expert index arrays are int32 or int64 (index_bytes 4 or 8); the kernels take the
// log2 of the size in 32-bit words.
inline bool index_shift(int index_bytes, int* shift) {
  *shift = index_bytes == 8 ? 1 : 0;
  return index_bytes == 4 || index_bytes == 8;
}

inline bool valid_act_dtype(int d) { return d == TT_F16 || d == TT_BF16; }
inline bool valid_out_dtype(int d) { return d == TT_F16 || d == TT_BF16 || d == TT_F32; }

// Attention scratch: kAttnCounters arrival counters of the single-launch path (one per
// KV head, at fixed offsets whatever the shape, left at zero by every call), then the
// chunk partials (m, l, o) per query head.
constexpr int kAttnCounters = 1024;

}  // namespace tt
