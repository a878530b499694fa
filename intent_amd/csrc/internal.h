// Host-side helpers shared by the entry points (error state, checks).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/intent_amd.h"

namespace intent {

// Records a formatted message for intent_amd_last_error() and returns `code`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

// Clears the thread's error message.
void clear_error();

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool aligned4(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0; }

// rows * stride_bytes stays below 2^31: the byte offsets of buffer loads are
// 32-bit and the kernels keep them non-negative ints.
inline bool fits_offset(int64_t rows, int64_t stride_bytes) {
  return rows >= 0 && stride_bytes >= 0 && (rows == 0 || stride_bytes <= ((int64_t)1 << 31) / rows) &&
         rows * stride_bytes < ((int64_t)1 << 31);
}

// Checks hipGetLastError() after a launch and records `kernel` as the
// thread's last launched kernel (intent_amd_last_kernel()).
int launch_status(const char* kernel);
// Same, with a printf-formatted kernel name (template parameters).
int launch_status_fmt(const char* fmt, ...) __attribute__((format(printf, 1, 2)));

// Writes `bits` (the low elem_bytes = 1, 2 or 4 bytes) to every element of a
// rows x cols matrix with a leading stride of ld elements: the output of a
// contraction over an empty K, which is its epilogue applied to zero.
int fill_launch(void* out, int64_t rows, int64_t cols, int64_t ld, int elem_bytes, uint32_t bits, void* stream);

// Compute units of the current device (queried once per device; 0 if the
// query fails, which callers treat as "no round-fitting").
int cu_count();

// By this the plans of one tiled kernel are ranked, in microseconds of a fit to
// measurements of it: base, plus per stage of the K loop a + b L while the L =
// workgroups / 256 do not exceed one per CU, and (a + b) times the rounds beyond
// (half a round's cost for a partly filled one, since its workgroups share a CU with
// those before them). It predicts no time: bandwidth, stores and how far workgroups
// that share a CU hide each other are left out. Over 700 random shapes (M 1..4096, K
// 256..16384, N 256..131072) the chosen plan reads 0.76 to 0.99 of its measured time
// in the median up to one workgroup per CU and 0.68 to 0.98 up to four, 0.3 where K is
// short and N very wide, and 47 us for the 35 of block-scaled FP8 at M = 300, N =
// 14336, K = 4096 (two workgroups on some CUs).
struct GridCost {
  double base, a, b;
  double us(int64_t workgroups, double stages) const {
    const double L = (double)workgroups / 256;
    return base + stages * (L <= 1 ? a + b * L : (a + b) * (L + (double)((workgroups + 255) / 256)) / 2);
  }
};

// Names of the kernels of a plan (tile and runs of K), recorded by launch_status.
struct PlanNames {
  const char* name[3][5];  // tiles of 256, 128 and 64 rows; 1, 2, 4, 8 and 16 runs
  const char* operator()(int rows, int runs) const {
    return name[rows == 256 ? 0 : rows == 128 ? 1 : 2][__builtin_ctz((unsigned)runs)];
  }
};

}  // namespace intent

#define INTENT_RUN_NAMES(tile) \
  { tile ">", tile ", 2 runs>", tile ", 4 runs>", tile ", 8 runs>", tile ", 16 runs>" }
// big: the 256-row tile; the others are 128x128 and 64x128.
#define INTENT_PLAN_NAMES(base, big) \
  {{INTENT_RUN_NAMES(base "<" big), INTENT_RUN_NAMES(base "<128x128"), INTENT_RUN_NAMES(base "<64x128")}}

#define INTENT_REQUIRE(cond, code, ...)            \
  do {                                             \
    if (!(cond)) return ::intent::fail(code, __VA_ARGS__); \
  } while (0)
