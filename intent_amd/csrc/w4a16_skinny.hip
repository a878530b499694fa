// W4A16 for 2 to 128 activation rows on the weight-streaming core (w4skinny.h):
// a workgroup owns 64 weight rows and one run of K, passes every activation row
// of the run through LDS and leaves f32 partial sums in scratch (1 KB contiguous
// per store), which w4_skinny_combine_kernel adds in order. Bound by latency at
// small N and by the weights' stream and the activation reads beyond. Both kernels
// together against what ran before: N = 11008, K = 4096, M = 12 17.2 -> 11.4 us
// (every 16 weight rows read all of x there); N = 4096, K = 14336, M = 16 23.3 ->
// 13.6; N = K = 4096, M = 32 13.7 -> 9.6, 77 20.3 -> 13.8, 128 21.0 -> 18.7 us. Two
// blocks of rows per wave were within 4% either way.
#include "common.h"
#include "internal.h"
#include "w4skinny.h"
#include <type_traits>

namespace {

constexpr int kRows = 64;  // weight rows per workgroup: one block of 16 per wave

struct ClampRows {
  int n0;
  int N;
  INTENT_DEVICE int operator()(int c) const {
    const int n = n0 + c;
    return n < N ? n : N - 1;
  }
};

template <int TB>
struct Cfg {
  static constexpr int HS = TB <= 2 ? 2 : 1;
  static constexpr int D = TB <= 2 ? 2 : TB <= 4 ? 3 : 2;
};

template <int TB, bool kPost>
__global__ __launch_bounds__(sk::kThreads, 2) void w4_skinny_kernel(
    const f16* __restrict__ x, int64_t ldx, int M, const uint8_t* __restrict__ wq, int64_t ldq,
    const f16* __restrict__ ws, const uint8_t* __restrict__ wz, int64_t ldp, int N, int K, int gs, sk::GroupDiv div,
    int vec, int unit, float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int p = blockIdx.y, S = gridDim.y, units = K / unit;
  const int k0 = (int)((int64_t)p * units / S) * unit, k1 = (int)((int64_t)(p + 1) * units / S) * unit;
  const int g0 = k0 / gs, groups = (k1 - k0) / gs;
  const sk::W4Src w{wq + k0 / 2, ldq, ws + g0, wz + g0, ldp, groups, vec != 0 && g0 % 4 == 0 && groups % 4 == 0, div};
  const ClampRows rows{(int)blockIdx.x * kRows, N};
  f32x4 acc[1][TB];
  sk::w4_mainloop<1, TB, TB, Cfg<TB>::HS, Cfg<TB>::D, kPost>(
      lds, x + k0, [&](int r) { return (uint32_t)((r < M ? r : M - 1) * ldx * 2); }, w, rows, (k1 - k0) / 128, acc);
  float* out = part + (((int64_t)p * gridDim.x + blockIdx.x) * sk::kWaves + (threadIdx.x >> 6)) * (TB * 256) +
               (threadIdx.x & 63) * 4;
#pragma unroll
  for (int t = 0; t < TB; ++t) *reinterpret_cast<f32x4*>(out + t * 256) = acc[0][t];
}

// y = f16(runs added in order): workgroup (tile, t), its wave w the 16 x 16 block
// of activation rows 16 t .. and weight rows 64 tile + 16 w ...
template <int TB, bool kPost>
__global__ __launch_bounds__(256) void w4_skinny_combine_kernel(const float* __restrict__ part, int S, int tiles, int M,
                                                                int N, f16* __restrict__ y, int64_t ldy, int vec) {
  const int t = blockIdx.x % TB, tile = blockIdx.x / TB;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float* src = part + ((int64_t)tile * sk::kWaves + wave) * (TB * 256) + t * 256 + lane * 4;
  const int64_t stride = (int64_t)tiles * sk::kWaves * (TB * 256);
  f32x4 v = *reinterpret_cast<const f32x4*>(src);
#pragma unroll 4
  for (int p = 1; p < S; ++p) {
    const f32x4 o = *reinterpret_cast<const f32x4*>(src + p * stride);
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] += o[c];
  }
  const int nb = tile * kRows + wave * 16;
  if constexpr (kPost) {
    const int n = nb + (lane & 15), m = 16 * t + 4 * (lane >> 4);
    if (n >= N) return;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (m + c < M) y[(int64_t)(m + c) * ldy + n] = (f16)v[c];
  } else {
    const int m = 16 * t + (lane & 15), n = nb + 4 * (lane >> 4);
    if (m >= M) return;
    f16* dst = y + (int64_t)m * ldy + n;
    if (vec && n + 3 < N) {
      *reinterpret_cast<u32x2*>(dst) = u32x2{bit_cast<uint32_t>(__builtin_convertvector(f32x2{v[0], v[1]}, f16x2)),
                                             bit_cast<uint32_t>(__builtin_convertvector(f32x2{v[2], v[3]}, f16x2))};
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (n + c < N) dst[c] = (f16)v[c];
    }
  }
}

struct Plan {
  int tb;         // activation rows / 16, rounded up to an instantiated count
  int splits;     // runs of K
  int64_t unit;   // K is cut at multiples of it (0: the kernel does not take the call)
  int lds;
};

constexpr int64_t kMaxPartialBytes = 64 << 20;  // as the tiled kernels' split
int64_t partial_bytes(const Plan& p, int64_t N) {
  return p.splits * ((N + kRows - 1) / kRows) * kRows * 16 * p.tb * 4;
}

template <class F>
auto with_rows(int tb, F&& f) {
  switch (tb) {
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    case 4: return f(std::integral_constant<int, 4>{});
    case 5: return f(std::integral_constant<int, 5>{});
    case 6: return f(std::integral_constant<int, 6>{});
    default: return f(std::integral_constant<int, 8>{});
  }
}

// Runs of about 1024 k (the longest that still give two workgroups per CU at N =
// 4096 were the fastest: N = 4096, K = 4096, M = 77: 4 runs 13.8 us, 2 16.9, 8 16.1),
// shorter ones down to 512 k while there are fewer than 128 workgroups; fewer where
// the partial sums would pass 64 MB (wide N has workgroups enough without).
Plan skinny_plan(int64_t M, int64_t N, int64_t K, int64_t gs) {
  Plan p{(int)((M + 15) / 16), 1, 0, 0};
  if (p.tb > 6) p.tb = 8;
  int64_t unit = gs % 128 == 0 ? gs : 128 % gs == 0 ? 128 : 0;
  if (M > 128 || gs % 32 != 0 || unit == 0 || K % unit != 0 || K / 32 >= 65536) return p;
  if (K % (4 * unit) == 0 && K / (4 * unit) >= 8) unit *= 4;  // runs of four groups: vector parameter loads
  const int64_t tiles = (N + kRows - 1) / kRows;
  while (K / (2 * p.splits) >= 1024 && p.splits < 16) p.splits *= 2;
  while (tiles * p.splits < 128 && K / (2 * p.splits) >= 512 && p.splits < 16) p.splits *= 2;
  while (p.splits > K / unit) p.splits /= 2;
  while (p.splits > 1 && partial_bytes(p, N) > kMaxPartialBytes) p.splits /= 2;
  if (partial_bytes(p, N) > kMaxPartialBytes) return p;
  const int64_t longest = (K / unit + p.splits - 1) / p.splits * unit;
  if (longest / gs > 256) return p;
  p.lds = with_rows(p.tb, [&](auto TB) {
    constexpr int kTB = decltype(TB)::value;
    return sk::lds_bytes<1, kTB, Cfg<kTB>::HS>((int)(longest / gs));
  });
  if (p.lds <= 81920) p.unit = unit;  // two workgroups per CU
  return p;
}

}  // namespace

namespace intent {

// Microseconds of a fit to 60 shapes (M 2..128, N 1024..14336, K 2048..14336); over
// 121 other ones (N 310..131072, K 256..16384) that it takes, four in five of the
// fits are 0.80 to 1.02 of the measured time. 0 where the kernel does not take the
// call. bytes: its scratch.
double w4a16_skinny_us(int64_t M, int64_t N, int64_t K, int64_t gs, size_t* bytes) {
  const Plan p = skinny_plan(M, N, K, gs);
  if (p.unit == 0) return 0;
  *bytes = (size_t)partial_bytes(p, N);
  const double work = (double)((N + kRows - 1) / kRows) * (double)(K / 128) / 8;
  // Runs that are not whole quads of groups load the parameters one by one: 1 to 2.5 us
  // more. Up to 6 rows that decides against one round of the GEMV for K below 10240 (N =
  // 2304, M = 6: K = 8320 10.6 us against 9.6, 9344 11.1 against 10.5, 10368 11.5 against
  // 11.4), at 7 rows below 9216 (N = 3072, K = 9344 10.8 against 11.3); not at M = 8 (K =
  // 8320 10.7 against 10.6), nor while one workgroup per CU does (M = 6, N = 2048 8.5
  // against 9.6).
  const bool gemv_round = N > 2048 && N <= 4096 && (M <= 6 ? K < 10240 : M == 7 && K < 9216);
  const bool quads = p.unit % (4 * gs) == 0 || (p.splits == 1 && K % (4 * gs) == 0);
  const double singles = gemv_round && !quads ? 3 : 0;
  // The partial sums' way through memory, which the fit has in its terms of K from 1024
  // on (N = 106112, K = 256, M = 26 18.3 us against 14.6 in tiles; N = 22848, K = 768, M =
  // 17 10.8 against 9.5; the other way round at N = 8192, K = 512: 6.6 against 6.9).
  const double sums = M > 16 && K < 1024 && (N > 16384 || !quads) ? 0.27e-6 * (double)partial_bytes(p, N) : 0;
  return 5.2 + 0.6 * p.tb + work * (0.0046 + 0.0034 * p.tb) + singles + sums;
}

// A w4a16_fast call whose plan exists, with 31-bit offsets checked by the caller.
int w4a16_skinny_launch(const void* x, int64_t M, int64_t K, int64_t x_ld, const uint8_t* packed, int64_t N,
                        int64_t packed_ld, const void* scales, const uint8_t* zeros, int64_t qparam_ld, int64_t gs,
                        void* y, int64_t y_ld, void* ws, void* stream) {
  const Plan p = skinny_plan(M, N, K, gs);
  const int64_t tiles = (N + kRows - 1) / kRows;
  const int vec = qparam_ld % 4 == 0 && (reinterpret_cast<uintptr_t>(scales) & 7) == 0 && aligned4(zeros);
  const int vout = y_ld % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 7) == 0;
  hipStream_t st = (hipStream_t)stream;
  return with_rows(p.tb, [&](auto TBc) -> int {
    constexpr int TB = decltype(TBc)::value;
    const auto go = [&](auto post) -> int {
      constexpr bool kPost = decltype(post)::value;
      const auto kernel = w4_skinny_kernel<TB, kPost>;
      if (p.lds > 65536) {
        const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, p.lds);
        INTENT_REQUIRE(e == hipSuccess, INTENT_ERR_LAUNCH, "w4a16: %d bytes of LDS refused (%s)", p.lds,
                       hipGetErrorString(e));
      }
      hipLaunchKernelGGL(kernel, dim3((unsigned)tiles, p.splits), dim3(sk::kThreads), p.lds, st, (const f16*)x, x_ld,
                         (int)M, packed, packed_ld, (const f16*)scales, zeros, qparam_ld, (int)N, (int)K, (int)gs,
                         sk::group_div(gs), vec, (int)p.unit, (float*)ws);
      const int s = launch_status("w4a16_skinny");
      if (s != INTENT_OK) return s;
      hipLaunchKernelGGL((w4_skinny_combine_kernel<TB, kPost>), dim3((unsigned)(tiles * TB)), dim3(256), 0, st,
                         (const float*)ws, p.splits, (int)tiles, (int)M, (int)N, (f16*)y, y_ld, vout);
      return launch_status("w4a16_skinny");
    };
    return gs % 128 == 0 ? go(std::true_type{}) : go(std::false_type{});
  });
}

}  // namespace intent
