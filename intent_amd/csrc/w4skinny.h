// W4 x few rows: the main loop of the projections whose time is the stream of
// packed weights (a handful to 64 activation rows against every weight row).
//
// A workgroup of four waves owns 64 * NB weight rows and up to 16 * TB
// activation rows; a wave owns NB blocks of 16 weight rows. Packed weights go
// straight to registers, 16 bytes per lane: lane (n = l % 16, q = l / 16) of
// block b loads bytes 16q .. 16q + 15 of a 64-byte run of row n, so one
// instruction covers 128 k of 16 rows and the two instructions of a stage of
// HS = 2 halves (256 k) whole 128-byte lines. The lane's dword j (8 k) is the A fragment of
// one v_mfma_f32_16x16x32_f16, whose k slots 8q .. 8q + 7 then stand for
// k = 32q + 8j .. + 7; the activation fragment is read from the same k, so the
// order inside an MFMA is the only thing that changes.
//
// What bounds it is bytes in flight and VALU issue, not MFMAs: D stages of
// weights (2 KB per block and stage) are in flight per wave with two or more
// workgroups per CU, and the decode is 13 operations per 8 weights: (d & mask)
// | magic pairs (1024 + q0, 1024 + q4), (64 + q1, 64 + q5) and the same of d >> 8,
// each less (1024 + z) or (64 + z), exact in f16, times the scale (one
// rounding, as dequant8). That pairing puts the weights in the order 0 4 1 5 2 6
// 3 7, so the activations are stored to LDS in that order (four v_perm per 16
// bytes, once per workgroup). Activation rows are padded by 16 bytes: sixteen
// rows' 16-byte reads of one chunk then cover the 64 banks once.
//
// Scales and zeros of the workgroup's rows and K range are staged once in LDS
// as (scale f16, 1024 + zero f16) dwords: per-stage loads of 2 + 1 bytes per
// row would double the vector memory instructions of the loop.
#pragma once

#include "common.h"

namespace sk {

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;

INTENT_DEVICE f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// LDS writes of this wave done, then a workgroup barrier; loads stay in flight.
INTENT_DEVICE void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Groups per row of a K range of nh * 128, and the LDS of one workgroup.
__host__ __device__ constexpr int param_stride(int groups) { return groups | 1; }  // odd: 16 rows in 16 banks
// LDS bytes of one activation row of a stage of HS * 128 k.
template <int HS>
constexpr int kXRow = HS * 256 + 16;
template <int NB, int TB, int HS>
__host__ __device__ constexpr int lds_bytes(int groups) {
  return 64 * NB * param_stride(groups) * 4 + 2 * TB * 16 * kXRow<HS>;
}

// u / gu by multiplication (u < 2^16): magic = floor(2^32 / gu) + 1; gu = 1 passes u through.
struct GroupDiv {
  uint32_t gu, magic;
  INTENT_DEVICE uint32_t operator()(uint32_t u) const { return gu == 1 ? u : __umulhi(u, magic); }
};
inline GroupDiv group_div(int64_t gs) {
  const uint64_t gu = (uint64_t)gs / 32;
  return GroupDiv{(uint32_t)gu, gu == 1 ? 0u : (uint32_t)((1ull << 32) / gu + 1)};
}

struct W4Src {
  const uint8_t* q;   // packed weights, row 0 at the first k of the range
  int64_t ldq;        // bytes per packed row
  const f16* s;       // scales and zeros, row 0 at the range's first group
  const uint8_t* z;
  int64_t ldp;        // groups per row
  int groups;         // groups of the range
  bool vec;           // 4-group runs of every row are 8-byte (scales) and 4-byte (zeros) aligned, groups % 4 == 0
  GroupDiv div;
};

// Decodes one dword (8 weights) in the order 0 4 1 5 2 6 3 7.
template <bool kScale>
INTENT_DEVICE f16x8 decode8(uint32_t d, uint32_t magic, uint32_t mhi, f16x2 za, f16x2 zb, f16x2 sc) {
  const uint32_t d8 = d >> 8;
  f16x2 a = bit_cast<f16x2>(bfi(0x000F000Fu, d, magic)) - za;
  f16x2 b = bit_cast<f16x2>(bfi(0x00F000F0u, d, mhi)) - zb;
  f16x2 c = bit_cast<f16x2>(bfi(0x000F000Fu, d8, magic)) - za;
  f16x2 e = bit_cast<f16x2>(bfi(0x00F000F0u, d8, mhi)) - zb;
  if constexpr (kScale) {
    a *= sc;
    b *= sc;
    c *= sc;
    e *= sc;
  }
  return f16x8{a[0], a[1], b[0], b[1], c[0], c[1], e[0], e[1]};
}

// acc[b][t], summed over nh * 128 k. kPost false: lane l holds activation row
// 16 t + l % 16 and weight rows (of the wave's block b) 4 (l / 16) + 0..3.
// kPost true (groups of whole 128 k): the weights enter the MFMAs as the exact
// q - z and each 128-k sum is scaled once in f32, so no weight is rounded to f16;
// the operands are swapped, so that a lane's sums share one weight row and
// scale: lane l holds weight row l % 16 and activation rows 16 t + 4 (l / 16) + 0..3.
// x: activation rows at the range's first k; trow(p): byte offset of row p
// (< 16 TU, every one readable); wrow(r): weight row of workgroup row r.
// TU: 16-row blocks computed (<= TB).
template <int NB, int TB, int TU, int HS, int D, bool kPost, class WRow, class TRow>
INTENT_DEVICE void w4_mainloop(char* lds, const void* x, const TRow& trow, const W4Src& w, const WRow& wrow, int nh,
                               f32x4 (&acc)[NB][TB]) {
  static_assert(TU >= 1 && TU <= TB, "computed blocks");
  constexpr int ROWS = 64 * NB;
  constexpr int XR = kXRow<HS>;
  constexpr int XB = TB * 16 * XR;
  constexpr int CPR = 16 * HS;             // 16-byte pieces of an activation row and stage
  constexpr int RPI = kThreads / CPR;      // rows per load instruction of the workgroup
  constexpr int NX = TU * 16 / RPI;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, q = lane >> 4;
  const int ps = param_stride(w.groups);
  uint32_t* par = reinterpret_cast<uint32_t*>(lds);
  char* xlds = lds + ROWS * ps * 4;

  // ---- parameters first (they are waited for first) ----
  const auto put = [&](int r, int g, uint32_t s16, uint32_t z8) {
    const f16 za = (f16)(float)(1024u + z8);
    par[r * ps + g] = s16 | ((uint32_t)bit_cast<uint16_t>(za) << 16);
  };
  uint32_t voff[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) voff[b] = (uint32_t)((int64_t)wrow((wave * NB + b) * 16 + n) * w.ldq + q * 16);
  const int xrow = tid / CPR, xcol = (tid % CPR) * 16;
  uint32_t xoff[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) xoff[i] = (uint32_t)(trow(i * RPI + xrow) + xcol);
  // With HS = 2 and an odd nh the last stage holds one half: its second half
  // re-reads the first, and is not computed.
  const int nst = (nh + HS - 1) / HS;
  u32x4 wr[D][NB][HS];
  u32x4 xr[D][NX];
  // Loads are issued on every path, so that the wait counts of the loop stay
  // exact; past the range they go through a resource of no records, which
  // returns zeros without a memory access.
  const auto rsrc_at = [&](const void* base, int st) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, st < nst ? 0x7fffffff : 0, 0x00020000);
  };
  const auto load_w = [&](int st, u32x4 (&r)[NB][HS]) {
    const auto rq = rsrc_at(w.q, st);
    const uint32_t o = st < nst ? (uint32_t)st * (64u * HS) : 0u;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int h = 0; h < HS; ++h)
        r[b][h] = __builtin_amdgcn_raw_buffer_load_b128(rq, voff[b], HS * st + h < nh ? o + 64u * h : o, 0);
  };
  const auto load_x = [&](int st, u32x4 (&r)[NX]) {
    const auto rx = rsrc_at(x, st);
    const uint32_t o = st < nst ? (uint32_t)st * (256u * HS) : 0u;
    const uint32_t back = (HS * st + HS - 1 < nh || xcol < 256) ? 0u : 256u;
#pragma unroll
    for (int i = 0; i < NX; ++i) r[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, xoff[i] - back, o, 0);
  };

  // Group quads of the range, a row's quads on neighbouring lanes, so that an
  // instruction reads each line once (a row per lane touched 64 lines), and in
  // flight over the first weight loads: down of E = 8, K = 14336, N = 4096 at 16
  // rows 61 -> 57 us, the layer at T = 1 65.5 -> 62. 80 KB of LDS less 17 KB of
  // activations hold at most 4032 quads: PB per thread cover them.
  constexpr int PB = 16;
  static_assert(4 * 4 * PB * kThreads + 2 * 16 * kXRow<2> >= 81920, "quads of the largest range");
  u32x2 s4[PB];
  uint32_t z4[PB];
  const uint32_t nq = (uint32_t)w.groups >> 2;
  const int quads = ROWS * (int)nq;
  const uint32_t qmagic = nq > 1 ? 0xFFFFFFFFu / nq + 1 : 0;
  const auto quad_row = [&](int i) { return nq > 1 ? (int)__umulhi((uint32_t)i, qmagic) : i; };
  if (w.vec) {
#pragma unroll
    for (int k = 0; k < PB; ++k) {
      if (kThreads * k >= quads) break;
      const int i = kThreads * k + tid < quads ? kThreads * k + tid : quads - 1;
      const int r = quad_row(i);
      const int64_t o = (int64_t)wrow(r) * w.ldp + (i - r * (int)nq) * 4;
      s4[k] = *reinterpret_cast<const u32x2*>(w.s + o);
      z4[k] = *reinterpret_cast<const uint32_t*>(w.z + o);
    }
  } else {
    const int items = ROWS * w.groups;
    constexpr int BATCH = 8;
    for (int i0 = tid; i0 < items; i0 += kThreads * BATCH) {
      f16 s1[BATCH];
      uint8_t z1[BATCH];
#pragma unroll
      for (int k = 0; k < BATCH; ++k) {
        const int i = i0 + kThreads * k < items ? i0 + kThreads * k : i0;
        const int64_t o = (int64_t)wrow(i / w.groups) * w.ldp + i % w.groups;
        s1[k] = w.s[o];
        z1[k] = w.z[o];
      }
#pragma unroll
      for (int k = 0; k < BATCH; ++k) {
        const int i = i0 + kThreads * k;
        if (i >= items) break;
        put(i / w.groups, i % w.groups, bit_cast<uint16_t>(s1[k]), z1[k]);
      }
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d) {
    load_x(d, xr[d]);
    load_w(d, wr[d]);
  }
  if (w.vec) {
#pragma unroll
    for (int k = 0; k < PB; ++k) {
      if (kThreads * k >= quads) break;
      const int i = kThreads * k + tid;
      const int r = quad_row(i), g = (i - r * (int)nq) * 4;
      if (i < quads) {
#pragma unroll
        for (int c = 0; c < 4; ++c) put(r, g + c, (s4[k][c >> 1] >> (16 * (c & 1))) & 0xFFFFu, (z4[k] >> (8 * c)) & 0xFFu);
      }
    }
  }

#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int t = 0; t < TU; ++t) acc[b][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t magic = 0x64006400u, mhi = 0x54005400u;
  asm("" : "+v"(magic));
  asm("" : "+v"(mhi));
  const uint32_t* prow[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) prow[b] = par + ((wave * NB + b) * 16 + n) * ps;

  const auto compute_half = [&](int st, int hh, const u32x4 (&r)[NB][HS], const char* xb) {
    const uint32_t g = w.div((uint32_t)((st * HS + hh) * 4 + q));
    f16x2 za[NB], zb[NB], sc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint32_t p = prow[b][g];
      sc[b] = splat2(bit_cast<f16>((uint16_t)(p & 0xFFFFu)));
      za[b] = splat2(bit_cast<f16>((uint16_t)(p >> 16)));
      zb[b] = za[b] - splat2((f16)960.f);
    }
    f32x4 sum[NB][TU];  // kPost: the half's own sums
    if constexpr (kPost) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int t = 0; t < TU; ++t) sum[b][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f16x8 xf[TU];
#pragma unroll
      for (int t = 0; t < TU; ++t)
        xf[t] = *reinterpret_cast<const f16x8*>(xb + (t * 16 + n) * XR + hh * 256 + q * 64 + j * 16);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const f16x8 wf = decode8<!kPost>(r[b][hh][j], magic, mhi, za[b], zb[b], sc[b]);
#pragma unroll
        for (int t = 0; t < TU; ++t) {
          if constexpr (kPost)
            sum[b][t] = mfma16(xf[t], wf, sum[b][t]);
          else
            acc[b][t] = mfma16(wf, xf[t], acc[b][t]);
        }
      }
    }
    if constexpr (kPost) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const float sf = (float)sc[b][0];
#pragma unroll
        for (int t = 0; t < TU; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[b][t][e] = __builtin_fmaf(sum[b][t][e], sf, acc[b][t][e]);
      }
    }
  };

  const auto stage = [&](int st, u32x4 (&xs)[NX], u32x4 (&ws)[NB][HS], bool more) {
    char* xb = xlds + (st & 1) * XB;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const u32x4 v = xs[i];
      const u32x4 o{__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
                    __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)};
      *reinterpret_cast<u32x4*>(xb + (i * RPI + xrow) * XR + xcol) = o;
    }
    if (more) load_x(st + D, xs);
    lds_barrier();  // also orders the parameter writes before their first read
#pragma unroll
    for (int h = 0; h < HS; ++h)
      if (h == 0 || HS * st + h < nh) compute_half(st, h, ws, xb);
    if (more) load_w(st + D, ws);
  };
  const int whole = nst / D * D;
  for (int s0 = 0; s0 < whole; s0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) stage(s0 + d, xr[d], wr[d], true);
  }
#pragma unroll
  for (int d = 0; d + 1 < D; ++d)
    if (whole + d < nst) stage(whole + d, xr[d], wr[d], false);
  // The sums are complete here, under the whole wave: a caller's branch per lane
  // must not take a last stage's fragment reads with it (mp::settle; the sums are
  // in VGPRs here).
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int t = 0; t < TU; ++t) asm volatile("" : "+v"(acc[b][t]));
}

}  // namespace sk
