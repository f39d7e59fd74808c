// dq_rows32.hip -- the decode-batch GEMV of the 32-value weight types for gfx950: Q8_0 / Q4_0
// weights x per-32 activations for 2..16 activation rows per pass, on int8 MFMA.
//
// Arithmetic per output and 32-value block b (kernels_generic.cpp:210-239): P_b, the exact
// integer dot of the codes (Q4_0: nibble - 8), t = dw_b da_b rounded to fp32, acc = acc + t
// (float)P_b over the blocks of a K slice in order, the slices added in order. Slices and roundings
// are the VALU GEMV's (gemv_splits ranges of gemv_waves32 slices), so an output has the same bits
// from either kernel, whatever the row count, the row range or the route.
//
// MFMA mapping (v_mfma_i32_16x16x64_i8: lane l supplies row / column l % 16 and 16 K values of
// lane group l / 16; result lane l holds column l % 16, rows 4 (l / 16) .. + 3). A step takes
// four blocks, one per lane group: a lane's 16 bytes of weights are then one whole load (Q8_0:
// two) of its row, with no exchange between lanes, and a lane's activation operand is a whole
// block of its activation row. Block g's dot is the MFMA with the activation operand zeroed
// outside group g (eight `and`s a block, shared by the step's TC weight tiles); t = dw da of the
// four blocks' 16 x 16 outputs is one v_mfma_f32_16x16x1_4b_f32 on the scales, group g's for block
// g (one product per output, rounded once); Q4_0's -8 sum(a) is the same MFMA against a constant
// -8, once per block, as the accumulator the tiles start from. That leaves 12 VALU per block and
// tile (convert, multiply, add) and Q4_0's 12 a step to split nibbles.
//
// The activations come quantized (one launch for the call): quantizing a lane's own block in
// here, 32 values at ~8 VALU each in every workgroup, took 19.6 us a call against 15.
//
// Work split: a workgroup owns 16 TC weight rows and all of K; TC = 4 (the weight load
// instructions read 1 KB runs, the activations are prepared once per 64 weight rows) where
// narrower ones would need a second round on the CUs, else 2 or 1 (N = 11008 Q8_0 at 8 rows 12.2 us
// against 15.8 with 32-row workgroups). A wave's slices are contiguous in K. Of two short slices
// (16 of a whole row) each takes two lane groups, which leaves no lane group idle at a slice's end;
// one after the other they took 3.9 us instead of 3.0 at K = 1024, N = 4096. Slice by slice go the
// long rows of few row groups (two ranges and more) and Q8_0's slices of 12 blocks and more: a load
// of four consecutive blocks touches half the cache lines of four slices' (Q8_0 K = 14336, N = 5120
// at 8 rows 30.3 us against 34.2; K = 7360, N = 14336 at 12 rows 22.2 against 24.1), on 16 waves
// where one workgroup fills a CU (N = 2048, Q4_0 14.6 against 16.6).
// What bounds it: Q4_0 K = 4096, N = 14336 at 8 rows takes 10.8 us for 33 MB (3.1 TB/s; the
// VALU GEMV, which pays its dots for every row, 15.3). A wave's four steps are 44 MFMAs (768 clocks)
// and ~350 VALU (1,400) each; loads one or two steps ahead measured alike.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dq_device.h"
#include "dq_internal.h"
#include "dq_mfma.h"
#include "dq_quant.h"

namespace dq {

namespace {

typedef float v4f_t __attribute__((ext_vector_type(4)));
typedef float v16f_t __attribute__((ext_vector_type(16)));
typedef u32 v4ua __attribute__((ext_vector_type(4), aligned(4)));  // loads of 4-byte aligned rows
constexpr u32 kNoLoad = 0xFFFFFFF0u;  // a buffer offset past every resource: the load returns zeros

// One lane's activation block: codes of values 0..15 and 16..31, the scale.
struct ActBlk {
  v4u lo, hi;
  float d;
};

struct ActRaw {  // ActBlockQ8 {float d; int32 sum; int8 q[32]}
  v4u q[2];
  float d;
  DQ_DEV void load(const uint8_t* row, int b) {
    const uint8_t* p = row + (int64_t)b * 40;
    d = *reinterpret_cast<const float*>(p);
    q[0] = *reinterpret_cast<const v4ua*>(p + 8);
    q[1] = *reinterpret_cast<const v4ua*>(p + 24);
  }
  DQ_DEV ActBlk block() const { return ActBlk{q[0], q[1], d}; }
};

// A lane's weights of one step and tile.
template <int WT>
struct WBlk {
  v4u q[WT == kQ8_0 ? 2 : 1];
  u32 d;
  DQ_DEV void load(__amdgpu_buffer_rsrc_t rq, __amdgpu_buffer_rsrc_t rd, u32 gb, u32 r, int b, int end) {
    const u32 blk = gb + (u32)b;
    const bool in = b < end;
    if constexpr (WT == kQ8_0) {
      q[0] = ld16nt(rq, in ? (blk * 2 * 64 + r) * 16 : kNoLoad);
      q[1] = ld16nt(rq, in ? ((blk * 2 + 1) * 64 + r) * 16 : kNoLoad);
    } else {
      q[0] = ld16nt(rq, in ? (blk * 64 + r) * 16 : kNoLoad);
    }
    d = ld2nt(rd, in ? (blk * 64 + r) * 2 : kNoLoad);
  }
  DQ_DEV v4u lo() const { return WT == kQ8_0 ? q[0] : q[0] & 0x0F0F0F0Fu; }
  DQ_DEV v4u hi() const { return WT == kQ8_0 ? q[WT == kQ8_0 ? 1 : 0] : (q[0] >> 4) & 0x0F0F0F0Fu; }
};

}  // namespace

// Workgroup i: weight rows [16 (t0 + i TC), + 16 TC); acts: m <= 16 ActBlockQ8 rows `stride`
// bytes apart; kSplits K-ranges of WR slices. A wave's slices, contiguous in K, go in kRounds
// rounds of G at once: the lane groups take 4 / G blocks of each of the G a step, `steps` steps a round.
template <int WT, int TC, int kWaves, int kSplits, int WR, int G>
__global__ __launch_bounds__(64 * kWaves) void k_rows32(const uint8_t* __restrict__ p0, const uint8_t* __restrict__ p1,
                                                        int nblk, int64_t n_pad, int64_t t0, int64_t n0, int64_t n1,
                                                        const uint8_t* __restrict__ acts, int64_t stride, int m,
                                                        float* __restrict__ y, int64_t ys,
                                                        const float* __restrict__ bias, int steps) {
  extern __shared__ __align__(16) float red[];
  const int t = threadIdx.x, lane = t & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t tile0 = t0 + (int64_t)blockIdx.x * TC;
  const auto rq = rsrc(p0, (u32)(n_pad * nblk * plane_unit(WT, 0)));
  const auto rd = rsrc(p1, (u32)(n_pad * nblk * 2));
  u32 gb[TC], r[TC];
#pragma unroll
  for (int i = 0; i < TC; ++i) {
    const int64_t n = 16 * (tile0 + i) + c;
    gb[i] = (u32)((n >> 6) * nblk);
    r[i] = (u32)(n & 63);
  }
  const uint8_t* row = acts + (int64_t)(c < m ? c : m - 1) * stride;  // rows past m repeat the last one (not stored)

  // the lane group's slice of a round, [b, end); its block of step q is b + kB q
  constexpr int kB = 4 / G, kPer = kSplits * WR / kWaves, kRounds = kPer / G;
  static_assert(kPer * kWaves == kSplits * WR && kPer % G == 0, "whole rounds");
  int b, end;
  auto round = [&](int r) {
    const int i = kPer * wave + G * r + g / kB, sk = i / WR, wl = i % WR;
    const int k0 = sk * nblk / kSplits, k1 = (sk + 1) * nblk / kSplits;
    b = k0 + wl * (k1 - k0) / WR + g % kB;
    end = k0 + (wl + 1) * (k1 - k0) / WR;
  };
  round(0);
  v4f_t acc[G][TC];
#pragma unroll
  for (int i = 0; i < G * TC; ++i) acc[i / TC][i % TC] = v4f_t{};
  // the next kD steps' loads in flight (one where two would spill registers), step q in set q %
  // kD; blocks past the slice repeat some block's codes, with weights and scales of zero (an
  // infinite scale times a zero weight is NaN)
  constexpr int kD = TC == 4 ? 1 : 2;
  WBlk<WT> w[kD][TC];
  ActRaw a[kD];
  int lq = 0, lr = 0;  // the step to load: step lq of round lr
  const int total = kRounds * steps;
  auto load = [&](int set) {
    a[set].load(row, b < nblk ? b : nblk - 1);
    if (b >= end) a[set].d = 0.0f;
#pragma unroll
    for (int i = 0; i < TC; ++i) w[set][i].load(rq, rd, gb[i], r[i], b, end);
    b += kB;
    if (kRounds > 1 && ++lq == steps) {
      lq = 0;
      round(++lr);
    }
  };
#pragma unroll
  for (int q = 0; q < kD; ++q) {
    if (q < total) load(q);
  }
  // a round's sums: element (tile i, lane, e) of slice j at ((j TC + i) 64 + lane) 4 + e
  auto put_slices = [&](int r) {
#pragma unroll
    for (int i = 0; i < G * TC; ++i) {
      *reinterpret_cast<v4f_t*>(red + (((kPer * wave + G * r + i / TC) * TC + i % TC) * 64 + lane) * 4) =
          acc[i / TC][i % TC];
      acc[i / TC][i % TC] = v4f_t{};
    }
  };
  int cq = 0, cr = 0;  // the step to compute
  auto step = [&](int q, int set) {
    const ActBlk x = a[set].block();
    v4u lo[TC], hi[TC];
    float dw[TC];
#pragma unroll
    for (int i = 0; i < TC; ++i) {
      lo[i] = w[set][i].lo();
      hi[i] = w[set][i].hi();
      dw[i] = h2f(w[set][i].d);
    }
    if (q + kD < total) load(set);
    // t = dw da of the four blocks' 16 x 16 outputs: [block][4 rows]
    v16f_t sc[TC];
#pragma unroll
    for (int i = 0; i < TC; ++i) sc[i] = __builtin_amdgcn_mfma_f32_16x16x1f32(x.d, dw[i], v16f_t{}, 0, 0, 0);
#pragma unroll
    for (int gg = 0; gg < 4; ++gg) {
      const u32 mask = g == gg ? 0xFFFFFFFFu : 0u;
      const v4u al = x.lo & mask, ah = x.hi & mask;
      v4i_t c0 = {};
      if constexpr (WT == kQ4_0) {
        const v4u m8 = {0xF8F8F8F8u, 0xF8F8F8F8u, 0xF8F8F8F8u, 0xF8F8F8F8u};
        c0 = mfma(ah, m8, mfma(al, m8, c0));
      }
#pragma unroll
      for (int i = 0; i < TC; ++i) {
        const v4i_t P = mfma(ah, hi[i], mfma(al, lo[i], c0));
        v4f_t& s = acc[gg / kB][i];
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = s[e] + sc[i][4 * gg + e] * (float)P[e];
      }
    }
    if (kRounds > 1 && ++cq == steps) {
      put_slices(cr++);
      cq = 0;
    }
  };
#pragma unroll 1
  for (int q = 0; q < total; q += kD) {
    step(q, 0);
    if (kD == 2 && q + 1 < total) step(q + 1, kD - 1);
  }
  if (kRounds == 1) put_slices(0);

  // each K-range's slices in order, then the ranges
  __syncthreads();
  for (int e = t; e < TC * 256; e += 64 * kWaves) {
    const int l = (e >> 2) & 63, mr = 4 * (l >> 4) + (e & 3);
    const int64_t n = 16 * (tile0 + (e >> 8)) + (l & 15);
    float v = 0;
    for (int sk = 0; sk < kSplits; ++sk) {
      float u = 0;
#pragma unroll
      for (int k = 0; k < WR; ++k) u = u + red[(sk * WR + k) * TC * 256 + e];
      v = v + u;
    }
    if (mr < m && n >= n0 && n < n1) y[mr * ys + n] = bias ? v + bias[n] : v;
  }
}

namespace {

template <int WT, int TC, int kWaves, int kSplits, int WR, int G>
hipError_t launch1(const WeightDev& w, const uint8_t* acts, int64_t stride, int64_t m, int64_t n0, int64_t n1, float* y,
                   int64_t ys, const float* bias, hipStream_t s) {
  static_assert(kSplits * WR * TC <= 64, "64 KB of LDS");
  const int64_t t0 = n0 / 16, wgs = ((n1 + 15) / 16 - t0 + TC - 1) / TC;
  const int64_t range = (w.nblk + kSplits - 1) / kSplits, slice = (range + WR - 1) / WR;
  hipLaunchKernelGGL((k_rows32<WT, TC, kWaves, kSplits, WR, G>), dim3((unsigned)wgs), dim3(64 * kWaves),
                     kSplits * WR * TC * 1024, s, w.plane[0], w.plane[1], (int)w.nblk, w.n_pad, t0, n0, n1, acts,
                     stride, (int)m, y, ys, bias, (int)((slice * G + 3) / 4));
  return hipGetLastError();
}

template <int WT>
hipError_t launch_type(const WeightDev& w, const uint8_t* acts, int64_t stride, int64_t m, int64_t n0, int64_t n1,
                       float* y, int64_t ys, const float* bias, hipStream_t s) {
  const int64_t tiles = w.n_pad / 16, cus = w.cus > 0 ? w.cus : 256;
  const int tc = tiles > 2 * cus ? 4 : 2 * tiles >= 3 * cus ? 2 : 1;
#define DQ_ROWS32(...) launch1<WT, __VA_ARGS__>(w, acts, stride, m, n0, n1, y, ys, bias, s)
  switch (gemv_splits(w, kActPer32)) {
    case 1:
      if (gemv_waves32(w, kActPer32) == 8) return DQ_ROWS32(4, 8, 1, 8, 1);
      if constexpr (WT == kQ8_0) {
        // long slices one after the other where that takes (nearly) no more steps
        const int64_t slice = (w.nblk + 15) / 16;
        if (slice >= 20 || (slice >= 12 && (slice + 1) % 4 <= 1)) {
          return tc == 4 ? DQ_ROWS32(4, 8, 1, 16, 1) : tc == 2 ? DQ_ROWS32(2, 8, 1, 16, 1) : DQ_ROWS32(1, 8, 1, 16, 1);
        }
      }
      return tc == 4 ? DQ_ROWS32(4, 8, 1, 16, 2) : tc == 2 ? DQ_ROWS32(2, 8, 1, 16, 2) : DQ_ROWS32(1, 8, 1, 16, 2);
    case 2: return tc == 1 ? DQ_ROWS32(1, 8, 2, 8, 1) : DQ_ROWS32(2, 8, 2, 8, 1);
    case 3: return DQ_ROWS32(1, 8, 3, 8, 1);
    case 4: return DQ_ROWS32(1, 16, 4, 8, 1);
    case 5: return DQ_ROWS32(1, 10, 5, 8, 1);
    case 6: return DQ_ROWS32(1, 16, 6, 8, 1);
    case 7: return DQ_ROWS32(1, 14, 7, 8, 1);
    case 8: return DQ_ROWS32(1, 16, 8, 8, 1);
    default: return hipErrorInvalidValue;
  }
#undef DQ_ROWS32
}

}  // namespace

// Against the VALU GEMV's passes of up to 8 rows, measured for K = 64 .. 14336, N = 256 .. 32000 (us).
//  - Rows to quantize first (a launch more; a call from Python, K = 4096): 5 rows and more always
//    (the VALU GEMV then takes a second pass; its one pass of 8 rows wins below K = 256): N = 4096
//    Q4_0 at 3 / 4 / 5 / 8 / 12 rows 10.4 / 8.1 / 8.2 / 8.2 / 8.7 against 8.2 / 9.9 / 14.4 / 16.6 /
//    26.1, K = 1024 at 3 / 4 / 5 / 8 rows 10.4 / 10.4 / 7.7 / 7.7 against 5.3 / 6.3 / 9.6 / 10.0; N =
//    11008 Q8_0 at 4 / 5 / 8 rows 15.7 / 13.9 / 14.3 against 11.0 / 18.9 / 17.2. At 4 rows only K
//    >= 4096 pays, on workgroups of at most two tiles (K = 14336, N = 4096 Q8_0 18.9 against 21.5).
//  - Quantized rows (dq_gemv, GPU time): also 3 and 4 rows of those weights, 3 not on the longest rows:
//    K = N = 4096 Q4_0 6.0 / 5.8 against 7.0 / 8.3; K = 14336, N = 3072 Q4_0 at 3 rows 15.3 against
//    12.8; N = 14336 at 4 rows 10.7 against 9.6.
// (From 13 rows the calls that may take the block GEMM do.)
bool rows32_pays(const WeightDev& w, int af, int64_t m, bool quantize) {
  if ((w.dtype != kQ8_0 && w.dtype != kQ4_0) || af != kActPer32 ||
      w.n_pad * w.nblk * plane_unit(w.dtype, 0) >= (int64_t)kNoLoad) {
    return false;
  }
  const bool wide = w.n_pad / 16 > 2 * (w.cus > 0 ? w.cus : 256);
  if (m >= 5) return m > 8 || w.k >= 256 || !(wide || (quantize && m == 8));
  if (wide) return false;
  return quantize ? m == 4 && w.k >= 4096 : m == 4 || (m == 3 && w.k <= 8192);
}

hipError_t launch_rows32(const WeightDev& w, const uint8_t* acts, int64_t arb, int64_t m, int64_t n0, int64_t n1,
                         float* y, int64_t ys, const float* bias, hipStream_t s) {
  if ((w.dtype != kQ8_0 && w.dtype != kQ4_0) || m < 1 || m > kRows32Max || n1 <= n0) return hipErrorInvalidValue;
  return w.dtype == kQ8_0 ? launch_type<kQ8_0>(w, acts, arb, m, n0, n1, y, ys, bias, s)
                          : launch_type<kQ4_0>(w, acts, arb, m, n0, n1, y, ys, bias, s);
}

}  // namespace dq
