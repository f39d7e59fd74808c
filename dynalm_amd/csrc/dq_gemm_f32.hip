// dq_gemm_f32.hip -- the fp32-activation prefill GEMM on the matrix cores (the
// "expand + GEMM" accuracy class, dynacore's kF32ExpandGemm:
// dynacore/cpu/cpu_device.cpp:1114-1152 with gemm_panel, kernels_avx2.cpp:146-230).
//
// The weight values are the reference's x86 expansion (kernels_avx2.cpp:370-466,
// store_scaled = fma(q, scale, offset)):
//   Q4_K  fma((float)q, d * sc_j, -(dmin * m_j))        q in 0..15
//   Q6_K  (float)q * (d * sc_g)                          q in -32..31
//   Q8_0  (float)q * d,  Q4_0  (float)(nibble - 8) * d
// i.e. an integer code, which bf16 holds exactly, times a scale that all 32 (Q6_K: 16)
// values of a block share. The products therefore run on the bf16 matrix cores, 16 times
// the rate of v_mfma_f32: each fp32 activation times 2^24 splits exactly into three bf16 parts
// (8 + 8 + 8 significand bits, round to nearest), 2^24 x = hi + mid + lo, and one block's
//   S = sum_k 2^24 x_k q_k
// is three bf16 MFMAs per K-step into one fp32 accumulator. Every product is exact (8 x at
// most 8 bits), so S has fp32 rounding only, and acc = fma(scale, S, acc) applies the
// scale once per block. Q4_K's offsets are Mn = sum_j m_j X_j, X_j the block's fp32
// activation sum (split the same way, one MFMA per super-block and tile), folded as
// fma(-dmin, Mn, acc). scale * q is exact in fp32 for every type with an offset (11 + 6 + 4
// bits), so a one-hot row returns the expanded weight bit for bit, in whichever order the
// two are added. Error against the exact product at K = 4096 (N(0, 1)-like rows): 2-norm
// relative 2.9e-7, against 1.1e-6 for v_mfma_f32_32x32x2_f32 over expanded weights (2048
// dependent fp32 additions per output; here 128 plus the sums inside an MFMA). The 2^24, taken off
// the finished sum, keeps the parts of every fp32 value, subnormal ones too, in bf16's normal range
// (unscaled, rows near 1e-36 came out 2e-5 off and near 1e-39 2e-2); it costs one of the split's 6.5
// VALU per value (K = 4096, N = 14336, M = 512: 174.7 -> 175.3 us, N = 4096, M = 16: 62.6 -> 65.3).
//
// Work split: a workgroup has 8 waves over 32 RG activation rows x 32 NTW (4 / RG) weight
// rows. Waves w and w + 4 (one SIMD) hold the same output tiles and take the two 32-value
// blocks of each 64-value chunk; their sums are added at the end, so an output's order of
// additions depends on K alone, not on the tile shape, the row count or the row. A wave
// splits its own 32 rows' activations (6.5 VALU per value) for NTW tiles, through LDS that no
// other wave touches; the weight codes become bf16 once per workgroup, in two LDS buffers.
// The split in the kernel keeps the call free of workspaces, launches and library state.
//
// Non-finite and huge inputs: an infinity has no exact split (its mid part is inf - inf) and 2^24 x
// overflows from 2^104 (2e31) on, so the tiles of outputs that come out infinite or NaN are run
// again on v_mfma_f32_32x32x2 over expanded weights, and those outputs taken from there. With
// every row holding a NaN or an infinity M = 512, K = 4096, N = 14336 takes 1110 us
// (all of it on v_mfma_f32 600; one dot per lane and output, as it was, 33500).
//
// Q4_K, K = 4096, N = 14336, M = 512: 543 -> 167-173 us (111 -> 355 TFLOP/s; over weights in turn
// 214-227, in the same number of clocks at a lower rate); Q6_K K = 14336, N = 4096: 1207 -> 290; Q8_0 4096 x
// 4096: 306 -> 79; M = 16 at N = 14336: 314 -> 69. What bounds it now: VALU issue beside the MFMAs. A
// wave's chunk is 44 MFMAs and 364 VALU, 8 per MFMA, where a register-only loop of 2 waves per
// SIMD hides 4 to 6; the matrix pipe is busy 54% of the clocks and has a VALU op beside it in 55% of
// those. Timing-only copies (before the scaling): the MFMAs alone 81 us of 172, with operand reads and
// barriers 117, with the folds too 123; without only the activation split 32 less, the weight
// conversion 26, the offsets 20, the folds 20.
//
// MFMA lane layout (v_mfma_f32_32x32x16_bf16): lane l supplies row (A) / column (B) l % 32
// and K = 8 (l / 32) .. + 7; result register r of lane l is row 8 (r / 4) + 4 (l / 32) +
// r % 4, column l % 32.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "dq_device.h"
#include "dq_f16mma.h"
#include "dq_internal.h"

namespace dq {

namespace {

typedef float v4f_t __attribute__((ext_vector_type(4)));

constexpr int kKc = 32;               // K values per block: a block (Q8_0, Q4_0) or sub-block (K-quants)
constexpr int kThreadsF = 512;
constexpr float kXScale = 0x1p24f;    // of the activations (see the split above)
constexpr u32 kNoLoad = 0xFFFFFFF0u;  // a buffer offset past every resource: the load returns zeros

// The exact three-part split of two floats: a pair of bf16 per part.
DQ_DEV void split3(float a, float b, u32& hi, u32& mid, u32& lo) {
  hi = bf_pair(a, b);
  a -= as_f(hi << 16);
  b -= as_f(hi & 0xFFFF0000u);
  mid = bf_pair(a, b);
  a -= as_f(mid << 16);
  b -= as_f(mid & 0xFFFF0000u);
  lo = bf_pair(a, b);
}
// Four bytes 0..15 as bf16: read as fp8 (e4m3), a byte b < 16 is b * 2^-9 (subnormals up to
// 7, then the first binade), which the conversion's scale undoes.
DQ_DEV void nibbles_bf(u32 w, u32& a, u32& b) {
  a = __builtin_bit_cast(u32, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 512.0f, false));
  b = __builtin_bit_cast(u32, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 512.0f, true));
}
// Four signed bytes as bf16.
DQ_DEV void bytes_bf(u32 w, u32& a, u32& b) {
  a = bf_pair((float)(int8_t)(w & 0xFFu), (float)(int8_t)((w >> 8) & 0xFFu));
  b = bf_pair((float)(int8_t)((w >> 16) & 0xFFu), (float)(int8_t)(w >> 24));
}

// The 32-value block that wave group g takes of 64-value chunk t.
template <int WT>
DQ_DEV int chunk_block(int t, int g) {
  if constexpr (WT == kQ6_K) return 8 * (t >> 2) + 4 * ((t >> 1) & 1) + (t & 1) + 2 * g;
  return 2 * t + g;
}

// The raw bytes one thread converts per chunk: weight row r of its 64-row group, whose
// blocks start at block index gb of the plane (G * nblk), and a half `sel` of the chunk.
// The resources span whole planes; rows past the weight's padded rows and blocks past the
// row read zeros. put writes the half's 32 codes as bf16 operands: op(g, s) is the 1 KB
// operand block of wave group g's block and K-step s (values 16 s .. + 15) for the row's
// tile, at lane 32 h + row % 32 for values 8 h .. + 7; and the scales.
template <int WT>
struct Raw;

DQ_DEV void put_op(uint8_t* op, u32 a0, u32 a1, u32 a2, u32 a3, u32 b0, u32 b1, u32 b2, u32 b3) {
  *reinterpret_cast<v4u*>(op) = v4u{a0, a1, a2, a3};
  *reinterpret_cast<v4u*>(op + 512) = v4u{b0, b1, b2, b3};
}
DQ_DEV void put_nibbles(uint8_t* op, v4u w) {  // 16 bytes 0..15
  u32 a[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) nibbles_bf(w[i], a[2 * i], a[2 * i + 1]);
  put_op(op, a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7]);
}
DQ_DEV void put_bytes(uint8_t* op, v4u w) {  // 16 signed bytes
  u32 a[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) bytes_bf(w[i], a[2 * i], a[2 * i + 1]);
  put_op(op, a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7]);
}

// Q4_K: chunk t = sub-blocks 2 (t % 4) and + 1 of super-block t / 4, the low and high
// nibbles of qs bytes 32 (t % 4) .. + 31; sel = the 16-byte half (K-step).
template <>
struct Raw<kQ4_K> {
  v4u qs, hd;
  DQ_DEV void load(const __amdgpu_buffer_rsrc_t* rs, u32 gb, int, int t, int sel, int r) {
    const u32 b = gb + (u32)(t >> 2);
    qs = ld16(rs[0], ((b * 8 + 2 * (u32)(t & 3) + (u32)sel) * 64 + (u32)r) * 16);
    hd = ld16(rs[1], (b * 64 + (u32)r) * 16);
  }
  template <int kPart, class Op>
  DQ_DEV void put(int t, int sel, Op op, float* ds, int rows, int row) const {
    const u32 m4 = 0x0F0F0F0Fu;
    if constexpr (kPart == 0) {
      put_nibbles(op(0, sel), qs & m4);
    } else {
      put_nibbles(op(1, sel), ((qs >> 4) & m4) ^ 0x08080808u);  // the plane stores the high nibble XOR 8
      // get_scale_min_k4 (quant_formats.h:62-70) from the scale bytes s[0..3] = hd.y,
      // s[4..7] = hd.z, s[8..11] = hd.w: this thread's share is group sel's sub-blocks
      const int j = 2 * (t & 3) + sel, sh = 8 * (j & 3);
      const u32 lo6 = hd.y >> sh;
      // (both forms and a mask: a branch would split the step's schedule)
      const u32 up = 0u - ((u32)t >> 1 & 1u), hi4 = ((hd.w >> sh) & 15u) | (((lo6 >> 6) & 3u) << 4);
      ds[sel * rows + row] = h2f(hd.x) * (float)(((lo6 & 63u) & ~up) | (hi4 & up));
    }
  }
  // the super-block's mins: group sel's m_j in chunk order, and dmin
  static DQ_DEV void put_mins(v4u hd, int sel, uint8_t* mins, int rows, int row) {
    const u32 a = hd.z >> (8 * sel), b = hd.w >> (8 * sel);
    const int m0 = (int)(a & 63u), m1 = (int)((a >> 16) & 63u);
    const int m2 = (int)(((b >> 4) & 15u) | (((a >> 6) & 3u) << 4));
    const int m3 = (int)(((b >> 20) & 15u) | (((a >> 22) & 3u) << 4));
    *reinterpret_cast<v2u*>(mins + (sel * rows + row) * 8) =
        v2u{bf_pair((float)m0, (float)m1), bf_pair((float)m2, (float)m3)};
    if (sel == 0) reinterpret_cast<float*>(mins + 16 * rows)[row] = h2f(hd.x >> 16);
  }
};

// Q6_K: chunk t = values 128 h + 32 p + (0..31) and + 64 of super-block t / 4 (h = bit 1, p =
// bit 0 of t % 4; quant_formats.cpp:192-216): low and high nibbles of ql bytes 64 h + 32 p ..
// + 31 with two bits of qh bytes 32 h .. + 31 (bits 2 p and 4 + 2 p); sel = the 16-byte half.
template <>
struct Raw<kQ6_K> {
  v4u ql, qh;
  v2u sc;
  u32 dw;
  DQ_DEV void load(const __amdgpu_buffer_rsrc_t* rs, u32 gb, int, int t, int sel, int r) {
    const u32 b = gb + (u32)(t >> 2), c = 2 * (u32)(t & 3) + (u32)sel, h = (u32)(t >> 1) & 1, rr = (u32)r;
    ql = ld16(rs[0], ((b * 8 + c) * 64 + rr) * 16);
    qh = ld16(rs[1], ((b * 4 + 2 * h + (u32)sel) * 64 + rr) * 16);
    sc = ld8(rs[2], (b * 64 + rr) * 16 + 8 * h);
    dw = ld2(rs[3], (b * 64 + rr) * 2);
  }
  template <int kPart, class Op>
  DQ_DEV void put(int t, int sel, Op op, float* ds, int rows, int row) const {
    const int p = t & 1;
    const v4u hs = qh >> (2 * p + 4 * kPart);
    const v4u q = ((ql >> (4 * kPart)) & 0x0F0F0F0Fu) | ((hs & 0x03030303u) << 4);
    put_bytes(op(kPart, sel), (q + 0x60606060u) ^ 0x80808080u);  // q - 32 as signed bytes
    const float sc1 = (float)(int8_t)((sc[kPart] >> (8 * (2 * p + sel))) & 0xFFu);
    ds[(2 * kPart + sel) * rows + row] = h2f(dw) * sc1;
  }
};

// Q8_0: chunk t = blocks 2 t and 2 t + 1; sel = the 16-value half of both.
template <>
struct Raw<kQ8_0> {
  v4u qs[2];
  u32 dw;
  DQ_DEV void load(const __amdgpu_buffer_rsrc_t* rs, u32 gb, int nblk, int t, int sel, int r) {
    const u32 b = gb + 2 * (u32)t, rr = (u32)r;
    const bool two = 2 * t + 1 < nblk;
    qs[0] = ld16(rs[0], ((b * 2 + (u32)sel) * 64 + rr) * 16);
    qs[1] = ld16(rs[0], two ? ((b * 2 + 2 + (u32)sel) * 64 + rr) * 16 : kNoLoad);
    dw = ld2(rs[1], sel == 0 || two ? ((b + (u32)sel) * 64 + rr) * 2 : kNoLoad);
  }
  template <int kPart, class Op>
  DQ_DEV void put(int, int sel, Op op, float* ds, int rows, int row) const {
    put_bytes(op(kPart, sel), qs[kPart]);
    if (kPart == 0) ds[sel * rows + row] = h2f(dw);
  }
};

// Q4_0: chunk t = blocks 2 t and 2 t + 1; sel = the block, whose low nibbles are values
// 0..15 and high ones 16..31 (quant_formats.cpp:12-20).
template <>
struct Raw<kQ4_0> {
  v4u qs;
  u32 dw;
  DQ_DEV void load(const __amdgpu_buffer_rsrc_t* rs, u32 gb, int nblk, int t, int sel, int r) {
    const u32 b = gb + 2 * (u32)t + (u32)sel, rr = (u32)r;
    const bool in = 2 * t + sel < nblk;
    qs = ld16(rs[0], in ? (b * 64 + rr) * 16 : kNoLoad);
    dw = ld2(rs[1], in ? (b * 64 + rr) * 2 : kNoLoad);
  }
  template <int kPart, class Op>
  DQ_DEV void put(int, int sel, Op op, float* ds, int rows, int row) const {
    const v4u q = (qs >> (4 * kPart)) & 0x0F0F0F0Fu;
    put_bytes(op(sel, kPart), (q + 0x78787878u) ^ 0x80808080u);  // q - 8 as signed bytes
    if (kPart == 0) ds[sel * rows + row] = h2f(dw);
  }
};

// The expanded weights k .. k + 3 (k % 4 == 0) of the row at (gb, r): the plain fp32 path.
template <int WT>
DQ_DEV v4f_t expand4(const __amdgpu_buffer_rsrc_t* rs, u32 gb, u32 r, u32 k) {
  v4f_t w;
  if constexpr (WT == kQ4_K) {
    const u32 b = gb + k / 256, j = k / 32 % 8, l = k % 32;
    const v4u hd = ld16(rs[1], (b * 64 + r) * 16);
    const u32 q = ld4(rs[0], ((b * 8 + 2 * (j >> 1) + l / 16) * 64 + r) * 16 + l % 16) ^ 0x80808080u;
    int sc, mn;
    scale_min_k4((int)j, hd.y, hd.z, hd.w, sc, mn);
    const float d = h2f(hd.x) * (float)sc, o = -(h2f(hd.x >> 16) * (float)mn);
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = fmaf((float)((q >> (8 * e + 4 * (j & 1))) & 15u), d, o);
  } else if constexpr (WT == kQ6_K) {
    const u32 b = gb + k / 256, u = k / 32 % 8, p = u >> 2, s = u & 3, l = k % 32;
    const u32 ql = ld4(rs[0], ((b * 8 + 4 * p + 2 * (s & 1) + l / 16) * 64 + r) * 16 + l % 16) >> (4 * (s >> 1));
    const u32 qh = ld4(rs[1], ((b * 4 + 2 * p + l / 16) * 64 + r) * 16 + l % 16) >> (2 * s);
    const int sc = (int8_t)__builtin_amdgcn_raw_buffer_load_b8(rs[2], (b * 64 + r) * 16 + k / 16 % 16, 0, 0);
    const float d = h2f(ld2(rs[3], (b * 64 + r) * 2)) * (float)sc;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w[e] = (float)((int)(((ql >> (8 * e)) & 15u) | (((qh >> (8 * e)) & 3u) << 4)) - 32) * d;
  } else {
    const u32 b = gb + k / 32, l = k % 32;
    const float d = h2f(ld2(rs[1], (b * 64 + r) * 2));
    const u32 q = WT == kQ8_0 ? ld4(rs[0], ((b * 2 + l / 16) * 64 + r) * 16 + l % 16)
                              : ld4(rs[0], (b * 64 + r) * 16 + l % 16) >> (l < 16 ? 0 : 4);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w[e] = (float)(WT == kQ8_0 ? (int)(int8_t)((q >> (8 * e)) & 0xFFu) : (int)((q >> (8 * e)) & 15u) - 8) * d;
  }
  return w;
}

// A wave's activation operands: block (s, part) of K-step s at 3904 s + 1280 part, lane
// 32 h + r of it at 640 h + 16 r: h and s are 128 and 64 B apart modulo the 256 B of the
// banks, so that 32 lanes writing 4 rows' 8-byte pieces meet no conflict.
constexpr int kXblk = 1280, kXs = 3 * kXblk + 64, kXop = kXs + 3 * kXblk;

// A workgroup's tile: 32 RG activation rows x 32 NTT weight rows, each wave 32 rows x NTW
// weight tiles. LDS: two buffers of bf16 operands (4 KB per tile) and scales, Q4_K's mins
// of two super-blocks, and each wave's activation operands; at the end the waves exchange half their sums in the same memory.
// The conversion works on whole 64-row blocks; rows past the tile go to operands that no
// wave reads.
template <int WT, int RG, int NTW>
struct F32Tile {
  static constexpr int kBM = 32 * RG, kCG = 4 / RG, kNTT = NTW * kCG, kBN = 32 * kNTT;
  static constexpr int kRows = 64 * ((kBN + 63) / 64);
  static constexpr int kItems = 2 * kRows;  // (row, half) items of a chunk
  static constexpr int kPasses = (kItems + kThreadsF - 1) / kThreadsF;
  // chunks whose loads are in flight: the narrow tiles' chunks take less than a load's latency
  static constexpr int kDepth = NTW <= 2 ? 2 : 1;
  static constexpr int kScales = WT == kQ6_K ? 4 : 2;
  static constexpr int kOpT = kRows / 32;  // tiles of LDS operands
  static constexpr int kOps = kOpT * 4096, kBuf = kOps + kScales * kRows * 4;
  static constexpr int kMins = WT == kQ4_K ? kRows * 20 : 0;
  static constexpr int kXm = WT == kQ4_K ? 2048 : 0;  // a wave's X_j operands of two super-blocks
  static constexpr int kOffMins = 2 * kBuf, kOffX = kOffMins + 2 * kMins, kOffXm = kOffX + 8 * kXop;
  static constexpr int kHalf = (NTW + 1) / 2;  // tiles a wave hands over
  static constexpr int kLoop = kOffXm + 8 * kXm, kRed = 8 * kHalf * 4096;
  static constexpr int kLds = kLoop > kRed ? kLoop : kRed;
  static_assert(kItems % kThreadsF == 0 || kItems < kThreadsF, "whole passes");
  static_assert(kLds <= 160 * 1024, "LDS");
};

}  // namespace

// One workgroup: activation rows [mbase, mbase + 32 RG) x weight rows [nbase, nbase + kBN).
// x: fp32 rows of stride xs floats; nslices = K / 32.
template <int WT, int RG, int NTW>
__global__ __launch_bounds__(kThreadsF) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_gemm_f32(
    const uint8_t* __restrict__ p0, const uint8_t* __restrict__ p1, const uint8_t* __restrict__ p2,
    const uint8_t* __restrict__ p3, int nblk, int k, int nslices, int64_t nbase0, int64_t n_pad, int64_t n0, int64_t n1,
    const float* __restrict__ x, int64_t xs, int64_t m, float* y, int64_t ys, const float* __restrict__ bias,
    int tiles_m, int xcd_map) {
  using T = F32Tile<WT, RG, NTW>;
  extern __shared__ __align__(16) uint8_t smem[];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 31, lg = lane >> 5;
  const int g = wave >> 2, rg = (wave & 3) % RG, cg = (wave & 3) / RG;

  // the activation tiles of one weight tile on one XCD (workgroups are dealt to the 8 XCDs
  // round-robin), so that its L2 serves the weight re-reads
  const int L = blockIdx.x;
  int tn, tm;
  if (xcd_map) {
    tn = 8 * (L / (8 * tiles_m)) + (L & 7);
    tm = (L >> 3) % tiles_m;
  } else {
    tn = L / tiles_m;
    tm = L - tn * tiles_m;
  }
  tn = __builtin_amdgcn_readfirstlane(tn);
  tm = __builtin_amdgcn_readfirstlane(tm);
  const int64_t nbase = nbase0 + (int64_t)T::kBN * tn;
  const int64_t mbase = (int64_t)tm * T::kBM;
  const int64_t mrows = m - mbase < T::kBM ? m - mbase : T::kBM;

  __amdgpu_buffer_rsrc_t rs[4];
  {
    const uint8_t* pl[4] = {p0, p1, p2, p3};
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int unit = plane_unit(WT, p);
      rs[p] = unit > 0 ? rsrc(pl[p], (u32)(n_pad * nblk * unit)) : rsrc(p0, 0u);
    }
  }

  // ---- conversion role: item i = 512 p + t: 64-row block i >> 7, half (i >> 6) & 1, row i & 63
  const bool conv = T::kItems >= kThreadsF || wave < T::kItems / 64;
  int erow[T::kPasses], esel[T::kPasses], er[T::kPasses];
  u32 egb[T::kPasses];
#pragma unroll
  for (int p = 0; p < T::kPasses; ++p) {
    const int i = kThreadsF * p + t;
    erow[p] = 64 * (i >> 7) + (i & 63);
    esel[p] = __builtin_amdgcn_readfirstlane((i >> 6) & 1);
    const int64_t n = nbase + erow[p];
    er[p] = (int)(n & 63);
    egb[p] = (u32)((n >> 6) * nblk);
  }
  Raw<WT> raw[T::kDepth][T::kPasses];
  auto load_w = [&](int c, int set) {
    if (!conv) return;
#pragma unroll
    for (int p = 0; p < T::kPasses; ++p) raw[set][p].load(rs, egb[p], nblk, c, esel[p], er[p]);
  };
  auto put_w = [&](int c, int dst, int set, auto part) {  // chunk c's bytes, into chunk dst's buffer
    if (!conv) return;
    uint8_t* buf = smem + (dst & 1) * T::kBuf;
#pragma unroll
    for (int p = 0; p < T::kPasses; ++p) {
      const int row = erow[p];
      auto op = [&](int gg, int s) {
        return buf + ((gg * 2 + s) * T::kOpT + (row >> 5)) * 1024 + (row & 31) * 16;
      };
      raw[set][p].template put<decltype(part)::value>(c, esel[p], op, reinterpret_cast<float*>(buf + T::kOps), T::kRows, row);
    }
  };

  // ---- this wave's activation rows: load i takes rows 8 i + lane / 8 of its 32, 16 bytes a
  // lane, so that a row's 32-value block is one 128-byte line (a lane loading its own
  // operand row would touch 32 lines per load: Q8_0 4096 x 4096 at M = 512 91 us against 79).
  // Rows past m repeat the last one
  // (their outputs are not stored), blocks past K the last block (its weights are zero).
  // The parts go to the wave's operand blocks in LDS, which no other wave touches.
  const auto rx = rsrc(x + mbase * xs, (u32)(((mrows - 1) * xs + k) * 4));
  u32 x_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 32 * rg + 8 * i + (lane >> 3);
    x_off[i] = (u32)(((row < mrows ? row : (int)mrows - 1) * xs + 4 * (lane & 7)) * 4);
  }
  v4u xv[T::kDepth][4];
  auto load_x = [&](int c, int set, int i) {
    const int b = chunk_block<WT>(c, g);
    xv[set][i] = __builtin_bit_cast(
        v4u, __builtin_amdgcn_raw_buffer_load_b128(rx, x_off[i], (b < nslices ? b : nslices - 1) * kKc * 4, 0));
  };
  uint8_t* const xop = smem + T::kOffX + wave * kXop;
  uint8_t* const x_wr =
      xop + ((lane >> 2) & 1) * kXs + ((lane >> 1) & 1) * 640 + (lane >> 3) * 16 + (lane & 1) * 8;
  float xsum[4] = {0, 0, 0, 0};
  auto split_x = [&](int set, int i) {
    v4f_t v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = as_f(xv[set][i][j]) * kXScale;
    v2u hi, mid, lo;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      u32 h, md, l;
      split3(v[2 * j], v[2 * j + 1], h, md, l);
      hi[j] = h;
      mid[j] = md;
      lo[j] = l;
    }
    *reinterpret_cast<v2u*>(x_wr + 128 * i) = hi;
    *reinterpret_cast<v2u*>(x_wr + 128 * i + kXblk) = mid;
    *reinterpret_cast<v2u*>(x_wr + 128 * i + 2 * kXblk) = lo;
    if constexpr (WT == kQ4_K) xsum[i] = red8f((v.x + v.y) + (v.z + v.w));
  };
  // Q4_K: the block's X_j as three bf16 (lane l the row 8 (l % 4) + l / 8) into slot c % 4 of
  // the super-block's operand: lane r hi (bytes 0..7) and mid (8..15), lane 32 + r lo and 0
  uint8_t* const xmop = smem + T::kOffXm + wave * T::kXm;
  auto put_xsum = [&](int c) {
    if constexpr (WT == kQ4_K) {
      const float a = (lane & 1) ? xsum[1] : xsum[0], b = (lane & 1) ? xsum[3] : xsum[2];
      u32 hi, mid, lo;
      split3((lane & 2) ? b : a, 0.0f, hi, mid, lo);
      uint8_t* d = xmop + ((c >> 2) & 1) * 1024 + (8 * (lane & 3) + (lane >> 3)) * 16 + 2 * (c & 3);
      *reinterpret_cast<uint16_t*>(d) = (uint16_t)hi;
      *reinterpret_cast<uint16_t*>(d + 8) = (uint16_t)mid;
      *reinterpret_cast<uint16_t*>(d + 512) = (uint16_t)lo;
    }
  };
  if constexpr (WT == kQ4_K) {  // the zero halves
    *reinterpret_cast<v4u*>(xmop + lane * 16) = v4u{};
    *reinterpret_cast<v4u*>(xmop + 1024 + lane * 16) = v4u{};
  }
  // the A operands of a block: [K-step][part: hi, mid, lo]
  v4u A[2][3];
  auto read_a = [&](int p) {
#pragma unroll
    for (int s = 0; s < 2; ++s) A[s][p] = lds16(xop + s * kXs + p * kXblk + lg * 640 + li * 16);
  };

  v16f_t acc[NTW];
#pragma unroll
  for (int j = 0; j < NTW; ++j) acc[j] = v16f_t{};
  const v16f_t zero{};
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;

  v4u mhd[T::kPasses];  // Q4_K: the chunk's headers, past the reload of raw
  auto keep_hd = [&](int set) {
    if constexpr (WT == kQ4_K) {
#pragma unroll
      for (int p = 0; p < T::kPasses; ++p) mhd[p] = raw[set][p].hd;
    }
  };
  auto put_mins = [&](int sb) {
    if constexpr (WT == kQ4_K) {
      if (!conv) return;
#pragma unroll
      for (int p = 0; p < T::kPasses; ++p)
        Raw<WT>::put_mins(mhd[p], esel[p], smem + T::kOffMins + (sb & 1) * T::kMins, T::kRows, erow[p]);
    }
  };

  // chunk 0 into buffer 0; the next kDepth chunks' loads in flight (chunk c in set c % kDepth)
  const int nch = (nslices + 1) / 2;
  auto clamp = [&](int c) { return c < nch ? c : nch - 1; };
#pragma unroll
  for (int d = 0; d < T::kDepth; ++d) {
    load_w(clamp(d), d);
#pragma unroll
    for (int i = 0; i < 4; ++i) load_x(clamp(d), d, i);
  }
  put_w(0, 0, 0, P0{});
  put_w(0, 0, 0, P1{});
  keep_hd(0);
  put_mins(0);
#pragma unroll
  for (int i = 0; i < 4; ++i) split_x(0, i);
  put_xsum(0);
  load_w(clamp(T::kDepth), 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) load_x(clamp(T::kDepth), 0, i);
  __syncthreads();
  const int b_off = (g * 2 * T::kOpT + cg * NTW) * 1024 + lane * 16;
  const int d_off = T::kOps + ((WT == kQ6_K ? 2 : 1) * g * T::kRows + cg * NTW * 32 + li) * 4;
  // the B operands and scales of the next tile
  v4u b0, b1;
  float f0 = 0, f1 = 0;
  auto read_b = [&](const uint8_t* buf, int n) {
    b0 = lds16(buf + b_off + n * 1024);
    b1 = lds16(buf + b_off + (T::kOpT + n) * 1024);
    f0 = *reinterpret_cast<const float*>(buf + d_off + n * 128);
    if (WT == kQ6_K) f1 = *reinterpret_cast<const float*>(buf + d_off + (T::kRows + n * 32) * 4);
  };
  read_b(smem, 0);
#pragma unroll
  for (int p = 0; p < 3; ++p) read_a(p);
  // One tile's step: its 6 MFMAs, the fold of the previous tile's sums and a share of the
  // next chunk's conversion; the next step's operands are read at its start. A wave issues in
  // order, and an MFMA that waits for the one before it blocks the wave's VALU, so the
  // fences place an even share of the step's VALU after each MFMA (without them the compiler
  // put each tile's MFMAs in one run and all folds at the loop's end: 238 us against 172).
  constexpr int kLastTile = NTW - 1;
  constexpr int kFolds = WT == kQ6_K ? 32 : 16;
  v16f_t sp0{}, sp1{};  // the previous tile's sums and scales
  float fp0 = 0, fp1 = 0;
  auto fold = [&](int n) {
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[n][r] = fmaf(fp0, sp0[r], acc[n][r]);
    if constexpr (WT == kQ6_K) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[n][r] = fmaf(fp1, sp1[r], acc[n][r]);
    }
  };
  auto chunk = [&](int c, int set) {
    const uint8_t* buf = smem + (c & 1) * T::kBuf;
    const uint8_t* nbuf = smem + ((c + 1) & 1) * T::kBuf;
    // chunk c + 1 (past the end: the last chunk's bytes again, still into the buffer, mins and
    // offsets of c + 1, which no one reads then) is converted between the MFMAs of chunk c; its
    // registers are reloaded for chunk c + 1 + kDepth as soon as they are read
    const int cn = clamp(c + 1), cl = clamp(c + 1 + T::kDepth);
#pragma unroll
    for (int n = 0; n < NTW; ++n) {
      const v4u c0 = b0, c1 = b1;
      const float g0 = f0, g1 = f1;
      constexpr int kLast = kLastTile;
      if (n < kLast) {
        read_b(buf, n + 1);
      } else if (NTW > 1) {
        read_b(nbuf, 0);
      }
      v16f_t s0 = mfma_bf(A[0][2], c0, zero), s1 = zero;
      if constexpr (WT == kQ6_K) {
        s1 = mfma_bf(A[1][2], c1, zero);
        s0 = mfma_bf(A[0][1], c0, s0);
        s1 = mfma_bf(A[1][1], c1, s1);
        s0 = mfma_bf(A[0][0], c0, s0);
        s1 = mfma_bf(A[1][0], c1, s1);
      } else {
        s0 = mfma_bf(A[1][2], c1, s0);
        s0 = mfma_bf(A[0][1], c0, s0);
        s0 = mfma_bf(A[1][1], c1, s0);
        s0 = mfma_bf(A[0][0], c0, s0);
        s0 = mfma_bf(A[1][0], c1, s0);
      }
      fold(n > 0 ? n - 1 : kLast);
      asm volatile("" : "+v"(acc[n > 0 ? n - 1 : kLast]));
      // the next chunk's share of this step: pieces 0, 1 the weights, 2..5 the activations
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        if (q * (kLast > 0 ? kLast : 1) / 6 != n) continue;
        if (q == 0) put_w(cn, c + 1, set, P0{});
        if (q == 1) {
          put_w(cn, c + 1, set, P1{});
          keep_hd(set);
          load_w(cl, set);
        }
        if (q >= 2) {
          split_x(set, q - 2);
          load_x(cl, set, q - 2);
        }
        if (q == 5) put_xsum(c + 1);
      }
      if (n == kLast && NTW > 1) {
#pragma unroll
        for (int p = 2; p >= 0; --p) read_a(p);
      }
      if (NTW >= 4) {
        constexpr int kShare = NTW > 1 ? 32 * 6 / (NTW > 1 ? NTW - 1 : 1) : 0;
        if (n < kLast) {
#pragma unroll
          for (int i = 0; i < 6; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, (kFolds + kShare + 5) / 6, 0);
          }
        } else {
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, (kFolds + 5) / 6, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, (kFolds + 5) / 6, 0);
          }
        }
      }
      sp0 = s0;
      sp1 = s1;
      fp0 = g0;
      fp1 = g1;
      __builtin_amdgcn_sched_barrier(0);
      // every read of buf has been issued and all of nbuf written
      if (n == (NTW > 1 ? NTW - 2 : 0)) lds_barrier();
    }
    if (NTW == 1) {
      read_b(nbuf, 0);
#pragma unroll
      for (int p = 2; p >= 0; --p) read_a(p);
    }
    if constexpr (WT == kQ4_K) {
      if ((c & 3) == 3) {  // the super-block's offsets; the next one's mins
        const uint8_t* mins = smem + T::kOffMins + ((c >> 2) & 1) * T::kMins;
        const float* dm = reinterpret_cast<const float*>(mins + 16 * T::kRows) + cg * NTW * 32 + li;
        const uint8_t* mb = mins + (g * T::kRows + cg * NTW * 32 + li) * 8;
        put_mins((c + 1) >> 2);
        const v4u xm = lds16(xmop + ((c >> 2) & 1) * 1024 + lane * 16);
        fold(kLastTile);  // before its offsets, as the other tiles' sums
        fp0 = 0;
#pragma unroll
        for (int n = 0; n < NTW; ++n) {
          const v2u mm = *reinterpret_cast<const v2u*>(mb + n * 256);
          const float nd = -dm[n * 32];
          const v16f_t mn = mfma_bf(xm, v4u{mm.x, mm.y, mm.x, mm.y}, zero);
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[n][r] = fmaf(nd, mn[r], acc[n][r]);
        }
      }
    }
  };
#pragma unroll 1
  for (int c = 0; c < nch; c += T::kDepth) {
    chunk(c, 1 % T::kDepth);
    if (T::kDepth == 2 && c + 1 < nch) chunk(c + 1, 0);
  }
  fold(kLastTile);

  // ---- the two groups' sums: group 0 finishes tiles [0, kHalf), group 1 the rest; each
  // hands the other its sums of those tiles
  __syncthreads();
  {
    v4u* mine = reinterpret_cast<v4u*>(smem) + (size_t)wave * T::kHalf * 256 + lane;
    const v4u* theirs = reinterpret_cast<const v4u*>(smem) + (size_t)(wave ^ 4) * T::kHalf * 256 + lane;
#pragma unroll
    for (int n = 0; n < NTW; ++n) {
      if ((n >= T::kHalf) == (g == 0)) {
        const int i = n >= T::kHalf ? n - T::kHalf : n;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          mine[i * 256 + 64 * q] = v4u{as_u(acc[n][4 * q]), as_u(acc[n][4 * q + 1]), as_u(acc[n][4 * q + 2]), as_u(acc[n][4 * q + 3])};
      }
    }
    __syncthreads();
    bool bad = false;
#pragma unroll
    for (int n = 0; n < NTW; ++n) {
      if ((n >= T::kHalf) != (g == 0)) {
        const int i = n >= T::kHalf ? n - T::kHalf : n;
        const int64_t nn = nbase + 32 * (cg * NTW + n) + li;
        const bool in = nn >= n0 && nn < n1;
        const float bv = bias && in ? bias[nn] : 0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const v4u o = theirs[i * 256 + 64 * q];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * q + e, row = 32 * rg + 8 * q + 4 * lg + e;
            const float v = (acc[n][r] + as_f(o[e])) * (1.0f / kXScale);
            if (in && row < mrows) {
              bad |= !(fabsf(v) <= 3.40282347e38f);
              y[(mbase + row) * ys + nn] = bias ? v + bv : v;
            }
          }
        }
      }
    }
    // outputs that are infinite or NaN: their tile on v_mfma_f32_32x32x2 over the expanded weights
    // (lane l supplies row / column l % 32 and K value l / 32 of each pair, here 4 lg + e of eight)
    if (__builtin_expect(__ballot(bad) != 0, 0)) {
      const int64_t xrow = 32 * rg + li < mrows ? 32 * rg + li : mrows - 1;
#pragma unroll 1
      for (int n = g == 0 ? 0 : T::kHalf; n < (g == 0 ? T::kHalf : NTW); ++n) {
        const int64_t nn = nbase + 32 * (cg * NTW + n) + li;
        const bool in = nn >= n0 && nn < n1;
        float* out = y + (mbase + 32 * rg + 4 * lg) * ys + nn;
        u32 redo = 0;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int dr = 8 * (r >> 2) + (r & 3);
          if (in && 32 * rg + 4 * lg + dr < mrows && !(fabsf(out[dr * ys]) <= 3.40282347e38f)) redo |= 1u << r;
        }
        if (__ballot(redo != 0) == 0) continue;
        const u32 gb = (u32)((nn >> 6) * nblk), rr = (u32)(nn & 63);
        v16f_t v{};
#pragma unroll 2
        for (int kk = 0; kk < k; kk += 8) {
          const v4u xq = ld16(rx, (u32)((xrow * xs + kk + 4 * lg) * 4));
          const v4f_t wq = expand4<WT>(rs, gb, rr, (u32)(kk + 4 * lg));
#pragma unroll
          for (int e = 0; e < 4; ++e) v = __builtin_amdgcn_mfma_f32_32x32x2f32(as_f(xq[e]), wq[e], v, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          if ((redo >> r) & 1u) out[(8 * (r >> 2) + (r & 3)) * ys] = bias ? v[r] + bias[nn] : v[r];
        }
      }
    }
  }
}

namespace {

template <int WT, int RG, int NTW>
hipError_t launch_f32(const WeightDev& w, const float* x, int64_t xs, int64_t m, int64_t n0, int64_t n1, float* y,
                      int64_t ys, const float* bias, hipStream_t s) {
  using T = F32Tile<WT, RG, NTW>;
  const int64_t nbase0 = n0 / kRowGroup * kRowGroup;
  const int64_t tiles_n = (n1 - nbase0 + T::kBN - 1) / T::kBN;
  const int64_t tiles_m = (m + T::kBM - 1) / T::kBM;
  const int nslices = (int)(w.k / kKc);
  const void* fn = reinterpret_cast<const void*>(&k_gemm_f32<WT, RG, NTW>);
  const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, T::kLds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_gemm_f32<WT, RG, NTW>), dim3((unsigned)(tiles_n * tiles_m)), dim3(kThreadsF), T::kLds, s,
                     w.plane[0], w.plane[1], w.plane[2], w.plane[3], (int)w.nblk, (int)w.k, nslices, nbase0, w.n_pad, n0,
                     n1, x, xs, m, y, ys, bias, (int)tiles_m, tiles_n % 8 == 0 ? 1 : 0);
  return hipGetLastError();
}

template <int WT>
hipError_t launch_f32_type(const WeightDev& w, const float* x, int64_t xs, int64_t m, int64_t n0, int64_t n1, float* y,
                           int64_t ys, const float* bias, hipStream_t s) {
  // The tile whose rounds of workgroups (one per CU) times its measured time per round is
  // least. One round at K = 4096 (us; Q4_K / Q6_K): 128 x 224 142 / 200, 128 x 128 106 / 107,
  // 128 x 64 74 / 84, 64 x 64 65 / 80 (the Q6_K 128 x 224 kernel spills 12 registers). So at
  // M = 512, N = 14336 the widest (256 workgroups, 182 us; 128 x 128 takes two rounds, 245), at
  // N = 4096 128 x 64 (93 against 115 and 144), at M = 64, N = 14336 64 x 64 (72 against 83 and
  // 109). 32-row tiles were never the fastest (M = 32, N = 4096: 69 against 65).
  const int64_t cus = w.cus > 0 ? w.cus : 256;
  const int64_t nbase0 = n0 / kRowGroup * kRowGroup;
  auto cost = [&](int bm, int bn, int t) {
    const int64_t tiles = (n1 - nbase0 + bn - 1) / bn * ((m + bm - 1) / bm);
    return (tiles + cus - 1) / cus * t;
  };
  constexpr bool q6 = WT == kQ6_K;
  const int64_t c7 = cost(128, 224, q6 ? 200 : 142), c4 = cost(128, 128, q6 ? 107 : 106);
  const int64_t c2 = cost(128, 64, q6 ? 84 : 74), c1 = cost(64, 64, q6 ? 80 : 65);
  if (c7 < c4 && c7 < c2 && c7 < c1) return launch_f32<WT, 4, 7>(w, x, xs, m, n0, n1, y, ys, bias, s);
  if (c4 < c2 && c4 < c1) return launch_f32<WT, 4, 4>(w, x, xs, m, n0, n1, y, ys, bias, s);
  if (c2 < c1) return launch_f32<WT, 4, 2>(w, x, xs, m, n0, n1, y, ys, bias, s);
  return launch_f32<WT, 2, 1>(w, x, xs, m, n0, n1, y, ys, bias, s);
}

}  // namespace

hipError_t launch_gemm_f32(const WeightDev& w, const float* x, int64_t xs, int64_t m, int64_t n0, int64_t n1, float* y,
                           int64_t ys, const float* bias, hipStream_t s) {
  if (m == 0 || n1 <= n0) return hipSuccess;
  // 32-bit buffer offsets: each plane of the whole weight (below kNoLoad) and one tile's
  // activation rows
  for (int p = 0; p < num_planes(w.dtype); ++p) {
    if (w.n_pad * w.nblk * plane_unit(w.dtype, p) >= (int64_t)kNoLoad) return hipErrorInvalidValue;
  }
  if ((127 * xs + w.k) * 4 >= (int64_t)kNoLoad || w.k % kKc != 0 ||
      (m + 31) / 32 * ((n1 - n0) / 128 + 2) >= (1ll << 31)) {
    return hipErrorInvalidValue;
  }
  switch (w.dtype) {
    case kQ4_K: return launch_f32_type<kQ4_K>(w, x, xs, m, n0, n1, y, ys, bias, s);
    case kQ6_K: return launch_f32_type<kQ6_K>(w, x, xs, m, n0, n1, y, ys, bias, s);
    case kQ8_0: return launch_f32_type<kQ8_0>(w, x, xs, m, n0, n1, y, ys, bias, s);
    case kQ4_0: return launch_f32_type<kQ4_0>(w, x, xs, m, n0, n1, y, ys, bias, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace dq
