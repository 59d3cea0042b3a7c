// Mixer projections on the int8 matrix cores, for calls of several tokens.
//
//   y[t][row] = sum_g s[row][g] * sum_{i in g} code(row, i) * x[t][i]
//
// over int4 rows in groups of 128 or int8 rows with one scale, fp32
// activations.  Each 128-column group of a token's activations is held as
// 30-bit fixed-point numbers q = rint(x * 2^k), 2^k the power of two that
// brings the largest magnitude among them into [2^29, 2^30).  q is cut into
// four balanced base-256 digits, each an MFMA B operand; the four int32 dots
// with the (small, exact) weight codes are exact, and are put together in fp32
// as (c1 * 256 + c2) * 2^16 + (c3 * 256 + c4), times 2^-k (exact): three
// roundings for the group (both conversions and the FMA), then one FMA with
// the row's group scale.
//
// A value is exact down to 2^-6 of the largest and off by at most 2^-31 of the
// largest below.  That is less than the roundings of an fp32 sum as long as
// the group's larger values are several, since then every row's sum has terms of
// their size: with eight values that are at least 2^-6 of the largest, the
// others' errors (112 of them, codes of RMS 4.6) come to 6.5e-8 of the sum of
// a row whose code is 0 for the largest, where an fp32 chain of the group is
// 1.1e-7 off.  So a leading range (within 2^-5 of the largest's binade) of
// fewer than kDigBulk values that would cost the rest any bit leaves the
// digits, the next range is tried, and what left (outliers, an infinity, a
// NaN, all of a group below 2^-91) is added column by column by fp32 FMAs.
// With it the error of a row follows the sum of its own terms' magnitudes,
// whatever else the group holds: one value of 1e6 among N(0, 1), rows with the
// code 0 there, 2.8e-4 of the sum without, 1e-7 so.  Groups of N(0, 1) values
// and the layers' own activations hardly ever have such a column.
//
// k_mix_digits forms the digits once per call in the MFMA's own lane order;
// k_mix_mfma and k_mix_gemm run the weights against them.
#pragma once

#include "sw_device.h"
#include "sw_lds_dma.h"

namespace sw {

constexpr int kDigPlanes = 8;  // four digits x two 64-column halves of a group
constexpr int kDigTile = 16;   // tokens of one MFMA B operand

constexpr int kDigBulk = 8;    // values a range needs to stay in the digits

// What k_mix_digits leaves behind of `tokens` rows of `cols`: the digits, the
// group scales [tile][group][16 tokens] (sign set: the token has columns
// outside the digits), the bits of those columns [tile][group][16 tokens][128]
// (only of such tokens) and their values [token][cols] (only those).
struct MixDigits {
  unsigned char *dig;
  float *asc;
  unsigned char *mask;
  float *out;
};
inline size_t mix_digit_bytes(int tokens, int cols) {
  const size_t units = (size_t)((tokens + kDigTile - 1) / kDigTile) * (cols / 128);
  return units * (kDigPlanes * 1024 + kDigTile * (4 + 16 + 128 * 4));
}
inline MixDigits mix_digits_at(unsigned char *p, int tokens, int cols) {
  const size_t units = (size_t)((tokens + kDigTile - 1) / kDigTile) * (cols / 128);
  MixDigits d;
  d.dig = p;
  d.asc = (float *)(d.dig + units * (kDigPlanes * 1024));
  d.mask = (unsigned char *)(d.asc + units * kDigTile);
  d.out = (float *)(d.mask + units * kDigTile * 16);
  return d;
}

// over the 16 lanes of a DPP row, in every lane
__device__ __forceinline__ unsigned row_max_u32(unsigned v) {
#define SW_ROW_MAX(ctrl)                                            \
  {                                                                 \
    const unsigned o_ = (unsigned)SW_DPP_I(0, (int)v, ctrl, 0xF, true); \
    v = o_ > v ? o_ : v;                                            \
  }
  SW_ROW_MAX(0xB1) SW_ROW_MAX(0x4E) SW_ROW_MAX(0x141) SW_ROW_MAX(0x140)
#undef SW_ROW_MAX
  return v;
}
__device__ __forceinline__ int row_sum_i32(int v) {
  v += SW_DPP_I(0, v, 0xB1, 0xF, true);
  v += SW_DPP_I(0, v, 0x4E, 0xF, true);
  v += SW_DPP_I(0, v, 0x141, 0xF, true);
  v += SW_DPP_I(0, v, 0x140, 0xF, true);
  return v;
}

struct DigitArgs {
  const float *x;  // token t at x + t * ldx
  int ldx, cols, T;
  MixDigits d;
  // optional per-(token, head) factor 1/sqrt(sum(msp) / hw + eps)
  const float *msp;
  int nsp, hw;
  float eps;
};

// Sixteen lanes take one (token, group), eight columns each; a wave takes
// four tokens of one group.  Digit planes, per (16-token tile, group):
// [digit d][half h][lane kb * 16 + token][16 bytes].  ROWS8 0 (int4 rows):
// byte j of half h is column 32 kb + 2 j + h, the low (0) or high (1) nibble
// of byte j of the 16 that a lane loads; 1 (int8 rows): column
// 32 kb + 16 h + j.  Columns outside the digits have the digits 0.
// Latency-bound: 4.5 us up to 16 tokens.
// grid (cols / 128, 4 * tiles), 64 threads.
template <int ROWS8>
__global__ __launch_bounds__(64) void k_mix_digits(DigitArgs a) {
  const int lane = threadIdx.x, i = lane & 15, kb = i >> 2;
  const int g = blockIdx.x, tile = blockIdx.y >> 2, n = (blockIdx.y & 3) * 4 + (lane >> 4);
  const int G = a.cols >> 7, t = tile * kDigTile + n, tc = t < a.T ? t : a.T - 1;
  const int col = g * 128 + 8 * i;
  const float4 v0 = *(const float4 *)(a.x + (size_t)tc * a.ldx + col);
  const float4 v1 = *(const float4 *)(a.x + (size_t)tc * a.ldx + col + 4);
  float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
  if (a.msp) {
    const float *m = a.msp + ((size_t)tc * (a.cols / a.hw) + col / a.hw) * a.nsp;
    float ms = 0.0f;
    for (int k = 0; k < a.nsp; k++) ms += m[k];
    const float r = 1.f / sqrtf(ms / (float)a.hw + a.eps);
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] *= r;
  }
  // A column that leaves: its value is stored and is 0 in the digits.  Each
  // turn takes one out of one token's digits at least, or is the last; the
  // first is the last for nearly every group.
  unsigned left = 0, mb;  // mb: the largest magnitude in the digits, as an integer
  int k;
  float scale;
#pragma unroll 1
  for (;;) {
    mb = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const unsigned b = __float_as_uint(v[e]) & 0x7fffffffu;
      mb = b > mb ? b : mb;
    }
    mb = row_max_u32(mb);
    // below 2^-91 the scale would leave the normal range: all of it goes out;
    // infinities and NaNs (which order above them) go first
    const int E = (int)(mb >> 23);
    const bool bad = E == 255, tiny = E < 36;
    k = tiny ? 120 : 29 + 127 - E;
    scale = __uint_as_float((unsigned)(k + 127) << 23);
    const unsigned lo = bad ? 0x7f800000u : tiny ? 1 : (unsigned)(E - 5) << 23;
    int cnt = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) cnt += (__float_as_uint(v[e]) & 0x7fffffffu) >= lo;
    bool drop = mb != 0 && (row_sum_i32(cnt) < kDigBulk || bad || tiny);
    if (__builtin_expect(__ballot(drop) == 0, 1)) break;
    bool lossy = bad || tiny;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float r = v[e] * scale;
      lossy |= r != __builtin_rintf(r);
    }
    drop = drop && (__ballot(lossy) >> (lane & 48) & 0xffff) != 0;
    if (__ballot(drop) == 0) break;
#pragma unroll
    for (int e = 0; e < 8; e++)
      if (drop && (__float_as_uint(v[e]) & 0x7fffffffu) >= lo) {
        if (t < a.T) a.d.out[(size_t)t * a.cols + col + e] = v[e];
        v[e] = 0.0f;
        left |= 1u << e;
      }
  }
  if (t >= a.T) left = 0;  // an absent token of the tile
  unsigned d[4][2] = {};
#pragma unroll
  for (int e = 0; e < 8; e++) {
    int q = (int)__builtin_rintf(v[e] * scale);
    const int w = ROWS8 ? e >> 2 : e & 1, sh = 8 * (ROWS8 ? e & 3 : e >> 1);
#pragma unroll
    for (int p = 3; p > 0; p--) {
      const int lo = (int)(signed char)(q & 255);
      d[p][w] |= (unsigned)(lo & 255) << sh;
      q = (q - lo) >> 8;
    }
    d[0][w] |= (unsigned)(q & 255) << sh;
  }
  unsigned *const out = (unsigned *)a.d.dig + ((size_t)tile * G + g) * (kDigPlanes * 256) + (kb * 16 + n) * 4;
#pragma unroll
  for (int p = 0; p < 4; p++)
#pragma unroll
    for (int w = 0; w < 2; w++) {
      const int half = ROWS8 ? (i & 3) >> 1 : w, dw = ROWS8 ? 2 * (i & 1) + w : i & 3;
      out[(2 * p + half) * 256 + dw] = d[p][w];
    }
  const size_t at = ((size_t)tile * G + g) * kDigTile + n;
  const unsigned some = (unsigned)(__ballot(left != 0) >> (lane & 48)) & 0xffffu;
  if (__builtin_expect(some != 0, 0)) a.d.mask[at * 16 + i] = (unsigned char)left;
  // int4 codes enter the MFMA as 16 * (nibble - 8)
  if (i == 0) {
    const float sc = mb == 0 ? 0.0f : __builtin_ldexpf(ROWS8 ? 1.0f : 0.0625f, -k);
    a.d.asc[at] = some ? -sc : sc;
  }
}

// The columns of one token and group that are outside the digits: their
// products with the codes of this lane's four rows, code(e, column).
template <class Code>
__device__ __forceinline__ void add_left_out(const float *asc, const unsigned char *mask, const float *out, const v4f &s4,
                                             v4f &acc, Code code) {
  if (!(__float_as_uint(*asc) >> 31)) return;
  const uint4 m = *(const uint4 *)mask;
  const unsigned w[4] = {m.x, m.y, m.z, m.w};
#pragma unroll 1
  for (int i = 0; i < 4; i++)
    for (unsigned u = i == 0 ? w[0] : i == 1 ? w[1] : i == 2 ? w[2] : w[3]; u; u &= u - 1) {
      const int c = 32 * i + __builtin_ctz(u);
      const float x = out[c];
#pragma unroll
      for (int e = 0; e < 4; e++) acc[e] = __builtin_fmaf(code(e, c) * x, s4[e], acc[e]);
    }
}
// code of column c (of a group) in its byte
template <int FMT>
__device__ __forceinline__ float code_of(unsigned char b, int c) {
  return FMT == 4 ? (float)((int)((b >> (4 * (c & 1))) & 15) - 8) : (float)(signed char)b;
}

// What one token of a Gated DeltaNet call reads and writes in the causal
// convolution's ring (K <= 4): where each tap's raw value comes from, and
// whether the token's own raw value is the last one written to its ring word.
struct ConvTok {
  signed char src[4];  // -2: before the sequence, -1: the ring in memory, else a token of this call
  signed char word[4];  // ring word of each tap
  int slot;
  short own;   // ring word the token writes
  short last;  // 1: no later token of the call writes that word
};

struct MfmaProj {
  const unsigned char *q;
  const float *s;
  float *y;  // y[t * ldy + row]
  int rows, rb, ng, ldy;
  int tile0;  // first 16-row tile of the matrix
};

struct MfmaArgs {
  MfmaProj m[3];
  int nm;
  int tiles;  // 16-row tiles of all matrices
  int G, T;   // 128-column groups; tokens
  MixDigits d;
  // causal convolution on matrix 0
  float *conv_state;    // [slot][K][channels]
  const float *conv_w;  // [channels][K]
  float *mix;           // [T][channels]
  int K;
  long long conv_slot_stride;
  ConvTok tok[kDigTile];
};

// A persistent workgroup of W waves walks 16-row tiles, b, b + grid, ...;
// wave w owns GW consecutive 128-column groups of every tile (whole 128-byte
// lines of a row).  The wave copies its share of the next NR - 1 tiles
// (weights, group scales, and for the convolution the ring words and tap
// weights that its own lanes will need) into its slots of an LDS ring
// (global_load_lds), so the bytes in flight hold no registers and the loop
// body exists once: launches of a few tiles a workgroup would otherwise spend
// their time fetching unrolled code.  With 8 waves the tokens' digits stay in
// registers for the whole launch and come from L2 once per workgroup (8 KB a
// group against 1 KB of int4 weights a tile); with 16 waves, for launches of
// one tile a workgroup, they are read for each tile, two groups at a time.
// Per group: two unpacked A operands (the nibbles, offset by XOR and kept in
// the high half of their byte), eight MFMAs, one fp32 step.  The waves' sums
// meet in LDS in wave order, one barrier a tile that leaves the copies in
// flight; waves 0..3 finish an even tile, 4..7 an odd one, a thread per
// (row, token).
// HBM-bound on the weights up to 16 tokens.  Measured at 16 tokens, S397: qkv
// and z (44.6 MB) 216 -> 17.7 us, out (17.8 MB) 117 -> 12.6 us against the fp32
// FMA kernel; at one group of registers in flight instead of the ring 25 to
// 30 and 14 us, with the loop unrolled over register buffers 21 and 17 us.
// grid (min(tiles, compute units), token tiles), 64 W threads.
constexpr int kMfmaMaxGroups = 64;  // 128-column groups of a row (W 16, GW 4)
constexpr int kMfmaPitch = 20;      // floats per token in LDS (16 rows, padded)
constexpr int kConvCopies = 4;      // dword copies of a tile's convolution: tap weights, three ring words

template <int FMT, int W, int GW, bool CONV>
struct MfmaRing {
  static constexpr int NA = FMT == 4 ? 1 : 2;
  static constexpr int scales = FMT == 4 ? (GW * 16 + 63) / 64 : 1;  // dword copies of a wave's scales
  static constexpr int wave = GW * NA * 1024 + scales * 256 + (CONV ? kConvCopies * 256 : 0);
  static constexpr int slot = wave * W;
  static constexpr int parities = slot > 100 * 1024 ? 1 : 2;  // buffers of the waves' sums
  static constexpr int red = parities * W * kDigTile * kMfmaPitch * 4;
  static constexpr int fit = (158 * 1024 - red - 256) / slot;
  static constexpr int slots = fit < 4 ? fit : 4;
  static constexpr int lds = slots * slot + red + 256;
};

template <int FMT, int W, int GW, bool CONV>
__global__ __launch_bounds__(64 * W) void k_mix_mfma(MfmaArgs a) {
  typedef MfmaRing<FMT, W, GW, CONV> Ring;
  constexpr int NA = Ring::NA, NR = Ring::slots, NS = Ring::scales;
  constexpr int kMfmaRed = Ring::red;
  constexpr int ND = W == 8 || GW < 2 ? GW : 2;  // digit buffers
  constexpr bool RES = ND == GW;                 // digits resident
  constexpr int OPS = GW * NA + NS;              // copies of a tile, at least
  static_assert(NR >= 1, "a tile fits the LDS");
  extern __shared__ __align__(16) unsigned char smem[];
  float *const red = (float *)smem;  // [parity][wave][token][pitch]
  uint64_t *const etab = (uint64_t *)(smem + kMfmaRed);
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kb = lane >> 4;
  // in a scalar register, and what follows from it (W 16, GW 4 spills without:
  // the 16-token S397 out projection 14.5 against 11.7 us)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char *const ring = smem + kMfmaRed + 256 + wave * (NR * Ring::wave);
  const int t0 = blockIdx.y * kDigTile, nt = a.T - t0 < kDigTile ? a.T - t0 : kDigTile;
  const int g0 = wave * GW, tiles = a.tiles, step = gridDim.x;
  if (CONV && tid < 32) etab[tid] = kExp2Tab[tid];
  // the token and row that this thread finishes; waves 0..3 even tiles of the
  // workgroup, 4..7 odd ones
  const int ft = (tid & 255) >> 4, fr = tid & 15, fpar = wave >> 2;  // waves 8.. finish none
  ConvTok ct;
  if (CONV) ct = a.tok[ft < nt ? ft : 0];

  auto mat_of = [&](int t) {
    int m = 0;
    if (a.nm > 1 && t >= a.m[1].tile0) m = 1;
    if (a.nm > 2 && t >= a.m[2].tile0) m = 2;
    return m;
  };
  // lanes of groups past the row read its last group: inside the row, unused
  auto copy = [&](int t, int i) {
    const int m = mat_of(t);
    const MfmaProj &pm = a.m[m];
    const int row0 = (t - pm.tile0) * 16, row = row0 + n < pm.rows ? row0 + n : pm.rows - 1;
    unsigned char *const slot = ring + (i % NR) * Ring::wave;
    const unsigned char *q = pm.q + (size_t)row * pm.rb + (FMT == 4 ? 16 : 32) * kb;
#pragma unroll
    for (int j = 0; j < GW; j++) {
      const int g = g0 + j < a.G ? g0 + j : a.G - 1;
#pragma unroll
      for (int h = 0; h < NA; h++)
        dma_b128(q + (size_t)g * (FMT == 4 ? 64 : 128) + 16 * h, lds_addr(slot + (j * NA + h) * 1024));
    }
#pragma unroll
    for (int j = 0; j < NS; j++) {
      const int gs = g0 + 4 * j + kb, g = gs < a.G && 4 * j + kb < GW ? gs : a.G - 1;
      dma_b32(FMT == 4 ? pm.s + (size_t)row * pm.ng + g : pm.s + row, lds_addr(slot + GW * NA * 1024 + j * 256));
    }
    if (CONV && m == 0 && (i & 1) == fpar) {
      const int ch = row0 + fr < pm.rows ? row0 + fr : pm.rows - 1, k = lane >> 4;
      unsigned char *const cw = slot + GW * NA * 1024 + NS * 256;
      dma_b32(a.conv_w + (size_t)ch * a.K + (k < a.K ? k : 0), lds_addr(cw));
      const float *cs = a.conv_state + (size_t)ct.slot * a.conv_slot_stride + ch;
#pragma unroll
      for (int j = 0; j < 3; j++) dma_b32(cs + (size_t)ct.word[j] * pm.rows, lds_addr(cw + (j + 1) * 256));
    }
  };

  copy(blockIdx.x, 0);
  // lanes of absent tokens read token 0's digits: no more lines
  const unsigned char *const dp =
      a.d.dig + (size_t)blockIdx.y * a.G * (kDigPlanes * 1024) + (kb * 16 + (n < nt ? n : 0)) * 16;
  const float *const ap = a.d.asc + (size_t)blockIdx.y * a.G * kDigTile + (n < nt ? n : 0);
  v4i dv[ND][kDigPlanes];
  float av[GW];
  auto digits = [&](int b, int g) {
    const int gc = g < a.G ? g : a.G - 1;
#pragma unroll
    for (int d = 0; d < kDigPlanes; d++) dv[b][d] = *(const v4i *)(dp + ((size_t)gc * kDigPlanes + d) * 1024);
  };
#pragma unroll
  for (int i = 0; i < GW; i++) av[i] = g0 + i < a.G ? ap[(size_t)(g0 + i) * kDigTile] : 0.0f;
  if (RES) {
#pragma unroll
    for (int i = 0; i < ND; i++) digits(i, g0 + i);
#pragma unroll
    for (int i = 0; i < ND; i++)
#pragma unroll
      for (int d = 0; d < kDigPlanes; d++) asm volatile("" : "+v"(dv[i][d]));
  }
  unsigned left = 0;  // groups in which a token has columns outside the digits
#pragma unroll
  for (int i = 0; i < GW; i++) {
    if (__ballot(__float_as_uint(av[i]) >> 31) != 0) left |= 1u << i;
    av[i] = fabsf(av[i]);
    asm volatile("" : "+v"(av[i]));
  }
  for (int i = 1; i < NR - 1; i++)
    if ((int)blockIdx.x + i * step < tiles) copy(blockIdx.x + i * step, i);

  for (int t = blockIdx.x, i = 0; t < tiles; t += step, i++) {
    const int m = mat_of(t), p = i & 1;
    const MfmaProj &pm = a.m[m];
    // the slot the next copy fills was read a tile ago
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const bool more = t + (NR - 1) * step < tiles;
    if (NR > 1 ? more : i > 0) copy(t + (NR - 1) * step, i + NR - 1);
    // this tile's copies are done when no more than the younger tiles' are left
    if (NR > 1 && more) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NR - 1) * OPS) : "memory");
    } else {
      wait_dma();
    }
    const unsigned char *const slot = ring + (i % NR) * Ring::wave;
    const float *const sc = (const float *)(slot + GW * NA * 1024);
    v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
    auto group = [&](int j, int b, float as) {
      v4i a0, a1;
      if (FMT == 4) {
        const v4u w = *(const v4u *)(slot + j * 1024 + 16 * lane);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const unsigned x = w[e] ^ 0x88888888u;
          a0[e] = (int)((x << 4) & 0xF0F0F0F0u);
          a1[e] = (int)(x & 0xF0F0F0F0u);
        }
      } else {
        a0 = *(const v4i *)(slot + (2 * j) * 1024 + 16 * lane);
        a1 = *(const v4i *)(slot + (2 * j + 1) * 1024 + 16 * lane);
      }
      v4i c[4];
#pragma unroll
      for (int d = 0; d < 4; d++) c[d] = mfma_i8(a0, dv[b][2 * d], v4i{0, 0, 0, 0});
#pragma unroll
      for (int d = 0; d < 4; d++) c[d] = mfma_i8(a1, dv[b][2 * d + 1], c[d]);
      v4f s4 = v4f{1.f, 1.f, 1.f, 1.f};
      if (FMT == 4) s4 = *(const v4f *)(sc + 16 * j + 4 * kb);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float f = __builtin_fmaf((float)(c[0][e] * 256 + c[1][e]), 65536.0f, (float)(c[2][e] * 256 + c[3][e]));
        acc[e] = FMT == 4 ? __builtin_fmaf(f * as, s4[e], acc[e]) : __builtin_fmaf(f, as, acc[e]);
      }
    };
    // groups past the row add their scale 0
    if (RES) {
#pragma unroll
      for (int j = 0; j < GW; j++) group(j, j % ND, av[j]);
    } else {
      digits(0, g0);
#pragma unroll
      for (int j = 0; j < GW; j += 2) {
        digits(1, g0 + j + 1);
        group(j, 0, av[j]);
        if (j + 2 < GW) digits(0, g0 + j + 2);
        group(j + 1, 1, av[j + 1]);
      }
    }
#pragma unroll 1
    for (unsigned u = left; __builtin_expect(u != 0, 0); u &= u - 1) {
      const int j = __builtin_ctz(u);
      int l = lane;
      asm volatile("" : "+v"(l));  // addresses formed here, not held in registers through the launch
      const int ln = l & 15, row = 4 * (l >> 4), tok = ln < nt ? ln : 0;
      const size_t at = ((size_t)blockIdx.y * a.G + g0 + j) * kDigTile + tok;
      add_left_out(a.d.asc + at, a.d.mask + at * 16,
                   a.d.out + ((size_t)(t0 + tok) * a.G + g0 + j) * 128,
                   FMT == 4 ? *(const v4f *)(sc + 16 * j + row) : v4f{1.f, 1.f, 1.f, 1.f}, acc, [&](int e, int c) {
                     const int at = FMT == 4 ? j * 1024 + ((c & 31) >> 1) : (2 * j + (c >> 4 & 1)) * 1024 + (c & 15);
                     return code_of<FMT>(slot[at + 16 * ((c >> 5) * 16 + row + e)], c);
                   });
    }
    *(v4f *)(red + ((p % Ring::parities * W + wave) * kDigTile + n) * kMfmaPitch + 4 * kb) = acc;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int row = (t - pm.tile0) * 16 + fr;
    if (p == fpar && ft < nt && row < pm.rows) {
      auto raw = [&](int tok) {
        const float *r = red + (p % Ring::parities * W * kDigTile + tok) * kMfmaPitch + fr;
        float v = r[0];
#pragma unroll
        for (int w = 1; w < W; w++) v += r[w * kDigTile * kMfmaPitch];
        return v;
      };
      const float own = raw(ft);
      if (!CONV || m != 0) {
        pm.y[(size_t)(t0 + ft) * pm.ldy + row] = FMT == 8 ? own * sc[fr] : own;
      } else {
        // the taps in order (c/qwen.c:3018-3023)
        const float *cw = (const float *)(slot + GW * NA * 1024 + NS * 256);
        float sconv = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int src = ct.src[k];
          if (k >= a.K || src == -2) continue;
          const float v = src == ft ? own : src >= 0 ? raw(src) : cw[64 * (k < 3 ? k + 1 : 0) + lane];
          sconv = __builtin_fmaf(cw[16 * k + fr], v, sconv);
        }
        a.mix[(size_t)ft * pm.rows + row] = silu_ref_t(sconv, etab);
        // tokens of one sequence share ring words: all of the tile's were
        // copied to LDS before the barrier
        if (ct.last) a.conv_state[(size_t)ct.slot * a.conv_slot_stride + (size_t)ct.own * pm.rows + row] = own;
      }
    }
    if (Ring::parities == 1) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
}

// The same product for prompt chunks: a workgroup of 8 waves computes 128 rows
// x 128 tokens, a wave 64 rows x 32 tokens (two waves along the rows).  Per
// 128-column group the workgroup's digit planes (64 KB) and scales go to one
// of two LDS buffers by global_load_lds while the previous group is worked on;
// a wave's own weight bytes go to registers.  A wave unpacks a row tile once
// for its two token tiles and reads a token tile's digits once for its four
// row tiles.  Workgroups of one token block follow each other by the number
// of token blocks, so that with eight of them an XCD's L2 keeps one block's
// digits.
// Bound by MFMA (64 of 16 cycles a wave and group) and the fp32 steps (28 VALU
// instructions per eight MFMAs) that two waves a SIMD overlap only in part:
// 2.9 us a group where the MFMAs alone take 0.85.  1,000 tokens, S397: q, k and
// v 736 -> 464 us, o 628 -> 180 us against k_mix_mfma, 1.3 int8 POP/s.
// grid row blocks x token blocks, 512 threads.
constexpr int kGemmRows = 128, kGemmTokens = 128;
constexpr int kGemmTiles = kGemmTokens / kDigTile;
constexpr int kGemmScales = kGemmTiles * kDigPlanes * 1024;  // activation, then row scales
constexpr int kGemmBuf = kGemmScales + kGemmTokens * 4 + kGemmRows * 4;
constexpr int kGemmLds = 2 * kGemmBuf;

template <int FMT>
__global__ __launch_bounds__(512) void k_mix_gemm(MfmaArgs a) {
  constexpr int NA = FMT == 4 ? 1 : 2, RT = 4, NTW = 2;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kb = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int ttiles = (a.T + kDigTile - 1) / kDigTile, tb = (ttiles + kGemmTiles - 1) / kGemmTiles;
  const int rb = blockIdx.x / tb, tile0 = (blockIdx.x % tb) * kGemmTiles;
  int mi = 0;
  if (a.nm > 1 && rb >= a.m[1].tile0) mi = 1;
  if (a.nm > 2 && rb >= a.m[2].tile0) mi = 2;
  const MfmaProj &pm = a.m[mi];
  const int row0 = (rb - pm.tile0) * kGemmRows, rlast = pm.rows - 1;
  const unsigned char *qp[RT];
#pragma unroll
  for (int r = 0; r < RT; r++) {
    const int row = row0 + 64 * wm + 16 * r + n;
    qp[r] = pm.q + (size_t)(row < rlast ? row : rlast) * pm.rb + (FMT == 4 ? 16 : 32) * kb;
  }
  v4u w[RT][NA], wn1[RT][NA];
  auto weights = [&](int g) {
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int h = 0; h < NA; h++) wn1[r][h] = *(const v4u *)(qp[r] + (size_t)g * (FMT == 4 ? 64 : 128) + 16 * h);
  };
  // one group's digits and scales; token tiles past the last repeat it
  auto copy = [&](int g, int b) {
    unsigned char *const buf = smem + b * kGemmBuf;
#pragma unroll
    for (int j = 0; j < kGemmTiles; j++) {  // wave w copies plane w of every tile
      const int tt = tile0 + j < ttiles ? tile0 + j : ttiles - 1;
      dma_b128(a.d.dig + (((size_t)tt * a.G + g) * kDigPlanes + wave) * 1024 + 16 * lane,
               lds_addr(buf + (j * kDigPlanes + wave) * 1024));
    }
    if (wave < NTW) {
      const int j = 4 * wave + kb, tt = tile0 + j < ttiles ? tile0 + j : ttiles - 1;
      dma_b32(a.d.asc + ((size_t)tt * a.G + g) * kDigTile + n, lds_addr(buf + kGemmScales + wave * 256));
    }
    if (FMT == 4 && wave >= 6) {
      const int row = row0 + 64 * (wave - 6) + lane;
      dma_b32(pm.s + (size_t)(row < rlast ? row : rlast) * pm.ng + g,
              lds_addr(buf + kGemmScales + kGemmTokens * 4 + (wave - 6) * 256));
    }
  };
  v4f acc[RT][NTW];
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int j = 0; j < NTW; j++) acc[r][j] = v4f{0.f, 0.f, 0.f, 0.f};
  unsigned long long left[NTW] = {};  // groups in which a token has columns outside the digits (G <= kMfmaMaxGroups)
  copy(0, 0);
  weights(0);
  for (int g = 0; g < a.G; g++) {
    const unsigned char *const buf = smem + (g & 1) * kGemmBuf;
    // this group's copies have landed and every wave has left the other buffer
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int h = 0; h < NA; h++) w[r][h] = wn1[r][h];
    if (g + 1 < a.G) {
      copy(g + 1, (g + 1) & 1);
      weights(g + 1);
    }
    v4i aop[RT][2];
    v4f s4[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
      if (FMT == 4) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const unsigned x = w[r][0][e] ^ 0x88888888u;
          aop[r][0][e] = (int)((x << 4) & 0xF0F0F0F0u);
          aop[r][1][e] = (int)(x & 0xF0F0F0F0u);
        }
        s4[r] = *(const v4f *)(buf + kGemmScales + kGemmTokens * 4 + (64 * wm + 16 * r + 4 * kb) * 4);
      } else {
        aop[r][0] = __builtin_bit_cast(v4i, w[r][0]);
        aop[r][1] = __builtin_bit_cast(v4i, w[r][NA - 1]);
        s4[r] = v4f{1.f, 1.f, 1.f, 1.f};
      }
    }
#pragma unroll
    for (int j = 0; j < NTW; j++) {
      const int tl = wn * NTW + j;
      v4i d[kDigPlanes];
#pragma unroll
      for (int p = 0; p < kDigPlanes; p++) d[p] = *(const v4i *)(buf + (tl * kDigPlanes + p) * 1024 + 16 * lane);
      const float sas = *(const float *)(buf + kGemmScales + (tl * kDigTile + n) * 4), as = fabsf(sas);
      if (__ballot(__float_as_uint(sas) >> 31) != 0) left[j] |= 1ull << g;
#pragma unroll
      for (int r = 0; r < RT; r++) {
        v4i c[4];
#pragma unroll
        for (int p = 0; p < 4; p++) c[p] = mfma_i8(aop[r][0], d[2 * p], v4i{0, 0, 0, 0});
#pragma unroll
        for (int p = 0; p < 4; p++) c[p] = mfma_i8(aop[r][1], d[2 * p + 1], c[p]);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float f = __builtin_fmaf((float)(c[0][e] * 256 + c[1][e]), 65536.0f, (float)(c[2][e] * 256 + c[3][e]));
          acc[r][j][e] = FMT == 4 ? __builtin_fmaf(f * as, s4[r][e], acc[r][j][e]) : __builtin_fmaf(f, as, acc[r][j][e]);
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NTW; j++) {
    const int tl = tile0 + wn * NTW + j, tt = tl < ttiles ? tl : ttiles - 1, t = tt * kDigTile + n;
#pragma unroll 1
    for (unsigned long long u = left[j]; __builtin_expect(u != 0, 0); u &= u - 1) {
      const int g = __builtin_ctzll(u);
#pragma unroll
      for (int r = 0; r < RT; r++) {
        const unsigned char *q[4];
        v4f s4;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int row = row0 + 64 * wm + 16 * r + 4 * kb + e, rc = row < rlast ? row : rlast;
          q[e] = pm.q + (size_t)rc * pm.rb + (size_t)g * (FMT == 4 ? 64 : 128);
          s4[e] = FMT == 4 ? pm.s[(size_t)rc * pm.ng + g] : 1.0f;
        }
        const size_t at = ((size_t)tt * a.G + g) * kDigTile + n;
        add_left_out(a.d.asc + at, a.d.mask + at * 16,
                     a.d.out + ((size_t)(t < a.T ? t : 0) * a.G + g) * 128, s4, acc[r][j],
                     [&](int e, int c) { return code_of<FMT>(q[e][FMT == 4 ? c >> 1 : c], c); });
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NTW; j++) {
    const int t = (tile0 + wn * NTW + j) * kDigTile + n;
    if (t >= a.T) continue;
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int row = row0 + 64 * wm + 16 * r + 4 * kb + e;
        if (row <= rlast) pm.y[(size_t)t * pm.ldy + row] = FMT == 8 ? acc[r][j][e] * pm.s[row] : acc[r][j][e];
      }
  }
}

}  // namespace sw
