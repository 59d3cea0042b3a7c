// The output head on gfx950: the final norm and the int8 lm_head projection
// of the reference's decode and prefill output (c/qwen.c:4505-4516,
// 4613-4616; the device glue cuda_resident_output_try, 1097-1124), with the
// CPU path's arithmetic bit for bit:
//   n = rmsnorm_zero(x, norm_w): ms = serial fp32 sum of rn(x_i*x_i) in
//       element order, r = 1/sqrtf(ms/n + eps), n_i = (x_i*r)*(1+w_i)
//       (c/qwen.c:1780-1784);
//   logits[v] = ((float)dot(q_v, xq) * scale[v]) * sx, xq = qrow_i8(n): the
//       IDOT of qmat_mul_ex / qmat_mul_batch for an int8 matrix
//       (c/qwen.c:1696-1705, 1765-1768, 3313-3319; allow_idot = 1 at 4512-4513
//       and 4616).
// The projection streams the vocab x hidden int8 matrix (HBM-bound: 1.02 GB
// for 248,320 x 4096), once per 16 tokens on the matrix cores (k_head_mfma) and
// for one to three tokens by VALU dots (k_head_q8): each lane keeps
// its 16-byte column chunks of the quantised activations in registers; a
// wave takes kHeadRows rows (one: 1, 2, 4 and 8 measured 5,750, 5,680, 5,520
// and 5,420 calls/s at S397), loads every chunk of them before the first
// dot, and reduces the exact int32 sums across the wave by DPP.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sw_backend.h"
#include "sw_device.h"

using namespace sw;

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

// rmsnorm_zero then qrow_i8, one token per block.  The sum of squares is the
// reference's serial chain, run by one wave over products computed in
// parallel (each product rounds once, as x[i]*x[i] does before the add).
__global__ __launch_bounds__(256) void k_head_norm(signed char *xq, float *sx, float *hidden, const float *x,
                                                   const float *w, int n, float eps, int pitch) {
  extern __shared__ float hp[];  // [n, to the next kSerialStep]: squares, then the normalised row
  __shared__ float s_r, red[4];
  const float *xs = x + (size_t)blockIdx.x * n;
  const int np = (n + kSerialStep - 1) / kSerialStep * kSerialStep;
  for (int i = threadIdx.x; i < np; i += blockDim.x) hp[i] = i < n ? xs[i] * xs[i] : 0.0f;
  __syncthreads();
  if (threadIdx.x < 64) {
    // 6, 12: eight rows of 4,096 30.6 -> 29.6 us with 64 logits, 29.1 without a bound
    const float ms = serial_sum_nonneg<6, 12>(hp, n, 0.0f);
    if (threadIdx.x == 0) s_r = 1.0f / sqrtf(ms / (float)n + eps);
  }
  __syncthreads();
  const float r = s_r;
  float m = 0.0f;
  float *hs = hidden ? hidden + (size_t)blockIdx.x * n : nullptr;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const float v = (xs[i] * r) * (1.0f + w[i]);
    hp[i] = v;
    if (hs) hs[i] = v;
    m = fmaxf(m, fabsf(v));
  }
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  float a = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float s = a / 127.0f;
  if (s < 1e-12f) s = 1e-12f;
  const float inv = 1.0f / s;
  if (threadIdx.x == 0) sx[blockIdx.x] = s;
  signed char *qs = xq + (size_t)blockIdx.x * pitch;
  for (int i = threadIdx.x; i < pitch; i += blockDim.x) qs[i] = i < n ? (signed char)__builtin_rintf(hp[i] * inv) : 0;
}

#ifndef SW_HEAD_DPP
#define SW_HEAD_DPP 1
#endif
#ifndef SW_HEAD_ROWS
#define SW_HEAD_ROWS 1
#endif
constexpr int kHeadRows = SW_HEAD_ROWS;  // rows per wave

__device__ __forceinline__ int dot16(const v4i w, const v4i x, int acc) {
  acc = __builtin_amdgcn_sdot4(w.x, x.x, acc, false);
  acc = __builtin_amdgcn_sdot4(w.y, x.y, acc, false);
  acc = __builtin_amdgcn_sdot4(w.z, x.z, acc, false);
  return __builtin_amdgcn_sdot4(w.w, x.w, acc, false);
}

// NB tokens, NCH chunks of 1024 columns (64 lanes x 16 bytes) per row.
// grid ceil(rows / (4 * kHeadRows)), 256 threads.  Requires cols % 16 == 0,
// row_bytes % 16 == 0, q 16-byte aligned and cols <= 1024 * NCH.
template <int NB, int NCH>
__global__ __launch_bounds__(256) void k_head_q8(float *logits, const signed char *xq, const float *sx, int pitch,
                                                 const signed char *q, const float *scales, int rows, int cols,
                                                 int row_bytes) {
  const int lane = threadIdx.x & 63;
  const int r0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * kHeadRows;
  if (r0 >= rows) return;
  v4i wv[kHeadRows][NCH];
#pragma unroll
  for (int i = 0; i < kHeadRows; i++) {
    const int row = r0 + i < rows ? r0 + i : rows - 1;
#pragma unroll
    for (int c = 0; c < NCH; c++) {
      const int col = 1024 * c + 16 * lane;
      wv[i][c] = col < cols ? __builtin_nontemporal_load((const v4i *)(q + (size_t)row * row_bytes + col))
                            : v4i{0, 0, 0, 0};
    }
  }
  v4i xr[NB][NCH];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int c = 0; c < NCH; c++) {
      const int col = 1024 * c + 16 * lane;
      xr[b][c] = col < cols ? *(const v4i *)(xq + (size_t)b * pitch + col) : v4i{0, 0, 0, 0};
    }
#pragma unroll
  for (int i = 0; i < kHeadRows; i++) {
    const int row = r0 + i;
#pragma unroll
    for (int b = 0; b < NB; b++) {
      int acc = 0;
#pragma unroll
      for (int c = 0; c < NCH; c++) acc = dot16(wv[i][c], xr[b][c], acc);
#if SW_HEAD_DPP
      acc = wave_sum_dpp(acc);
#else
      acc = wave_sum_i(acc);
#endif
      if (lane == 0 && row < rows) logits[(size_t)b * rows + row] = ((float)acc * scales[row]) * sx[b];
    }
  }
}

// Several tokens: exact int32 dots of 16 rows x up to 16 tokens by
// v_mfma_i32_16x16x64_i8, so the matrix is streamed once per 16 tokens and the
// dots leave the VALU (8 tokens, S397: two passes of VALU dots at 268 us each
// before, one of 203 us now, 5.0 TB/s; eight steps in flight against 4 and 16,
// nontemporal loads against plain ones: 224 against 232, 223 and 229 us a call).  The quantised activations wait in LDS in the
// MFMA's lane order ([64-column step][lane][16 bytes], zero past cols and
// batch); a wave walks 16-row tiles, eight steps (512 contiguous bytes of each
// row) of weights in flight ahead of the eight it works on, also across
// tiles.  HBM-bound.  Two workgroups a compute unit fit up to 4,096 columns.
// grid workgroups of 8 waves, cols % 64 == 0, 16-byte rows.
constexpr int kHeadSteps = 8;   // steps of 64 columns in flight
constexpr int kHeadTokens = 16;
__host__ __device__ inline int head_cols(int cols) { return (cols + 64 * kHeadSteps - 1) / (64 * kHeadSteps) * (64 * kHeadSteps); }

__global__ __launch_bounds__(512) void k_head_mfma(float *logits, const signed char *xq, const float *sx, int pitch,
                                                   int batch, const signed char *q, const float *scales, int rows,
                                                   int cols, int row_bytes) {
  extern __shared__ __align__(16) unsigned char hx[];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kb = lane >> 4;
  const int tiles = (rows + 15) / 16, step = gridDim.x * 8, chunks = head_cols(cols) / (64 * kHeadSteps);
  int tile = blockIdx.x * 8 + (tid >> 6);
  v4i cur[kHeadSteps], nxt[kHeadSteps];
  auto load = [&](int t, int c) {
    const int row = 16 * t + n < rows ? 16 * t + n : rows - 1;
    const signed char *p = q + (size_t)row * row_bytes;
#pragma unroll
    for (int j = 0; j < kHeadSteps; j++) {
      const int col = (c * kHeadSteps + j) * 64 + 16 * kb;
      nxt[j] = __builtin_nontemporal_load((const v4i *)(p + (col < cols ? col : 0)));
    }
  };
  if (tile < tiles) load(tile, 0);
  for (int u = tid; u < head_cols(cols); u += 512) {
    const int t = u & 15, col = (u >> 6) * 64 + ((u >> 4) & 3) * 16;
    ((v4i *)hx)[u] = t < batch && col < cols ? *(const v4i *)(xq + (size_t)t * pitch + col) : v4i{0, 0, 0, 0};
  }
  __syncthreads();
  const float sn = sx[n < batch ? n : 0];
  for (; tile < tiles; tile += step) {
    v4i acc = v4i{0, 0, 0, 0};
    float sc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) sc[i] = scales[16 * tile + 4 * kb + i < rows ? 16 * tile + 4 * kb + i : rows - 1];
    for (int c = 0; c < chunks; c++) {
#pragma unroll
      for (int j = 0; j < kHeadSteps; j++) cur[j] = nxt[j];
      if (c + 1 < chunks)
        load(tile, c + 1);
      else if (tile + step < tiles)
        load(tile + step, 0);
#pragma unroll
      for (int j = 0; j < kHeadSteps; j++) acc = mfma_i8(cur[j], ((const v4i *)hx)[(c * kHeadSteps + j) * 64 + lane], acc);
    }
    if (n < batch) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int row = 16 * tile + 4 * kb + i;
        if (row < rows) logits[(size_t)n * rows + row] = ((float)acc[i] * sc[i]) * sn;
      }
    }
  }
}

// any shape: one wave per (row, token), dword dots where aligned
__global__ __launch_bounds__(256) void k_head_q8_any(float *logits, const signed char *xq, const float *sx,
                                                     int pitch, const signed char *q, const float *scales,
                                                     int rows, int cols, int row_bytes) {
  const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6), b = blockIdx.y;
  if (row >= rows) return;
  const signed char *w = q + (size_t)row * row_bytes, *xb = xq + (size_t)b * pitch;
  int acc = 0;
  for (int j = lane; j < cols; j += 64) acc += (int)w[j] * (int)xb[j];
  acc = wave_sum_i(acc);
  if (lane == 0) logits[(size_t)b * rows + row] = ((float)acc * scales[row]) * sx[b];
}

template <int NB>
int launch_head(int nch, float *logits, const signed char *xq, const float *sx, int pitch, const signed char *q,
                const float *scales, int rows, int cols, int row_bytes, hipStream_t st) {
  const unsigned blocks = (unsigned)((rows + 4 * kHeadRows - 1) / (4 * kHeadRows));
  switch (nch) {
    case 1: k_head_q8<NB, 1><<<blocks, 256, 0, st>>>(logits, xq, sx, pitch, q, scales, rows, cols, row_bytes); break;
    case 2: k_head_q8<NB, 2><<<blocks, 256, 0, st>>>(logits, xq, sx, pitch, q, scales, rows, cols, row_bytes); break;
    case 4: k_head_q8<NB, 4><<<blocks, 256, 0, st>>>(logits, xq, sx, pitch, q, scales, rows, cols, row_bytes); break;
    default: k_head_q8<NB, 8><<<blocks, 256, 0, st>>>(logits, xq, sx, pitch, q, scales, rows, cols, row_bytes); break;
  }
  return 0;
}

}  // namespace

extern "C" int coli_cuda_output_head_q8(ColiCuda *ctx, float *logits, float *hidden, const float *x,
                                        const float *norm_w, float eps, int batch, const signed char *q,
                                        const float *scales, int vocab, int cols, int row_bytes) {
  if (!ctx || !logits || !x || !norm_w || !q || !scales || batch <= 0 || vocab <= 0 || cols <= 0 ||
      row_bytes < cols)
    return fail_arg("coli_cuda_output_head_q8: invalid argument");
  if (cols > 16384) return fail_arg("coli_cuda_output_head_q8: hidden %d exceeds 16384", cols);
  const int pitch = (cols + 15) & ~15;
  const size_t qbytes = ((size_t)batch * pitch + 255) & ~(size_t)255;
  if (ensure_scratch(ctx, kScrHead, qbytes + (size_t)batch * sizeof(float), "output head activation allocation"))
    return -1;
  signed char *xq = (signed char *)ctx->scratch[kScrHead];
  float *sx = (float *)((char *)ctx->scratch[kScrHead] + qbytes);
  hipStream_t st = ctx->stream;
  const size_t lds = (size_t)((cols + kSerialStep - 1) / kSerialStep * kSerialStep) * sizeof(float);
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void *)k_head_norm, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail_hip("output head norm attributes", e);
  }
  k_head_norm<<<batch, 256, lds, st>>>(xq, sx, hidden, x, norm_w, cols, eps, pitch);
  const bool fast = cols % 16 == 0 && row_bytes % 16 == 0 && ((uintptr_t)q & 15) == 0 && cols <= 8192;
  const int nch = (cols + 1023) / 1024;
  const int nchp = nch <= 1 ? 1 : nch <= 2 ? 2 : nch <= 4 ? 4 : 8;
  // 1 / 2 / 4 / 8 tokens, MFMA against VALU dots: 2,048 columns 105 / 106 / 108 /
  // 114 against 95 / 115 / 154 / 293 us, 4,096 columns 210 / 211 / 215 / 224 against
  // 165 / 189 / 278 / 534 (three tokens 113 against 105 at a vocabulary of 100,003).
  // Vocabulary 151,936, two tokens at 512 / 1,024 / 1,536 columns 23 / 39 / 59 against
  // 44 / 51 / 68, four at 2,560 / 3,072 / 5,120 / 8,192 99 / 111 / 192 / 263 against 144 /
  // 150 / 243 / 355; three there take 110 / 117 / 205 / 288 by VALU dots
  if (fast && batch >= (cols <= 2048 ? 2 : 4) && cols % 64 == 0) {
    const int hl = head_cols(cols) * 16, cus = ctx->sm_count > 0 ? ctx->sm_count : 256;
    const hipError_t e = hipFuncSetAttribute((const void *)k_head_mfma, hipFuncAttributeMaxDynamicSharedMemorySize, hl);
    if (e != hipSuccess) return fail_hip("output head attributes", e);
    const int wgs = (vocab + 127) / 128, most = cus * (hl <= 72 * 1024 ? 2 : 1);
    for (int b0 = 0; b0 < batch; b0 += kHeadTokens)
      k_head_mfma<<<wgs < most ? wgs : most, 512, hl, st>>>(logits + (size_t)b0 * vocab, xq + (size_t)b0 * pitch, sx + b0,
                                                           pitch, batch - b0 < kHeadTokens ? batch - b0 : kHeadTokens, q,
                                                           scales, vocab, cols, row_bytes);
    return launch_status("coli_cuda_output_head_q8");
  }
  for (int b0 = 0; b0 < batch; b0 += 4) {
    const int nb = batch - b0 < 4 ? batch - b0 : 4;
    float *lg = logits + (size_t)b0 * vocab;
    const signed char *xb = xq + (size_t)b0 * pitch;
    const float *sb = sx + b0;
    if (!fast) {
      k_head_q8_any<<<dim3((vocab + 3) / 4, nb), 256, 0, st>>>(lg, xb, sb, pitch, q, scales, vocab, cols, row_bytes);
      continue;
    }
    switch (nb) {
      case 1: launch_head<1>(nchp, lg, xb, sb, pitch, q, scales, vocab, cols, row_bytes, st); break;
      case 2: launch_head<2>(nchp, lg, xb, sb, pitch, q, scales, vocab, cols, row_bytes, st); break;
      case 3: launch_head<3>(nchp, lg, xb, sb, pitch, q, scales, vocab, cols, row_bytes, st); break;
      default: launch_head<4>(nchp, lg, xb, sb, pitch, q, scales, vocab, cols, row_bytes, st); break;
    }
  }
  return launch_status("coli_cuda_output_head_q8");
}
