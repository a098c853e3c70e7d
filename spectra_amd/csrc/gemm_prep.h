// The activation pre-pass of the prefill GEMM paths (gemm.hip, dequant.hip): blockwise FWHT of a
// row in fp32, scaled and rounded.
#pragma once
#include "common.h"

namespace spectra {

constexpr int kPrepThreads = 256;

// One workgroup of 256 threads per activation row.  The row's 8-element chunks are spread
// over the threads (chunk c = tid + 256 u, up to 16 per thread), so a Hadamard block of b
// <= 512 elements lies in b / 8 consecutive lanes of one wave: stages h = 1, 2, 4 run on
// register bits and h = 8 .. 256 across lanes (each stage one fp32 add or subtract, the
// reference's order and rounding); blocks of 1024 finish their last stage through LDS.
// The row is scaled by a power of two (max |x_rot| -> [2^14, 2^15)), rounded to fp16 and
// written in packed-byte pair order.
constexpr int kPrepMaxU = 16;  // K <= 256 * 8 * 16 = 32768

// raw_dt >= 0 (the library-GEMM path): no scale (F = 0), the rotated row rounded to raw_dt
// (SPECTRA_F16 or SPECTRA_BF16), the compute dtype of the reference's GEMM; marlin must be 0.
// With no row-wide scale to find, sg then picks a segment of kPrepThreads * 8 * kPrepU
// elements of the row (a multiple of every Hadamard block size), so a long row spreads over
// several workgroups; the scaled mode runs with sg = 0 (the whole row).
// fs: LDS, [k] fp32 for 1024-blocks (their last stage), [k] fp16 for marlin (pair-order write).
template <int kPrepU>
__device__ __forceinline__ void gemm_prep_row(const void* __restrict__ a, int64_t lda, int dt, int k, int log_had,
                                              float div, int marlin, int vec, uint16_t* __restrict__ a16,
                                              int32_t* __restrict__ fexp, int raw_dt, int64_t row, int sg, float* fs) {
  __shared__ float wmax[kPrepThreads / 64];
  const int tid = threadIdx.x;
  const int64_t seg0 = (int64_t)sg * (kPrepThreads * 8 * kPrepU);  // first element
  const int n8 = (int)min((int64_t)k - seg0, (int64_t)kPrepThreads * 8 * kPrepU) >> 3;
  float v[kPrepU][8];
#pragma unroll
  for (int u = 0; u < kPrepU; ++u) {
    const int c = tid + u * kPrepThreads;
    if (c < n8) {
      if (vec) {
        const uint4 q = ((const uint4*)((const uint16_t*)a + row * lda + seg0))[c];
        const uint32_t w4[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[u][2 * e] = to_f32_16((uint16_t)(w4[e] & 0xffffu), dt);
          v[u][2 * e + 1] = to_f32_16((uint16_t)(w4[e] >> 16), dt);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] = load_elem(a, row * lda + seg0 + 8 * c + e, dt);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[u][e] = 0.0f;
    }
  }
  // compressor.py:34-39: stages h = 1, 2, 4, ...: (u, v) -> (u + v, u - v) in fp32
  // (stage loops unrolled with compile-time strides: the register array stays in registers)
#pragma unroll
  for (int lh = 0; lh < 3; ++lh) {
    if (lh < log_had) {
      const int h = 1 << lh;
#pragma unroll
      for (int u = 0; u < kPrepU; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if ((e & h) == 0) {
            const float x0 = v[u][e], x1 = v[u][e | h];
            v[u][e] = x0 + x1;
            v[u][e | h] = x0 - x1;
          }
    }
  }
  // stages h = 8 .. 256 across the lanes of a block (lane bit lh - 3)
  const int lane = tid & 63;
  float sgn = 1.0f;
  auto side = [&](int lb) { const bool hi = (tid & lb) != 0; if (hi) sgn = -sgn; return hi ? -1.0f : 1.0f; };
  if (log_had > 3) prep_fly<1>(v, side(1), lane);
  if (log_had > 4) prep_fly<2>(v, side(2), lane);
  if (log_had > 5) prep_fly<4>(v, side(4), lane);
  if (log_had > 6) prep_fly<8>(v, side(8), lane);
  if (log_had > 7) prep_fly<16>(v, side(16), lane);
  if (log_had > 8) prep_fly<32>(v, side(32), lane);
  if (log_had > 9) {  // 1024-blocks: the stage across waves through LDS
#pragma unroll
    for (int u = 0; u < kPrepU; ++u)
      if (tid + u * kPrepThreads < n8)
#pragma unroll
        for (int e = 0; e < 8; ++e) fs[8 * (tid + u * kPrepThreads) + e] = v[u][e];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPrepU; ++u) {
      const int c = tid + u * kPrepThreads;
      if (c < n8) {
        const float cc = (c & 64) != 0 ? -1.0f : 1.0f;  // element bit 9 = chunk bit 6 (same for every u)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] = __builtin_fmaf(fs[8 * (c ^ 64) + e], cc, v[u][e]);
      }
    }
    __syncthreads();
    if (tid & 64) sgn = -sgn;  // every chunk of this thread has the same bit 6 (256 | 64)
  }
  // the normalisation by sqrt(block) (compressor.py:40-41) rides on the output scale below
  float mx = 0.0f;
#pragma unroll
  for (int u = 0; u < kPrepU; ++u)
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[u][e]));
  mx = wave_max(mx);
  if ((tid & 63) == 0) wmax[tid >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  if (log_had > 0) mx = mx / div;  // the normalised row's max |x_rot|
  const uint32_t bits = __builtin_bit_cast(uint32_t, mx);
  const int eb = (int)(bits >> 23);
  const int E = eb == 0 ? -126 : eb - 127;
  int F = bits == 0 ? 0 : 14 - E;  // max |x_rot| * 2^F in [2^14, 2^15): exact scaling, no overflow
  F = F < -126 ? -126 : (F > 126 ? 126 : F);
  if (raw_dt >= 0) F = 0;
  const float f2 = __builtin_bit_cast(float, (uint32_t)(F + 127) << 23);
  // output scale: 2^F / sqrt(block) (one rounding), with the lane's butterfly sign
  const float f = sgn * (log_had > 0 ? f2 / div : f2);
  uint16_t* xs = (uint16_t*)fs;
  if (marlin) {  // natural order into LDS, then pairs (k, k + 16) of each 32-run
#pragma unroll
    for (int u = 0; u < kPrepU; ++u) {
      const int c = tid + u * kPrepThreads;
      if (c < n8) {
        uint32_t d[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          d[e] = (uint32_t)f2h(v[u][2 * e] * f) | ((uint32_t)f2h(v[u][2 * e + 1] * f) << 16);
        *(uint4*)(xs + 8 * c) = make_uint4(d[0], d[1], d[2], d[3]);
      }
    }
    __syncthreads();
    // output chunk c (positions 8 c .. 8 c + 7) = bytes 4 c .. 4 c + 3: run c / 4, j = 4 (c % 4) + i
#pragma unroll
    for (int u = 0; u < kPrepU; ++u) {
      const int c = tid + u * kPrepThreads;
      if (c < n8) {
        const uint16_t* run = xs + 32 * (c >> 2);
        const int j0 = 4 * (c & 3);
        uint32_t d[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i] = (uint32_t)run[j0 + i] | ((uint32_t)run[j0 + i + 16] << 16);
        *(uint4*)(a16 + row * k + seg0 + 8 * c) = make_uint4(d[0], d[1], d[2], d[3]);
      }
    }
  } else {  // byte j = (k 2j, k 2j + 1): pair order is the natural order
#pragma unroll
    for (int u = 0; u < kPrepU; ++u) {
      const int c = tid + u * kPrepThreads;
      if (c < n8) {
        uint32_t d[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          d[e] = raw_dt >= 0 ? (uint32_t)from_f32_16(v[u][2 * e] * f, raw_dt) |
                                   ((uint32_t)from_f32_16(v[u][2 * e + 1] * f, raw_dt) << 16)
                             : (uint32_t)f2h(v[u][2 * e] * f) | ((uint32_t)f2h(v[u][2 * e + 1] * f) << 16);
        *(uint4*)(a16 + row * k + seg0 + 8 * c) = make_uint4(d[0], d[1], d[2], d[3]);
      }
    }
  }
  if (tid == 0) fexp[row] = F;
}

}  // namespace spectra
