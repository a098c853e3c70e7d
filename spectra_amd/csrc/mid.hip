// Mid-size batches of the GEMM family (17 <= m < 512: batched serving, chunks of prompts):
//   out = FWHT(a) . W_eff^T + bias
// for both weight formats (replaces kernels.py:187-389 at these sizes).
//
// What bounds it: a few dozen to a few hundred rows over a 4-bit weight need little HBM
// (QKV at 48 rows: 9.6 MB, 2 us) and little MFMA time (1 us); what a 256-row tile with a
// barrier per 32 k costs is latency and padding.  So here
//
// 1. mid_prep_kernel rotates, scales (a power of two per row) and rounds the activations to
//    fp16 and stores them as MFMA A fragments -- 1 KB per (32 rows, 16 k), in the order the
//    packed bytes decode -- plus, for weights with outliers, a k-major copy; further
//    workgroups of the same launch turn the outlier entries (CSR entries or outlier columns)
//    into (column, value - decoded code) pairs.
// 2. mid_kernel: 128 columns (weight rows), up to 256 activation rows and a range of K per
//    workgroup.  A lane takes the packed bytes of its own weight row (one 32-run; the wave's
//    halves take the two runs of a 64-k chunk), decodes them in registers
//    (NF4: nibble-pair LUT in LDS, Format A: integer bits to fp16), applies the block scale
//    with one fp16 rounding and uses the result as the B operand for every row tile: decoded
//    weights never pass through LDS.
// 3. mid_reduce_kernel sums the K splits' fp32 partials in order, adds the outliers (one
//    coalesced read of the k-major activations per entry), undoes the row scale, adds the
//    bias and rounds once.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"

namespace spectra {

typedef _Float16 m8h_t __attribute__((ext_vector_type(8)));
typedef _Float16 m2h_t __attribute__((ext_vector_type(2)));
typedef float m16f_t __attribute__((ext_vector_type(16)));
typedef uint32_t mu4_t __attribute__((ext_vector_type(4)));
typedef uint16_t mus2_t __attribute__((ext_vector_type(2)));

constexpr int kMidThreads = 512;
constexpr int kMidBN = 128;      // columns per workgroup
constexpr int kMidLut = 65536;   // nibble-pair LUT at LDS address 0 (NF4)

struct MidParams {
  const uint16_t* frag;  // A fragments [row tile][64-k chunk][4][64 lanes][8]
  const uint16_t* xk;    // k-major fp16 [k][mp] (outliers only)
  const uint2* meta;     // outlier entries (column, fp32 value - decoded code)
  const void* sfrag;     // block scales [32-row group][64-k chunk][64 lanes]: fp16, Format A with -(1024 + z)
  const int32_t* fexp;
  const uint8_t* packed;
  int64_t ldp;
  const int32_t* rowptr;  // CSR; null: n_out entries per row
  const void* bias;
  void* out;
  int64_t ldo;
  float* part;  // fp32 partials [ksplit][mp / 32][np / 32][32 x 32 in accumulator order]
  int m, n, k, mp, np;
  int n_out, has_o, cap, asym, marlin, bias_dt, act_dt;  // cap: entries of a row its own lanes add
  int ksplit, chunks;  // K splits (blockIdx.z) and 64-k chunks per split
};

// Four packed bytes -> the B operand of one MFMA step: byte i is the pair (fp16) of dword i, times
// the block scale (sz: its fp16 bits; Format A: fp16 -(1024 + z) in the high half)
template <int FMT>
__device__ __forceinline__ m8h_t mid_decode(uint32_t w, uint32_t sz, uint32_t lanebits) {
  const _Float16 sh = __builtin_bit_cast(_Float16, (uint16_t)sz);
  const m2h_t s2 = {sh, sh};
  uint32_t o[4];
  if constexpr (FMT == SPECTRA_FMT_NF4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t addr = __builtin_amdgcn_perm(w, lanebits, 0x0c0c0000u | ((4u + i) << 8));
      m2h_t c = __builtin_bit_cast(m2h_t, *(const __attribute__((address_space(3))) uint32_t*)(uintptr_t)addr);
      c = c * s2;  // one fp16 rounding
      o[i] = __builtin_bit_cast(uint32_t, c);
    }
  } else {
    // 0x6400 | q is the fp16 number 1024 + q: minus (1024 + z) is q - z exactly
    const _Float16 zh = __builtin_bit_cast(_Float16, (uint16_t)(sz >> 16));
    const m2h_t z2 = {zh, zh};
    const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t q = __builtin_amdgcn_perm(hi, lo, 0x0c000c00u | ((4u + i) << 16) | (uint32_t)i) | 0x64006400u;
      m2h_t c = __builtin_bit_cast(m2h_t, q) + z2;
      c = c * s2;
      o[i] = __builtin_bit_cast(uint32_t, c);
    }
  }
  const mu4_t o4 = {o[0], o[1], o[2], o[3]};
  return __builtin_bit_cast(m8h_t, o4);
}

// ---------------------------------------------------------------------------
// activation pre-pass
// ---------------------------------------------------------------------------
constexpr int kMidPrepThreads = 512, kMidPrepRows = 8, kMidPrepSeg = 512;
constexpr int kMidPrepWgs = 128;
constexpr int kMidEntryRows = 32;  // weight rows per entry workgroup

struct MidSide {
  const uint8_t* packed;
  int64_t ldp;
  const uint16_t* scales;
  int64_t lds;
  const uint8_t* zeros;  // Format A; null: NF4
  int64_t ldz;
  const int64_t* oidx;
  const void* ow;
  int64_t ldow;
  const int32_t* rowptr;  // CSR; null: outlier columns
  const int32_t* ccol;
  const uint16_t* cval;
  int n, gshift, n_out, ow_dt;
  uint2* meta;   // null: no outliers
  void* sfrag;
};

// Block scales of weight rows [32 b, 32 b + 32) into the order the MFMA kernel's lanes use them
// (lane (n, g) of chunk c: row n's scale of run 2 c + g; rows past the last repeat it), so that a
// wave's scales are one or two lines instead of 32.  32 chunks a workgroup.
__device__ __forceinline__ void mid_scales(const MidSide& en, int k, int b, int sg, int tid, uint32_t (*st)[65]) {
  const int n0 = b * kMidEntryRows, nc = k >> 6, s0 = 32 * sg;
  uint32_t v[2048 / kMidPrepThreads];
#pragma unroll
  for (int u = 0; u < 2048 / kMidPrepThreads; ++u) {
    const int i = tid + u * kMidPrepThreads, r = min(n0 + (i >> 6), en.n - 1), run = min(2 * s0 + (i & 63), 2 * nc - 1);
    v[u] = en.scales[(int64_t)r * en.lds + ((32 * run) >> en.gshift)];
    if (en.zeros) v[u] |= (uint32_t)en.zeros[(int64_t)r * en.ldz + run] << 16;
  }
#pragma unroll
  for (int u = 0; u < 2048 / kMidPrepThreads; ++u) {
    const int i = tid + u * kMidPrepThreads;
    if (en.zeros) v[u] = (v[u] & 0xffffu) | (uint32_t)f2h(-(float)(1024 + (int)(v[u] >> 16))) << 16;
    st[(i & 63) >> 1][(i & 1) * 32 + (i >> 6)] = v[u];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 2048 / kMidPrepThreads; ++u) {
    const int i = tid + u * kMidPrepThreads, c = s0 + (i >> 6);
    if (c < nc) {
      const int64_t o = ((int64_t)b * nc + c) * 64 + (i & 63);
      if (en.zeros)
        ((uint32_t*)en.sfrag)[o] = st[i >> 6][i & 63];
      else
        ((uint16_t*)en.sfrag)[o] = (uint16_t)st[i >> 6][i & 63];
    }
  }
}

// The entries of weight rows [32 b, 32 b + 32): an entry takes the place of the decoded code at
// its position, so what the product still lacks is (value - decoded code) x[column].  The
// decoded code rounds as the kernels' (one fp16 rounding of code * scale); columns outside K
// are dropped (delta 0).
__device__ __forceinline__ void mid_entries(const MidSide& en, int k, int marlin, int b, int sg, int nsg, int tid,
                                            int32_t* rp) {
  const int n0 = b * kMidEntryRows, nr = min(kMidEntryRows, en.n - n0);
  if (tid <= nr) rp[tid] = en.rowptr ? en.rowptr[n0 + tid] : (n0 + tid) * en.n_out;
  __syncthreads();
  for (int e = rp[0] + sg * kMidPrepThreads + tid; e < rp[nr]; e += nsg * kMidPrepThreads) {
    int lo = 0;  // last row whose first entry is <= e
#pragma unroll
    for (int h = kMidEntryRows / 2; h > 0; h >>= 1)
      if (lo + h < nr && rp[lo + h] <= e) lo += h;
    const int row = n0 + lo;
    int c;
    float v;
    if (en.rowptr) {
      c = en.ccol[e];
      v = h2f(en.cval[e]);
    } else {
      const int j = e - rp[lo];
      const int64_t ix = en.oidx[j];
      c = ix < 0 || ix >= k ? -1 : (int)ix;
      v = h2f(f2h(load_elem(en.ow, (int64_t)row * en.ldow + j, en.ow_dt)));
    }
    float dv = 0.0f;
    if ((unsigned)c < (unsigned)k) {
      int64_t bj;
      int hb;
      k_to_nibble(c, marlin, &bj, &hb);
      const int code = (en.packed[(int64_t)row * en.ldp + bj] >> (4 * hb)) & 15;
      const _Float16 sc = __builtin_bit_cast(_Float16, en.scales[(int64_t)row * en.lds + (c >> en.gshift)]);
      _Float16 w;
      if (en.zeros)
        w = (_Float16)(float)(code - (int)en.zeros[(int64_t)row * en.ldz + (c >> 5)]) * sc;
      else
        w = __builtin_bit_cast(_Float16, nf4_f16_bits(code)) * sc;
      dv = v - (float)w;
    } else {
      c = 0;
    }
    en.meta[e] = make_uint2((uint32_t)c, __builtin_bit_cast(uint32_t, dv));
  }
}

// Workgroups [0, sblocks): block scales and outlier entries; the others: 8 rows (one per wave) x
// segs 512-k segments (lane l: elements 8 l .. 8 l + 7 of each).  The row scale is every workgroup's
// own from the whole row.  max |x_rot| 2^F lies in [2^14, 2^15), or, where the raw row is even (every
// nonzero piece of 8 reaches 2^-10 of its maximum), the bound sqrt(b) max |x| does: a block's energy is
// then at least 2^-5 per element, 2^20 above what fp16 can drop there.  A bound alone cost a row
// with one large activation up to 4.5 octaves of its small blocks' range; the maximum alone, a
// transform of the whole row in every workgroup, QKV 0.8 us at 48 rows and down 3.  FWHT
// stages 1, 2, 4 run in registers, 8 .. 256 across lanes.  Fragments leave through LDS in whole
// 128-byte lines (8 rows x 16 bytes); the k-major copy in 16-byte pieces.
template <bool VEC, int DT>
__global__ void __launch_bounds__(kMidPrepThreads) mid_prep_kernel(const uint16_t* __restrict__ a, int64_t lda, int m,
                                                                    int k, int log_had, float div, int marlin,
                                                                    uint16_t* __restrict__ frag,
                                                                    uint16_t* __restrict__ xk, int mp,
                                                                    int32_t* __restrict__ fexp, int sblocks, int segs,
                                                                    const MidSide en) {
  __shared__ __align__(16) mu4_t tile[64][kMidPrepRows + 1];  // [16-byte unit][row]
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int nseg = (k + kMidPrepSeg - 1) / kMidPrepSeg;
  if ((int)blockIdx.x < sblocks) {
    const int ssegs = (k + 2047) / 2048, b = (int)blockIdx.x / ssegs, sg = (int)blockIdx.x % ssegs;
    mid_scales(en, k, b, sg, tid, (uint32_t(*)[65])tile);
    if (en.meta && b * kMidEntryRows < en.n) {
      __syncthreads();
      mid_entries(en, k, marlin, b, sg, ssegs, tid, (int32_t*)tile);
    }
    return;
  }
  const int xb = (int)blockIdx.x - sblocks, gsegs = (nseg + segs - 1) / segs;
  const int r0 = (xb / gsegs) * kMidPrepRows, s0 = (xb % gsegs) * segs;
  const uint16_t* arow = a + (int64_t)min(r0 + wv, m - 1) * lda;
  auto load8 = [&](int e) __attribute__((always_inline)) {
    const uint16_t* src = arow + e;
    mu4_t q;
    if constexpr (VEC) {
      q = *(const mu4_t*)src;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = (uint32_t)src[2 * i] | ((uint32_t)src[2 * i + 1] << 16);
    }
    return q;
  };
  // eight elements of the row, blockwise transformed but for the sign (returned) and 1 / sqrt(b):
  // stages 1, 2, 4, ...: (u, v) -> (u + v, u - v) in fp32 (compressor.py:34-39)
  auto rotate = [&](const mu4_t& x, float (&v)[1][8]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[0][2 * i] = to_f32_16((uint16_t)(x[i] & 0xffffu), DT);
      v[0][2 * i + 1] = to_f32_16((uint16_t)(x[i] >> 16), DT);
    }
#pragma unroll
    for (int lh = 0; lh < 3; ++lh) {
      if (lh < log_had) {
        const int h = 1 << lh;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if ((e & h) == 0) {
            const float x0 = v[0][e], x1 = v[0][e | h];
            v[0][e] = x0 + x1;
            v[0][e | h] = x0 - x1;
          }
      }
    }
    float sgn = 1.0f;
    auto side = [&](int lb) { const bool hi = (tid & lb) != 0; if (hi) sgn = -sgn; return hi ? -1.0f : 1.0f; };
    if (log_had > 3) prep_fly<1>(v, side(1), lane);
    if (log_had > 4) prep_fly<2>(v, side(2), lane);
    if (log_had > 5) prep_fly<4>(v, side(4), lane);
    if (log_had > 6) prep_fly<8>(v, side(8), lane);
    if (log_had > 7) prep_fly<16>(v, side(16), lane);
    if (log_had > 8) prep_fly<32>(v, side(32), lane);
    return sgn;
  };
  // the raw row: its largest magnitude, and the smallest one that a lane's nonzero piece of 8 reaches,
  // as 15-bit integers, two to an instruction (an infinity or a NaN is the largest)
  mus2_t mx = {0, 0};
  uint32_t mn = 0x7fff;  // less 1
  for (int e = 8 * lane; e < k; e += 16 * kMidPrepSeg) {  // sixteen loads in flight (past the end: the first again)
    mu4_t f[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) f[j] = load8(e + kMidPrepSeg * j < k ? e + kMidPrepSeg * j : e);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      mus2_t c = {0, 0};
#pragma unroll
      for (int i = 0; i < 4; ++i) c = __builtin_elementwise_max(c, __builtin_bit_cast(mus2_t, f[j][i] & 0x7fff7fffu));
      mx = __builtin_elementwise_max(mx, c);
      mn = min(mn, (uint32_t)max(c[0], c[1]) - 1u);
    }
  }
  // fp32 bits: an infinity above every number, NaN above all
  uint32_t mb = max(__builtin_bit_cast(uint32_t, to_f32_16(mx[0], DT)), __builtin_bit_cast(uint32_t, to_f32_16(mx[1], DT)));
  auto wave_max_bits = [&](uint32_t v) __attribute__((always_inline)) {
    auto with = [&](float o) { v = max(v, __builtin_bit_cast(uint32_t, o)); };
    with(lane_xor<32>(__builtin_bit_cast(float, v), lane));
    with(lane_xor<16>(__builtin_bit_cast(float, v), lane));
    with(lane_xor<8>(__builtin_bit_cast(float, v), lane));
    with(lane_xor<4>(__builtin_bit_cast(float, v), lane));
    with(lane_xor<2>(__builtin_bit_cast(float, v), lane));
    with(lane_xor<1>(__builtin_bit_cast(float, v), lane));
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
  };
  mb = wave_max_bits(mb);
  uint32_t bits = mb;
  if (log_had > 0) {
    const float raw = __builtin_bit_cast(float, mb), bound = raw * div * 1.0009765625f;
    const uint32_t least = 0x8000u - wave_max_bits(0x7fffu - mn);  // (0x8000: no nonzero piece)
    const bool even = log_had >= 3 && bound < __builtin_inff() &&
                      (least == 0x8000u || to_f32_16((uint16_t)least, DT) >= raw * 0x1p-10f);
    bits = __builtin_bit_cast(uint32_t, bound);
    if (!even) {
      mb = 0;
      // A maximum needs the block's outputs in no order and with no sign: lanes meet at distances
      // 1, 2, 7, 8 (all single DPP operands; a lane's sides are then bits 0 ^ 2, 1 ^ 2, 2, 3), and the
      // stage inside a dword comes last, max(|u + v|, |u - v|) = |u| + |v|.  What the order moves the
      // maximum by (2^-22) can turn the exponent at its edge only, inside fp16's spare octave.
      const float s1 = ((lane ^ (lane >> 2)) & 1) ? -1.0f : 1.0f, s2 = ((lane ^ (lane >> 1)) & 2) ? -1.0f : 1.0f;
      const float s4 = (lane & 4) ? -1.0f : 1.0f, s8 = (lane & 8) ? -1.0f : 1.0f;
      auto block_max = [&](const mu4_t& x) __attribute__((always_inline)) {
        float v[1][8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[0][2 * i] = to_f32_16((uint16_t)(x[i] & 0xffffu), DT);
          v[0][2 * i + 1] = to_f32_16((uint16_t)(x[i] >> 16), DT);
        }
#pragma unroll
        for (int lh = 1; lh < 3; ++lh)
          if (lh < log_had)
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if ((e & (1 << lh)) == 0) {
                const float x0 = v[0][e], x1 = v[0][e | (1 << lh)];
                v[0][e] = x0 + x1;
                v[0][e | (1 << lh)] = x0 - x1;
              }
        if (log_had > 3) prep_fly<1>(v, s1, lane);
        if (log_had > 4) prep_fly<2>(v, s2, lane);
        if (log_had > 5) prep_fly<7>(v, s4, lane);
        if (log_had > 6) prep_fly<8>(v, s8, lane);
        if (log_had > 7) prep_fly<16>(v, (lane & 16) ? -1.0f : 1.0f, lane);
        if (log_had > 8) prep_fly<32>(v, (lane & 32) ? -1.0f : 1.0f, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          mb = max(mb, __builtin_bit_cast(uint32_t, fabsf(v[0][2 * i]) + fabsf(v[0][2 * i + 1])) & 0x7fffffffu);
      };
      constexpr int B = 8;  // loads in flight; a lane past the end takes its piece of the first block again
      const int e0 = 8 * lane, back = e0 & ((1 << log_had) - 1);
      for (int b = 0; b < k; b += B * kMidPrepSeg) {
        mu4_t f[B];
#pragma unroll
        for (int j = 0; j < B; ++j) f[j] = load8(b + kMidPrepSeg * j + e0 < k ? b + kMidPrepSeg * j + e0 : back);
#pragma unroll
        for (int j = 0; j < B; ++j) {
          if (b + kMidPrepSeg * j >= k) break;
          block_max(f[j]);
        }
      }
      mb = wave_max_bits(mb);
      bits = __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, mb) / div);
    }
  }
  const int eb = (int)(bits >> 23);
  const int E = eb == 0 ? -126 : eb - 127;
  int F = bits == 0 || mb > 0x7f800000u ? 0 : 14 - E;  // (NaN takes the whole row at any scale)
  F = F < -126 ? -126 : (F > 126 ? 126 : F);
  if (s0 == 0 && lane == 0 && r0 + wv < m) fexp[r0 + wv] = F;
  const float f2 = __builtin_bit_cast(float, (uint32_t)(F + 127) << 23);
  // unit of this lane in its 32-run (lane & 3 = q holds elements 8 q .. 8 q + 7): plain order,
  // elements 8 q ..; Marlin order, the pairs (k, k + 16) for k = 4 d .. 4 d + 3, which the
  // lanes q and q ^ 2 build from each other's halves (d = 0, 2, 1, 3 for q = 0, 1, 2, 3)
  const int q = lane & 3;
  const int d = marlin ? ((q & 1) << 1) | (q >> 1) : q;
  const int nc = k >> 6, t = r0 >> 5, rl = r0 & 31;
  for (int sg = s0; sg < min(s0 + segs, nseg); ++sg) {
    const int k0 = sg * kMidPrepSeg;
    const mu4_t x = load8(k0 + 8 * lane < k ? k0 + 8 * lane : 0);  // k is a multiple of 64
    float v[1][8];
    const float sgn = rotate(x, v);
    const float f = sgn * (log_had > 0 ? f2 / div : f2);
    mu4_t w;
    if (marlin) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float own = (q & 2) ? v[0][4 + i] * f : v[0][i] * f, give = (q & 2) ? v[0][i] * f : v[0][4 + i] * f;
        const float got = lane_xor<2>(give, lane);
        w[i] = (uint32_t)f2h((q & 2) ? got : own) | ((uint32_t)f2h((q & 2) ? own : got) << 16);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        w[i] = (uint32_t)f2h(v[0][2 * i] * f) | ((uint32_t)f2h(v[0][2 * i + 1] * f) << 16);
    }
    if (sg > s0) __syncthreads();  // (the last segment has been read)
    tile[(lane & ~3) + d][wv] = w;
    __syncthreads();
    // fragments: unit ru = 4 run + d of the segment, 8 rows of 16 bytes = 128 contiguous bytes
    {
      const int ru = tid >> 3, r = tid & 7, run = (k0 >> 5) + (ru >> 2);
      if (run < (k >> 5)) {
        const int64_t o = (((int64_t)t * nc + (run >> 1)) * 4 + (ru & 3)) * 512 + ((run & 1) * 32 + rl + r) * 8;
        *(mu4_t*)(frag + o) = tile[ru][r];
      }
    }
    if (xk != nullptr && k0 + tid < k) {  // element tid of the segment
      const int es = tid & 31;
      const int b = marlin ? (es & 15) : (es >> 1), h = marlin ? (es >> 4) : (es & 1);
      const uint16_t* src = (const uint16_t*)&tile[(tid >> 5) * 4 + (b >> 2)][0] + 2 * (b & 3) + h;
      mu4_t o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = (uint32_t)src[16 * j] | ((uint32_t)src[16 * j + 8] << 16);
      *(mu4_t*)(xk + (int64_t)(k0 + tid) * mp + r0) = o;
    }
  }
}

// ---------------------------------------------------------------------------
// MFMA kernels
// ---------------------------------------------------------------------------
// 8 waves = 2 column halves of 64 x 4: for up to 64 rows (CS = 4) the four 64-k chunks of a stage,
// up to 128 (CS = 2) the two chunks x two halves of a chunk's MFMA steps, up to 256 (CS = 1) two
// halves of the rows x two halves of the steps.  A wave multiplies WT row tiles by 64 columns: a
// fragment read from LDS feeds two MFMAs, a decoded operand WT.  Fragments (a stage) and packed
// bytes (a quad of four chunks: whole 128-byte lines of each row, where the operand layout would
// touch 32 lines for 1 KB) pass through registers into two LDS buffers each, one barrier a stage,
// fragments three stages and packed bytes UQ quads ahead.  The waves that share outputs meet in
// LDS, in a fixed order.
template <int FMT, int WT, int CS>
__global__ void __launch_bounds__(kMidThreads) mid_kernel(const MidParams p) {
  constexpr int MT = CS == 1 ? 2 * WT : WT;       // row tiles
  constexpr int AF = MT * CS * 4 / 8;             // fragments a wave copies per stage
  constexpr int kStage = MT * CS * 4096, SPQ = 4 / CS, UQ = CS == 4 ? 4 : 2, ST = CS == 4 ? 4 : 2;
  constexpr int AS = WT == 4 && CS == 1 ? 1 : 2;  // fragment stages in registers (one where two would spill)
  typedef typename std::conditional<FMT == SPECTRA_FMT_NF4, uint16_t, uint32_t>::type scale_t;
  extern __shared__ __align__(16) uint8_t smem[];
  uint8_t* abuf = smem + kMidLut;
  uint8_t* wbuf = abuf + 2 * kStage;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1, sh = (wave >> 1) & 1, hh = wave >> 2;
  const int g = lane >> 5, ln = lane & 31;
  const int n0 = blockIdx.x * kMidBN, t0 = blockIdx.y * MT;
  const int NC = p.k >> 6;
  const int c0 = blockIdx.z * p.chunks, cend = min(c0 + p.chunks, NC);
  const int nq = (cend - c0 + 3) >> 2, ns = (cend - c0 + CS - 1) / CS;
  const int cw = CS == 4 ? 2 * hh + sh : CS == 2 ? hh : 0;  // this wave's chunk of a stage

  // packed bytes: rows 16 wave + 8 i + lane / 8, 16-byte piece lane % 8 of the quad's 128
  mu4_t wr[UQ][2];
  const uint8_t* wsrc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    wsrc[i] = p.packed + (int64_t)min(n0 + 16 * wave + 8 * i + (lane >> 3), p.n - 1) * p.ldp;
  auto wload = [&](int u, int q) __attribute__((always_inline)) {  // (past the row: its last piece again)
    const int o = 16 * min(2 * (c0 + 4 * q) + (lane & 7), 2 * NC - 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) wr[u][i] = *(const mu4_t*)(wsrc[i] + o);
  };
  // (piece x of row r at x ^ (r % 8): the operand reads take one piece of 32 rows)
  const int wdst = (16 * wave + (lane >> 3)) * 128 + 16 * ((lane & 7) ^ (lane >> 3));
  auto wstore = [&](int u, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) *(mu4_t*)(wbuf + buf * 16384 + i * 1024 + wdst) = wr[u][i];
  };
  // block scales in operand order (mid_prep_kernel)
  scale_t sr[4][2];
  const scale_t* ssrc = (const scale_t*)p.sfrag + ((int64_t)(n0 >> 5) + 2 * wn) * NC * 64 + lane;
  auto sload = [&](int u, int s) __attribute__((always_inline)) {
    const int cc = min(c0 + CS * s + cw, NC - 1);
#pragma unroll
    for (int j = 0; j < 2; ++j) sr[u][j] = ssrc[((int64_t)j * NC + cc) * 64];
  };
  // fragment f = wave + 8 i of a stage: (row tile f / (4 CS), chunk f / 4 % CS, step f % 4)
  mu4_t ar[AS][AF];
  const uint16_t* asrc = p.frag + ((int64_t)t0 * NC * 4 + (wave & 3)) * 512 + lane * 8;
  auto aload = [&](int set, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AF; ++i) {
      const int f = wave + 8 * i;
      const int cc = min(c0 + CS * s + ((f >> 2) % CS), NC - 1);
      ar[set][i] = *(const mu4_t*)(asrc + (int64_t)(f / (4 * CS) * NC + cc) * 2048);
    }
  };
  auto astore = [&](int set, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AF; ++i) *(mu4_t*)(abuf + buf * kStage + (wave + 8 * i) * 1024 + lane * 16) = ar[set][i];
  };
  wload(0, 0);
  aload(0, 0);
  sload(0, 0);
#pragma unroll
  for (int u = 1; u < UQ; ++u) wload(u, u);
  if constexpr (AS == 2) aload(1, 1);
#pragma unroll
  for (int u = 1; u < 4; ++u) sload(u, u);
  if constexpr (FMT == SPECTRA_FMT_NF4) build_pair_lut<FMT>(smem, wave, kMidThreads / 64, lane);
  wstore(0, 0);
  wload(0, UQ);
  if constexpr (SPQ == 1) {
    wstore(1, 1);
    wload(1, UQ + 1);
  }
  astore(0, 0);
  aload(0, AS);
  asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");  // LDS writes only: the loads stay in flight

  const uint32_t lanebits = (uint32_t)lane << 2;
  m16f_t acc[WT][2];
#pragma unroll
  for (int i = 0; i < WT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  // this wave's part of a stage: row tile i at + i kTile, its first step at abase; its packed bytes
  constexpr int kTile = CS * 4096;
  const uint8_t* abase = abuf + (CS == 1 ? hh * WT * 4096 : cw * 4096) + (CS == 4 ? 0 : sh * 2048) + lane * 16;
  const uint8_t* wbase = wbuf + (64 * wn + ln) * 128 + (CS == 4 ? 0 : 8 * sh);
  uint32_t w[2][ST];  // the packed bytes of the stage decoded next
  auto wread = [&](int qbuf, int sub) __attribute__((always_inline)) {
    const int piece = 16 * ((2 * (CS * sub + cw) + g) ^ (ln & 7));
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint8_t* wp = wbase + qbuf * 16384 + j * 4096 + piece;
      if constexpr (ST == 4) {
        const mu4_t t = *(const mu4_t*)wp;
#pragma unroll
        for (int d = 0; d < 4; ++d) w[j][d] = t[d];
      } else {
        const uint2 t = *(const uint2*)wp;
        w[j][0] = t.x;
        w[j][1] = t.y;
      }
    }
  };
  m8h_t b[2][ST][2];  // decoded operands of the stage and of the next
  auto decode = [&](m8h_t (&bd)[2], int d, int ss, int s) __attribute__((always_inline)) {
    const bool live = c0 + CS * s + cw < cend;
#pragma unroll
    for (int j = 0; j < 2; ++j) bd[j] = mid_decode<FMT>(w[j][d], live ? sr[ss][j] : (scale_t)0, lanebits);
  };
  wread(0, 0);
#pragma unroll
  for (int d = 0; d < ST; ++d) decode(b[0][d], d, 0, 0);
  sload(0, 4);
  // stage 0 of a one-stage quad writes over the first quad: its reads have arrived (Format A's
  // decode, plain arithmetic, may sink past the barrier and with it the wait for them)
  asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");
  // Stage s: the products of its operands, with the next stage's decoded, its fragments written
  // to the other buffer and the loads of s + 1 + AS (fragments), s + 5 (scales) and the quad UQ (+ 1)
  // ahead issued in between (past the range: its last chunk again).
  for (int q0 = 0; q0 < nq; q0 += UQ) {
#pragma unroll
    for (int uq = 0; uq < UQ; ++uq) {
      const int q = q0 + uq;
      if (q >= nq) break;
#pragma unroll
      for (int sub = 0; sub < SPQ; ++sub) {
        const int s = q * SPQ + sub;
        if (s >= ns) break;
        const int st = (uq * SPQ + sub) & 1, ss = (uq * SPQ + sub + 1) & 3;  // (ss: the next stage's scales)
        const uint8_t* ab = abase + st * kStage;
        wread(sub == SPQ - 1 ? (uq + 1) & 1 : uq & 1, (sub + 1) % SPQ);
        astore((1 - st) % AS, 1 - st);
        aload((1 - st) % AS, s + 1 + AS);
#pragma unroll
        for (int d = 0; d < ST; ++d) {
          m8h_t af[WT];
#pragma unroll
          for (int i = 0; i < WT; ++i) af[i] = *(const m8h_t*)(ab + i * kTile + d * 1024);
#pragma unroll
          for (int i = 0; i < WT; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], b[st][d][j], acc[i][j], 0, 0, 0);
          decode(b[1 - st][d], d, ss, s + 1);
        }
        sload(ss, s + 5);
        if (SPQ == 1) {  // (the buffer read a stage ago)
          wstore((uq + 2) % UQ, uq & 1);
          wload((uq + 2) % UQ, q + 2 + UQ);
        } else if (sub == SPQ - 2) {
          wstore((uq + 1) % UQ, (uq + 1) & 1);
          wload((uq + 1) % UQ, q + 1 + UQ);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");
      }
    }
  }

  // the waves that differ in sh meet: wave sh keeps column group sh and hands over the other
  float* red = (float*)smem;
  m16f_t y[WT];
#pragma unroll
  for (int i = 0; i < WT; ++i)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      float4 o;
      o.x = sh ? acc[i][0][4 * r4] : acc[i][1][4 * r4];
      o.y = sh ? acc[i][0][4 * r4 + 1] : acc[i][1][4 * r4 + 1];
      o.z = sh ? acc[i][0][4 * r4 + 2] : acc[i][1][4 * r4 + 2];
      o.w = sh ? acc[i][0][4 * r4 + 3] : acc[i][1][4 * r4 + 3];
      *(float4*)(red + (((wave ^ 2) * WT + i) * 4 + r4) * 256 + lane * 4) = o;
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < WT; ++i)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const float4 o = *(const float4*)(red + ((wave * WT + i) * 4 + r4) * 256 + lane * 4);
      y[i][4 * r4] = (sh ? acc[i][1][4 * r4] : acc[i][0][4 * r4]) + o.x;
      y[i][4 * r4 + 1] = (sh ? acc[i][1][4 * r4 + 1] : acc[i][0][4 * r4 + 1]) + o.y;
      y[i][4 * r4 + 2] = (sh ? acc[i][1][4 * r4 + 2] : acc[i][0][4 * r4 + 2]) + o.z;
      y[i][4 * r4 + 3] = (sh ? acc[i][1][4 * r4 + 3] : acc[i][0][4 * r4 + 3]) + o.w;
    }
  const int tw = t0 + (CS == 1 ? hh * WT : 0);
  float* part = p.part + (((int64_t)blockIdx.z * (p.mp >> 5) + tw) * (p.np >> 5) + (n0 >> 5) + 2 * wn + sh) * 1024;
  if constexpr (CS == 1) {
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        *(float4*)(part + (int64_t)i * (p.np >> 5) * 1024 + r4 * 256 + lane * 4) =
            make_float4(y[i][4 * r4], y[i][4 * r4 + 1], y[i][4 * r4 + 2], y[i][4 * r4 + 3]);
  } else {  // so do those that differ in hh: wave hh keeps r4 = 2 hh, 2 hh + 1 of each row tile
    __syncthreads();
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        float4 o;
        o.x = hh ? y[i][4 * q] : y[i][8 + 4 * q];
        o.y = hh ? y[i][4 * q + 1] : y[i][8 + 4 * q + 1];
        o.z = hh ? y[i][4 * q + 2] : y[i][8 + 4 * q + 2];
        o.w = hh ? y[i][4 * q + 3] : y[i][8 + 4 * q + 3];
        *(float4*)(red + (((wave ^ 4) * WT + i) * 2 + q) * 256 + lane * 4) = o;
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float4 o = *(const float4*)(red + ((wave * WT + i) * 2 + q) * 256 + lane * 4);
        float4 v;
        v.x = (hh ? y[i][8 + 4 * q] : y[i][4 * q]) + o.x;
        v.y = (hh ? y[i][8 + 4 * q + 1] : y[i][4 * q + 1]) + o.y;
        v.z = (hh ? y[i][8 + 4 * q + 2] : y[i][4 * q + 2]) + o.z;
        v.w = (hh ? y[i][8 + 4 * q + 3] : y[i][4 * q + 3]) + o.w;
        *(float4*)(part + (int64_t)i * (p.np >> 5) * 1024 + (2 * hh + q) * 256 + lane * 4) = v;
      }
  }
}

// Rows with an infinity have the scale exponent kMidInfF, which no finite row reaches.  Where the
// weight has outliers such a row's products are summed here, value x inf in place of code x inf (a
// code of 0 would make it NaN); what its finite activations add does not show beside an infinity.
constexpr int kMidInfF = 14 - 128;
__device__ __forceinline__ float mid_inf_row(const MidParams& p, int row, int col, float y0) {
  const int e0 = p.rowptr ? p.rowptr[col] : col * p.n_out, e1 = p.rowptr ? p.rowptr[col + 1] : e0 + p.n_out;
  const int NC = p.k >> 6;
  float y = 0.0f;
  bool any = false;
#pragma unroll 16
  for (int k = 0; k < p.k; ++k) {
    const uint16_t x = p.xk[(int64_t)k * p.mp + row];
    if ((x & 0x7c00) != 0x7c00) continue;
    any = true;
    int64_t bj;
    int hb;
    k_to_nibble(k, p.marlin, &bj, &hb);
    const int code = (p.packed[(int64_t)col * p.ldp + bj] >> (4 * hb)) & 15;
    const int64_t si = ((int64_t)(col >> 5) * NC + (k >> 6)) * 64 + (k & 32) + (col & 31);
    float w;
    if (p.asym) {
      const uint32_t sz = ((const uint32_t*)p.sfrag)[si];
      w = ((float)(1024 + code) + h2f((uint16_t)(sz >> 16))) * h2f((uint16_t)sz);
    } else {
      w = h2f(nf4_f16_bits(code)) * h2f(((const uint16_t*)p.sfrag)[si]);
    }
    w = h2f(f2h(w));
    float v = w;
    for (int e = e0; e < e1; ++e) {
      const uint2 m = p.meta[e];
      if ((int)m.x == k) v = w + __builtin_bit_cast(float, m.y);
    }
    y = __builtin_fmaf(v, h2f(x), y);
  }
  return any ? y : y0;
}

// out = act((sum over splits of the partials + outliers) 2^-F + bias), 32 columns x RB row tiles
// per workgroup, splits summed in order.  Groups of RB * 8 lanes (four rows a lane) own a
// column's entries, twelve reads of the k-major activations in flight; the 512 threads are
// 64 / RB such groups, CG of them (64 / RB / 32) sharing a column.  A row much longer than the others
// would run on alone: past p.cap entries (twice the average, at least 64) all groups share it.  48 rows
// of 3072 x 8192, 0.5% outliers: 37.7 us, one dense row 623 without that and 71 with it (the 256-row
// tiles: 74).
constexpr int kMidRedThreads = 512, kMidMaxSplit = 16;
template <int RB>
__global__ void __launch_bounds__(kMidRedThreads) mid_reduce_kernel(const MidParams p) {
  constexpr int LP = 8 * RB, CG = kMidRedThreads / LP / 32, RS = 32 * RB + 4;
  __shared__ __align__(16) float cor[CG][32][RS];
  __shared__ __align__(16) uint16_t ot[32 * RB][32 + 8];
  constexpr int NG = kMidRedThreads / LP;
  __shared__ __align__(16) float tail[NG][RS];  // long rows: the groups' sums
  __shared__ int2 rows[32];
  __shared__ int longer[kMidRedThreads / 64];
  const int tid = threadIdx.x;
  const int nb = blockIdx.y, n0 = 32 * nb, tb = blockIdx.x * RB, m0 = 32 * tb;
  const int NB = p.np >> 5, MB = p.mp >> 5;
  // pieces of a float4: (row tile, r4, lane); RB * 256 of them, at most one per thread
  const bool has_p = tid < RB * 256;
  const float* src = p.part + ((int64_t)(tb + (has_p ? tid >> 8 : 0)) * NB + nb) * 1024 + (tid & 255) * 4;
  const int64_t zs = (int64_t)MB * NB * 1024;
  float4 pb[8];
#pragma unroll
  for (int v = 0; v < 8; ++v) pb[v] = *(const float4*)(src + min(v, p.ksplit - 1) * zs);
  if (p.has_o) {
    const int grp = tid / LP, lr = tid % LP, cg = grp >> 5;
    const uint16_t* xsrc = p.xk + m0 + 4 * lr;
    // entries e, e + step, ... of [.., e1) into o
    auto gather = [&](int e, const int e1, const int step, float (&o)[4]) __attribute__((always_inline)) {
      constexpr int U = 12;
      uint2 md[U];  // the next turn's entries are read while this turn's activations are on the way
      if (e < e1)
#pragma unroll
        for (int v = 0; v < U; ++v) md[v] = p.meta[min(e + v * step, e1 - 1)];
      for (; e < e1; e += U * step) {
        uint2 x[U];
        float d[U];
#pragma unroll
        for (int v = 0; v < U; ++v) {
          x[v] = *(const uint2*)(xsrc + (int64_t)md[v].x * p.mp);
          d[v] = e + v * step < e1 ? __builtin_bit_cast(float, md[v].y) : 0.0f;
        }
#pragma unroll
        for (int v = 0; v < U; ++v) md[v] = p.meta[min(e + (U + v) * step, e1 - 1)];
#pragma unroll
        for (int v = 0; v < U; ++v)
          if (e + v * step < e1) {
            o[0] = __builtin_fmaf(d[v], h2f((uint16_t)x[v].x), o[0]);
            o[1] = __builtin_fmaf(d[v], h2f((uint16_t)(x[v].x >> 16)), o[1]);
            o[2] = __builtin_fmaf(d[v], h2f((uint16_t)x[v].y), o[2]);
            o[3] = __builtin_fmaf(d[v], h2f((uint16_t)(x[v].y >> 16)), o[3]);
          }
      }
    };
    const int c = min(n0 + (grp & 31), p.n - 1);
    const int e0 = p.rowptr ? p.rowptr[c] : c * p.n_out, e1 = p.rowptr ? p.rowptr[c + 1] : e0 + p.n_out;
    if (grp < 32 && lr == 0) rows[grp] = make_int2(e0, e1);
    float o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    gather(e0 + cg, e0 + min(e1 - e0, p.cap), CG, o);
    const bool any = __builtin_amdgcn_ballot_w64(e1 - e0 > p.cap) != 0;
    if ((tid & 63) == 0) longer[tid >> 6] = any;
    *(float4*)&cor[cg][grp & 31][4 * lr] = make_float4(o[0], o[1], o[2], o[3]);
    __syncthreads();
    int more = 0;
#pragma unroll
    for (int w = 0; w < kMidRedThreads / 64; ++w) more |= longer[w];
    if (more) {
      for (int j = 0; j < min(32, p.n - n0); ++j) {
        const int2 r = rows[j];
        if (r.y - r.x <= p.cap) continue;  // (uniform)
        float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        gather(r.x + p.cap + grp, r.y, NG, t);
        *(float4*)&tail[grp][4 * lr] = make_float4(t[0], t[1], t[2], t[3]);
        __syncthreads();
        if (tid < 32 * RB) {
          float v = cor[0][j][tid];
          for (int g = 0; g < NG; ++g) v += tail[g][tid];
          cor[0][j][tid] = v;
        }
        __syncthreads();
      }
    }
  }
  float y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int z0 = 0;;) {
#pragma unroll
    for (int v = 0; v < 8; ++v)
      if (z0 + v < p.ksplit) {
        y[0] += pb[v].x; y[1] += pb[v].y; y[2] += pb[v].z; y[3] += pb[v].w;
      }
    z0 += 8;
    if (z0 >= p.ksplit) break;
#pragma unroll
    for (int v = 0; v < 8; ++v) pb[v] = *(const float4*)(src + min(z0 + v, p.ksplit - 1) * zs);
  }
  const int col = n0 + (tid & 31);  // (the piece's lane % 32)
  const float bv = p.bias && col < p.n ? load_elem(p.bias, col, p.bias_dt) : 0.0f;
  if (has_p) {
    // D[row][col]: row = 8 r4 + 4 (lane / 32) + element, col = lane % 32
    const int rl = 32 * (tid >> 8) + 8 * ((tid >> 6) & 3) + 4 * ((tid >> 5) & 1);
    if (p.has_o) {
#pragma unroll
      for (int h = 0; h < CG; ++h) {
        const float4 o = *(const float4*)&cor[h][tid & 31][rl];
        y[0] += o.x; y[1] += o.y; y[2] += o.z; y[3] += o.w;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = min(m0 + rl + e, p.m - 1), F = p.fexp[row];
      if (p.has_o && F == kMidInfF && col < p.n) y[e] = mid_inf_row(p, row, col, y[e]);
      ot[rl + e][tid & 31] = from_f32_16(y[e] * __builtin_bit_cast(float, (uint32_t)(127 - F) << 23) + bv, p.act_dt);
    }
  }
  __syncthreads();
  for (int i = tid; i < 32 * RB * 4; i += kMidRedThreads) {  // 8 columns of one row
    const int r = i >> 2, c8 = 8 * (i & 3);
    if (m0 + r < p.m && n0 + c8 < p.n) {
      uint16_t* dst = (uint16_t*)p.out + (int64_t)(m0 + r) * p.ldo + n0 + c8;
      if (n0 + c8 + 8 <= p.n && (reinterpret_cast<uintptr_t>(dst) & 15) == 0)
        *(uint4*)dst = *(const uint4*)&ot[r][c8];
      else
        for (int e = 0; e < 8 && n0 + c8 + e < p.n; ++e) dst[e] = ot[r][c8 + e];
    }
  }
}

static size_t mid_align(size_t v) { return (v + 255) & ~(size_t)255; }

struct MidPlan {
  int cs, t, mt, nt, ksplit, chunks, mp;  // mid_kernel<t, cs>
};
static MidPlan plan_mid(int64_t m, int64_t n, int64_t k) {
  MidPlan g;
  const int tiles = (int)((m + 255) / 256);
  const int rows = (int)((m + tiles - 1) / tiles);
  g.cs = rows <= 64 ? 4 : rows <= 128 ? 2 : 1;
  g.t = g.cs == 1 ? (rows + 63) / 64 : (rows + 31) / 32;
  const int R = 32 * g.t * (g.cs == 1 ? 2 : 1);
  g.mt = (int)((m + R - 1) / R);
  g.mp = (g.mt * R + 63) & ~63;  // (whole row tiles of the reduce)
  g.nt = (int)((n + kMidBN - 1) / kMidBN);
  const int nq = (int)((k / 64 + 3) / 4), ncu = device_cu_count();
  // K splits (whole quads): the rounds of workgroups times a split's quads (us, measured), against
  // the partials' round trip.  A sweep of 1 .. 16 splits on ten shapes found the most splits that
  // still run in one round the best or within 0.5 us of it; a second round costs 6 to 10 us.
  double best = 1e30;
  int per = nq;
  for (int s = 1; s <= kMidMaxSplit && s <= nq; ++s) {
    const int qs = (nq + s - 1) / s;
    if ((nq + qs - 1) / qs != s) continue;
    const double rounds = (double)(((int64_t)g.mt * g.nt * s + ncu - 1) / ncu);
    const double quad = g.cs == 4 ? 0.45 + 0.25 * g.t : g.cs == 2 ? 0.55 + 0.3 * g.t : 0.9 + 0.6 * g.t;
    const double t = rounds * (5.5 + qs * quad) + (double)s * g.mp * n * 4 * 2 / 5e6;
    if (t < best) {
      best = t;
      per = qs;
    }
  }
  g.ksplit = (nq + per - 1) / per;
  g.chunks = 4 * per;
  return g;
}

// entries of the outlier side tensor (0: none)
static int64_t mid_entries_count(const spectra_qweight_t* w) {
  if (w->outlier_kind == SPECTRA_OUTLIERS_CSR) return w->csr_nnz;
  if (w->outlier_kind == SPECTRA_OUTLIERS_COLUMNS) return w->n * (int64_t)w->num_outliers;
  return 0;
}

// When this family runs.  Whole calls in graphs over 450 MB of layers, us, the 256-row-tile GEMM / this
// family, N x K = 5120 x 3072, 16384 x 3072, 3072 x 8192, 14336 x 4096:
//   NF4, none      32 rows  25 / 18   44 / 25   36 / 20   55 / 27    96 rows  30 / 26   50 / 36   41 / 27   61 / 38
//   NF4, 0.5%      32 rows  27 / 24   46 / 35   39 / 28   58 / 38    48 rows  29 / 29   48 / 42   40 / 34   59 / 45
//                  96 rows  33 / 34   53 / 56   42 / 38   64 / 59
//   NF4, 2%        32 rows  32 / 28   51 / 45   49 / 38   65 / 51    48 rows  32 / 36   53 / 57   50 / 51   67 / 67
//   Format A, 1%   32 rows  29 / 25   52 / 41   44 / 32   64 / 45    48 rows  31 / 30   54 / 48   45 / 40   65 / 55
//                  96 rows  35 / 36   58 / 63   48 / 43   69 / 72
// An outlier entry costs a read of every row's activation here and a fixed amount there, so the line is
// a density that falls with the rows; it lies twice as high for K >= 4096 (that GEMM's chain of K steps
// is what it is up against), and for Format A (its decode needs no table here) up to 64 rows or for
// K >= 8192, and small weights with short rows lose to the reduce's fixed part (2048 x 2048, 0.5%, 56
// rows 21.8 / 23.3).  Without outliers 160 rows are 33 / 30, 55 / 49, 42 / 36, 64 / 53, and 224 rows
// slower here.  Where that GEMM leaves most of the chip idle (it splits K at most eight ways, and not
// at all for N % 4 != 0) this family is faster at any size: N = 289, K = 12288 31
// against 259 at 130 rows, 43 against 279 at 400; N = 1001, K = 2112 36 against 67.
static bool mid_serves(const spectra_qweight_t* w, int64_t m, int64_t tile_wgs) {
  const int64_t entries = mid_entries_count(w);
  if (m < 17 || m >= 512 || w->n < 1 || w->k < 64 || w->k % 64 != 0 || w->k > 32768 || w->hadamard_block > 512 ||
      (w->format == SPECTRA_FMT_NF4 && w->group_size < 32) || entries >= (1LL << 31) - 4096 || w->n > 65535 * 32)
    return false;
  if (tile_wgs < device_cu_count() / 4) return true;
  if (entries == 0) return m <= 160;
  int64_t per = m <= 32 ? 40 : m <= 64 ? 160 : 320;  // weights to an entry, at least
  if (m > 32 && w->k >= 4096) per /= 2;
  if (m > 32 && (m <= 64 || w->k >= 8192) && w->format == SPECTRA_FMT_ASYM_G32) per /= 2;
  const int64_t fixed = m > 32 && w->k < 4096 ? 1 << 22 : 0;
  return m <= 96 && entries * per + fixed <= w->n * w->k;
}

struct MidWorkspace {
  size_t frag, xk, meta, sfrag, fexp, part, total;
};
static MidWorkspace mid_layout(const spectra_qweight_t* w, int64_t m, const MidPlan& g) {
  MidWorkspace l;
  const size_t act = mid_align((size_t)g.mp * w->k * 2);
  const int64_t ne = mid_entries_count(w);
  l.frag = 0;
  l.xk = act;
  l.meta = l.xk + (ne > 0 ? act : 0);
  l.sfrag = l.meta + mid_align((size_t)ne * 8);
  l.fexp = l.sfrag + mid_align((size_t)g.nt * kMidBN * (w->k / 32) * (w->format == SPECTRA_FMT_NF4 ? 2 : 4));
  l.part = l.fexp + mid_align((size_t)m * 4);
  l.total = l.part + (size_t)g.ksplit * g.mp * g.nt * kMidBN * 4;
  return l;
}

// tile_wgs: workgroups of the 256-row-tile GEMM for this call
size_t mid_workspace(const spectra_qweight_t* w, int64_t m, int64_t tile_wgs) {
  return mid_serves(w, m, tile_wgs) ? mid_layout(w, m, plan_mid(m, w->n, w->k)).total : 0;
}

bool mid_runs(const spectra_qweight_t* w, int64_t m, size_t workspace_bytes, int64_t tile_wgs) {
  return mid_serves(w, m, tile_wgs) && workspace_bytes >= mid_layout(w, m, plan_mid(m, w->n, w->k)).total;
}

template <int FMT>
static const void* mid_pick(const MidPlan& g) {
  if (g.cs == 1) return g.t == 3 ? (const void*)mid_kernel<FMT, 3, 1> : (const void*)mid_kernel<FMT, 4, 1>;
  if (g.cs == 2) return g.t == 3 ? (const void*)mid_kernel<FMT, 3, 2> : (const void*)mid_kernel<FMT, 4, 2>;
  return g.t == 1 ? (const void*)mid_kernel<FMT, 1, 4> : (const void*)mid_kernel<FMT, 2, 4>;
}

// SPECTRA_ERR_UNSUPPORTED (nothing launched): the caller runs the 256-row-tile GEMM
int mid_launch(const spectra_qweight_t* w, const void* a, int64_t lda, int64_t m, int act_dtype, void* out,
               int64_t ldo, void* workspace, size_t workspace_bytes, int64_t tile_wgs, hipStream_t s) {
  if (!mid_serves(w, m, tile_wgs)) return SPECTRA_ERR_UNSUPPORTED;
  const MidPlan g = plan_mid(m, w->n, w->k);
  const MidWorkspace l = mid_layout(w, m, g);
  if (workspace_bytes < l.total) return SPECTRA_ERR_UNSUPPORTED;  // (as mid_runs)
  const bool has_o = mid_entries_count(w) > 0, csr = w->outlier_kind == SPECTRA_OUTLIERS_CSR;
  uint8_t* ws = (uint8_t*)workspace;
  int gs = 0;
  while ((1 << gs) < w->group_size) ++gs;
  MidParams p;
  p.frag = (const uint16_t*)(ws + l.frag);
  p.xk = has_o ? (const uint16_t*)(ws + l.xk) : nullptr;
  p.meta = (const uint2*)(ws + l.meta);
  p.fexp = (const int32_t*)(ws + l.fexp);
  p.sfrag = ws + l.sfrag;
  p.packed = w->packed; p.ldp = w->packed_stride;
  p.rowptr = csr ? w->csr_rowptr : nullptr;
  p.bias = w->bias; p.out = out; p.ldo = ldo;
  p.part = (float*)(ws + l.part);
  p.m = (int)m; p.n = (int)w->n; p.k = (int)w->k; p.mp = g.mp; p.np = g.nt * kMidBN;
  p.n_out = w->num_outliers; p.has_o = has_o;
  p.cap = (int)std::max<int64_t>(64, 2 * mid_entries_count(w) / w->n);
  p.asym = w->format == SPECTRA_FMT_ASYM_G32; p.marlin = w->marlin_layout ? 1 : 0;
  p.bias_dt = w->bias_dtype; p.act_dt = act_dtype;
  p.ksplit = g.ksplit; p.chunks = g.chunks;
  MidSide en;
  en.packed = w->packed; en.ldp = w->packed_stride;
  en.scales = w->scales; en.lds = w->scales_stride;
  en.zeros = w->format == SPECTRA_FMT_ASYM_G32 ? w->zeros : nullptr; en.ldz = w->zeros_stride;
  en.oidx = w->outlier_idx; en.ow = w->outlier_w; en.ldow = w->outlier_w_stride; en.ow_dt = w->outlier_w_dtype;
  en.rowptr = p.rowptr; en.ccol = w->csr_col; en.cval = w->csr_val;
  en.n = p.n; en.gshift = gs; en.n_out = p.n_out; 
  en.meta = has_o ? (uint2*)(ws + l.meta) : nullptr; en.sfrag = ws + l.sfrag;

  int log_had = 0;
  while (w->hadamard_block > 1 && (1 << log_had) < w->hadamard_block) ++log_had;
  const float div = log_had > 0 ? (float)std::sqrt((double)w->hadamard_block) : 1.0f;
  const int vec = (reinterpret_cast<uintptr_t>(a) % 16) == 0 && lda % 8 == 0;
  // segments a workgroup takes: every workgroup reads its whole rows for their scale, so no more
  // workgroups than half the CUs can hold
  const int rg = (int)((m + kMidPrepRows - 1) / kMidPrepRows), nseg = (int)((w->k + kMidPrepSeg - 1) / kMidPrepSeg);
  const int segs = std::max(1, (rg * nseg + kMidPrepWgs - 1) / kMidPrepWgs);
  const int xblocks = rg * ((nseg + segs - 1) / segs);
  const int sblocks = g.nt * (kMidBN / kMidEntryRows) * (int)((w->k + 2047) / 2048);
  const void* prep = act_dtype == SPECTRA_BF16
                         ? (vec ? (const void*)mid_prep_kernel<true, SPECTRA_BF16> : (const void*)mid_prep_kernel<false, SPECTRA_BF16>)
                         : (vec ? (const void*)mid_prep_kernel<true, SPECTRA_F16> : (const void*)mid_prep_kernel<false, SPECTRA_F16>);
  const int mi = (int)m, marlin = w->marlin_layout ? 1 : 0;
  uint16_t *frag = (uint16_t*)(ws + l.frag), *xk = has_o ? (uint16_t*)(ws + l.xk) : nullptr;
  int32_t* fexp = (int32_t*)(ws + l.fexp);
  void* pargs[] = {(void*)&a, (void*)&lda, (void*)&mi, (void*)&p.k, (void*)&log_had, (void*)&div,
                   (void*)&marlin, (void*)&frag, (void*)&xk, (void*)&p.mp, (void*)&fexp, (void*)&sblocks, (void*)&segs, (void*)&en};
  SPECTRA_HIP_CHECK(hipLaunchKernel(prep, dim3((unsigned)(xblocks + sblocks)), dim3(kMidPrepThreads), pargs, 0, s));
  SPECTRA_HIP_CHECK(hipGetLastError());

  const void* kern = w->format == SPECTRA_FMT_NF4 ? mid_pick<SPECTRA_FMT_NF4>(g) : mid_pick<SPECTRA_FMT_ASYM_G32>(g);
  const int st = ensure_lds_limit(kern, true);
  if (st != SPECTRA_OK) return st;
  void* kargs[] = {(void*)&p};
  // LDS: the LUT and two stages; the waves' meeting place lies over both
  const size_t lds = (size_t)kMidLut + 2 * (size_t)(g.t * 4096 * (g.cs == 4 ? 4 : 2)) + 2 * 16384;
  SPECTRA_HIP_CHECK(hipLaunchKernel(kern, dim3((unsigned)g.nt, (unsigned)g.mt, (unsigned)g.ksplit),
                                    dim3(kMidThreads), kargs, lds, s));
  SPECTRA_HIP_CHECK(hipGetLastError());
  const int rb = m > 32 ? 2 : 1;
  const void* red = rb == 2 ? (const void*)mid_reduce_kernel<2> : (const void*)mid_reduce_kernel<1>;
  SPECTRA_HIP_CHECK(hipLaunchKernel(red, dim3((unsigned)((m + 32 * rb - 1) / (32 * rb)), (unsigned)((w->n + 31) / 32)),
                                    dim3(kMidRedThreads), kargs, 0, s));
  SPECTRA_HIP_CHECK(hipGetLastError());
  return SPECTRA_OK;
}

}  // namespace spectra
