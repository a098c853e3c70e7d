// Compressor-side kernels: blockwise FWHT, Format A (asymmetric INT4 group-32)
// quantizer and Format B (NF4 + Hadamard + CSR) quantizer.  All are bit-exact
// restatements of float32 reference arithmetic: compiled with -ffp-contract=off
// and the default correctly-rounded fp32 division, so each +,-,*,/ rounds once,
// exactly as torch's CPU float32 kernels do.
#include <algorithm>
#include <cmath>

#include "common.h"

namespace spectra {

constexpr int kQThreads = 256;

// In-LDS normalised FWHT of `nblk` consecutive blocks of `b` floats starting at s.
// Stage order h = 1, 2, 4, ... and the (u+v, u-v) butterfly follow
// compressor.py:34-39; normalisation is a division by fp32(sqrt(b)) (:40-41).
__device__ void fwht_lds(float* s, int nblk, int b, float div) {
  const int npairs = nblk * (b >> 1);
  for (int h = 1; h < b; h <<= 1) {
    __syncthreads();
    for (int p = threadIdx.x; p < npairs; p += blockDim.x) {
      const int blk = p / (b >> 1), w = p % (b >> 1);
      const int i = blk * b + (w / h) * 2 * h + (w % h);
      const float u = s[i], v = s[i + h];
      s[i] = u + v;
      s[i + h] = u - v;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nblk * b; i += blockDim.x) s[i] = s[i] / div;
  __syncthreads();
}

// ---------------------------------------------------------------------------
// spectra_fwht_rows: one workgroup transforms `seg` consecutive elements of one row
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kQThreads) fwht_rows_kernel(const void* __restrict__ x, int64_t ldx, int in_dt,
                                                                void* __restrict__ out, int64_t ldo, int out_dt,
                                                                int64_t k, int b, int seg, float div) {
  extern __shared__ float fs[];
  const int64_t segs_per_row = k / seg;
  const int64_t row = blockIdx.x / segs_per_row;
  const int64_t k0 = (blockIdx.x % segs_per_row) * seg;
  for (int i = threadIdx.x; i < seg; i += blockDim.x) fs[i] = load_elem(x, row * ldx + k0 + i, in_dt);
  fwht_lds(fs, seg / b, b, div);
  for (int i = threadIdx.x; i < seg; i += blockDim.x) store_elem(out, row * ldo + k0 + i, out_dt, fs[i]);
}

// ---------------------------------------------------------------------------
// shared pieces of the register quantizers: a wave owns 512 consecutive elements of a row, lane l
// the elements 8 l .. 8 l + 7, so a 32-group is 4 lanes and a 64-block 8
// ---------------------------------------------------------------------------
constexpr int kQSeg = 512, kQWaves = kQThreads / 64;

// eight consecutive elements in fp32 (vec: 16-byte aligned)
__device__ __forceinline__ void load8(const void* w, int64_t o, int dt, int vec, float (&v)[8]) {
  if (!vec) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = load_elem(w, o + e, dt);
  } else if (dt == SPECTRA_F32) {
    const float4 a = *(const float4*)((const float*)w + o), b = *(const float4*)((const float*)w + o + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
    const uint4 q = *(const uint4*)((const uint16_t*)w + o);
    const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = to_f32_16((uint16_t)(u[e >> 1] >> (16 * (e & 1))), dt);
  }
}

// a / b rounded to nearest, from y = 1 / b rounded to nearest: two Newton steps on the quotient,
// the first making it faithful, the second correctly rounded (P. Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", 1990, theorem 7.2).  Five
// instructions where the general division takes about ten; valid while nothing under- or
// overflows, which the callers see to.
__device__ __forceinline__ float div_by(float a, float b, float y) {
  float q = a * y;
  q = __builtin_fmaf(__builtin_fmaf(-q, b, a), y, q);
  return __builtin_fmaf(__builtin_fmaf(-q, b, a), y, q);
}

// Butterfly across lanes at distance LB: u + v low, u - v high, each one fp32 addition of the
// reference's operands (so zeros keep its signs)
template <int LB>
__device__ __forceinline__ void lane_fly(float (&v)[8], int lane) {
  const float c = (lane & LB) ? -1.0f : 1.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = __builtin_fmaf(v[e], c, lane_xor<LB>(v[e], lane));
}

// bytes (code e of `own` in byte e % 4) of the lane's eight codes, low dword elements 0 .. 3
__device__ __forceinline__ uint32_t pack_marlin(uint32_t c03, uint32_t c47, int lane) {
  // a 32-run is 4 lanes, q = lane % 4 holding elements 8 q ..; byte j = q[j] | q[j + 16] << 4:
  // lanes q and q ^ 2 trade halves, q < 2 keeping elements 0 .. 3 of both
  const bool up = (lane & 2) != 0;
  const uint32_t give = up ? c03 : c47, keep = up ? c47 : c03;
  const uint32_t got = (uint32_t)__builtin_amdgcn_mov_dpp((int)give, 0x4E, 0xF, 0xF, false);  // lane ^ 2
  return up ? got | (keep << 4) : keep | (got << 4);
}

// ---------------------------------------------------------------------------
// Format A quantizer (compressor.py:71-112).  HBM-bound (N K elements in, half a byte each out):
// wave-wide 16-byte loads and 4-byte stores, min / max and the nibble exchange across lanes.
// One thread per two groups, reading its own 128 bytes element by element, took 335 us for
// 3072 x 8192 bf16; this form 24 us (65 MB: 2.7 TB/s).  A wave keeps its columns for kQRows rows, so the outlier
// columns among a lane's eight are looked up once.
// ---------------------------------------------------------------------------
constexpr int kQRows = 8;

__global__ void __launch_bounds__(kQThreads) quant_g32_kernel(const void* __restrict__ w, int64_t ldw, int w_dt,
                                                                int64_t n, int64_t k, int vec,
                                                                const int64_t* __restrict__ oidx, int n_out,
                                                                uint8_t* __restrict__ packed,
                                                                uint16_t* __restrict__ scales,
                                                                uint8_t* __restrict__ pzeros) {
  const int lane = threadIdx.x & 63;
  const int64_t c0 = ((int64_t)blockIdx.x * kQWaves + (threadIdx.x >> 6)) * kQSeg + 8 * lane;
  const bool in = c0 < k;  // whole groups in or out (k is a multiple of 32)
  const int64_t G = k / 32, GP = (G + 1) / 2, g = c0 / 32;
  uint32_t omask = 0;  // outlier columns are zeroed before quantization (compressor.py:134-135)
  if (in && oidx != nullptr) {
    int lo = 0, hi = n_out;  // first idx >= c0 (idx ascending)
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (oidx[mid] < c0) lo = mid + 1; else hi = mid;
    }
    for (; lo < n_out && oidx[lo] < c0 + 8; ++lo) omask |= 1u << (oidx[lo] - c0);
  }
  const int64_t r1 = min(n, ((int64_t)blockIdx.y + 1) * kQRows);
  for (int64_t row = (int64_t)blockIdx.y * kQRows; row < r1; ++row) {
    float v[8];
    load8(w, row * ldw + (in ? c0 : 0), w_dt, vec, v);
    float wmin, wmax;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if ((omask >> e) & 1) v[e] = 0.0f;
      wmin = e == 0 ? v[0] : fminf(wmin, v[e]);
      wmax = e == 0 ? v[0] : fmaxf(wmax, v[e]);
    }
    wmin = fminf(wmin, lane_xor<1>(wmin, lane));
    wmax = fmaxf(wmax, lane_xor<1>(wmax, lane));
    wmin = fminf(wmin, lane_xor<2>(wmin, lane));
    wmax = fmaxf(wmax, lane_xor<2>(wmax, lane));
    const float diff = wmax - wmin;                       // :80
    const bool is_const = diff < 1e-8f;                   // :81 (scalar rounded to fp32)
    float s = is_const ? (wmin == 0.0f ? 1.0f : fabsf(wmin)) : diff / 15.0f;  // :83
    s = fmaxf(s, 1e-8f);                                  // :84
    uint32_t z;
    if (is_const)
      z = wmin < 0.0f ? 1 : 0;                            // :88
    else
      z = (uint32_t)fminf(fmaxf(rintf(-wmin / s), 0.0f), 15.0f);  // :89
    const float neg_zs = (-(float)z) * s;                 // -zeros.float() * scales   :95
    const float y = 1.0f / s;
    const bool plain = s > 0x1p-60f && s < 0x1p60f;       // (1e-8 <= s; an infinite or NaN group divides)
    uint32_t c03 = 0, c47 = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float t = v[e] - neg_zs;
      const float d = plain ? div_by(t, s, y) : t / s;
      const uint32_t q = is_const ? (wmin > 0.0f ? 1u : 0u)                            // :94
                                  : (uint32_t)fminf(fmaxf(rintf(d), 0.0f), 15.0f);     // :95
      if (e < 4) c03 |= q << (8 * e);
      else c47 |= q << (8 * (e - 4));
    }
    const uint32_t bytes = pack_marlin(c03, c47, lane);                                // :99-102
    const uint32_t zn = (uint32_t)__builtin_bit_cast(int, lane_xor<4>(__builtin_bit_cast(float, z), lane));
    if (in) {
      // lane q of the run: elements 0 .. 3 of lanes 0 and 2 are bytes 0 .. 3, and so on
      const int64_t o = row * (k / 2) + g * 16 + 8 * (lane & 1) + 2 * (lane & 2);
      uint8_t* dst = packed + o;
      if ((reinterpret_cast<uintptr_t>(dst) & 3) == 0) *(uint32_t*)dst = bytes;
      else
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = (uint8_t)(bytes >> (8 * e));
      if ((lane & 3) == 0) scales[row * G + g] = f2h(s);                               // :112
      if ((lane & 7) == 0)  // odd group count: high nibble stays 0 (compressor.py:106-107)
        pzeros[row * GP + (g >> 1)] = (uint8_t)(z | (g + 1 < G ? zn << 4 : 0));        // :108-110
    }
  }
}

// ---------------------------------------------------------------------------
// Format B quantizer: one workgroup per row segment of `seg` elements
// ---------------------------------------------------------------------------
__device__ __forceinline__ int nf4_nearest(float r) {
  // argmin_i |C_i - r| in fp32, lowest index on ties
  int best = 0;
  float bd = fabsf(-1.0f - r);
#pragma unroll
  for (int i = 1; i < 16; ++i) {
    const float d = fabsf(nf4_code_f32(i) - r);
    if (d < bd) {
      bd = d;
      best = i;
    }
  }
  return best;
}

__global__ void __launch_bounds__(kQThreads) quant_nf4_kernel(const void* __restrict__ w, int64_t ldw, int w_dt,
                                                                int64_t k, int seg, int bs, int had, float div,
                                                                int marlin, const int32_t* __restrict__ rowptr,
                                                                const int32_t* __restrict__ ccol,
                                                                uint16_t* __restrict__ cval,
                                                                uint8_t* __restrict__ packed,
                                                                uint16_t* __restrict__ absmax) {
  extern __shared__ float fs[];
  const int64_t segs_per_row = k / seg;
  const int64_t row = blockIdx.x / segs_per_row;
  const int64_t k0 = (blockIdx.x % segs_per_row) * seg;
  for (int i = threadIdx.x; i < seg; i += blockDim.x) fs[i] = load_elem(w, row * ldw + k0 + i, w_dt);
  __syncthreads();
  if (had) fwht_lds(fs, seg / had, had, div);
  // CSR outliers inside this segment: record fp16 value, then zero the position
  if (rowptr != nullptr) {
    const int e0 = rowptr[row], e1 = rowptr[row + 1];
    for (int e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
      const int64_t c = ccol[e];
      if (c >= k0 && c < k0 + seg) cval[e] = f2h(fs[c - k0]);
    }
    __syncthreads();
    for (int e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
      const int64_t c = ccol[e];
      if (c >= k0 && c < k0 + seg) fs[c - k0] = 0.0f;
    }
  }
  __syncthreads();
  // one thread per block: fp16 absmax, nearest codes, packed nibbles
  const int nblk = seg / bs;
  for (int b = threadIdx.x; b < nblk; b += blockDim.x) {
    const float* v = fs + b * bs;
    float m = 0.0f;
    for (int i = 0; i < bs; ++i) m = fmaxf(m, fabsf(v[i]));
    const uint16_t a16 = f2h(m);
    const float a = h2f(a16);
    absmax[row * (k / bs) + (k0 / bs) + b] = a16;
    // a block (>= 32, a multiple of 32) owns the contiguous bytes [kb/2, kb/2 + bs/2)
    // in both nibble layouts, and both nibbles of each of those bytes
    const int64_t kb = k0 + (int64_t)b * bs;
    uint8_t* pb = packed + row * (k / 2) + kb / 2;
    for (int jj = 0; jj < bs / 2; ++jj) {
      const int64_t j = kb / 2 + jj;
      const int elo = (int)(nibble_k(j, 0, marlin) - kb), ehi = (int)(nibble_k(j, 1, marlin) - kb);
      const int qlo = nf4_nearest(a > 0.0f ? v[elo] / a : 0.0f);
      const int qhi = nf4_nearest(a > 0.0f ? v[ehi] / a : 0.0f);
      pb[jj] = (uint8_t)(qlo | (qhi << 4));
    }
  }
}

// The same quantizer in registers for Hadamard and quantization blocks of at most 512 (whole
// blocks inside a wave's 512 elements).  Bound by VALU (about 35 instructions an element; HBM
// needs 2.6 bytes in and out): the transform runs on register bits (1, 2, 4) and across lanes
// (8 .. 256), its division by sqrt(block) and the division by absmax by div_by, the nearest code
// is a table lookup.  The LDS form above (a barrier per stage, one thread per block with 16
// distances an element) took 252 us for 3072 x 8192 bf16, block 128; this one 36 us (64 MB:
// 1.8 TB/s).
//
// Nearest code: as r grows, argmin |C_i - r| in fp32 steps from i to i + 1 at one float each
// (kNf4Step, found by bisection on the float lattice with the same arithmetic).  They lie at
// least 0.08 apart, so each of the bins of width 1/16 holds at most one, and the code of r is
// the bin's base plus (r >= the bin's step).  NaN falls into bin 0 without a step: code 0, as
// the distances' argmin.  |r| <= 1.5 (absmax rounds down by at most that, in fp16 subnormals).
constexpr uint32_t kNf4Step[15] = {0xbf591cd8u, 0xbf1c5270u, 0xbeeb847fu, 0xbeadea76u, 0xbe703cecu,
                                   0xbe0d38bbu, 0xbd3a7870u, 0x3d22fb00u, 0x3df64863u, 0x3e5067e1u,
                                   0x3e9582d5u, 0x3ec753fau, 0x3f006d04u, 0x3f248db0u, 0x3f5c89dau};
constexpr int kNf4Bins = 64;

__global__ void __launch_bounds__(kQThreads) quant_nf4_reg_kernel(
    const void* __restrict__ w, int64_t ldw, int w_dt, int64_t n, int64_t k, int vec, int log_bs, int log_had,
    float div, float inv, int marlin, const int32_t* __restrict__ rowptr, const int32_t* __restrict__ ccol,
    uint16_t* __restrict__ cval, uint8_t* __restrict__ packed, uint16_t* __restrict__ absmax) {
  __shared__ uint32_t step[kNf4Bins], base[kNf4Bins];
  __shared__ __align__(16) float fs[kQWaves][kQSeg];  // outlier segments only
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (tid < kNf4Bins) {
    uint32_t st = 0x7f800000u, bs = 0;  // (no step: +inf)
#pragma unroll
    for (int i = 0; i < 15; ++i) {
      const int bin = (int)(__builtin_bit_cast(float, kNf4Step[i]) * 16.0f + 17.0f);
      if (bin == tid) st = kNf4Step[i];
      if (bin < tid) ++bs;
    }
    step[tid] = st;
    base[tid] = bs;
  }
  __syncthreads();
  const int64_t nseg = (k + kQSeg - 1) / kQSeg, task = (int64_t)blockIdx.x * kQWaves + wv;
  if (task >= n * nseg) return;  // (no barrier below)
  const int64_t row = task / nseg, k0 = (task - row * nseg) * kQSeg;
  const bool in = k0 + 8 * lane < k;  // whole blocks in or out
  float v[8];
  load8(w, row * ldw + (in ? k0 + 8 * lane : 0), w_dt, vec, v);
  if (log_had > 0) {
    // compressor.py:34-39: stages h = 1, 2, 4, ...: (u, v) -> (u + v, u - v) in fp32
#pragma unroll
    for (int lh = 0; lh < 3; ++lh)
      if (lh < log_had) {
        const int h = 1 << lh;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if ((e & h) == 0) {
            const float x0 = v[e], x1 = v[e | h];
            v[e] = x0 + x1;
            v[e | h] = x0 - x1;
          }
      }
    if (log_had > 3) lane_fly<1>(v, lane);
    if (log_had > 4) lane_fly<2>(v, lane);
    if (log_had > 5) lane_fly<4>(v, lane);
    if (log_had > 6) lane_fly<8>(v, lane);
    if (log_had > 7) lane_fly<16>(v, lane);
    if (log_had > 8) lane_fly<32>(v, lane);
    // / sqrt(block) (:40-41)
    float lo = fabsf(v[0]), hi = lo;
#pragma unroll
    for (int e = 1; e < 8; ++e) {
      lo = fminf(lo, fabsf(v[e]));
      hi = fmaxf(hi, fabsf(v[e]));
    }
    if (lo > 0x1p-90f && hi < 0x1p90f) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = div_by(v[e], div, inv);
    } else {  // zeros, NaN and the ends of the range
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] / div;
    }
  }
  // CSR outliers inside this segment: record the fp16 value, then zero the position
  if (rowptr != nullptr) {
    const int e0 = rowptr[row], e1 = rowptr[row + 1];
    float* f = fs[wv];
    bool any = false;
    for (int e = e0 + lane; e < e1 + lane; e += 64) {  // (uniform trip count)
      const int64_t c = e < e1 ? ccol[e] : -1;
      const bool here = c >= k0 && c < k0 + kQSeg && c < k;
      if (__builtin_amdgcn_ballot_w64(here) == 0) continue;
      if (!any) {
        *(float4*)(f + 8 * lane) = make_float4(v[0], v[1], v[2], v[3]);
        *(float4*)(f + 8 * lane + 4) = make_float4(v[4], v[5], v[6], v[7]);
        any = true;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (one wave's LDS operations stay in order)
      if (here) cval[e] = f2h(f[c - k0]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (here) f[c - k0] = 0.0f;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (any) {
      const float4 a = *(const float4*)(f + 8 * lane), b = *(const float4*)(f + 8 * lane + 4);
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
      v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    }
  }
  float m = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(v[e]));
  if (log_bs > 3) m = fmaxf(m, lane_xor<1>(m, lane));
  if (log_bs > 4) m = fmaxf(m, lane_xor<2>(m, lane));
  if (log_bs > 5) m = fmaxf(m, lane_xor<4>(m, lane));
  if (log_bs > 6) m = fmaxf(m, lane_xor<8>(m, lane));
  if (log_bs > 7) m = fmaxf(m, lane_xor<16>(m, lane));
  if (log_bs > 8) m = fmaxf(m, lane_xor<32>(m, lane));
  const uint16_t a16 = f2h(m);
  const float a = h2f(a16), y = 1.0f / a;
  const bool plain = a > 0.0f && a < __builtin_inff();
  uint32_t c03 = 0, c47 = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    // (a value too small for div_by's exactness is far from every step)
    const float r = plain ? div_by(v[e], a, y) : a > 0.0f ? v[e] / a : 0.0f;
    const uint32_t bin = min((uint32_t)fmaxf(__builtin_fmaf(r, 16.0f, 17.0f), 0.0f), (uint32_t)(kNf4Bins - 1));
    const uint32_t q = base[bin] + (r >= __builtin_bit_cast(float, step[bin]) ? 1u : 0u);
    if (e < 4) c03 |= q << (8 * e);
    else c47 |= q << (8 * (e - 4));
  }
  if (!in) return;
  // a 32-run owns bytes [k / 2, k / 2 + 16) in both nibble orders
  uint32_t bytes;
  int64_t o = row * (k / 2) + (k0 + 8 * lane) / 2;  // plain: this lane's four bytes
  if (marlin) {
    bytes = pack_marlin(c03, c47, lane);
    o = row * (k / 2) + (k0 + 8 * (lane & ~3)) / 2 + 8 * (lane & 1) + 2 * (lane & 2);
  } else {
    const uint32_t t0 = c03 | (c03 >> 4), t1 = c47 | (c47 >> 4);  // byte 0 and byte 2 hold the pairs
    bytes = (t0 & 0xffu) | ((t0 >> 8) & 0xff00u) | ((t1 & 0xffu) << 16) | ((t1 << 8) & 0xff000000u);
  }
  uint8_t* dst = packed + o;
  if ((reinterpret_cast<uintptr_t>(dst) & 3) == 0) *(uint32_t*)dst = bytes;
  else
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[e] = (uint8_t)(bytes >> (8 * e));
  if ((8 * lane & ((1 << log_bs) - 1)) == 0) absmax[row * (k >> log_bs) + ((k0 + 8 * lane) >> log_bs)] = a16;
}

// ---------------------------------------------------------------------------
// CSR positions of a boolean mask: per-row counts, their scan into row pointers, the columns.
// One wave per row, 16 mask bytes a lane.  For 3072 x 8192 at 0.5%: 6 + 3 + 9 us (the mask is 25
// MB), where a generic nonzero, bincount, cumsum and casts took about 200 us in 15 launches.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint4 mask16(const uint8_t* row, int64_t c, int64_t k, int vec) {
  if (vec) {  // (any nonzero byte counts, as torch.nonzero)
    const uint4 q = *(const uint4*)(row + c);
    uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      u[e] |= u[e] >> 4;
      u[e] |= u[e] >> 2;
      u[e] = (u[e] | (u[e] >> 1)) & 0x01010101u;
    }
    return make_uint4(u[0], u[1], u[2], u[3]);
  }
  uint32_t w[4] = {0, 0, 0, 0};
  for (int e = 0; e < 16 && c + e < k; ++e) w[e >> 2] |= (uint32_t)(row[c + e] != 0) << (8 * (e & 3));
  return make_uint4(w[0], w[1], w[2], w[3]);
}

__global__ void __launch_bounds__(kQThreads) mask_count_kernel(const uint8_t* __restrict__ mask, int64_t ldm,
                                                                int64_t n, int64_t k, int vec,
                                                                int32_t* __restrict__ counts) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kQWaves + (threadIdx.x >> 6);
  if (row >= n) return;
  const uint8_t* src = mask + row * ldm;
  uint32_t cnt = 0;
  for (int64_t c = 16 * lane; c < k; c += 1024) {
    const uint4 m = mask16(src, c, k, vec);  // bytes 0 or 1
    cnt += __builtin_popcount(m.x) + __builtin_popcount(m.y) + __builtin_popcount(m.z) + __builtin_popcount(m.w);
  }
  for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
  if (lane == 0) counts[row] = (int32_t)cnt;
}

// one workgroup: rowptr[0 .. n] from the counts in rowptr[1 .. n] (in place), 4096 rows a turn
constexpr int kScanThreads = 1024;
__global__ void __launch_bounds__(kScanThreads) mask_scan_kernel(int32_t* __restrict__ rowptr, int64_t n) {
  __shared__ int32_t wsum[kScanThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int32_t carry = 0;
  if (tid == 0) rowptr[0] = 0;
  for (int64_t b = 0; b < n; b += 4 * kScanThreads) {
    int32_t v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t i = b + 4 * tid + e;
      v[e] = i < n ? rowptr[1 + i] : 0;
    }
    v[1] += v[0];
    v[2] += v[1];
    v[3] += v[2];
    int32_t inc = v[3];  // inclusive scan over the wave
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t t = __shfl_up(inc, o, 64);
      if (lane >= o) inc += t;
    }
    if (lane == 63) wsum[wv] = inc;
    __syncthreads();
    int32_t pre = carry + inc - v[3], all = 0;
#pragma unroll
    for (int q = 0; q < kScanThreads / 64; ++q) {
      if (q < wv) pre += wsum[q];
      all += wsum[q];
    }
    carry += all;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t i = b + 4 * tid + e;
      if (i < n) rowptr[1 + i] = pre + v[e];
    }
    __syncthreads();  // (wsum is read before the next turn writes it)
  }
}

__global__ void __launch_bounds__(kQThreads) mask_cols_kernel(const uint8_t* __restrict__ mask, int64_t ldm, int64_t n,
                                                               int64_t k, int vec, const int32_t* __restrict__ rowptr,
                                                               int32_t* __restrict__ col) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kQWaves + (threadIdx.x >> 6);
  if (row >= n) return;
  const uint8_t* src = mask + row * ldm;
  int32_t at = rowptr[row];
  if (rowptr[row + 1] == at) return;  // (uniform in the wave)
  for (int64_t b = 0; b < k; b += 1024) {
    const int64_t c = b + 16 * lane;
    const uint4 m = c < k ? mask16(src, c, k, vec) : make_uint4(0, 0, 0, 0);
    const uint32_t w[4] = {m.x, m.y, m.z, m.w};
    const int32_t cnt = __builtin_popcount(m.x) + __builtin_popcount(m.y) + __builtin_popcount(m.z) +
                        __builtin_popcount(m.w);
    int32_t inc = cnt;
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t t = __shfl_up(inc, o, 64);
      if (lane >= o) inc += t;
    }
    int32_t dst = at + inc - cnt;
    if (cnt > 0)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        for (uint32_t x = w[q]; x != 0; x &= x - 1) col[dst++] = (int32_t)(c + 4 * q + (__builtin_ctz(x) >> 3));
    at += __shfl(inc, 63, 64);
  }
}

}  // namespace spectra

using namespace spectra;

// 16-byte aligned rows
static int rows_aligned(const void* w, int64_t ldw, int dt) {
  return reinterpret_cast<uintptr_t>(w) % 16 == 0 && (ldw * elem_size(dt)) % 16 == 0;
}

static int ilog2(int64_t v) {
  int l = 0;
  while ((int64_t(1) << l) < v) ++l;
  return l;
}

static int fwht_seg(int64_t k, int b) {
  // largest segment <= 4096 elements made of whole blocks and dividing k
  int64_t seg = b;
  while (seg * 2 <= 4096 && k % (seg * 2) == 0) seg *= 2;
  return (int)seg;
}

extern "C" int spectra_fwht_rows(const void* x, int64_t ldx, int32_t in_dtype, int64_t rows, int64_t k,
                                 int32_t block, void* out, int64_t ldo, int32_t out_dtype,
                                 spectra_stream_t stream) {
  SPECTRA_REQUIRE(x && out, "NULL pointer");
  SPECTRA_REQUIRE(rows > 0 && k > 0, "rows and k must be positive");
  SPECTRA_REQUIRE(is_pow2(block) && block >= 2 && block <= 1024 && k % block == 0,
                  "block must be a power of two in [2, 1024] dividing k");
  SPECTRA_REQUIRE(in_dtype >= SPECTRA_F16 && in_dtype <= SPECTRA_F32 && out_dtype >= SPECTRA_F16 &&
                      out_dtype <= SPECTRA_F32, "bad dtype");
  SPECTRA_REQUIRE(ldx >= k && ldo >= k, "row stride smaller than k");
  const int seg = fwht_seg(k, block);
  const int64_t grid = rows * (k / seg);
  SPECTRA_REQUIRE(grid < (1LL << 31), "too many rows");
  const float div = (float)std::sqrt((double)block);
  hipLaunchKernelGGL(fwht_rows_kernel, dim3((unsigned)grid), dim3(kQThreads), seg * sizeof(float),
                     (hipStream_t)stream, x, ldx, (int)in_dtype, out, ldo, (int)out_dtype, k, (int)block, seg,
                     div);
  SPECTRA_HIP_CHECK(hipGetLastError());
  return SPECTRA_OK;
}

extern "C" int spectra_quantize_group32(const void* w, int64_t ldw, int32_t w_dtype, int64_t n, int64_t k,
                                        int32_t group_size, const int64_t* outlier_idx, int32_t n_out,
                                        uint8_t* packed, uint16_t* scales, uint8_t* packed_zeros,
                                        spectra_stream_t stream) {
  if (group_size != 32)  // compressor.py:53-54
    return fail(SPECTRA_ERR_INVALID, "SPECTRA currently requires group_size=32 (Group-32 microscales)");
  SPECTRA_REQUIRE(w && packed && scales && packed_zeros, "NULL pointer");
  SPECTRA_REQUIRE(n > 0 && k > 0 && k % 32 == 0, "k must be a positive multiple of 32");
  SPECTRA_REQUIRE(ldw >= k, "row stride smaller than k");
  SPECTRA_REQUIRE(w_dtype >= SPECTRA_F16 && w_dtype <= SPECTRA_F32, "bad dtype");
  SPECTRA_REQUIRE(outlier_idx == nullptr || n_out > 0, "n_out must be positive with outlier_idx");
  SPECTRA_REQUIRE((n + kQRows - 1) / kQRows < (1LL << 31), "matrix too large");
  const int vec = rows_aligned(w, ldw, w_dtype);
  // (the grid's y dimension holds 65535 blocks: more rows run as further launches)
  for (int64_t r0 = 0; r0 < n; r0 += 65535 * (int64_t)kQRows) {
    const int64_t nr = std::min(n - r0, 65535 * (int64_t)kQRows);
    hipLaunchKernelGGL(quant_g32_kernel,
                       dim3((unsigned)((k + kQSeg * kQWaves - 1) / (kQSeg * kQWaves)),
                            (unsigned)((nr + kQRows - 1) / kQRows)),
                       dim3(kQThreads), 0, (hipStream_t)stream,
                       (const void*)((const uint8_t*)w + r0 * ldw * elem_size(w_dtype)), ldw, (int)w_dtype, nr, k, vec,
                       outlier_idx, outlier_idx ? n_out : 0, packed + r0 * (k / 2), scales + r0 * (k / 32),
                       packed_zeros + r0 * ((k / 32 + 1) / 2));
    SPECTRA_HIP_CHECK(hipGetLastError());
  }
  SPECTRA_HIP_CHECK(hipGetLastError());
  return SPECTRA_OK;
}

extern "C" int spectra_quantize_nf4(const void* w, int64_t ldw, int32_t w_dtype, int64_t n, int64_t k,
                                    int32_t blocksize, int32_t hadamard_block, int32_t marlin_layout,
                                    const int32_t* csr_rowptr, const int32_t* csr_col, uint16_t* csr_val,
                                    uint8_t* packed, uint16_t* absmax, spectra_stream_t stream) {
  SPECTRA_REQUIRE(w && packed && absmax, "NULL pointer");
  SPECTRA_REQUIRE(n > 0 && k > 0, "n and k must be positive");
  SPECTRA_REQUIRE(is_pow2(blocksize) && blocksize >= 32 && k % blocksize == 0,
                  "blocksize must be a power of two >= 32 dividing k");
  SPECTRA_REQUIRE(hadamard_block == 0 || (is_pow2(hadamard_block) && hadamard_block >= 2 &&
                                          hadamard_block <= 1024 && k % hadamard_block == 0),
                  "hadamard_block must be 0 or a power of two in [2, 1024] dividing k");
  SPECTRA_REQUIRE(ldw >= k, "row stride smaller than k");
  SPECTRA_REQUIRE(w_dtype >= SPECTRA_F16 && w_dtype <= SPECTRA_F32, "bad dtype");
  SPECTRA_REQUIRE((csr_rowptr == nullptr) == (csr_col == nullptr) && (csr_rowptr == nullptr) == (csr_val == nullptr),
                  "CSR rowptr/col/val must be given together");
  const float div = hadamard_block ? (float)std::sqrt((double)hadamard_block) : 1.0f;
  if (blocksize <= kQSeg && hadamard_block <= kQSeg) {
    const int64_t tasks = n * ((k + kQSeg - 1) / kQSeg), wgs = (tasks + kQWaves - 1) / kQWaves;
    SPECTRA_REQUIRE(wgs < (1LL << 31), "matrix too large");
    hipLaunchKernelGGL(quant_nf4_reg_kernel, dim3((unsigned)wgs), dim3(kQThreads), 0, (hipStream_t)stream, w, ldw,
                       (int)w_dtype, n, k, rows_aligned(w, ldw, w_dtype), ilog2(blocksize),
                       hadamard_block ? ilog2(hadamard_block) : 0, div, 1.0f / div, (int)marlin_layout, csr_rowptr,
                       csr_col, csr_val, packed, absmax);
    SPECTRA_HIP_CHECK(hipGetLastError());
    return SPECTRA_OK;
  }
  // segment: whole rows up to 8192 elements, otherwise the largest power-of-two
  // multiple of max(blocksize, hadamard_block) dividing k
  int64_t unit = blocksize > hadamard_block ? blocksize : hadamard_block;
  int64_t seg = unit;
  while (seg * 2 <= 8192 && k % (seg * 2) == 0) seg *= 2;
  if (k <= 8192) seg = k;
  SPECTRA_REQUIRE(k % seg == 0 && seg % unit == 0, "unsupported k for the NF4 quantizer");
  const int64_t grid = n * (k / seg);
  SPECTRA_REQUIRE(grid < (1LL << 31), "matrix too large");
  hipLaunchKernelGGL(quant_nf4_kernel, dim3((unsigned)grid), dim3(kQThreads), seg * sizeof(float),
                     (hipStream_t)stream, w, ldw, (int)w_dtype, k, (int)seg, (int)blocksize, (int)hadamard_block,
                     div, (int)marlin_layout, csr_rowptr, csr_col, csr_val, packed, absmax);
  SPECTRA_HIP_CHECK(hipGetLastError());
  return SPECTRA_OK;
}

extern "C" int spectra_mask_rowptr(const uint8_t* mask, int64_t ldm, int64_t n, int64_t k, int32_t* rowptr,
                                   spectra_stream_t stream) {
  SPECTRA_REQUIRE(mask && rowptr, "NULL pointer");
  SPECTRA_REQUIRE(n > 0 && k > 0 && ldm >= k, "n and k must be positive, the row stride at least k");
  SPECTRA_REQUIRE(n < (1LL << 31), "too many rows");
  const int vec = reinterpret_cast<uintptr_t>(mask) % 16 == 0 && ldm % 16 == 0 && k % 16 == 0;
  hipLaunchKernelGGL(mask_count_kernel, dim3((unsigned)((n + kQWaves - 1) / kQWaves)), dim3(kQThreads), 0,
                     (hipStream_t)stream, mask, ldm, n, k, vec, rowptr + 1);
  SPECTRA_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(mask_scan_kernel, dim3(1), dim3(kScanThreads), 0, (hipStream_t)stream, rowptr, n);
  SPECTRA_HIP_CHECK(hipGetLastError());
  return SPECTRA_OK;
}

extern "C" int spectra_mask_columns(const uint8_t* mask, int64_t ldm, int64_t n, int64_t k, const int32_t* rowptr,
                                    int32_t* col, spectra_stream_t stream) {
  SPECTRA_REQUIRE(mask && rowptr && col, "NULL pointer");
  SPECTRA_REQUIRE(n > 0 && k > 0 && ldm >= k, "n and k must be positive, the row stride at least k");
  SPECTRA_REQUIRE(n < (1LL << 31), "too many rows");
  const int vec = reinterpret_cast<uintptr_t>(mask) % 16 == 0 && ldm % 16 == 0 && k % 16 == 0;
  hipLaunchKernelGGL(mask_cols_kernel, dim3((unsigned)((n + kQWaves - 1) / kQWaves)), dim3(kQThreads), 0,
                     (hipStream_t)stream, mask, ldm, n, k, vec, rowptr, col);
  SPECTRA_HIP_CHECK(hipGetLastError());
  return SPECTRA_OK;
}
