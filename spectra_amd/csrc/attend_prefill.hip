// Causal prefill attention of a Llama-shaped layer on the matrix cores (the reference runs the
// prompt through the model's own attention, engine.py:1387-1415 keeps its static cache):
//   out[t, h, :] = softmax(q[t, h] . K[0 .. p]^T / sqrt(hd)) . V[0 .. p],  p = pos[t]
// for rotated queries q [T, heads, hd] and the caches K, V [kv_heads, max_seq, hd], whose first
// `keys` positions are filled, fp16 with fp32 scores, softmax and sums.
//
// The work is small (777 tokens, 24 heads of 128: 3.7 GFLOP causal, 3 us of MFMA); as separate
// products it moved the scores eleven times through memory (225 us a layer at 777 tokens, seven
// of the launches elementwise).  Here they stay in registers: 777 tokens 23 us, 2040
// tokens 59 us.
//
// A workgroup of 4 waves owns 64 queries of one head: waves = 2 query halves of 32 x 2 halves of
// each 128-key step, so the longest row's chain of steps is half as long; the key halves meet in
// LDS at the end.  Scores are computed transposed, S^T = K . Q^T (v_mfma_f32_32x32x16_f16: K rows
// as A, the lane's query as B), so a lane holds 16 keys of one query per tile: maxima and sums
// cross only to the lane 32 away, and the exponentials are already the B operand of
// O^T = V^T . P^T when the contraction takes the keys in the accumulator's order (4 g + 0 .. 3,
// 8 + 4 g + 0 .. 3 of each 16).  V is transposed on its way into LDS.  The next step's rows
// are loaded into registers while this one computes.  Query tiles run longest first.
#include "common.h"

namespace spectra {

typedef _Float16 p8h_t __attribute__((ext_vector_type(8)));
typedef uint32_t p4u_t __attribute__((ext_vector_type(4)));
typedef float p16f_t __attribute__((ext_vector_type(16)));

constexpr int kPfThreads = 256, kPfQ = 64, kPfKeys = 128;
constexpr int kPfVRow = 264;  // bytes of a transposed V row (128 keys, padded: conflict-free 8-byte reads)

template <int HD>
__global__ void __launch_bounds__(kPfThreads, 2) attend_prefill_kernel(const uint16_t* __restrict__ q,
                                                                       const uint16_t* __restrict__ kc,
                                                                       const uint16_t* __restrict__ vc,
                                                                       const int64_t* __restrict__ pos, int T, int L,
                                                                       int heads, int kv_heads, int lmax, float scale2,
                                                                       uint16_t* __restrict__ out) {
  constexpr int CH = HD / 8, DT = HD / 32, KS = HD / 16;  // 16-byte chunks, 32-dim tiles, 16-dim steps
  constexpr int KL = kPfKeys * CH / kPfThreads;           // K chunks a thread copies
  constexpr int VL = 32 * CH / kPfThreads;                // (4 keys x 8 dims) pieces of V
  __shared__ __align__(16) uint8_t ks[kPfKeys * HD * 2];
  __shared__ __align__(16) uint8_t vs[HD * kPfVRow];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int qh = wave & 1, kh = wave >> 1, g = lane >> 5, ln = lane & 31;
  const int h = blockIdx.x, kvh = h / (heads / kv_heads);
  const int q0 = (gridDim.y - 1 - blockIdx.y) * kPfQ;
  const int qi = q0 + 32 * qh + ln;
  // last key of every query of the tile, of this wave's 32 (its first too) and of this lane's
  const int pl = (int)min(max(pos[min(q0 + lane, T - 1)], (int64_t)-1), (int64_t)L - 1);
  int hi = pl, lo = pl;
#pragma unroll
  for (int x = 16; x > 0; x >>= 1) {
    hi = max(hi, __shfl_xor(hi, x, 64));
    lo = min(lo, __shfl_xor(lo, x, 64));
  }
  const int qlast = __builtin_amdgcn_readfirstlane(max(hi, __shfl_xor(hi, 32, 64)));
  const int wlast = __builtin_amdgcn_readlane(hi, 32 * qh), wfirst = __builtin_amdgcn_readlane(lo, 32 * qh);
  const int qp = __shfl(pl, 32 * qh + ln, 64);
  const uint16_t* kb = kc + (int64_t)kvh * lmax * HD;
  const uint16_t* vb = vc + (int64_t)kvh * lmax * HD;
  // the lane's query, B operand of step s: dims 16 s + 8 g ..
  p8h_t qf[KS];
  const uint16_t* qrow = q + ((int64_t)min(qi, T - 1) * heads + h) * HD + 8 * g;
#pragma unroll
  for (int s = 0; s < KS; ++s) qf[s] = *(const p8h_t*)(qrow + 16 * s);

  p4u_t kr[KL], vr[VL][4];
  auto load = [&](int k0) __attribute__((always_inline)) {  // rows past the last key: its row (masked)
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      const int c = tid + i * kPfThreads;
      kr[i] = *(const p4u_t*)(kb + (int64_t)min(k0 + c / CH, L - 1) * HD + 8 * (c % CH));
    }
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int t = tid + i * kPfThreads, kq = t & 31, o = t >> 5;
#pragma unroll
      for (int j = 0; j < 4; ++j) vr[i][j] = *(const p4u_t*)(vb + (int64_t)min(k0 + 4 * kq + j, L - 1) * HD + 8 * o);
    }
  };
  auto store = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      const int c = tid + i * kPfThreads, key = c / CH;
      *(p4u_t*)(ks + key * (HD * 2) + 16 * ((c % CH) ^ (key & (CH - 1)))) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int t = tid + i * kPfThreads, kq = t & 31, o = t >> 5;
#pragma unroll
      for (int e = 0; e < 8; ++e) {  // dim 8 o + e of the four keys
        const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
        const uint2 w = make_uint2(__builtin_amdgcn_perm(vr[i][1][e >> 1], vr[i][0][e >> 1], sel),
                                   __builtin_amdgcn_perm(vr[i][3][e >> 1], vr[i][2][e >> 1], sel));
        *(uint2*)(vs + (8 * o + e) * kPfVRow + 8 * kq) = w;
      }
    }
  };

  p16f_t o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
  float m = -INFINITY, l = 0.0f;  // running maximum (of scores in log2 units) and sum
  load(0);
  for (int k0 = 0; k0 <= qlast; k0 += kPfKeys) {
    __syncthreads();  // (the last step's reads are done)
    store();
    __syncthreads();
    if (k0 + kPfKeys <= qlast) load(k0 + kPfKeys);
    const int kw = k0 + 64 * kh;  // this wave's 64 keys
    if (kw > wlast) continue;     // (uniform in the wave; no barrier below)
    p16f_t s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[t][r] = 0.0f;
      const int key = 64 * kh + 32 * t + ln;
#pragma unroll
      for (int st = 0; st < KS; ++st) {
        const p8h_t kf = *(const p8h_t*)(ks + key * (HD * 2) + 16 * ((2 * st + g) ^ (key & (CH - 1))));
        s[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[st], s[t], 0, 0, 0);
      }
    }
    // score r of tile t: key kw + 32 t + 8 (r / 4) + 4 g + r % 4
    float mn = m;
    if (kw + 63 > wfirst) {  // the causal edge crosses this tile
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (kw + 32 * t + 8 * (r >> 2) + 4 * g + (r & 3) > qp) s[t][r] = -INFINITY;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) mn = fmaxf(mn, s[t][r] * scale2);
    mn = fmaxf(mn, lane_xor<32>(mn, lane));
    const float mu = mn == -INFINITY ? 0.0f : mn;  // (a query with no key in its tiles yet)
    const float corr = __builtin_amdgcn_exp2f(m - mu);
    m = mn;
    float add = 0.0f;
    p8h_t pf[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][r], scale2, -mu));
        add += e;
        pf[t][r >> 3][r & 7] = (_Float16)e;
      }
    l = l * corr + (add + lane_xor<32>(add, lane));
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[d][r] *= corr;
    // O^T += V^T . P^T: step (t, u) contracts keys 32 t + 16 u + {4 g + 0 .. 3, 8 + 4 g + 0 .. 3}
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const uint8_t* vrow = vs + (32 * d + ln) * kPfVRow + 2 * (64 * kh + 4 * g);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint2 a = *(const uint2*)(vrow + 2 * (32 * t + 16 * u)), b = *(const uint2*)(vrow + 2 * (32 * t + 16 * u + 8));
          const p4u_t w = {a.x, a.y, b.x, b.y};
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(p8h_t, w), pf[t][u], o[d], 0, 0, 0);
        }
    }
  }

  // the key halves meet: half 1 leaves its sums, half 0 merges and writes
  __syncthreads();
  float* red = (float*)vs;       // [2 query halves][64 lanes][DT * 16]: in pieces of one 32-dim tile
  float* ml = (float*)ks;        // [2][64][2]
  if (kh == 1) {
    ml[(qh * 64 + lane) * 2] = m;
    ml[(qh * 64 + lane) * 2 + 1] = l;
  }
  float c0 = 1.0f, c1 = 0.0f;
#pragma unroll
  for (int d = 0; d < DT; ++d) {
    if (kh == 1)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *(float4*)(red + ((qh * 4 + r) * 64 + lane) * 4) =
            make_float4(o[d][4 * r], o[d][4 * r + 1], o[d][4 * r + 2], o[d][4 * r + 3]);
    __syncthreads();
    if (kh == 0) {
      if (d == 0) {  // half 0 has key 0: its maximum is finite, or NaN and the row with it (no keys: NaN)
        const float m1 = ml[(qh * 64 + lane) * 2], l1 = ml[(qh * 64 + lane) * 2 + 1];
        const float mm = fmaxf(m, m1);
        const float a0 = __builtin_amdgcn_exp2f(m - mm), a1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - mm);
        const float inv = 1.0f / (l * a0 + l1 * a1);
        c0 = a0 * inv;
        c1 = a1 * inv;
      }
      if (qi < T) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {  // dims 32 d + 8 r + 4 g + 0 .. 3
          const float4 x = *(const float4*)(red + ((qh * 4 + r) * 64 + lane) * 4);
          const uint32_t w0 = (uint32_t)f2h(o[d][4 * r] * c0 + x.x * c1) |
                              ((uint32_t)f2h(o[d][4 * r + 1] * c0 + x.y * c1) << 16);
          const uint32_t w1 = (uint32_t)f2h(o[d][4 * r + 2] * c0 + x.z * c1) |
                              ((uint32_t)f2h(o[d][4 * r + 3] * c0 + x.w * c1) << 16);
          *(uint2*)(out + ((int64_t)qi * heads + h) * HD + 32 * d + 8 * r + 4 * g) = make_uint2(w0, w1);
        }
      }
    }
    __syncthreads();
  }
}

}  // namespace spectra

using namespace spectra;

extern "C" int spectra_attend_prefill(const void* q, const int64_t* pos, int64_t tokens, int64_t keys, int32_t heads, int32_t kv_heads,
                                      int32_t head_dim, int32_t max_seq, const void* k_cache, const void* v_cache,
                                      void* out, spectra_stream_t stream) {
  SPECTRA_REQUIRE(q && pos && k_cache && v_cache && out, "NULL pointer");
  SPECTRA_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "heads must be a multiple of kv_heads");
  SPECTRA_REQUIRE(tokens > 0 && keys > 0 && keys <= max_seq, "tokens must be positive, keys in [1, max_seq]");
  SPECTRA_REQUIRE(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_cache) |
                    reinterpret_cast<uintptr_t>(v_cache) | reinterpret_cast<uintptr_t>(out)) % 16) == 0,
                  "operands must be 16-byte aligned");
  if (head_dim != 64 && head_dim != 128) return fail(SPECTRA_ERR_UNSUPPORTED, "head_dim must be 64 or 128");
  const int64_t tiles = (tokens + kPfQ - 1) / kPfQ;
  if (tiles > 65535) return fail(SPECTRA_ERR_UNSUPPORTED, "too many tokens");
  // scores in log2 units: log2(e) / sqrt(head_dim)
  const float scale2 = (float)(1.4426950408889634 / (head_dim == 64 ? 8.0 : 11.313708498984761));
  const void* kern = head_dim == 64 ? (const void*)attend_prefill_kernel<64> : (const void*)attend_prefill_kernel<128>;
  int T = (int)tokens, L = (int)keys;
  void* args[] = {(void*)&q, (void*)&k_cache, (void*)&v_cache, (void*)&pos, (void*)&T, (void*)&L, (void*)&heads, (void*)&kv_heads,
                  (void*)&max_seq, (void*)&scale2, (void*)&out};
  SPECTRA_HIP_CHECK(hipLaunchKernel(kern, dim3((unsigned)heads, (unsigned)tiles), dim3(kPfThreads), args, 0,
                                    (hipStream_t)stream));
  SPECTRA_HIP_CHECK(hipGetLastError());
  return SPECTRA_OK;
}
