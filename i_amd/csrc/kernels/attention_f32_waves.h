// FlashAttention forward for f32 inputs (full f32 arithmetic) on gfx950, for grids that give a CU little to do: a
// workgroup takes 16 query rows and its wavefronts take a part of the keys each.
//
// The kernels of attention_f32_direct.h give a workgroup 128 query rows: one head of 512 is 4 workgroups, every
// wavefront walks all keys, and a trip of 32 keys is a serial chain of 2.7 us (4.7 at d = 128).  Here the chain of a
// wavefront is an NW-th of the keys, a head of 512 is 32 workgroups, and the parts meet in LDS instead of in a second
// launch.  Bound by the matrix instructions of the CUs that have a workgroup (64 to 70 % of their rate) and the 4 to 7 us
// of launch, first loads and the end.  Before -> now, us: 512 x 64, one head 15.6 -> 9.6; 145 x 128 28 -> 10.4; 16 heads of 512 x
// 64 24.4 -> 16; 48 of 700 x 64 107 -> 71; one head of 1024 x 128 29 -> 17; 64 of 16 queries, 1000 keys of 128 45 -> 19.
//
//   matrix          v_mfma_f32_16x16x4_f32, S^T = K Q^T and O^T = V^T P^T: lane (c, g) = (lane % 16, lane / 16) holds query c
//                   and, of a block of 16 keys, the scores of keys 4 g + i in element i of the accumulator, which is what
//                   MFMA i of the second product takes as its B operand (its four k are the keys {4 g + i})
//   K, V            from global memory (L2) straight into the registers of the wavefront that needs them, nothing is shared:
//                   16 bytes per lane.  K: chunk 4 s + g of key c, element e feeds MFMA e of group s, so that the
//                   contraction runs over d in the order the Q operand follows.  V: chunk 16 u + c of key 4 g + i; element
//                   e feeds output tile 4 u + e, whose row r is column 64 u + 4 r + e of O.
//   Q               in LDS, in operand order: one conflict-free 16-byte read per four MFMAs and block of keys
//   pipeline        V of a step is requested before its scores are computed, K of the next one before its output product
//   end             every wavefront leaves (max, sum) of its rows and its O, rescaled to the workgroup's max, in LDS; all add
//                   them up in wavefront order
//
// p.kv_splits > 1: the keys also split over workgroups, as in the other kernels (`head` counts (head, part) pairs).
// PADDED: d = p.d and dv = p.dv are any multiples of 4 up to DPAD.  Chunks past the end of a row repeat its last one: the
// contraction clears them, and the output columns they reach are not stored.
#pragma once
#include "common.h"
#include "params.h"

// Both of two neighbouring groups of 16 lanes hold the larger / the sum of their values; as both_halves for 32 lanes.
__device__ __forceinline__ void both_quarters(float x, float& lo, float& hi) {
  float a = x, b = x;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  lo = a;
  hi = b;
}
__device__ __forceinline__ float quarters_max(float x) {
  float lo, hi;
  both_quarters(x, lo, hi);
  return half_max(fmaxf(lo, hi));
}
__device__ __forceinline__ float quarters_sum(float x) {
  float lo, hi;
  both_quarters(x, lo, hi);
  return half_sum(lo + hi);
}

template <int DPAD, int NW, bool PADDED>
__device__ __forceinline__ void attn_fwd_f32_waves_body(const AttnParams& p) {
  constexpr int BM = 16;
  constexpr int KB = 2;          // blocks of 16 keys per step
  constexpr int BN = 16 * KB;
  constexpr int G = DPAD / 16;   // 16-byte chunks of K and Q per lane and row: 16 d each over the four lane groups
  constexpr int U = DPAD / 64;   // 16-byte chunks of V per lane and row: 64 columns each over the 16 lanes
  constexpr int SLOTS = U * 4 * 64;  // 16-byte pieces of a wavefront's O
  __shared__ __attribute__((aligned(16))) f32x4 q_lds[G * 64];
  __shared__ __attribute__((aligned(16))) f32x4 o_lds[NW * SLOTS];
  __shared__ float ml_lds[2][NW][BM];

  uint32_t head, qt;
  xcd_map(blockIdx.x, p.nqt, p.bh, head, qt);
  if (head >= p.bh) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t c = lane & 15, g = lane >> 4;
  const uint32_t d = PADDED ? p.d : (uint32_t)DPAD, dv = PADDED ? p.dv : (uint32_t)DPAD;
  const uint32_t chunks = d / 4, chunks_v = dv / 4;

  uint32_t qhead = head, part_first = 0, nk = p.nk;
  if (p.kv_splits > 1) {
    qhead = head / p.kv_splits;
    part_first = (head - qhead * p.kv_splits) * p.kv_chunk;
    nk = p.nk - part_first < p.kv_chunk ? p.nk - part_first : p.kv_chunk;
  }
  // this wavefront's keys: first .. end (none where the part has fewer steps than wavefronts)
  const uint32_t chunk = (nk + NW * BN - 1) / (NW * BN) * BN;
  const uint32_t first = wave * chunk, end = first >= nk || nk - first < chunk ? nk : first + chunk;

  const float* __restrict__ Q = reinterpret_cast<const float*>(p.q) + (size_t)qhead * p.nq * d;
  const char* __restrict__ K = reinterpret_cast<const char*>(p.k) + ((size_t)qhead * p.nk + part_first) * d * 4;
  const char* __restrict__ V = reinterpret_cast<const char*>(p.v) + ((size_t)qhead * p.nk + part_first) * dv * 4;
  const float scale_raw = load_scale(p.scale_ptr, p.scale_value);
  const float qsign = scale_raw < 0.0f ? -1.0f : 1.0f;  // negative scale folded into Q (exact)
  const float scale_log2 = fabsf(scale_raw) * I_LOG2_E32;

  // rows past the end of the keys repeat the last one; their scores are masked and their V is cleared
  f32x4 kf[KB][G], vf[KB][4][U];
  auto load_k = [&](uint32_t key0) {
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      const uint32_t key = key0 + 16 * b + c, row = (key < nk ? key : nk - 1) * d * 4;
#pragma unroll
      for (int s = 0; s < G; ++s) {
        if (PADDED && 16u * s >= d) break;
        const uint32_t chunk = !PADDED || 4 * s + g < chunks ? 4 * s + g : chunks - 1;
        kf[b][s] = *reinterpret_cast<const f32x4*>(K + (row + 16 * chunk));
      }
    }
  };
  auto load_v = [&](uint32_t key0) {
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t key = key0 + 16 * b + 4 * g + i, row = (key < nk ? key : nk - 1) * dv * 4;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t chunk = !PADDED || 16 * u + c < chunks_v ? 16 * u + c : chunks_v - 1;
          vf[b][i][u] = *reinterpret_cast<const f32x4*>(V + (row + 16 * chunk));
        }
      }
  };
  if (first < end) load_k(first);

  for (uint32_t at = tid; at < G * 64; at += 64 * NW) {
    const uint32_t row = qt * BM + (at & 15), chunk = 4 * (at >> 6) + ((at >> 4) & 3);
    f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
    if (row < p.nq && chunk < chunks) z = *reinterpret_cast<const f32x4*>(Q + (size_t)row * d + 4 * chunk);
    q_lds[at] = z * qsign;
  }
  f32x4 o[4 * U];
#pragma unroll
  for (int t = 0; t < 4 * U; ++t) o[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = -INFINITY, l_run = 0.0f;
  __syncthreads();

  for (uint32_t key0 = first; key0 < end; key0 += BN) {
    load_v(key0);
    f32x4 sc[KB];
#pragma unroll
    for (int b = 0; b < KB; ++b) sc[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t from = lane;
    asm volatile("" : "+v"(from));  // (Q is read again for every step rather than held in 4 G registers)
#pragma unroll
    for (int s = 0; s < G; ++s) {
      if (PADDED && 16u * s >= d) break;
      const f32x4 q = q_lds[s * 64 + from];
      if (PADDED && 16u * s + 16 > d) {
#pragma unroll
        for (int b = 0; b < KB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) kf[b][s][e] = 4 * s + g < chunks ? kf[b][s][e] : 0.0f;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < KB; ++b) sc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b][s][e], q[e], sc[b], 0, 0, 0);
    }
    if (key0 + BN < end) load_k(key0 + BN);

    const bool masked = key0 + BN > end;
    if (masked) {
#pragma unroll
      for (int b = 0; b < KB; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool out = key0 + 16 * b + 4 * g + i >= end;
          sc[b][i] = out ? -INFINITY : sc[b][i];
#pragma unroll
          for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) vf[b][i][u][e] = out ? 0.0f : vf[b][i][u][e];
        }
    }
    float mx = sc[0][0];
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sc[b][i]);
    const float m_new = fmaxf(m_run, quarters_max(mx));
    const float alpha = m_run == -INFINITY ? 0.0f : fast_exp2((m_run - m_new) * scale_log2);
    // The difference is taken before the product with the scale: a score near the lowest f32 times the scale is infinite or
    // far from what the rounded product of the maximum cancels, and a step of nothing but such scores would sum to infinity,
    // which its weight of 0 in the end makes NaN.  (-inf: a step of nothing else weighs nothing.)
    const float m_from = m_new == -INFINITY ? 0.0f : m_new;
    m_run = m_new;
    float psum = 0.0f;
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float e = fast_exp2((sc[b][i] - m_from) * scale_log2);
        // spelled out rather than left to exp(-inf): a zero scale turns the masked score into 0 * inf
        if (masked && key0 + 16 * b + 4 * g + i >= end) e = 0.0f;
        sc[b][i] = e;
        psum += e;
      }
    l_run = l_run * alpha + psum;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
      for (int t = 0; t < 4 * U; ++t) o[t] *= alpha;
    }
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < 4 * U; ++t)
          o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[b][i][t / 4][t % 4], sc[b][i], o[t], 0, 0, 0);
  }

  // ---- the parts put together.  o[4 u + e][j] is O[c][64 u + 16 g + 4 j + e].
  const float sum = quarters_sum(l_run);
  if (g == 0) {
    ml_lds[0][wave][c] = m_run;
    ml_lds[1][wave][c] = sum;
  }
  __syncthreads();
  float top = ml_lds[0][0][c];
#pragma unroll
  for (int w = 1; w < NW; ++w) top = fmaxf(top, ml_lds[0][w][c]);
  float total = 0.0f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float m = ml_lds[0][w][c];
    total += (m == -INFINITY ? 0.0f : fast_exp2((m - top) * scale_log2)) * ml_lds[1][w][c];
  }
  // (A part over workgroups that sums to nothing, its scores all -inf, leaves O = 0 beside its lse of -inf: the merge weighs it
  // with 0, and a NaN would survive that.  Without parts, or with all of them so, the row is NaN.)
  const float divisor = p.kv_splits > 1 && total == 0.0f ? 1.0f : total;
  const float weight = (m_run == -INFINITY ? 0.0f : fast_exp2((m_run - top) * scale_log2)) / divisor;
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = o[4 * u + e][j] * weight;
      o_lds[wave * SLOTS + (u * 4 + j) * 64 + lane] = w;
    }
  if (p.kv_splits > 1 && tid < BM && qt * BM + tid < p.nq) p.lse[(size_t)head * p.nq + qt * BM + tid] = top * scale_log2 + log2f(total);
  __syncthreads();
  float* __restrict__ O = reinterpret_cast<float*>(p.o) + (size_t)head * p.nq * dv;
  for (uint32_t at = tid; at < SLOTS; at += 64 * NW) {
    const uint32_t row = at / (16 * U), chunk = at % (16 * U);  // 16 bytes of a row of O
    const uint32_t slot = ((chunk >> 4) * 4 + (chunk & 3)) * 64 + 16 * ((chunk & 15) >> 2) + row;
    f32x4 w = o_lds[slot];
#pragma unroll
    for (int n = 1; n < NW; ++n) w += o_lds[n * SLOTS + slot];
    if (qt * BM + row < p.nq && chunk < chunks_v) *reinterpret_cast<f32x4*>(O + (size_t)(qt * BM + row) * dv + 4 * chunk) = w;
  }
}
