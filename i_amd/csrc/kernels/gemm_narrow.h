// C[m,n] = sum_k A[m,k] * B[n,k]  (NN: B[k,n]) for a few rows of A, sums in f32: a layer applied to a few rows.  f32
// operands (NT up to 32 rows, NN up to 64) and, for small B, bf16 ones (NT, up to 16 rows).  Bound by HBM: B is read
// once and each of its elements meets at most 64 products.
//
// The tiled kernels serve such a product badly: 128 rows of LDS and of matrix instructions for m rows, B taken
// through LDS though nobody shares it, few workgroups, hence the k loop in parts and a second launch to add them up,
// and for f32 NN a transposed copy of B first.  Here B goes from memory straight into the registers of the one
// wavefront that needs it, many loads in flight, and a workgroup's W wavefronts take every W-th piece of k of the
// same columns; their sums meet in LDS at the end.  Measured, before -> now: f32 NN 16 x 9808 x 4288 198 -> 41 us
// (4.1 TB/s), 64 x 8192 x 8192 256 -> 133 (the f32 matrix rate), 1 x 16384 x 1024 73 -> 14; f32 NT 16 x 8192 x 8192
// 128 -> 66, 3 x 1688 x 8896 44 -> 21 (in 4 parts of k); bf16 NT 7 x 8040 x 1296 15.0 -> 11.8.
//
//   matrix      v_mfma_f32_16x16x32_bf16 / 16x16x4_f32, B's columns of C as the first operand and A's rows as the
//               second: a lane ends up with C[m = lane % 16][4 columns]
//   NT          lane (c, g) = (lane % 16, lane / 16) loads 16 bytes of row c of B at k = KV g (KV elements), which
//               is the bf16 instruction's operand; element e of it (f32) feeds matrix instruction e, whose four k
//               are then {KV g + e}: the same for A, so the sum is complete.  TN fragments of 16 columns per wave.
//   NN          (f32) lane (c, g) loads the 4 columns 4 c .. + 3 of rows k = 4 g + e, e < 4: value j of load e is the
//               operand of fragment j (columns 4 c + j) and k = 4 g + e.  64 columns per wave.
//   A           m k elements, read by every workgroup out of L2: what keeps the bf16 form to small B and few rows (16
//               x 8192 x 8192 takes 33 us here against 31 on the tiled kernel, which shares A between 128 columns)
// Requires k % KV == 0 and 16-byte aligned A and B; NN: n % 4 == 0.
#pragma once
#include <type_traits>

#include "common.h"
#include "params.h"

template <bool F32, bool NN, int MT, int TN, int W>
__device__ __forceinline__ void gemm_narrow_body(const GemmParams& p) {
  static_assert(!NN || (TN == 4 && F32), "an NN wave has four interleaved fragments of f32");
  constexpr int EL = F32 ? 4 : 2;       // bytes per element
  constexpr int KV = 16 / EL;           // k per 16-byte load
  constexpr int KSTEP = 4 * KV;         // k per A load of a wave
  constexpr int CS = NN ? 1 : 2;        // steps per piece: 128 bytes of a row of B (NT)
  constexpr int PIECE = KSTEP * CS;
  constexpr int BL = NN ? KV : TN;      // loads of B per step
    // pieces in flight per wave: about 96 registers of loads (48 with 16 waves, which have half the registers)
  constexpr int BUDGET = W > 8 ? 48 : 96, COST = CS * (BL + MT) * 4;
  constexpr int U = BUDGET / COST > 1 ? BUDGET / COST : 1;
  constexpr int NTILE = 16 * TN, RS = NTILE + 4;  // columns per workgroup; floats per row of the sums in LDS
  __shared__ __attribute__((aligned(16))) float red[W][16 * MT][RS];

  const uint32_t nsplit = p.splits > 1 ? p.splits : 1u;
  const uint32_t batch = blockIdx.y / nsplit, split = blockIdx.y - batch * nsplit;
  const uint32_t k_first = split * p.k_chunk;
  const uint32_t kk = nsplit > 1 ? (p.k - k_first < p.k_chunk ? p.k - k_first : p.k_chunk) : p.k;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t c = lane & 15, g = lane >> 4;
  // (workgroups go round the 8 XCDs: neighbouring columns, which share lines of B (NN), on the same one)
  const uint32_t tiles = (p.n + NTILE - 1) / NTILE, per_xcd = (tiles + 7) / 8;
  const uint32_t tile = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per_xcd || tile >= tiles) return;
  const uint32_t n0 = tile * NTILE;

  // per-lane pointers at k = k_first + KV g; rows and columns past the end repeat the last ones and are not stored
  const char* a_row[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const uint32_t r = 16 * i + c < p.m ? 16 * i + c : p.m - 1;
    a_row[i] = reinterpret_cast<const char*>(p.a) + (((size_t)batch * p.m + r) * p.k + k_first + KV * g) * EL;
  }
  constexpr int BP = NN ? 1 : TN;
  const char* b_row[BP];
  const size_t brow = (size_t)p.n * EL;  // NN: bytes per row of B
  if constexpr (NN) {
    const uint32_t col = n0 + 4 * c < p.n ? n0 + 4 * c : p.n - 4;
    b_row[0] = reinterpret_cast<const char*>(p.b) + ((size_t)batch * p.k + k_first + KV * g) * brow + (size_t)col * EL;
  } else {
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      const uint32_t r = n0 + 16 * t + c < p.n ? n0 + 16 * t + c : p.n - 1;
      b_row[t] = reinterpret_cast<const char*>(p.b) + (((size_t)batch * p.n + r) * p.k + k_first + KV * g) * EL;
    }
  }

  struct Piece {
    u32x4 a[CS][MT];
    u32x4 b[CS][BL];
  };
  auto load = [&](Piece& x, uint32_t piece, auto guarded) {
#pragma unroll
    for (int s = 0; s < CS; ++s) {
      const uint32_t k = piece * PIECE + s * KSTEP;
      // (a partial last piece: the lanes whose k lies past the end contribute zeros on both sides)
      const bool there = !decltype(guarded)::value || k + KV * g < kk;
#pragma unroll
      for (int l = 0; l < BL; ++l) {
        u32x4 v = {};
        if (there) {
          if constexpr (NN) v = *reinterpret_cast<const u32x4*>(b_row[0] + (size_t)(k + l) * brow);
          else v = *reinterpret_cast<const u32x4*>(b_row[l] + (size_t)k * EL);
        }
        x.b[s][l] = v;
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        u32x4 v = {};
        if (there) v = *reinterpret_cast<const u32x4*>(a_row[i] + (size_t)k * EL);
        x.a[s][i] = v;
      }
    }
  };

  f32x4 acc[MT][TN];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < TN; ++t) acc[i][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](const Piece& x) {
#pragma unroll
    for (int s = 0; s < CS; ++s) {
      if constexpr (F32) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int t = 0; t < TN; ++t) {
            const uint32_t b = NN ? x.b[s][e][t] : x.b[s][t][e];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
              const uint32_t a = x.a[s][i][e];
              acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, b), __builtin_bit_cast(float, a), acc[i][t], 0, 0, 0);
            }
          }
      } else {
#pragma unroll
        for (int t = 0; t < TN; ++t) {
#pragma unroll
          for (int i = 0; i < MT; ++i)
            acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x.b[s][t]), __builtin_bit_cast(bf16x8, x.a[s][i]), acc[i][t], 0, 0, 0);
        }
      }
    }
  };

  const uint32_t whole = kk / PIECE, pieces = (kk + PIECE - 1) / PIECE;
  uint32_t q = wave;
  for (; q + W * (U - 1) < whole; q += W * U) {
    Piece x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) load(x[u], q + W * u, std::false_type{});
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) multiply(x[u]);
  }
  for (; q < pieces; q += W) {
    Piece x;
    load(x, q, std::true_type{});
    multiply(x);
  }

  // ---- the waves' sums, added up in wave order.  NT: acc[i][t][r] is C[16 i + c][16 t + 4 g + r]; NN: fragment t
  // holds the columns 4 * + t, so it is C[16 i + c][16 g + 4 r + t].
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    float* row = red[wave][16 * i + c];
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      if constexpr (NN) *reinterpret_cast<f32x4*>(row + 16 * g + 4 * t) = f32x4{acc[i][0][t], acc[i][1][t], acc[i][2][t], acc[i][3][t]};
      else *reinterpret_cast<f32x4*>(row + 16 * t + 4 * g) = acc[i][t];
    }
  }
  __syncthreads();
  char* __restrict__ C = reinterpret_cast<char*>(p.c) + (size_t)blockIdx.y * p.m * p.n * (p.out_bf16 ? 2 : 4);
  const bool n4 = p.n % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
  for (uint32_t at = threadIdx.x; at < 16 * MT * (NTILE / 4); at += W * 64) {
    const uint32_t r = at / (NTILE / 4), quad = at % (NTILE / 4), col = n0 + 4 * quad;
    if (r >= p.m || col >= p.n) continue;
    f32x4 sum = *reinterpret_cast<const f32x4*>(&red[0][r][4 * quad]);
#pragma unroll
    for (int w = 1; w < W; ++w) sum += *reinterpret_cast<const f32x4*>(&red[w][r][4 * quad]);
    const size_t to = (size_t)r * p.n + col;
    if (n4 && !p.out_bf16) {
      *reinterpret_cast<f32x4*>(C + 4 * to) = sum;
    } else if (n4) {
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (bf16_t)sum[e];
      *reinterpret_cast<bf16x4*>(C + 2 * to) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < p.n) {
          if (p.out_bf16) reinterpret_cast<bf16_t*>(C)[to + e] = (bf16_t)sum[e];
          else reinterpret_cast<float*>(C)[to + e] = sum[e];
        }
    }
  }
}
