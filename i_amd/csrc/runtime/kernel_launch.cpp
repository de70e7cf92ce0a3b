#include "kernel_launch.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <initializer_list>
#include <cstdint>
#include <string>

#include "../kernels/params.h"

namespace ihip {
namespace {
constexpr size_t kMaxGrid = 0x7fffffffu;

bool fits_u32(size_t v) { return v <= 0xffffffffull; }
bool aligned16(const void* ptr) { return reinterpret_cast<uintptr_t>(ptr) % 16 == 0; }
}  // namespace

Err set_kernel_option(KernelOptions& o, const std::string& name, int value) {
  auto one_of = [&](std::initializer_list<int> allowed) {
    for (int a : allowed)
      if (a == value) return true;
    return false;
  };
  auto bad = [&](const char* allowed) { return "program option '" + name + "' must be " + allowed + ", not " + std::to_string(value); };
  if (name == "attention.f32_scale") {
    o.attention_f32_scale = value != 0;
  } else if (name == "attention.kv_parts") {
    if (value < 0) return bad("0 (the launcher decides), 1 (never) or a number of parts");
    o.attention_kv_parts = value;
  } else if (name == "attention.waves") {
    if (!one_of({0, 2, 4, 8, 64})) return bad("0, 2, 4 or 8 (or 64: the 64-queries-per-wave kernel for d = 64)");
    o.attention_waves = value;
  } else if (name == "attention.direct") {
    o.attention_direct = value != 0;
  } else if (name == "gemm.k_parts") {
    if (value < 0) return bad("0 (the launcher decides), 1 (never) or a number of parts");
    o.gemm_k_parts = value;
  } else if (name == "gemm.waves") {
    if (!one_of({0, 4, 8})) return bad("0, 4 or 8");
    o.gemm_waves = value;
  } else if (name == "gemm.tile") {
    if (!one_of({0, 128, 192, 256})) return bad("0, 128, 192 (192 x 256) or 256");
    o.gemm_tile = value;
  } else if (name == "gemm.tile_n") {
    if (!one_of({0, 128, 192, 256})) return bad("0 (what goes with gemm.tile), 128, 192 (256 x 192) or 256");
    o.gemm_tile_n = value;
  } else if (name == "gemm.direct") {
    o.gemm_direct = value != 0;
  } else if (name == "generated.only") {
    o.generated_only = value != 0;
  } else if (name == "generated.wave") {
    if (!one_of({-1, 0, 1})) return bad("-1 (the launcher decides), 0 or 1");
    o.generated_wave = value;
  } else if (name == "generated.parts") {
    if (value < 0 || value > 4096) return bad("0 (the launcher decides), 1 (never) or a number of parts up to 4096");
    o.generated_parts = value;
  } else {
    return "unknown program option '" + name +
           "' (known: attention.f32_scale, attention.kv_parts, attention.waves, attention.direct, gemm.k_parts, gemm.waves, "
           "gemm.tile, gemm.tile_n, gemm.direct, generated.only, generated.wave, generated.parts)";
  }
  return {};
}

Err parse_kernel_options(const char* text, KernelOptions* options) {
  if (!text) return {};
  const std::string all(text);
  size_t at = 0;
  auto separator = [](char c) { return c == ' ' || c == ',' || c == ';' || c == '\t' || c == '\n'; };
  while (at < all.size()) {
    while (at < all.size() && separator(all[at])) ++at;
    size_t end = at;
    while (end < all.size() && !separator(all[end])) ++end;
    if (end == at) break;
    const std::string pair = all.substr(at, end - at);
    at = end;
    const size_t eq = pair.find('=');
    if (eq == std::string::npos || eq == 0 || eq + 1 == pair.size()) return "option '" + pair + "' is not of the form name=value";
    char* tail = nullptr;
    const long value = std::strtol(pair.c_str() + eq + 1, &tail, 10);
    if (*tail != '\0') return "option '" + pair + "' has no integer value";
    if (Err e = set_kernel_option(*options, pair.substr(0, eq), (int)value); !e.empty()) return e;
  }
  return {};
}

Err launch_shader_clock_probe(unsigned long long* ticks, unsigned microseconds, hipStream_t stream) {
  if (!ticks) return "clock probe: null device pointer";
  if (reinterpret_cast<uintptr_t>(ticks) % 8 != 0) return "clock probe: the counters must be 8-byte aligned";
  if (microseconds > 2000000u) return "clock probe: at most two seconds";
  ClockProbeParams p{ticks, microseconds * 100u};
  hipFunction_t fn;
  if (Err e = builtin_function("shader_clock_probe", &fn); !e.empty()) return e;
  return launch(fn, 1, 1, 1, 64, &p, sizeof(p), stream);
}

bool attention_supported(DType in_dtype, size_t d, size_t dv, const KernelOptions& knobs) {
  if (d == 0 || dv == 0) return false;
  // head sizes above 128 up to 256: bf16, on the direct kernels only
  if (d > 128 || dv > 128)
    return in_dtype == BF16 && d <= 256 && dv <= 256 && d % 8 == 0 && dv % 8 == 0 && knobs.attention_direct;
  if (in_dtype == BF16) return d % 8 == 0 && dv % 8 == 0;
  return true;
}

// f32 attention: which kernel, and into how many parts over workgroups the keys go.
struct F32AttentionPlan {
  unsigned waves;   // 4 | 8: the kernel whose wavefronts take a part of the keys each (attention_f32_waves.h); 0: query tiles of 128
  unsigned splits;
};
static unsigned attention_tile_splits(DType in_dtype, size_t bh, size_t nq, size_t nk, const AttentionOptions& options);
static bool f32_waves_supported(size_t nk, size_t d, size_t dv, const KernelOptions& knobs) {
  const size_t dmax = d > dv ? d : dv;
  return d % 4 == 0 && dv % 4 == 0 && dmax <= 128 && nk * dmax * 4 < (size_t(1) << 32) && knobs.attention_direct && knobs.attention_kv_parts == 0;
}
// A model of the time in us.  Query tiles of 128: 4, and per trip of 32 keys 2.7 (4.7 above 64 columns, 2.4 up to 32) for a
// CU's only workgroup, 2.3 (4.3, 1.75) for each of several.  16 rows per workgroup: a CU's only one is a chain of steps of 32
// keys per wavefront; of several, each costs its share of the matrix instructions and of a step.  A split over workgroups
// costs 6 for the second launch and its pass at 3 TB/s.  Over 1212 shapes from 1 x 1 x 21 x 8 to 512 x 700 x 700 x 128 this choice is 1.98 times as fast as query
// tiles alone in the mean, and nowhere slower by more than 4 % but for calls of 10 us that wait for the host.  Both sides at
// the line, us: 160 heads of 512 x 128 219 on tiles, 241 on rows; 16 of 1024 x 64 54 and 47.
static F32AttentionPlan f32_attention_plan(size_t bh, size_t nq, size_t nk, size_t d, size_t dv, const AttentionOptions& options, bool may_split) {
  const size_t dmax = d > dv ? d : dv;
  auto merge = [&](size_t splits) { return splits > 1 ? 6.0 + (double)(bh * splits * nq * dv * 4) / 3e6 : 0.0; };
  auto of_cu = [](size_t workgroups) { return (double)((workgroups + 255) / 256); };
  F32AttentionPlan best{0, dmax > 32 && may_split ? attention_tile_splits(F32, bh, nq, nk, options) : 1};
  if (!f32_waves_supported(nk, d, dv, options.knobs)) return best;
  const double tiles = of_cu(bh * ((nq + 127) / 128) * best.splits), trips = (double)(((nk + best.splits - 1) / best.splits + 31) / 32);
  const double alone = dmax <= 32 ? 2.4 : dmax <= 64 ? 2.7 : 4.7, shared = dmax <= 32 ? 1.75 : dmax <= 64 ? 2.3 : 4.3;
  double least = 0.97 * (4.0 + trips * std::max(alone, shared * tiles) + merge(best.splits));
  const size_t rows = bh * ((nq + 15) / 16);
  for (unsigned waves : {8u, 4u}) {
    if (waves == 8 && dmax > 64) continue;
    //                      fixed, a step of a CU's only workgroup, per workgroup of several, and per step of it
    const double cost[4] = {dmax > 64 ? 7.0 : waves == 8 ? 4.2 : 4.0, dmax > 64 ? 2.6 : waves == 8 ? 2.65 : 1.56,
                            dmax > 64 ? 2.4 : waves == 8 ? 0.8 : 0.45, dmax > 64 ? 2.35 : waves == 8 ? 2.5 : 1.27};
    for (size_t s = 1; s <= 32 && (s == 1 || (may_split && nk / s >= 32 * waves && rows * s <= 1024)); ++s) {
      const size_t chunk = s == 1 ? nk : ((nk + s - 1) / s + 63) / 64 * 64, parts = (nk + chunk - 1) / chunk, blocks = (chunk + 31) / 32;
      const double t = cost[0] + std::max((double)((blocks + waves - 1) / waves) * cost[1], of_cu(rows * parts) * (cost[2] + (double)blocks / waves * cost[3])) + merge(parts);
      if (t < least) {
        least = t;
        best = {waves, (unsigned)parts};
      }
    }
  }
  return best;
}

// bf16: into how many parts a workgroup's waves take the keys (1: all waves walk all keys).  A model of the time in us
// where every CU has at most one workgroup: a fixed part and a chain of trips, of 64 keys (32 above 128 columns) for the kernels
// with 128 query rows, of 32 or 64 keys times the groups for these.  Their K/V tiles fill the LDS of a CU, so grids of more
// workgroups than CUs stay where they are (400 heads of 1 x 1500 x 128: 55 us, in groups 61), and so do loops that are long
// enough for parts over workgroups.  Measured, us: one head of 1500 x
// 128 24.5 -> 18.5, x 64 18.3 -> 12; 84 heads of 1 x 1500, d = 64 18.5 -> 11.9, 128 24.3 -> 19.8, 184 42.7 -> 36; but 200 of 1 x
// 2048 x 128, where reading K and V is the bound, 34.2 and 35.8.
static unsigned attention_key_groups(size_t bh, size_t nq, size_t nk, size_t dmax, const AttentionOptions& options) {
  const KernelOptions& knobs = options.knobs;
  const size_t tile = options.query_tile;
  if (knobs.attention_f32_scale || knobs.attention_waves || knobs.attention_kv_parts || tile == 64 || tile == 128 || tile == 256 || tile == 512) return 1;
  const size_t rows64 = bh * ((nq + 63) / 64), rows32 = bh * ((nq + 31) / 32);
  if (rows64 > 256 || attention_tile_splits(BF16, bh, nq, nk, options) > 1) return 1;
  auto chain = [nk](double fixed, size_t keys, double trip) { return fixed + (double)((nk + keys - 1) / keys) * trip; };
  if (dmax <= 64) {
    const double whole = chain(4.5, 64, 0.56);
    if (rows32 <= 256 && nk >= 256 && chain(7.2, 256, 0.53) < 0.97 * whole) return 8;
    return nk >= 256 && chain(8.0, 256, 0.7) < 0.97 * whole ? 4 : 1;
  }
  if (dmax <= 128) return nk >= 128 && rows64 <= 192 && chain(8.5, 128, 0.66) < 0.97 * chain(6.3, 64, 0.72) ? 4 : 1;
  return nk >= 64 && chain(14.0, 64, 0.9) < 0.97 * chain(8.8, 32, 0.72) ? 2 : 1;
}

Err launch_attention(const void* q, const void* k, const void* v, void* o, DType in_dtype, DType out_dtype, size_t bh,
                     size_t nq, size_t nk, size_t d, size_t dv, const float* scale_ptr, float scale, hipStream_t stream,
                     const AttentionOptions& options, LaunchNote* note) {
  const KernelOptions& knobs = options.knobs;
  if (!attention_supported(in_dtype, d, dv, knobs))
    return "attention kernel: unsupported operands (need 0 < d, dv <= 128, or bf16 with d, dv <= 256; bf16 needs d, dv % 8 == 0)";
  if ((d > 128 || dv > 128) && nk * (d > dv ? d : dv) * 2 >= (size_t(1) << 32))
    return "attention kernel: too many keys for a head size above 128";
  if (!std::isfinite(scale)) return "attention kernel: unsupported scale (must be finite)";
  if (in_dtype == F32 && out_dtype != F32) return "attention kernel: f32 inputs produce f32 output";
  if (bh == 0 || nq == 0) return {};
  if (nk == 0) return "attention kernel: no keys";
  if (!fits_u32(bh) || !fits_u32(nq) || !fits_u32(nk)) return "attention kernel: extent exceeds 32 bits";
  if (!q || !k || !v || !o) return "attention kernel: null device pointer";
  // every bf16 kernel moves 16 bytes per lane (the direct ones straight into LDS) and stores 8 (bf16) or 16 (f32)
  if (in_dtype == BF16 && (!aligned16(q) || !aligned16(k) || !aligned16(v) || reinterpret_cast<uintptr_t>(o) % (out_dtype == BF16 ? 8 : 16) != 0))
    return "attention kernel: bf16 operands must be 16-byte aligned (the output 8-byte for bf16, 16-byte for f32)";

  const size_t dmax = d > dv ? d : dv;
  const size_t query_tile = options.query_tile, key_tile = options.key_tile;
  // Kernel choice for bf16:
  //   d == dv in {64, 128}: direct-to-LDS kernels, templated on the workgroup's query rows (64 / 128 / 256 = 2 / 4 / 8
  //     waves) and on the key tile in LDS (32 / 64).  The schedule's tile decides when such a kernel exists.
  //     Without a usable request: 64-key tiles, and 256 query rows (half the L2 -> LDS traffic per query) on long
  //     key loops when that still leaves at least two workgroups per CU and does not pad nq by much, else 128.
  //     d == 64 on grids with at least two 512-query workgroups per CU (or a schedule tile of 512 x 32): the
  //     64-queries-per-wave kernel, which reads every K/V operand from LDS once for two MFMAs.
  //   any other d, dv that are multiples of 8 up to 128: the 4- and 8-wave kernels with 64-key tiles and their LDS
  //     rows padded to 64 or 128 columns (the larger of d and dv decides).
  //   d or dv above 128 up to 256 (multiples of 8): the kernel for 256-column rows (padded below 256), 4 waves, one
  //     per SIMD, 32-key tiles; nothing else exists above 128, so callers ask attention_supported() first.
  //   otherwise (knobs.attention_direct == 0, key offsets beyond 32 bits): register-staged kernel with guarded
  //     columns (always multiplies the scores in f32)
  // knobs.attention_waves = 2 | 4 | 8 forces the workgroup size of the direct kernel (64: the 64-queries-per-wave
  // kernel, d == 64 only) and knobs.attention_direct = 0 the register-staged kernel; both exist so that tests and
  // searches can reach every kernel with small inputs.
  unsigned bm = 128, bn = 64;
  bool q64 = false;
  const bool exact = in_dtype == BF16 && d == dv && (d == 64 || d == 128);
  const bool wide = in_dtype == BF16 && dmax > 128;  // (supported: d, dv <= 256, multiples of 8)
  const bool padded = in_dtype == BF16 && !exact && d % 8 == 0 && dv % 8 == 0 && !(d == 256 && dv == 256);
  // per-head K/V byte offsets are 32-bit in the direct-to-LDS kernel
  const bool direct = (exact || padded || wide) && nk * dmax * 2 < (size_t(1) << 32) && knobs.attention_direct;
  const bool f32_scale = knobs.attention_f32_scale != 0;
  if (direct && wide) {
    bm = 128;  // 4 waves, one per SIMD
    bn = 32;
  } else if (direct && padded) {
    // 64-key tiles; 256 query rows per workgroup on the grids where the unpadded kernels take them, else 128
    if (query_tile == 256 || (query_tile != 128 && bh * ((nq + 255) / 256) >= 2 * 256 && nk >= 2560 &&
                              10 * ((nq + 255) / 256 * 256) <= 11 * ((nq + 127) / 128 * 128)))
      bm = 256;
    if (const int waves = knobs.attention_waves) {
      if (waves != 4 && waves != 8) return "attention kernel: attention.waves must be 4 or 8 for a padded head size";
      bm = 32u * (unsigned)waves;
    }
  } else if (direct) {
    const bool tile_known = query_tile == 64 || query_tile == 128 || query_tile == 256;
    if (key_tile == 32 && !f32_scale && tile_known && !(d == 64 && query_tile == 256)) bn = 32;
    if (tile_known && !(f32_scale && query_tile == 64)) bm = (unsigned)query_tile;  // the schedule's i split
    else if (d == 64 && !f32_scale &&
             ((query_tile == 512 && (key_tile == 32 || key_tile == 0)) ||
              (query_tile == 0 && bh * ((nq + 511) / 512) >= 2 * 256 &&
               10 * ((nq + 511) / 512 * 512) <= 11 * ((nq + 127) / 128 * 128))))
      q64 = true;
    else if (bh * ((nq + 255) / 256) >= 2 * 256 && nk >= 2560 &&
             10 * ((nq + 255) / 256 * 256) <= 11 * ((nq + 127) / 128 * 128))
      bm = 256;  // ... on long key loops (two resident 4-wave workgroups hide each other's prologue and epilogue,
                 // which wins up to about 2048 keys), and unless rounding nq up to 256 instead of 128 adds more
                 // than 10 % of idle query rows
    if (const int waves = knobs.attention_waves) {
      q64 = waves == 64 && d == 64 && !f32_scale;
      if (!q64) {
        if (waves != 2 && waves != 4 && waves != 8) return "attention kernel: attention.waves must be 2, 4 or 8 (or 64 for d = 64)";
        bm = 32u * (unsigned)waves;
        if (f32_scale && bm == 64) bm = 128;
        if (d == 64 && bm == 256) bn = 64;
      }
    }
    if (q64) { bm = 512; bn = 32; }
  }
  // ... and where nothing is asked for and a chain over all keys is what a call waits for: groups of waves on parts of the keys
  const unsigned groups = direct && !q64 && options.kv_splits <= 1 ? attention_key_groups(bh, nq, nk, dmax, options) : 1;
  if (groups > 1) {
    bm = groups == 8 ? 32 : 64;
    bn = groups == 4 && dmax <= 64 ? 64 : 32;
  }
  // f32: the direct-to-LDS kernel for d, dv multiples of 4 up to 128, the larger above 32 (16-byte aligned operands,
  // 32-bit byte offsets inside a head; up to 32 the register-staged kernel with 32-column tiles is the faster one), the
  // register-staged kernel with guarded columns otherwise (and with knobs.attention_direct == 0)
  const bool f32_direct = in_dtype == F32 && d % 4 == 0 && dv % 4 == 0 && dmax > 32 && dmax <= 128 &&
                          nk * dmax * 4 < (size_t(1) << 32) && aligned16(q) && aligned16(k) && aligned16(v) && aligned16(o) &&
                          knobs.attention_direct;
  // ... or, where its tiles of 128 query rows leave the CUs little to do, the kernel with 16 rows per workgroup
  unsigned f32_waves = 0;
  if (in_dtype == F32 && f32_waves_supported(nk, d, dv, knobs) && aligned16(q) && aligned16(k) && aligned16(v) && aligned16(o))
    f32_waves = f32_attention_plan(bh, nq, nk, d, dv, options, options.kv_splits > 1).waves;
  if (f32_waves) bm = 16;
  AttnParams p{};
  p.q = q; p.k = k; p.v = v; p.o = o;
  p.bh = (uint32_t)bh; p.nq = (uint32_t)nq; p.nk = (uint32_t)nk; p.d = (uint32_t)d; p.dv = (uint32_t)dv;
  p.nqt = (uint32_t)((nq + bm - 1) / bm);
  p.out_bf16 = out_dtype == BF16 ? 1u : 0u;
  p.scale_ptr = scale_ptr;
  p.scale_value = scale;
  p.clock = knobs.clock_ticks;
  // the keys of a head in several parts: the direct kernels take (head, part) pairs for heads and write to the
  // caller's temporaries; attn_kv_merge follows.  (A request that the kernel chosen above cannot honour, the
  // register-staged ones and the 64-queries-per-wave kernel, is ignored: the result is the same.)
  unsigned splits = 1;
  if (options.kv_splits > 1 && ((in_dtype == BF16 && direct && !q64) || f32_direct || f32_waves)) {
    if (!options.partial_o || !options.partial_lse) return "attention kernel: a split needs its temporaries";
    p.kv_chunk = (uint32_t)(((nk + options.kv_splits - 1) / options.kv_splits + 63) / 64 * 64);
    splits = (unsigned)((nk + p.kv_chunk - 1) / p.kv_chunk);  // (rounding the parts up to whole tiles may leave fewer)
    if (splits > 1) {
      if (!fits_u32(bh * splits)) return "attention kernel: extent exceeds 32 bits";
      p.kv_splits = splits;
      p.bh = (uint32_t)(bh * splits);
      p.o = options.partial_o;
      p.lse = options.partial_lse;
      p.out_bf16 = 0;
    }
  }

  std::string name;
  unsigned threads = 2 * bm;  // one query per lane of a half-wave: 32 queries per wave
  if (in_dtype == BF16) {
    if (direct && q64) {
      name = "attn_fwd_bf16_d64_bn32_q64";
      threads = bm;
    } else if (direct) {
      name = "attn_fwd_bf16_d" + std::to_string(wide ? 256 : padded ? (dmax <= 64 ? 64 : 128) : d) + "_bn" + std::to_string(bn) + "_direct";
      if (bm <= 64) name += bm == 64 ? "_w2" : "_w1";
      if (groups > 1) {
        name += "_k" + std::to_string(groups);
        threads *= groups;
      }
      if (bm == 256) name += "_w8";
      if (f32_scale) name += "_f32scale";
      if (padded) name += "_pad";
    } else if (exact) name = d == 64 ? "attn_fwd_bf16_d64_bn64" : "attn_fwd_bf16_d128_bn64";
    else name = dmax <= 64 ? "attn_fwd_bf16_d64_bn64_any" : "attn_fwd_bf16_d128_bn64_any";
  } else {
    if (f32_waves) {
      name = (dmax <= 64 ? "attn_fwd_f32_d64_bn32_direct" : "attn_fwd_f32_d128_bn32_direct") + std::string(d == dv && (d == 64 || d == 128) ? "" : "_pad") + "_waves" + std::to_string(f32_waves);
      threads = 64 * f32_waves;
    } else if (f32_direct) {
      // (head sizes other than d == dv in {64, 128}: the same kernel with its LDS rows padded to 64 or 128 columns)
      name = dmax <= 64 ? "attn_fwd_f32_d64_bn32_direct" : "attn_fwd_f32_d128_bn32_direct";
      if (!(d == dv && (d == 64 || d == 128))) name += "_pad";
    }
    else name = dmax <= 32 ? "attn_fwd_f32_d32_bn32" : dmax <= 64 ? "attn_fwd_f32_d64_bn32" : "attn_fwd_f32_d128_bn32";
    bn = 32;
  }
  // padded head sizes of which 96 columns cover d and dv: the form that computes no more (its report names it so)
  const bool columns96 = in_dtype == BF16 && direct && padded && !wide && dmax > 64 && dmax <= 96;
  const std::string parts = f32_waves ? (splits > 1 ? std::to_string(splits) + " x " : "") + std::to_string(f32_waves) : std::to_string(splits);
  if (note) *note = LaunchNote{name + (columns96 ? " (96 columns)" : "") + (splits > 1 || f32_waves ? " (keys in " + parts + " parts)" : ""), bm, bn};
  if (columns96) name += "96";

  const size_t grid = (size_t(p.bh) * p.nqt + 7) / 8 * 8;  // the query tiles of all heads in 8 equal runs, one per XCD
  if (grid > kMaxGrid) return "attention kernel: grid too large";
  hipFunction_t fn;
  if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
  if (Err e = launch(fn, (unsigned)grid, 1, 1, threads, &p, sizeof(p), stream); !e.empty() || splits == 1) return e;
  AttnMergeParams m{options.partial_o, options.partial_lse, o, (uint32_t)bh, splits, (uint32_t)nq, (uint32_t)dv, out_dtype == BF16 ? 1u : 0u};
  if (Err e = builtin_function("attn_kv_merge", &fn); !e.empty()) return e;
  size_t mgrid = (bh * nq * (dv / 4) + 255) / 256;
  if (mgrid > 65536) mgrid = 65536;
  return launch(fn, (unsigned)mgrid, 1, 1, 256, &m, sizeof(m), stream);
}

// Into how many parts to split the keys of each head (1: do not).  A grid of bh * ceil(nq / 128) workgroups that
// leaves most of the 256 CUs without one (a single head, a few sequences, a few queries against many keys)
// finishes sooner when parts of the key loop run side by side: as many parts as fill the CUs once, of at least 512
// keys each, at most 32, and only for loops of 2048 keys and more (below that the second launch takes what the
// split gains).  Measured, enqueued back to back, d = 128: one head of 8192 x 8192 92 -> 46 us (4 parts), of
// 4096 x 4096 48 -> 27, 128 queries x 8192 keys 91 -> 23 (16 parts), 8 heads of 128 x 16384 176 -> 32; from 256
// workgroups on nothing is gained (16 heads of 4096: 127 -> 146 us with 2 parts).  An f32 workgroup spends four times
// as long on half the keys, so f32 loops on these tiles are split from 256 keys on, into parts of at least 64: 2 heads of
// 128 queries x 8192 keys of 128, 1136 -> 64 us in 32.  Only where the direct kernels run (launch_attention's own
// conditions); f32_attention_plan has the last word on f32.
static unsigned attention_tile_splits(DType in_dtype, size_t bh, size_t nq, size_t nk, const AttentionOptions& options) {
  const KernelOptions& knobs = options.knobs;
  // an f32 workgroup takes about 2.8 us per 32 keys (a bf16 one 0.7 us per 64): much shorter loops are worth parts
  const size_t least_loop = in_dtype == BF16 ? 2048 : 256, least_part = in_dtype == BF16 ? 512 : 64;
  size_t want;
  if (knobs.attention_kv_parts > 1) {
    want = (size_t)knobs.attention_kv_parts;  // forced, still bounded by whole 64-key tiles below
  } else {
    const size_t bm = in_dtype == BF16 && (options.query_tile == 64 || options.query_tile == 256) ? options.query_tile : 128;
    const size_t groups = bh * ((nq + bm - 1) / bm);
    if (nk < least_loop || nk < least_loop / 64 * groups) return 1;  // (half the CUs busy: two parts pay from twice the least loop on)
    want = std::min<size_t>(std::min<size_t>(256 / groups, nk / least_part), 32);
  }
  if (want < 2 || nk < 128) return 1;
  want = std::min<size_t>(want, nk / 64);
  if (want < 2) return 1;
  const size_t chunk = ((nk + want - 1) / want + 63) / 64 * 64;
  return (unsigned)((nk + chunk - 1) / chunk);
}

unsigned attention_kv_splits(DType in_dtype, size_t bh, size_t nq, size_t nk, size_t d, size_t dv, const AttentionOptions& options) {
  const KernelOptions& knobs = options.knobs;
  if (bh == 0 || nq == 0 || nk == 0 || d == 0 || dv == 0 || !knobs.attention_direct || knobs.attention_kv_parts == 1) return 1;
  const size_t dmax = d > dv ? d : dv;
  if (in_dtype == BF16) {
    if (d % 8 != 0 || dv % 8 != 0 || d > 256 || dv > 256 || !(nk * dmax * 2 < (size_t(1) << 32))) return 1;
    if (knobs.attention_waves == 64) return 1;
    if (options.query_tile == 512) return 1;  // (may select the 64-queries-per-wave kernel)
    return attention_tile_splits(in_dtype, bh, nq, nk, options);
  }
  if (f32_waves_supported(nk, d, dv, knobs)) return f32_attention_plan(bh, nq, nk, d, dv, options, true).splits;
  // (f32: the direct kernels' head sizes; operands they cannot take for their alignment run unsplit)
  if (d % 4 != 0 || dv % 4 != 0 || dmax <= 32 || dmax > 128 || !(nk * dmax * 4 < (size_t(1) << 32))) return 1;
  return attention_tile_splits(in_dtype, bh, nq, nk, options);
}

bool gemm_nt_bf16_supported(size_t k) { return k > 0 && k % 8 == 0; }

// 256 x 256 tiles (one workgroup per CU, 256 at a time) or 128 x 128 tiles (two per CU, 512 at a time) for a
// problem with enough of either?  The larger tile is about 20 % more efficient per flop (1442 against 1237 TFLOP/s
// at 4096^3, whole rounds of either), but its last round of workgroups may leave most of the chip idle: 4608^3 is
// 1.27 rounds of 256-tiles (measured 1061 TFLOP/s) and 2.53 rounds of 128-tiles (1092).  Rounds of the two-per-CU
// kernel count in halves.  A round that leaves part of the chip idle runs its tiles faster (the clock rises when
// fewer CUs draw power): 1600 per filled CU-round against 1460 for full rounds.  (A model, within 3 % of the
// better tile from 1024^3 to 8192^3 in steps of 512.)
static unsigned pick_direct_tile(size_t t256, size_t t128) {
  const double r256 = (double)t256 / 256.0, r128 = (double)t128 / 512.0;
  const double fill256 = r256 / std::ceil(r256);
  const double e256 = (fill256 > 0.95 ? 1460.0 : 1600.0) * fill256;
  const double e128 = (r128 < 1.0 ? 1250.0 : 1150.0) * r128 / (std::ceil(2.0 * r128) / 2.0);
  return e256 >= e128 ? 256 : 128;
}

// A model of a launch's time in us, by which the 192 x 256 tile is weighed against the one chosen above: a fixed
// part (launch, first slab, the store of C), plus the slabs of the k loop times the time of a slab for a full round
// of workgroups (1.5 us on a 256 x 256 tile, 1.154 on 192 x 256, 0.95 on two 128 x 128 tiles per CU), times the
// rounds, a partly empty round counting for 0.55 + half of its fill (fewer busy CUs run a higher clock and share
// L2 and the fabric among fewer); less than one round of 128-tiles is cheaper still (one workgroup per CU).
// Fitted to cubes from 1792 to 8192, where it is within 5 % of the measured times of all three tiles but for the
// 192 x 256 tile from 7168 on, which it flatters by 8 %: that tile has to win by 8 % to be taken.  It is taken at
// 3072^3 (64 against 71 us), 4608^3 (170 against 190) and 6144^3 (344 against 382), and nowhere from 5120 to 5632
// or from 6400 on.
static double direct_tile_time(unsigned tile, size_t tiles, size_t slabs) {
  const double slots = tile == 128 ? 512.0 : 256.0;
  const double slab_us = tile == 128 ? 0.95 : tile == 192 ? 1.154 : 1.5;
  const double r = (double)tiles / slots, whole = std::floor(r), part = r - whole;
  double rounds = whole + (part > 0.0 ? std::min(1.0, 0.55 + 0.5 * part) : 0.0);
  if (tile == 128 && r <= 1.0) rounds = std::min(1.0, 0.25 + 0.85 * r);
  return (tile == 128 ? 9.0 : 12.0) + rounds * (double)slabs * slab_us;
}

Err launch_gemm_nt_bf16(const void* a, const void* b, void* c, size_t bh, size_t m, size_t n, size_t k,
                        hipStream_t stream, size_t tile_m, size_t tile_n, LaunchNote* note, DType out_dtype,
                        const KernelOptions& knobs) {
  if (!gemm_nt_bf16_supported(k)) return "gemm_nt kernel: k must be a positive multiple of 8";
  if (bh == 0 || m == 0 || n == 0) return {};
  if (!fits_u32(m) || !fits_u32(n) || !fits_u32(k) || !fits_u32(bh)) return "gemm_nt kernel: extent exceeds 32 bits";
  if (!a || !b || !c) return "gemm_nt kernel: null device pointer";
  if (!aligned16(a) || !aligned16(b)) return "gemm_nt kernel: operands must be 16-byte aligned";
  GemmParams p{};
  p.a = a; p.b = b; p.c = c;
  p.bh = (uint32_t)bh; p.m = (uint32_t)m; p.n = (uint32_t)n; p.k = (uint32_t)k;
  p.out_bf16 = out_dtype == BF16 ? 1u : 0u;
  // Direct global -> LDS kernels (64-wide k slabs, 32-bit byte offsets inside a tile's rows):
  //   256 x 256 tiles  long k loops on grids that fill at least half of the CUs (its prologue and its
  //                    unoverlapped store only pay off there)
  //   128 x 128 tiles  everything else, two workgroups per CU (down to one tile and one slab it is the faster
  //                    128-tile kernel: 4.3 against 5.9 us at 128 x 128 x 64, 9.4 against 17.0 at 128 x 128 x 1024)
  // (k that is no multiple of 64: their _ktail forms, the last slab partial)
  // and the register-staged 128 x 128 kernel beyond their offset ranges (k > 2^22, more than 65535 batches).
  // The schedule's i, j splits (256 x 256, 192 x 256, 256 x 192 or 128 x 128) decide when given; knobs.gemm_tile
  // = 256 | 192 | 128 (with knobs.gemm_tile_n = 192 for 256 x 192) and
  // knobs.gemm_direct = 0 force a kernel so that tests and searches can reach each of them at small sizes.
  {
    const size_t t256 = ((m + 255) / 256) * ((n + 255) / 256) * bh, t128 = ((m + 127) / 128) * ((n + 127) / 128) * bh;
    // the two rectangular tiles: 192 rows of A against 256 of B, or 256 against 192, whichever leaves fewer tiles
    const size_t t192m = ((m + 191) / 192) * ((n + 255) / 256) * bh, t192n = ((m + 255) / 256) * ((n + 191) / 192) * bh;
    unsigned tile = 128, across = 0;  // rows of A and of B per tile (across 0: as many as of A; tile 0: register-staged kernel)
    if (k >= 512 && t256 >= 64) {
      tile = pick_direct_tile(t256, t128);
      const size_t slabs = (k + 63) / 64;
      if (1.08 * direct_tile_time(192, std::min(t192m, t192n), slabs) < direct_tile_time(tile, tile == 256 ? t256 : t128, slabs)) {
        tile = t192m <= t192n ? 192 : 256;
        across = t192m <= t192n ? 256 : 192;
      }
    }
    if (tile_m == 128 && tile_n == 128) tile = 128, across = 0;
    if ((tile_m == 256 || tile_m == 192) && (tile_n == 256 || tile_n == 192) && tile_m + tile_n >= 448) tile = (unsigned)tile_m, across = (unsigned)tile_n;
    if (knobs.gemm_tile) tile = (unsigned)knobs.gemm_tile, across = (unsigned)knobs.gemm_tile_n;
    if (!across) across = tile == 192 ? 256 : tile;
    if (tile == 192 && across != 256) return "gemm_nt kernel: a 192-row tile goes with 256 columns";
    if (tile == 128 && across != 128) return "gemm_nt kernel: a 128-row tile goes with 128 columns";
    if (tile == 256 && across != 256 && across != 192) return "gemm_nt kernel: a 256-row tile goes with 256 or 192 columns";
    if (!knobs.gemm_direct) tile = 0;
    const bool ktail = k % 64 != 0;
    if (tile && k <= (size_t(1) << 22) && bh <= 65535) {
      p.tiles_m = (uint32_t)((m + tile - 1) / tile);
      p.tiles_n = (uint32_t)((n + across - 1) / across);
      const size_t grid = (size_t(p.tiles_m) * p.tiles_n + 7) / 8 * 8;  // the tiles in 8 equal runs, one per XCD
      if (grid > kMaxGrid) return "gemm_nt kernel: grid too large";
      hipFunction_t fn;
      // the 256 x 256 tile runs with four waves of 128 x 128 (knobs.gemm_waves = 8: the form with eight of 128 x 64,
      // kept for comparison: equal on one round of tiles, 5-10 % behind on several); the rectangular ones with four
      // of 96 x 128 or 128 x 96
      const bool w4 = tile + across == 448 || (tile == 256 && knobs.gemm_waves != 8);
      const std::string name = "gemm_nt_bf16_" + std::to_string(tile) + "x" + std::to_string(across) + "x64_direct" +
                               (ktail ? "_ktail" : "") + (w4 ? "_w4" : "");
      if (note) *note = LaunchNote{name, tile, across};
      if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
      return launch(fn, (unsigned)grid, (unsigned)bh, 1, w4 || tile == 128 ? 256 : 512, &p, sizeof(p), stream);
    }
  }
  p.tiles_m = (uint32_t)((m + 127) / 128);
  p.tiles_n = (uint32_t)((n + 127) / 128);
  const size_t tiles = (size_t)p.tiles_m * p.tiles_n;
  const size_t grid = ((tiles + 7) / 8 * 8) * bh;
  if (grid > kMaxGrid) return "gemm_nt kernel: grid too large";
  hipFunction_t fn;
  if (note) *note = LaunchNote{"gemm_nt_bf16_128x128x64", 128, 128};
  if (Err e = builtin_function("gemm_nt_bf16_128x128x64", &fn); !e.empty()) return e;
  return launch(fn, (unsigned)grid, 1, 1, 256, &p, sizeof(p), stream);
}

// A model of a product's time in us on 128 x 128 or 256 x 256 tiles with k in `parts` of `slabs` 64-wide slabs: a workgroup
// spends 0.7 us per slab on a 128 x 128 tile (0.8 when the operands, beyond the 32 MB of the L2s, come from HBM, whose latency a
// CU's only workgroup waits for; 0.95 when two share a CU) plus two slabs' worth before and after its loop, 1.4 us per slab and
// 9 on a 256 x 256 tile; the chip holds 512 / 256 of them at a time; the second launch costs 5 us and the pass over the
// partial products runs at 3 TB/s.  The workgroups that count are those launched, the tiles of a batch and part rounded up to
// one per XCD (fewer than four small ones: to four): the empty ones leave at once but leave holes (8 x 27 x 704 x 7960, 6 tiles
// a batch: 25 us in 8 parts = 512 workgroups, 34 in 9; 64 x 16 x 512 x 1024, 4 tiles: 16 whole, 22 in 2).
static double split_k_time(unsigned tile, size_t bh, size_t m, size_t n, size_t k, size_t parts, size_t slabs) {
  const size_t tiles = ((m + tile - 1) / tile) * ((n + tile - 1) / tile);  // of a batch
  const size_t workgroups = (tile == 128 && tiles < 4 ? 4 : (tiles + 7) / 8 * 8) * bh * parts;
  const double rounds = (double)((workgroups + (tile == 128 ? 511 : 255)) / (tile == 128 ? 512 : 256));
  const bool far = bh * (m + n) * k * 2 > (size_t(32) << 20);
  const double loop = tile == 256 ? (double)slabs * 1.4 + 9.0 : (double)(slabs + 2) * (workgroups > 256 ? 0.95 : far ? 0.8 : 0.7);
  return rounds * loop + (parts > 1 ? 5.0 + (double)(bh * parts * m * n * 4) / 3e6 : 0.0);
}

// Tile of a product whose k loop is in parts.  The large one only where both extents fill it and the parts are long: on 110
// products from 20 x 100 x 512 to 3500 x 3500 x 12000 the best of all parts of 128-tiles is 1.19 times as fast as the best of
// 256-tiles, which lead on one (2854 x 1184 x 3880, 50.5 against 51.4 us; 402 x 896 x 2080 takes 14.2 on 128-tiles, 26.4 on those).
static unsigned split_k_tile(size_t bh, size_t m, size_t n, size_t k, unsigned splits) {
  if (m < 192 || n < 192) return 128;
  const size_t slabs = ((k + splits - 1) / splits + 63) / 64;
  return split_k_time(256, bh, m, n, k, splits, slabs) < split_k_time(128, bh, m, n, k, splits, slabs) ? 256 : 128;
}

// Into how many parts to cut k: by the model, parts of at least two slabs, where that gains 10 %.  Examples (whole -> parts):
// 64 x 8192 x 8192 79 -> 30 us in 8, 512 x 512 x 4096 52 -> 16, 461 x 1535 x 4592 55 -> 24 in 5, 256 x 256 x 65536 576 -> 32 in
// 32, 2 x 9304 x 2904 37 -> 17 in 5; left whole: 1024^3 (10 us), 2048^3 (28; 40 in 2).  The choice is 2.7 % behind the best of
// all parts in the mean of those 110 products; with 256-tiles wherever they fit and parts of at least 512 it was 20 %.
unsigned gemm_nt_bf16_split_k(size_t bh, size_t m, size_t n, size_t k, const KernelOptions& knobs) {
  if (bh == 0 || m == 0 || n == 0 || k % 8 != 0 || knobs.gemm_k_parts == 1) return 1;
  auto chunk_of = [k](size_t want) { return (k / want + 63) / 64 * 64; };  // what one part contracts: whole slabs
  if (knobs.gemm_k_parts > 1) {  // (tests, searches and measurements: that many parts)
    const size_t want = std::min<size_t>((size_t)knobs.gemm_k_parts, k / 64);
    if (want < 2 || bh * want > 65535) return 1;
    return (unsigned)((k + chunk_of(want) - 1) / chunk_of(want));
  }
  if (k < 1024 || k > (size_t(1) << 22)) return 1;  // (short loops: 45 x 936 x 880 9.9 us whole, 11.1 in 5 parts)
  const size_t slabs = (k + 63) / 64, t256 = ((m + 255) / 256) * ((n + 255) / 256);
  double best = split_k_time(128, bh, m, n, k, 1, slabs);
  if (t256 * bh >= 64) best = std::min(best, split_k_time(256, bh, m, n, k, 1, slabs));
  best *= 0.9;
  size_t splits = 1;
  for (size_t s = 2; s <= 32 && k / s >= 128 && bh * s <= 65535; ++s) {
    const size_t chunk = chunk_of(s), parts = (k + chunk - 1) / chunk;
    double t = split_k_time(128, bh, m, n, k, parts, chunk / 64);
    if (m >= 192 && n >= 192) t = std::min(t, split_k_time(256, bh, m, n, k, parts, chunk / 64));
    if (t < best) {
      best = t;
      splits = parts;
    }
  }
  return (unsigned)splits;
}

Err launch_gemm_nt_bf16_split_k(const void* a, const void* b, void* c, float* partial, unsigned splits, size_t bh, size_t m,
                                size_t n, size_t k, hipStream_t stream, LaunchNote* note, DType out_dtype) {
  if (!gemm_nt_bf16_supported(k)) return "gemm_nt kernel: k must be a positive multiple of 8";
  if (splits < 2 || bh * splits > 65535 || !fits_u32(m) || !fits_u32(n) || k > (size_t(1) << 22)) return "gemm_nt kernel: bad split";
  if (!a || !b || !c || !partial) return "gemm_nt kernel: null device pointer";
  if (!aligned16(a) || !aligned16(b)) return "gemm_nt kernel: operands must be 16-byte aligned";
  GemmParams p{};
  p.a = a; p.b = b; p.c = partial;
  p.bh = (uint32_t)bh; p.m = (uint32_t)m; p.n = (uint32_t)n; p.k = (uint32_t)k;
  p.k_chunk = (uint32_t)(((k + splits - 1) / splits + 63) / 64 * 64);
  splits = (unsigned)((k + p.k_chunk - 1) / p.k_chunk);  // (rounding the parts up to whole slabs may leave fewer of them)
  if (splits < 2) return "gemm_nt kernel: bad split";
  p.splits = splits;
  const unsigned tile = split_k_tile(bh, m, n, k, splits);
  p.tiles_m = (uint32_t)((m + tile - 1) / tile);
  p.tiles_n = (uint32_t)((n + tile - 1) / tile);
  const size_t grid = (size_t(p.tiles_m) * p.tiles_n + 7) / 8 * 8;
  if (grid > kMaxGrid) return "gemm_nt kernel: grid too large";
  const bool ktail = k % 64 != 0;  // (only the last split is partial; the others run whole slabs through the same code)
  const std::string name = std::string(tile == 256 ? "gemm_nt_bf16_256x256x64_direct" : "gemm_nt_bf16_128x128x64_direct") +
                           (ktail ? "_ktail" : "") + (tile == 256 ? "_w4" : "");
  if (note) *note = LaunchNote{name + " (k in " + std::to_string(splits) + " parts)", tile, tile};
  hipFunction_t fn;
  if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
  if (Err e = launch(fn, (unsigned)grid, (unsigned)(bh * splits), 1, 256, &p, sizeof(p), stream); !e.empty()) return e;
  SplitReduceParams r{partial, c, (uint32_t)bh, splits, (uint64_t)m * n, out_dtype == BF16 ? 1u : 0u};
  if (Err e = builtin_function("splitk_reduce", &fn); !e.empty()) return e;
  size_t rgrid = (bh * ((m * n + 3) / 4) + 255) / 256;
  if (rgrid > 65536) rgrid = 65536;
  return launch(fn, (unsigned)rgrid, 1, 1, 256, &r, sizeof(r), stream);
}

static unsigned gemm_nn_tile(size_t bh, size_t m, size_t n, size_t k, size_t tile_m, size_t tile_n, const KernelOptions& knobs, size_t b_cols) {
  if (k == 0 || k % 8 != 0 || b_cols % 8 != 0 || b_cols < n || b_cols > (size_t(1) << 24) || k > (size_t(1) << 22) || n > (size_t(1) << 24) || bh > 65535) return 0;
  if (!fits_u32(m) || !fits_u32(n)) return 0;
  const size_t t256 = ((m + 255) / 256) * ((n + 255) / 256) * bh, t128 = ((m + 127) / 128) * ((n + 127) / 128) * bh;
  unsigned tile = t256 >= 128 ? pick_direct_tile(t256, t128) : 128;
  if (tile_m == 256 && tile_n == 256) tile = 256;
  if (tile_m == 128 && tile_n == 128) tile = 128;
  if (knobs.gemm_tile) tile = knobs.gemm_tile == 192 ? 256u : (unsigned)knobs.gemm_tile;  // (192 x 256 exists for bf16 NT products only)
  if (!knobs.gemm_direct) tile = 0;  // (no register-staged form of this product: callers transpose and use the NT kernels)
  return tile;
}

bool gemm_nn_bf16_supported(size_t bh, size_t m, size_t n, size_t k, const KernelOptions& knobs) {
  return gemm_nn_tile(bh, m, n, k, 0, 0, knobs, n) != 0;
}

Err launch_gemm_nn_bf16(const void* a, const void* b, void* c, size_t bh, size_t m, size_t n, size_t k,
                        hipStream_t stream, size_t tile_m, size_t tile_n, LaunchNote* note, DType out_dtype, float* partial,
                        unsigned splits, const KernelOptions& knobs, size_t b_cols) {
  if (b_cols == 0) b_cols = n;
  unsigned tile = gemm_nn_tile(bh, m, n, k, tile_m, tile_n, knobs, b_cols);
  if (tile == 0) return "gemm_nn kernel: needs k % 8 == 0 and rows of B of a multiple of 8 elements (and extents within its offset range)";
  if (bh == 0 || m == 0 || n == 0) return {};
  if (!a || !b || !c) return "gemm_nn kernel: null device pointer";
  if (!aligned16(a) || !aligned16(b)) return "gemm_nn kernel: operands must be 16-byte aligned";
  GemmParams p{};
  p.a = a; p.b = b; p.c = c;
  p.bh = (uint32_t)bh; p.m = (uint32_t)m; p.n = (uint32_t)n; p.k = (uint32_t)k;
  p.out_bf16 = out_dtype == BF16 ? 1u : 0u;
  p.b_cols = (uint32_t)b_cols;
  // the k loop in parts over workgroups (gemm_nt_bf16_split_k says when, for this form too): f32 partial products
  // in the caller's temporary, added up by splitk_reduce
  if (splits > 1) {
    if (!partial) return "gemm_nn kernel: a split needs its temporary";
    p.k_chunk = (uint32_t)(((k + splits - 1) / splits + 63) / 64 * 64);
    splits = (unsigned)((k + p.k_chunk - 1) / p.k_chunk);  // (rounding the parts up to whole slabs may leave fewer of them)
    if (bh * splits > 65535) return "gemm_nn kernel: extent too large";
  }
  if (splits > 1) {
    p.splits = splits;
    p.c = partial;
    p.out_bf16 = 0;
    tile = split_k_tile(bh, m, n, k, splits);
  }
  p.tiles_m = (uint32_t)((m + tile - 1) / tile);
  p.tiles_n = (uint32_t)((n + tile - 1) / tile);
  const size_t grid = (size_t(p.tiles_m) * p.tiles_n + 7) / 8 * 8;  // the tiles in 8 equal runs, one per XCD
  if (grid > kMaxGrid) return "gemm_nn kernel: grid too large";
  hipFunction_t fn;
  const bool w4 = tile == 256 && knobs.gemm_waves != 8;  // (as for the NT kernels: four waves unless 8 are asked for)
  const std::string name = std::string(tile == 256 ? "gemm_nn_bf16_256x256x64_direct" : "gemm_nn_bf16_128x128x64_direct") +
                           (k % 64 != 0 ? "_ktail" : "") + (w4 ? "_w4" : "");
  if (note) *note = LaunchNote{splits > 1 ? name + " (k in " + std::to_string(splits) + " parts)" : name, tile, tile};
  if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
  if (Err e = launch(fn, (unsigned)grid, (unsigned)(bh * (splits > 1 ? splits : 1)), 1, tile == 256 && !w4 ? 512 : 256, &p, sizeof(p), stream);
      !e.empty() || splits <= 1)
    return e;
  SplitReduceParams r{partial, c, (uint32_t)bh, splits, (uint64_t)m * n, out_dtype == BF16 ? 1u : 0u};
  if (Err e = builtin_function("splitk_reduce", &fn); !e.empty()) return e;
  size_t rgrid = (bh * ((m * n + 3) / 4) + 255) / 256;
  if (rgrid > 65536) rgrid = 65536;
  return launch(fn, (unsigned)rgrid, 1, 1, 256, &r, sizeof(r), stream);
}

// Where B's one pass through registers beats the tiled kernels (us, tiled -> narrow).  f32 NT up to 32 rows: 30 x 4096
// x 4096 41 -> 28, 16 x 8192 x 8192 128 -> 66; from 33 rows on nothing is gained (64 x 8192 x 8192 130 -> 137).  f32 NN
// up to 64 rows, where the tiled kernel needs a transposed copy of B: 64 x 1024 x 16384 78 -> 42.  bf16, whose tiled
// kernel reads a large B at 5 TB/s, only where the tiled form's second launch weighs as much as B: NT, up to 16 rows,
// B of at most 40 MB and k up to 8192 (4 x 16384 x 1024 17.4 -> 11.8, 15 x 1248 x 4528 14.9 -> 11.8; 8 x 1024 x
// 16384 would go 16 -> 27).
bool gemm_narrow_usable(DType dtype, bool nn, size_t bh, size_t m, size_t n, size_t k, const KernelOptions& knobs) {
  if (knobs.gemm_tile || knobs.gemm_waves || knobs.gemm_k_parts || !knobs.gemm_direct) return false;  // (a tiled kernel is asked for)
  if (bh == 0 || bh > 65535 / 32 || m == 0 || n < 512 || k < 512 || !fits_u32(n) || k > (size_t(1) << 22)) return false;
  if (dtype == BF16) {
    // Batches of whole 64-wide slabs with many columns in all, or whose 128-tiles make one full round of workgroups: the
    // tiled kernels fill the chip then, unsplit, and read A once for 128 or 256 columns where this kernel reads it for every 32 (tiled -> narrow, us: 64
    // batches of 16 x 4096 x 512 66 -> 85, of 16 x 512 x 512 9.9 -> 11.5, 512 of 16 x 1024 x 1024 255 -> 284; but 64 of 1 x 4096
    // x 2048 255 -> 194, of 8 x 768 x 1024 41 -> 23, and off the slabs of 16 x 4096 x 520 91 -> 75).
    if (bh > 1 && k % 64 == 0) {
      const size_t t128 = bh * ((n + 127) / 128);
      if (n >= 2048 && bh * n >= 32768 && (k <= 1024 || m > 8)) return false;
      if (n >= 1024 && bh * n >= 262144 && k <= 1024 && m > 8) return false;
      if (m > 4 && t128 > 192 && t128 <= 256) return false;
    }
    return !nn && m <= 16 && k % 8 == 0 && k <= 8192 && n * k * 2 <= size_t(40) * 1000 * 1000;
  }
  return k % 4 == 0 && (nn ? m <= 64 && n % 4 == 0 : m <= 32);
}

// Columns of an NT workgroup: 32 (A is read half as often) where that leaves 192 workgroups or k is in parts, else 16: 16
// x 8192 x 8192 f32 79 us with 16, 66 with 32.
static size_t narrow_nt_tile(size_t bh, size_t n, unsigned splits) { return splits <= 1 && (n + 31) / 32 * bh < 192 ? 16 : 32; }

// f32 NT: the k loop in parts over workgroups of 32 columns, added up by a second launch, where the columns alone leave CUs
// idle or a last round nearly empty.  A workgroup's 16 wavefronts fill a CU, so the time goes by whole rounds of 256
// workgroups: 4 us, and per element of k 3.2 ns on 16 columns, 6 on 32 (5.6 and 9.5 above 16 rows); a split costs 4.5 more,
// and its many workgroups read B at 5 TB/s at most.  A single round has to hold every workgroup that is launched, the tiles of a batch and
// part rounded up to one per XCD (85 tiles in 3 parts are 264, and some CU gets two: 2 x 2713 x 14136 59 us so, 48 in 6 or whole);
// in later rounds the empty ones cost nothing (2 x 2345 x 9628, 74 tiles: 24.2 in 10 parts, 29.0 in 3).  Whole -> in parts, us: 12 x 4904 x 6696 60 -> 43, 3 x 1688 x 8896
// 31 -> 21, 5 x 2000 x 16000 56 -> 34, 24 x 1500 x 9000 54 -> 29, 31 x 1024 x 16000 98 -> 29; left whole: 30 x 4096 x 4096
// (28; 28 in 2), 16 x 8192 x 8192 (65; 73), 1 x 12952 x 6288 (69; 75 in 11).
static unsigned narrow_nt_f32_parts(size_t bh, size_t m, size_t n, size_t k) {
  auto time_of = [&](size_t tile, size_t parts) {
    const size_t tiles = (n + tile - 1) / tile, launched = (tiles + 7) / 8 * 8 * bh * parts;
    const double rounds = std::max((double)((tiles * bh * parts + 255) / 256), launched > 256 ? 2.0 : 1.0);
    const double loops = rounds * (double)(k / parts) * 1e-3 * (m <= 16 ? (tile == 16 ? 3.2 : 6.0) : (tile == 16 ? 5.6 : 9.5));
    return parts > 1 ? 8.5 + std::max(loops, (double)(bh * n * k) * 4 / 5e6) : 4 + loops;
  };
  double least = 0.9 * time_of(narrow_nt_tile(bh, n, 1), 1);
  unsigned best = 1;
  for (size_t s = 2; s <= 16 && k / s >= 512 && bh * s <= 65535; ++s)
    if (const double t = time_of(32, s); t < least) {
      least = t;
      best = (unsigned)s;
    }
  if (best < 2) return 1;
  const size_t chunk = ((k + best - 1) / best + 63) / 64 * 64;
  return (unsigned)((k + chunk - 1) / chunk);
}

// An NN workgroup takes 64 columns, and the k loop is cut into parts of at least 256, added up by a second launch, until
// there are three workgroups per CU (16 x 9808 x 4288 is 153 column tiles: 50 us in 2 parts, 41 in 6; 20 x 9000 x 6000
// 108 and 78).
unsigned gemm_narrow_parts(DType dtype, bool nn, size_t bh, size_t m, size_t n, size_t k) {
  if (!nn) return dtype == F32 ? narrow_nt_f32_parts(bh, m, n, k) : 1;
  const size_t tiles = (n + 63) / 64 * bh;
  if (tiles >= 576 || (tiles >= 192 && k < 2048)) return 1;  // (1 x 16384 x 1024: 14 us whole, 17 in 3 parts)
  const size_t want = std::min<size_t>(std::min<size_t>((768 + tiles - 1) / tiles, k / 256), 32);
  if (want < 2) return 1;
  const size_t chunk = (k / want + 63) / 64 * 64;
  return (unsigned)((k + chunk - 1) / chunk);
}

Err launch_gemm_narrow(const void* a, const void* b, void* c, DType dtype, bool nn, size_t bh, size_t m, size_t n, size_t k,
                       hipStream_t stream, LaunchNote* note, DType out_dtype, float* partial, unsigned splits) {
  if (m > (nn ? 64 : dtype == BF16 ? 16 : 32) || (nn && dtype == BF16) || bh * std::max(splits, 1u) > 65535 || k > (size_t(1) << 22) || !fits_u32(n)) return "narrow gemm kernel: extent too large";
  if (k % (dtype == BF16 ? 8 : 4) != 0 || (nn && n % 4 != 0)) return "narrow gemm kernel: unsupported extents";
  if (bh == 0 || m == 0 || n == 0) return {};
  if (!a || !b || !c) return "narrow gemm kernel: null device pointer";
  if (!aligned16(a) || !aligned16(b)) return "narrow gemm kernel: operands must be 16-byte aligned";
  GemmParams p{};
  p.a = a; p.b = b; p.c = c;
  p.bh = (uint32_t)bh; p.m = (uint32_t)m; p.n = (uint32_t)n; p.k = (uint32_t)k;
  p.out_bf16 = out_dtype == BF16 ? 1u : 0u;
  if (splits > 1) {
    if (!partial) return "narrow gemm kernel: a split needs its temporary";
    p.k_chunk = (uint32_t)(((k + splits - 1) / splits + 63) / 64 * 64);
    splits = (unsigned)((k + p.k_chunk - 1) / p.k_chunk);  // (rounding the parts up may leave fewer of them)
  }
  if (splits > 1) {
    p.splits = splits;
    p.c = partial;
    p.out_bf16 = 0;
  }
  const size_t tile = nn ? 64 : narrow_nt_tile(bh, n, splits);
  const std::string name = std::string(nn ? "gemm_nn_" : "gemm_nt_") + (dtype == BF16 ? "bf16" : "f32") + "_narrow" +
                           (m <= 16 ? "16x" : m <= 32 ? "32x" : "64x") + std::to_string(tile);
  if (note) *note = LaunchNote{splits > 1 ? name + " (k in " + std::to_string(splits) + " parts)" : name, 0, 0};
  hipFunction_t fn;
  if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
  if (Err e = launch(fn, (unsigned)(((n + tile - 1) / tile + 7) / 8 * 8), (unsigned)(bh * std::max(splits, 1u)), 1, tile < 64 ? 1024 : 512, &p, sizeof(p), stream);
      !e.empty() || splits <= 1)
    return e;
  SplitReduceParams r{partial, c, (uint32_t)bh, splits, (uint64_t)m * n, out_dtype == BF16 ? 1u : 0u};
  if (Err e = builtin_function("splitk_reduce", &fn); !e.empty()) return e;
  const size_t rgrid = std::min<size_t>((bh * ((m * n + 3) / 4) + 255) / 256, 65536);
  return launch(fn, (unsigned)rgrid, 1, 1, 256, &r, sizeof(r), stream);
}

bool gemm_nt_f32_supported(size_t k) { return k > 0 && k % 4 == 0 && k <= (size_t(1) << 21); }

// Tile and parts of k of an f32 product, by a model of the time in us.  Its matrix instructions are the bound (157
// TFLOP/s, a sixteenth of bf16) and the workgroups of a CU share them, so the time is what the fullest CU has to do: 1.7
// per 32-wide slab of a 128 x 128 tile, a quarter of it, 0.46, of a 64 x 64 one, plus two slabs' worth before and after
// the loop.  A workgroup has one slab in flight, though, and operands beyond the 32 MB of the L2s take 0.7 to arrive: a
// CU with a single small tile waits for them.  A split costs 4 for the second launch and the pass over the partial
// products at 3 TB/s, parts have at least 64 of k, and a split has to gain 15 %.  256 x 256 tiles where they fill at
// least half of the CUs.  Measured (128 x 128 tiles in parts -> this rule): 1000 x 1500 x 700 34 -> 26 us, 1024^3 27 ->
// 18 (118 TFLOP/s), 128 x 128 x 4096 28 -> 16 in 32 parts, 777 x 999 x 1001 with a row-major right operand, padded
// copies included, 88 -> 30; 100 x 8000 x 8000 takes 176 on whole 64-tiles, a CU each, and 129 on 128-tiles in 4
// parts; 64 x 8192 x 8192 105 on 64-tiles in 2 parts, 88 in 4.
struct F32Plan {
  unsigned tile, splits;
};
static F32Plan f32_plan(size_t bh, size_t m, size_t n, size_t k, const KernelOptions& knobs, bool whole) {
  const size_t t256 = ((m + 255) / 256) * ((n + 255) / 256) * bh;
  auto parts_of = [&](size_t want) -> unsigned {
    if (whole || want < 2 || bh * want > 65535) return 1;
    const size_t chunk = (k / want + 63) / 64 * 64;  // what one split contracts: whole slabs
    return (unsigned)((k + chunk - 1) / chunk);
  };
  const unsigned asked = knobs.gemm_tile == 0 ? 0u : knobs.gemm_tile == 192 ? 256u : (unsigned)knobs.gemm_tile;  // (192 x 256 exists for bf16 NT products only)
  if (knobs.gemm_k_parts > 1) return {asked ? asked : t256 >= 128 ? 256u : 128u, parts_of(std::min<size_t>((size_t)knobs.gemm_k_parts, k / 64))};
  if ((asked == 256 || !asked) && t256 >= 128) return {256, 1};
  const size_t slabs = (k + 31) / 32;
  const bool far = bh * (m + n) * k * 4 > (size_t(32) << 20);
  F32Plan best{asked ? asked : 128u, 1};
  double best_time = 1e30;
  for (unsigned tile : {256u, 128u, 64u}) {
    if (asked ? tile != asked : tile == 256) continue;
    const size_t tiles = ((m + tile - 1) / tile) * ((n + tile - 1) / tile) * bh;
    for (size_t s = 1; s <= 32 && (s == 1 || (!whole && knobs.gemm_k_parts != 1 && k / s >= 64 && bh * s <= 65535)); ++s) {
      // (A single round of parts of large tiles has to hold every workgroup that is launched, the tiles of a batch and part rounded up
      // to one per XCD: 85 tiles of 128 in 3 parts are 264, and some CU gets two.  605 x 2151 x 3224 136 us so, 90 on 64-tiles.  Of
      // those a second one costs little: 815 x 122 x 1560, 26 tiles, 12.3 in 9 parts, 14.2 in 7.)
      const bool crowded = tile >= 128 && s > 1 && (tiles / bh + 7) / 8 * 8 * bh * s > 256;
      const double resident = std::max((double)((tiles * s + 255) / 256), crowded ? 2.0 : 1.0);
      double t = (double)((slabs + s - 1) / s + 2) * std::max(resident * (tile == 256 ? 6.8 : tile == 128 ? 1.7 : 0.46), far ? 0.7 : 0.0);
      if (s > 1) t = (t + 4.0 + (double)(bh * s * m * n * 4) / 3e6) / 0.85;
      if (t < best_time) {
        best_time = t;
        best = {tile, (unsigned)s};
      }
    }
  }
  best.splits = parts_of(best.splits);
  return best;
}

unsigned gemm_nt_f32_split_k(size_t bh, size_t m, size_t n, size_t k, const KernelOptions& knobs) {
  if (bh == 0 || m == 0 || n == 0 || !gemm_nt_f32_supported(k) || knobs.gemm_k_parts == 1) return 1;
  return f32_plan(bh, m, n, k, knobs, false).splits;
}

Err launch_gemm_nt_f32(const float* a, const float* b, float* c, size_t bh, size_t m, size_t n, size_t k,
                       hipStream_t stream, LaunchNote* note, float* partial, unsigned splits, const KernelOptions& knobs, size_t b_cols) {
  if (!gemm_nt_f32_supported(k)) return "gemm_nt f32 kernel: k must be a positive multiple of 4 (at most 2^21)";
  if (reinterpret_cast<uintptr_t>(a) % 16 != 0 || reinterpret_cast<uintptr_t>(b) % 16 != 0)
    return "gemm_nt f32 kernel: operands must be 16-byte aligned";
  if (bh == 0 || m == 0 || n == 0) return {};
  if (!fits_u32(m) || !fits_u32(n) || bh > 65535) return "gemm_nt f32 kernel: extent too large";
  if (!a || !b || !c) return "gemm_nt f32 kernel: null device pointer";
  const bool nn = b_cols != 0;
  if (nn && (b_cols % 4 != 0 || b_cols < n || b_cols > (size_t(1) << 24))) return "gemm_nn f32 kernel: needs rows of B of a multiple of 4 elements (at most 2^24)";
  GemmParams p{};
  p.a = a; p.b = b; p.c = c;
  p.bh = (uint32_t)bh; p.m = (uint32_t)m; p.n = (uint32_t)n; p.k = (uint32_t)k;
  p.b_cols = (uint32_t)b_cols;
  const unsigned tile = f32_plan(bh, m, n, k, knobs, splits <= 1).tile;
  // the k loop in parts over workgroups (gemm_nt_f32_split_k says when): partial products in the caller's temporary
  if (splits > 1) {
    if (!partial) return "gemm_nt f32 kernel: a split needs its temporary";
    p.k_chunk = (uint32_t)(((k + splits - 1) / splits + 63) / 64 * 64);
    splits = (unsigned)((k + p.k_chunk - 1) / p.k_chunk);  // (rounding the parts up to whole slabs may leave fewer of them)
    if (bh * splits > 65535) return "gemm_nt f32 kernel: extent too large";
  }
  if (splits > 1) {
    p.splits = splits;
    p.c = partial;
  }
  p.tiles_m = (uint32_t)((m + tile - 1) / tile);
  p.tiles_n = (uint32_t)((n + tile - 1) / tile);
  const size_t grid = (size_t(p.tiles_m) * p.tiles_n + 7) / 8 * 8;  // the tiles in 8 equal runs, one per XCD
  if (grid > kMaxGrid) return "gemm_nt f32 kernel: grid too large";
  hipFunction_t fn;
  const std::string edge = std::to_string(tile);
  const std::string name = "gemm_nt_f32_" + edge + "x" + edge + "x32_direct" + (k % 32 != 0 ? "_ktail" : "") + (nn ? "_brow" : "");
  // (_ktail: a partial last slab of 32 k; of the last part, when split)
  if (note) *note = LaunchNote{splits > 1 ? name + " (k in " + std::to_string(splits) + " parts)" : name, tile, tile};
  if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
  if (Err e = launch(fn, (unsigned)grid, (unsigned)(bh * (splits > 1 ? splits : 1)), 1, tile == 256 ? 512 : 256, &p, sizeof(p), stream);
      !e.empty() || splits <= 1)
    return e;
  SplitReduceParams r{partial, c, (uint32_t)bh, splits, (uint64_t)m * n, 0u};
  if (Err e = builtin_function("splitk_reduce", &fn); !e.empty()) return e;
  size_t rgrid = (bh * ((m * n + 3) / 4) + 255) / 256;
  if (rgrid > 65536) rgrid = 65536;
  return launch(fn, (unsigned)rgrid, 1, 1, 256, &r, sizeof(r), stream);
}

// Into how many parts to cut each row of a softmax (1: do not): fewer rows than half the CUs, each of 2^17 columns
// and more, which one workgroup per row would leave to a few CUs; parts of at least 2^15 columns, as many as give
// every CU a workgroup.
unsigned row_softmax_parts(size_t rows, size_t cols, int mode) {
  if ((mode != 0 && mode != 4) || rows == 0 || rows > 128 || cols < (size_t(1) << 17)) return 1;
  const size_t parts = std::min<size_t>(std::min<size_t>(256 / rows, cols >> 15), 64);
  return parts < 2 ? 1u : (unsigned)parts;
}

// Groups of 8 elements that a row of the row_*_any_* kernels spans at most, `shift` being where its operand starts
// (in elements past a 16-byte boundary).
static size_t row_groups(size_t cols, unsigned shift) { return cols % 8 == 0 && shift == 0 ? cols / 8 : (cols + 14) / 8; }

bool row_softmax_any_supported(size_t cols) { return cols <= 65536; }

Err launch_row_softmax(const void* x, void* y, size_t rows, size_t cols, hipStream_t stream, int mode, LaunchNote* note,
                       const float* scale_ptr, float scale, float* stats, unsigned parts, DType in_dtype, DType out_dtype) {
  if (rows == 0 || cols == 0) return {};
  if (!fits_u32(rows) || !fits_u32(cols)) return "row_softmax kernel: extent exceeds 32 bits";
  if (!x || !y) return "row_softmax kernel: null device pointer";
  if (mode < 0 || mode > 4) return "row_softmax kernel: unknown mode";
  if (mode == 4 && !std::isfinite(scale)) return "row_softmax kernel: unsupported scale (must be finite)";
  static const char* const kOps[5] = {"softmax", "shift", "norm", "exp", "scaled_softmax"};
  SoftmaxParams p{x, y, (uint32_t)rows, (uint32_t)cols, scale_ptr, scale};
  hipFunction_t fn;
  const bool f32 = in_dtype == F32 && out_dtype == F32;
  if (!f32 && (!row_softmax_any_supported(cols) || mode == 4)) return "row_softmax kernel: bf16 rows are too long (or scaled)";
  const bool vec = f32 && cols % 4 == 0 && (reinterpret_cast<uintptr_t>(x) % 16 == 0) && (reinterpret_cast<uintptr_t>(y) % 16 == 0);
  if (f32 && parts > 1 && (mode == 0 || mode == 4)) {
    // every row in parts over workgroups: the parts' (max, sum) pairs into `stats`, then a second launch that
    // combines them and writes
    if (!stats) return "row_softmax kernel: rows in parts need their temporary";
    const size_t chunks = vec ? cols / 4 : cols;
    p.part_chunks = (uint32_t)((chunks + parts - 1) / parts);
    p.parts = (uint32_t)((chunks + p.part_chunks - 1) / p.part_chunks);
    p.stats = stats;
    if (rows * p.parts > kMaxGrid) return "row_softmax kernel: grid too large";
    const std::string base = std::string("row_") + kOps[mode] + "_parts_";
    if (note) *note = LaunchNote{base + "stats" + (vec ? "_v" : "") + " + " + base + "apply" + (vec ? "_v" : "") + " (rows in " + std::to_string(p.parts) + " parts)", 0, 0};
    if (Err e = builtin_function((base + "stats" + (vec ? "_v" : "")).c_str(), &fn); !e.empty()) return e;
    if (Err e = launch(fn, (unsigned)(rows * p.parts), 1, 1, 1024, &p, sizeof(p), stream); !e.empty()) return e;
    if (Err e = builtin_function((base + "apply" + (vec ? "_v" : "")).c_str(), &fn); !e.empty()) return e;
    return launch(fn, (unsigned)(rows * p.parts), 1, 1, 1024, &p, sizeof(p), stream);
  }
  // f32 rows whose length is a multiple of 4 and that start on 16-byte boundaries: float4 chunks.  Every other row
  // that registers hold (odd lengths, other alignments, bf16 on either side): groups of 8 elements; but f32 rows of
  // at most 128 columns keep the form with few lanes per row (2000000 x 31: 114 against 209 us).
  if (!vec && mode != 4 && row_softmax_any_supported(cols) && !(f32 && cols <= 128)) {
    const size_t in_elem = in_dtype == BF16 ? 2 : 4, out_elem = out_dtype == BF16 ? 2 : 4;
    const size_t x_shift = reinterpret_cast<uintptr_t>(x) % 16 / in_elem, y_shift = reinterpret_cast<uintptr_t>(y) % 16 / out_elem;
    p.in_bf16 = in_dtype == BF16;
    p.out_bf16 = out_dtype == BF16;
    p.x_shift = (uint32_t)x_shift;
    p.y_wide = (8 + x_shift - y_shift) % (16 / out_elem) == 0;
    const size_t groups = row_groups(cols, p.x_shift);
    // Lanes per row and groups per lane: one group per lane up to 32 groups, a wavefront up to 512, then workgroups
    // of 256 and 1024 lanes, with the least number of groups per lane that covers the row.
    size_t lanes = 2, each = 1;
    std::string form;
    if (groups <= 32) {
      while (lanes < groups) lanes *= 2;
      form = "lanes_s" + std::to_string(lanes);
    } else {
      lanes = groups <= 512 ? 64 : groups <= 2048 ? 256 : 1024;
      static const size_t kEach[3][6] = {{1, 2, 3, 4, 6, 8}, {3, 4, 8, 8, 8, 8}, {3, 4, 6, 9, 9, 9}};
      for (size_t n : kEach[lanes == 64 ? 0 : lanes == 256 ? 1 : 2]) {
        each = n;
        if (lanes * n >= groups) break;
      }
      form = lanes == 64 ? "wave_s" + std::to_string(2 * each) : "group_s" + std::to_string(8 * lanes * each / 4096);
    }
    const std::string name = std::string("row_") + kOps[mode] + "_" + form;
    if (note) *note = LaunchNote{name, 0, 0};
    if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
    const size_t threads = lanes > 256 ? lanes : 256, grid = (rows * lanes + threads - 1) / threads;
    if (grid > kMaxGrid) return "row_softmax kernel: grid too large";
    return launch(fn, (unsigned)grid, 1, 1, (unsigned)threads, &p, sizeof(p), stream);
  }
  if (f32 && cols <= 128) {
    // G lanes per row, one float4 chunk each: 64 / G rows per wavefront
    size_t g = 1;
    while (4 * g < cols) g *= 2;
    const std::string name = std::string("row_") + kOps[mode] + "_sub_" + (vec ? "v" : "s") + std::to_string(g);
    if (note) *note = LaunchNote{name, 0, 0};
    if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
    const size_t grid = (rows * g + 255) / 256;
    if (grid > kMaxGrid) return "row_softmax kernel: grid too large";
    return launch(fn, (unsigned)grid, 1, 1, 256, &p, sizeof(p), stream);
  }
  if (vec && cols <= 8192) {
    int nv = 1;
    while ((size_t)256 * nv < cols) nv *= 2;
    const std::string name = std::string("row_") + kOps[mode] + "_wave_v" + std::to_string(nv);
    if (note) *note = LaunchNote{name, 0, 0};
    if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
    const size_t grid = (rows + 3) / 4;  // four wavefronts (rows) per workgroup
    if (grid > kMaxGrid) return "row_softmax kernel: grid too large";
    return launch(fn, (unsigned)grid, 1, 1, 256, &p, sizeof(p), stream);
  }
  if (rows > kMaxGrid) return "row_softmax kernel: grid too large";
  if (vec && cols <= 65536) {
    // the row still fits the registers of one workgroup of 16 wavefronts: one read and one write per element
    const int nv = cols <= 16384 ? 4 : cols <= 32768 ? 8 : 16;
    const std::string name = std::string("row_") + kOps[mode] + "_group_v" + std::to_string(nv);
    if (note) *note = LaunchNote{name, 0, 0};
    if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
    return launch(fn, (unsigned)rows, 1, 1, 1024, &p, sizeof(p), stream);
  }
  // wider rows: two passes over the row (one for exp, elementwise)
  const std::string name = std::string("row_") + kOps[mode] + (vec ? "_block_v" : "_block");
  if (note) *note = LaunchNote{name, 0, 0};
  if (Err e = builtin_function(name.c_str(), &fn); !e.empty()) return e;
  return launch(fn, (unsigned)rows, 1, 1, 1024, &p, sizeof(p), stream);
}

Err launch_transpose(const void* src, void* dst, size_t bh, size_t rows, size_t cols, size_t elem_bytes,
                     hipStream_t stream) {
  if (elem_bytes != 2 && elem_bytes != 4) return "transpose kernel: element size must be 2 or 4 bytes";
  if (bh == 0 || rows == 0 || cols == 0) return {};
  if (!fits_u32(bh) || !fits_u32(rows) || !fits_u32(cols)) return "transpose kernel: extent exceeds 32 bits";
  if (!src || !dst) return "transpose kernel: null device pointer";
  TransposeParams p{};
  p.src = src; p.dst = dst;
  p.bh = (uint32_t)bh; p.rows = (uint32_t)rows; p.cols = (uint32_t)cols;
  p.tiles_r = (uint32_t)((rows + 63) / 64);
  p.tiles_c = (uint32_t)((cols + 63) / 64);
  const size_t grid = bh * p.tiles_r * p.tiles_c;
  if (grid > kMaxGrid) return "transpose kernel: grid too large";
  hipFunction_t fn;
  if (Err e = builtin_function(elem_bytes == 2 ? "transpose_b16" : "transpose_b32", &fn); !e.empty()) return e;
  return launch(fn, (unsigned)grid, 1, 1, 256, &p, sizeof(p), stream);
}

Err launch_convert(const void* src, void* dst, DType from, DType to, size_t n, hipStream_t stream) {
  if (n == 0) return {};
  if (from == to) return "convert kernel: identical dtypes";
  ConvertParams p{src, dst, (uint64_t)n};
  hipFunction_t fn;
  if (Err e = builtin_function(from == F32 ? "convert_f32_to_bf16" : "convert_bf16_to_f32", &fn); !e.empty()) return e;
  size_t grid = (n + 255) / 256;
  if (grid > 65536) grid = 65536;
  return launch(fn, (unsigned)grid, 1, 1, 256, &p, sizeof(p), stream);
}

Err launch_pad_rows(const void* src, void* dst, size_t rows, size_t cols, size_t cols_padded, size_t elem_bytes,
                    hipStream_t stream) {
  if (elem_bytes != 2 && elem_bytes != 4) return "pad kernel: element size must be 2 or 4 bytes";
  if (rows == 0 || cols_padded == 0) return {};
  if (!fits_u32(cols_padded) || cols > cols_padded) return "pad kernel: bad extents";
  if (!src || !dst) return "pad kernel: null device pointer";
  PadParams p{src, dst, (uint64_t)rows, (uint32_t)cols, (uint32_t)cols_padded};
  hipFunction_t fn;
  if (Err e = builtin_function(elem_bytes == 2 ? "pad_rows_b16" : "pad_rows_b32", &fn); !e.empty()) return e;
  size_t grid = (rows * cols_padded + 255) / 256;
  if (grid > 65536) grid = 65536;
  return launch(fn, (unsigned)grid, 1, 1, 256, &p, sizeof(p), stream);
}

Err launch_pad_pair(const PadPair& pair, unsigned count, size_t batches, size_t elem_bytes, hipStream_t stream) {
  if (count < 1 || count > 2) return "pad kernel: one operand or two";
  if (elem_bytes != 2 && elem_bytes != 4) return "pad kernel: element size must be 2 or 4 bytes";
  PadPairParams p{};
  p.batches = (uint32_t)batches;
  size_t most = 0;
  for (unsigned o = 0; o < count; ++o) {
    if (pair.cols[o] > pair.cols_padded[o] || pair.rows[o] > pair.rows_padded[o] || pair.cols_padded[o] * elem_bytes % 16 != 0) return "pad kernel: bad extents";
    const size_t chunks = batches * pair.rows_padded[o] * (pair.cols_padded[o] * elem_bytes / 16);
    if (chunks == 0) return "pad kernel: bad extents";
    if (chunks >= (size_t(1) << 31) || !fits_u32(pair.cols_padded[o])) return "pad kernel: extent too large";
    if (!pair.src[o] || !pair.dst[o]) return "pad kernel: null device pointer";
    if (!aligned16(pair.dst[o])) return "pad kernel: the copies must be 16-byte aligned";
    most = std::max(most, chunks);
    p.src[o] = pair.src[o];
    p.dst[o] = pair.dst[o];
    p.rows[o] = (uint32_t)pair.rows[o];
    p.rows_padded[o] = (uint32_t)pair.rows_padded[o];
    p.cols[o] = (uint32_t)pair.cols[o];
    p.cols_padded[o] = (uint32_t)pair.cols_padded[o];
  }
  hipFunction_t fn;
  if (Err e = builtin_function(elem_bytes == 2 ? "pad_pair_b16" : "pad_pair_b32", &fn); !e.empty()) return e;
  // (index arithmetic in 32 bits: at most 2^31 chunks and 2^24 work-items past them)
  const size_t grid = std::min<size_t>((most + 255) / 256, 65536);
  return launch(fn, (unsigned)grid, count, 1, 256, &p, sizeof(p), stream);
}

}  // namespace ihip
