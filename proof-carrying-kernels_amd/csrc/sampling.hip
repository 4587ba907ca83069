// Set-sampling checker: checks that a sampler's selected set is a valid top-k set, or a valid
// minimal top-p nucleus, of each row of FP32 logits.  The GPU form of the CPU checker
// (reference src/pck/sampling.py:91-122); the reference's kernel is
// src/pck/cuda/csrc/sampling_kernel.cu:38-229.
//
// For row b with selection sel[b, 0 .. len[b]) over V logits:
//   top-k passes iff the selection is well formed (every index in range, none twice, length k),
//     no logit is NaN and min(selected) >= max(rejected) (-inf when nothing is rejected);
//   top-p also needs mass >= p - slack and mass_without_smallest < p + slack, where
//     mass = sum_sel e / sum_all e and mass_without_smallest drops e of the smallest selected
//     logit, e = exp((l - M) / T), M the row maximum.  `slack` comes from the host: the
//     sampler's declared error plus the bound below for this kernel's own rounding.
// min(selected) and max(rejected) are exact (FP32 comparisons).  Each e is an FP32
// 2^d on the split argument d = (l - m) log2(e) / T = hi + lo in two floats, within 0.8 FP32 ulps
// for every |d| (an FP32 argument alone would lose |d| ulps), 0 for e < 2^-150 (masked -inf logits
// among them); the sums are FP64.
//
// Launches on the caller's stream; nothing depends on scheduling:
//   mark:    (selections longer than kLdsSelect only) one lane per selected entry sets its bit
//            in the row's bitmap (caller-zeroed scratch) with a device-scope atomic OR.  An
//            index out of range, or one whose bit was already set, marks the row malformed (a
//            plain store of 1 to the row's flag).
//   segment: a workgroup per (row, segment of ceil(V / S) logits).  For selections of at most
//            kLdsSelect entries it first builds its segment's bitmap in LDS from the selection
//            itself (LDS atomic OR: a bit already set is a duplicate; segment 0 also flags
//            indices out of range), so those calls need no scratch and no mark launch.  It then
//            forms the exact min over the selected, max over the rejected and over all logits,
//            a NaN flag and, for top-p, the FP64 sums of e^((l - m_s) / T) over all and over
//            the selected logits relative to the segment's own maximum m_s, in a fixed order
//            (lane, then wave butterfly, then the waves' sums rescaled from each wave's own
//            maximum to m_s with one FP64 exp and multiply).
//   finish:  a wave per row; lane i merges segments i, i + 64, ... in order (M = max m_s,
//            z_s e^((m_s - M) / T) with FP64 exp, multiply and add), the lanes meet in a fixed
//            butterfly, and lane 0 decides.
// The reference merges in the last segment to finish through an atomic ticket; here a third
// launch does it, so no workgroup waits on another's writes across the per-XCD L2 caches.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

#include "exp2_term.h"
#include "pck_hip.h"

namespace pck {
namespace {

constexpr int kThreads = 256;
constexpr int kWave = 64;
constexpr int kWaves = kThreads / kWave;
constexpr int kAhead = 8;  // logits in flight per lane
constexpr int64_t kLdsSelect = 4096;      // selections up to this length are read per segment
constexpr int64_t kLdsBits = 1 << 18;     // the largest segment bitmap kept in LDS (32 KiB)
constexpr uint32_t kNanFlag = 1u, kMalformedFlag = 2u;

struct Partial {
  float min_sel, max_rej, max_all;
  uint32_t flags;  // kNanFlag, kMalformedFlag
  double z, z_sel;
};
static_assert(sizeof(Partial) == 32, "partial layout");

struct Args {
  const float* logits;
  const int64_t* sel;
  const int64_t* len;  // (rows,), or NULL: every row is max_len long
  int64_t rows, vocab, max_len, k;
  int top_p;
  double p, temperature, slack;
  int64_t segments, seg_len, words;
  uint32_t* bitmap;  // (rows, words); unused when the selection bitmap is built in LDS
  uint32_t* flags;   // (rows,): nonzero = malformed
  Partial* partials; // (rows, segments)
  uint8_t* passed;
  float* min_sel;
  float* max_rej;
  double* mass;
  double* without;
};

// The selection length of a row (every row is max_len long without a lengths array).
__device__ __forceinline__ int64_t row_length(const Args& a, int64_t row) {
  return a.len ? a.len[row] : a.max_len;
}

__global__ void __launch_bounds__(kThreads) mark_kernel(const Args a) {
  const int64_t row = blockIdx.y;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  const int64_t n = row_length(a, row) < a.max_len ? row_length(a, row) : a.max_len;
  if (i >= n) return;
  const int64_t idx = a.sel[row * a.max_len + i];
  if (idx < 0 || idx >= a.vocab) {
    a.flags[row] = 1u;
    return;
  }
  const uint32_t bit = 1u << (idx & 31);
  if (atomicOr(&a.bitmap[row * a.words + (idx >> 5)], bit) & bit) a.flags[row] = 1u;
}

__device__ __forceinline__ bool selected(const uint32_t* bits, int64_t j) {
  return (bits[j >> 5] >> (j & 31)) & 1u;
}

// The first kAhead kThreads entries of a row's selection, requested ahead of the logits (loads
// return in order, so entries requested behind them would wait for them); an entry past the
// selection reads the last one and is not used.
__device__ __forceinline__ void request_selection(const int64_t* sel, int64_t max_len,
                                                  int64_t (&v)[kAhead]) {
#pragma unroll
  for (int e = 0; e < kAhead; ++e) {
    const int64_t i = static_cast<int>(threadIdx.x) + e * kThreads;
    v[e] = sel[i < max_len ? i : max_len - 1];
  }
}

// Builds the segment's selection bitmap in LDS from the row's selection (bit j - j0 for index
// j in [j0, j1)), whose first entries are in v; returns this lane's malformed finding (a
// duplicate in the segment, or, in segment 0, an index out of range).
__device__ __forceinline__ bool build_lds_bitmap(const Args& a, int64_t row, int64_t seg,
                                                 int64_t j0, int64_t j1, int64_t n, uint32_t* lds,
                                                 int64_t (&v)[kAhead]) {
  const int t = static_cast<int>(threadIdx.x);
  const int words = static_cast<int>((j1 - j0 + 31) / 32);
  for (int w = t; w < words; w += kThreads) lds[w] = 0u;
  __syncthreads();
  const int64_t* sel = a.sel + row * a.max_len;
  bool bad = false;
  auto mark = [&](int64_t i0) {
#pragma unroll
    for (int e = 0; e < kAhead; ++e) {
      const bool live = i0 + e * kThreads < n;
      const uint64_t off = static_cast<uint64_t>(v[e] - j0);
      bad |= seg == 0 && live && static_cast<uint64_t>(v[e]) >= static_cast<uint64_t>(a.vocab);
      if (live && off < static_cast<uint64_t>(j1 - j0)) {
        const uint32_t bit = 1u << (off & 31);
        bad |= (atomicOr(&lds[off >> 5], bit) & bit) != 0u;
      }
    }
  };
  mark(t);
  for (int64_t i0 = t + kAhead * kThreads; i0 < n; i0 += kAhead * kThreads) {
#pragma unroll
    for (int e = 0; e < kAhead; ++e) {
      const int64_t i = i0 + static_cast<int64_t>(e) * kThreads;
      v[e] = sel[i < n ? i : n - 1];
    }
    mark(i0);
  }
  __syncthreads();
  return bad;
}

// log2(e) / T as an unevaluated sum of two floats (48 bits).
struct InvT {
  float hi, lo;
};
constexpr double kLog2E = 1.4426950408889634074;
__device__ __forceinline__ InvT inverse(double temperature) {
  const double v = kLog2E / temperature;
  const float hi = static_cast<float>(v);
  return InvT{hi, static_cast<float>(v - static_cast<double>(hi))};
}

// Whether d = (l - m) log2(e) / T is formed in two floats; in FP64 for a temperature whose
// inverse, or whose products, could leave the FP32 range.
__device__ __forceinline__ bool float_quotient(double temperature) {
  return temperature >= 0x1p-40 && temperature <= 0x1p40;
}

// e^((l - m) / T) = 2^d, d = hi + lo (exp2_term.h).  l - m is exact (Knuth's TwoSum) and the product
// with log2(e) / T within 2^-44 relative, so d is within 2^-36 at |d| = 150 against the 2^-24 of the
// FP32 terms.  log2(e) rides in the constant, so no term pays a reduction of its own base.
template <bool kFloats>
__device__ __forceinline__ double term(float l, float m, const InvT& inv, double temperature) {
  float hi, lo;
  if constexpr (!kFloats) {
    const double d = (static_cast<double>(l) - static_cast<double>(m)) / temperature * kLog2E;
    hi = static_cast<float>(d);
    lo = static_cast<float>(d - static_cast<double>(hi));
  } else {
    const float nm = -m;
    const float s = l + nm;
    const float bv = s - l;
    const float err = (l - (s - bv)) + (nm - bv);
    hi = s * inv.hi;
    lo = __builtin_fmaf(s, inv.hi, -hi);
    lo = __builtin_fmaf(s, inv.lo, lo);
    lo = __builtin_fmaf(err, inv.hi, lo);
  }
  return exp2_pair(hi, lo);  // 0 for -inf logits; a NaN logit is flagged elsewhere
}

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) v = fminf(v, __shfl_xor(v, o, kWave));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
  return v;
}
// The same bits on every lane: at each level both partners add the same two values.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) v = v + __shfl_xor(v, o, kWave);
  return v;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_any __attribute__((aligned(4)));  // a segment may start at any logit

// The selection bits of logits j .. j + 3 (below `end`).  kLds: j is a multiple of 4 (relative
// to the segment), so they are one nibble of one word.
template <bool kLds>
__device__ __forceinline__ uint32_t selected4(const uint32_t* bits, int64_t j, int64_t end) {
  if constexpr (kLds) {
    const int i = static_cast<int>(j), last = static_cast<int>(end) - 1;
    const uint32_t nib = (bits[(i < last ? i : last) >> 5] >> (i & 31)) & 15u;
    return i <= last ? nib : 0u;
  } else {
    uint32_t n = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) n |= (j + k < end && selected(bits, j + k) ? 1u : 0u) << k;
    return n;
  }
}

// The larger of v and its DPP partner; four steps reduce a row of 16 lanes.
template <int kCtrl>
__device__ __forceinline__ float dpp_max(float v) {
  return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xF, 0xF,
                                                             false)));
}
__device__ __forceinline__ float lane_float(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// The wave's maximum, uniform, in VALU moves.
__device__ __forceinline__ float uniform_max(float v) {
  v = dpp_max<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v = dpp_max<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v = dpp_max<0x124>(v);  // row_ror 4
  v = dpp_max<0x128>(v);  // row_ror 8
  return fmaxf(fmaxf(lane_float(v, 0), lane_float(v, 16)),
               fmaxf(lane_float(v, 32), lane_float(v, 48)));
}

// A workgroup reads its segment once, kChunk logits at a time in registers (16-byte loads at any
// 4-byte address), the next chunk's loads in flight while one is used: its extremes, then, for
// top-p, its terms relative to the wave's largest logit so far (a wave's sums are rescaled in
// FP64 when a chunk raises that).  Top-k is bound by the loads, top-p by the terms' arithmetic
// (about 28 instructions a logit), so a wave without a selected logit in its chunk (nearly all)
// skips what the selection needs.  The selection's entries are requested ahead of the logits and
// every load is unconditional: loads return in order, and a branch around one makes all later
// uses wait for everything in flight.  Both launches at 151,936 logits a row, against two passes
// over memory with an FP64 division and an LDS read per logit: top-p 64 rows 22.1 against 33.3
// us, 256 rows 49.4 against 108; top-k 50 256 rows 30.1 against 47.4 us (5.2 TB/s).
//
// kQuads: 16-byte loads per lane and chunk.  kOne: every segment is at most one chunk, so there is no
// next one to request; launch_segments has the forms.
constexpr int kLongQuads = 5;  // of segments of several chunks

template <bool kLds, int kQuads, bool kOne>
__global__ void __launch_bounds__(kThreads) segment_kernel(const Args a) {
  constexpr int kChunk = kQuads * 4 * kThreads;  // logits per chunk
  extern __shared__ uint32_t lds_bits[];  // kLds: the segment's bitmap
  __shared__ float fred[3][kWaves];
  __shared__ double dred[2][kWaves];
  __shared__ uint32_t any_flag;
  const int t = static_cast<int>(threadIdx.x);
  const int wave = t / kWave, lane = t % kWave;
  const int64_t row = blockIdx.y, seg = blockIdx.x;
  const float* l = a.logits + row * a.vocab;
  const int64_t j0 = seg * a.seg_len < a.vocab ? seg * a.seg_len : a.vocab;
  const int64_t j1 = j0 + a.seg_len < a.vocab ? j0 + a.seg_len : a.vocab;
  const int64_t count = j1 - j0;
  const float* s0 = l + j0;

  // x[q] holds the four logits from quad_at(c0 + (q kThreads + t) 4) of the segment: the quad
  // itself, or the four that end the segment where it is the last, partial one (they may begin
  // before the segment).  Every load is unconditional, also those of chunks past the end (all
  // lanes then read the last quad), so that the loads in flight are counted exactly.
  auto quad_at = [&](int64_t j) { return j + 4 <= count ? j : count - 4; };
  // Where four logits do not exist before the segment's end, the loads read this launch's own
  // output instead (16 bytes that no logit comes from) and the logits are read singly.
  const bool no_quad = row * a.vocab + j1 < 4;
  const float* quads = no_quad ? reinterpret_cast<const float*>(a.partials) : s0;
  auto load = [&](f32x4 (&x)[kQuads], int64_t c0) {
#pragma unroll
    for (int q = 0; q < kQuads; ++q) {
      const int64_t at = quad_at(c0 + (q * kThreads + t) * 4);
      x[q] = __builtin_nontemporal_load(
          reinterpret_cast<const f32x4_any*>(quads + (no_quad ? 0 : at)));
    }
  };
  // the row's length is waited for first: it would wait for every load requested ahead of it
  int64_t length = row_length(a, row);
  length = length < a.max_len ? length : a.max_len;
  __asm__ volatile("" ::"s"(__builtin_amdgcn_readfirstlane(static_cast<int>(length))));
  int64_t first_sel[kAhead];
  if constexpr (kLds) request_selection(a.sel + row * a.max_len, a.max_len, first_sel);
  __builtin_amdgcn_sched_barrier(0);
  f32x4 xa[kQuads], xb[kQuads];  // xb: the next chunk (not kOne)
  load(xa, 0);
  if constexpr (!kOne) load(xb, kChunk);
  if (no_quad) {  // at most three logits, in lane 0's first quad
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float v = count > 0 ? s0[count - 4 + k > 0 ? count - 4 + k : 0] : -INFINITY;
      __asm__ volatile("" : "+v"(v));  // waited for here, not by every later use of xa
      xa[0][k] = v;
    }
  }
  if (t == 0) any_flag = 0u;
  bool malformed = false;
  if constexpr (kLds) malformed = build_lds_bitmap(a, row, seg, j0, j1, length, lds_bits, first_sel);
  // bit of logit j: kLds, bit j - j0 of the LDS bitmap; else bit j of the row's bitmap
  const uint32_t* bits = kLds ? lds_bits : a.bitmap + row * a.words;
  const int64_t base = kLds ? 0 : j0;
  const int64_t end = kLds ? count : j1;
  const InvT inv = inverse(a.temperature);
  const bool floats = float_quotient(a.temperature);

  float mn = INFINITY, mx_rej = -INFINITY, mx = -INFINITY;  // mx: the wave's, uniform
  bool nan = false;
  double z = 0.0, z_sel = 0.0;
  auto use = [&](f32x4 (&x)[kQuads], int64_t c0) {
    uint32_t nibs[kQuads];  // bit k: logit k of quad q is selected
    float top = -INFINITY;
#pragma unroll
    for (int q = 0; q < kQuads; ++q)
      nibs[q] = selected4<kLds>(bits, base + c0 + (q * kThreads + t) * 4, end);
    if (c0 + kChunk > count) {  // uniform: the segment's last chunk
#pragma unroll
      for (int q = 0; q < kQuads; ++q) {
        // the logits of x[q] before its own quad belong to other lanes: -inf here
        const int64_t j = c0 + (q * kThreads + t) * 4;
        const int64_t over64 = j - quad_at(j);
        const int over = over64 < 4 ? static_cast<int>(over64) : 4;
#pragma unroll
        for (int k = 0; k < 4; ++k) x[q][k] = k >= over ? x[q][k] : -INFINITY;
        nibs[q] = (nibs[q] << over) & 15u;
      }
    }
    uint32_t any = 0;
#pragma unroll
    for (int q = 0; q < kQuads; ++q) {
      nan |= (x[q][0] != x[q][0]) | (x[q][1] != x[q][1]) | (x[q][2] != x[q][2]) |
             (x[q][3] != x[q][3]);
      top = fmaxf(top, fmaxf(fmaxf(x[q][0], x[q][1]), fmaxf(x[q][2], x[q][3])));
      any |= nibs[q];
    }
    const bool some = __ballot(any != 0) != 0;  // some logit of the wave's chunk is selected
    if (!some) {
      mx_rej = fmaxf(mx_rej, top);
    } else {
#pragma unroll
      for (int q = 0; q < kQuads; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool in = (nibs[q] >> k) & 1u;
          mn = fminf(mn, in ? x[q][k] : INFINITY);
          mx_rej = fmaxf(mx_rej, in ? -INFINITY : x[q][k]);
        }
    }
    top = uniform_max(top);
    const float before = mx;
    mx = fmaxf(mx, top);
    if (!a.top_p || !(mx > -INFINITY)) return;  // uniform
    if (mx > before && before > -INFINITY) {
      const double scale =
          exp((static_cast<double>(before) - static_cast<double>(mx)) / a.temperature);
      z = z * scale;
      z_sel = z_sel * scale;
    }
    auto terms = [&](auto mode) {
#pragma unroll
      for (int q = 0; q < kQuads; ++q) {
        double v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          v[k] = term<decltype(mode)::value>(x[q][k], mx, inv, a.temperature);
          z = z + v[k];
        }
        if (some) {
#pragma unroll
          for (int k = 0; k < 4; ++k) z_sel = z_sel + ((nibs[q] >> k) & 1u ? v[k] : 0.0);
        }
      }
    };
    if (floats)
      terms(std::true_type{});
    else
      terms(std::false_type{});
  };
  if constexpr (kOne) {
    if (count > 0) use(xa, 0);
  } else {
    for (int64_t c0 = 0; c0 < count; c0 += 2 * kChunk) {
      use(xa, c0);
      load(xa, c0 + 2 * kChunk);
      if (c0 + kChunk < count) use(xb, c0 + kChunk);
      load(xb, c0 + 3 * kChunk);
    }
  }
  mn = -uniform_max(-mn);
  mx_rej = uniform_max(mx_rej);
  if (a.top_p) {
    z = wave_sum(z);
    z_sel = wave_sum(z_sel);
  }
  const bool wave_nan = __any(nan);
  const bool wave_bad = __any(malformed);
  __syncthreads();  // any_flag is cleared before any wave sets it
  if (lane == 0) {
    fred[0][wave] = mn;
    fred[1][wave] = mx_rej;
    fred[2][wave] = mx;
    dred[0][wave] = z;
    dred[1][wave] = z_sel;
    if (wave_nan) atomicOr(&any_flag, kNanFlag);
    if (wave_bad) atomicOr(&any_flag, kMalformedFlag);
  }
  __syncthreads();
  if (t >= kWaves) return;
  // Lanes 0 .. 3 take one wave each: its sums relative to the segment's maximum.
  mn = fminf(fminf(fred[0][0], fred[0][1]), fminf(fred[0][2], fred[0][3]));
  mx_rej = fmaxf(fmaxf(fred[1][0], fred[1][1]), fmaxf(fred[1][2], fred[1][3]));
  mx = fmaxf(fmaxf(fred[2][0], fred[2][1]), fmaxf(fred[2][2], fred[2][3]));
  if (a.top_p) {
    const float own = fred[2][t];
    const double scale =
        own > -INFINITY
            ? exp((static_cast<double>(own) - static_cast<double>(mx)) / a.temperature)
            : 0.0;
    z = dred[0][t] * scale;
    z_sel = dred[1][t] * scale;
    z = z + __shfl_xor(z, 1, kWaves);
    z = z + __shfl_xor(z, 2, kWaves);
    z_sel = z_sel + __shfl_xor(z_sel, 1, kWaves);
    z_sel = z_sel + __shfl_xor(z_sel, 2, kWaves);
  }
  if (t == 0) a.partials[row * a.segments + seg] = Partial{mn, mx_rej, mx, any_flag, z, z_sel};
}

__global__ void __launch_bounds__(kThreads) finish_kernel(const Args a, int lds_select) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kWaves + threadIdx.x / kWave;
  const int lane = static_cast<int>(threadIdx.x) % kWave;
  if (row >= a.rows) return;  // whole waves
  const Partial* ps = a.partials + row * a.segments;
  float min_sel = INFINITY, max_rej = -INFINITY, mx = -INFINITY;
  uint32_t flags = 0u;
  for (int64_t s = lane; s < a.segments; s += kWave) {
    min_sel = fminf(min_sel, ps[s].min_sel);
    max_rej = fmaxf(max_rej, ps[s].max_rej);
    mx = fmaxf(mx, ps[s].max_all);
    flags |= ps[s].flags;
  }
  min_sel = wave_min(min_sel);
  max_rej = wave_max(max_rej);
  mx = wave_max(mx);
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) flags |= __shfl_xor(flags, o, kWave);
  const int64_t n_sel = row_length(a, row);
  const bool malformed = lds_select ? (flags & kMalformedFlag) != 0u : a.flags[row] != 0u;
  const bool well_formed = !malformed && n_sel >= 1 && n_sel <= a.max_len && n_sel <= a.vocab &&
                           (a.top_p || n_sel == a.k);
  bool ok = well_formed && (flags & kNanFlag) == 0u && min_sel >= max_rej;
  double mass = 0.0, without = 0.0;
  if (a.top_p && ok) {  // uniform over the wave
    const double big_m = static_cast<double>(mx);
    double big_z = 0.0, big_z_sel = 0.0;
    for (int64_t s = lane; s < a.segments; s += kWave) {  // this lane's segments in order
      if (ps[s].max_all > -INFINITY) {
        const double scale = exp((static_cast<double>(ps[s].max_all) - big_m) / a.temperature);
        big_z = big_z + ps[s].z * scale;
        big_z_sel = big_z_sel + ps[s].z_sel * scale;
      }
    }
    big_z = wave_sum(big_z);
    big_z_sel = wave_sum(big_z_sel);
    const double e_min = exp((static_cast<double>(min_sel) - big_m) / a.temperature);
    mass = big_z_sel / big_z;
    without = (big_z_sel - e_min) / big_z;
    ok = mass >= a.p - a.slack && without < a.p + a.slack;
  }
  if (lane != 0) return;
  a.passed[row] = ok ? 1u : 0u;
  a.min_sel[row] = min_sel;
  a.max_rej[row] = max_rej;
  a.mass[row] = mass;
  a.without[row] = without;
}

// The segment launch.  Segments of at most 4,096 logits (the default for rows that already fill the
// GPU, or are short) are one chunk: without the next chunk's registers seven waves fit a SIMD instead
// of three, so all of 1,024 workgroups run at once, and nothing is requested past the segment.
// Against the form of several chunks, which has the shortest rows wait for ten loads a lane: top-k 50
// of 128 x 32,000 logits 9.8 against 12.8 us, top-p 14.3 / 17.5; of 512 x 1,000 (one load a lane) top-p
// 9.8 / 12.9.
template <bool kLds>
hipError_t launch_segments(const Args& a, size_t lds, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.segments), static_cast<unsigned>(a.rows));
  if (a.seg_len <= 4 * kThreads)
    segment_kernel<kLds, 1, true><<<grid, dim3(kThreads), lds, s>>>(a);
  else if (a.seg_len <= 16 * kThreads)
    segment_kernel<kLds, 4, true><<<grid, dim3(kThreads), lds, s>>>(a);
  else
    segment_kernel<kLds, kLongQuads, false><<<grid, dim3(kThreads), lds, s>>>(a);
  return hipGetLastError();
}

}  // namespace
}  // namespace pck

extern "C" int pck_sampling_needs_scratch(int64_t vocab, int64_t max_len, int64_t segments) {
  if (vocab < 1 || max_len < 1 || segments < 1 || segments > vocab) return -1;
  const int64_t seg_len = (vocab + segments - 1) / segments;
  return max_len <= pck::kLdsSelect && seg_len <= pck::kLdsBits ? 0 : 1;
}

extern "C" int64_t pck_sampling_scratch_words(int64_t vocab) {
  return vocab < 1 ? -1 : (vocab + 31) / 32 + 1;
}

extern "C" int64_t pck_sampling_partial_bytes(void) {
  return static_cast<int64_t>(sizeof(pck::Partial));
}

extern "C" int pck_sampling_check(const float* logits, const int64_t* selected,
                                  const int64_t* lengths, int64_t rows, int64_t vocab,
                                  int64_t max_len, int64_t k, int top_p, double p,
                                  double temperature, double slack, int64_t segments,
                                  uint32_t* scratch, void* partials, uint8_t* passed,
                                  float* min_selected, float* max_rejected, double* mass,
                                  double* mass_without_smallest, void* stream) {
  using namespace pck;
  const int64_t seg_len = (vocab + segments - 1) / segments;
  const bool lds_select = max_len <= kLdsSelect && seg_len <= kLdsBits;
  if (!logits || !selected || (!scratch && !lds_select) || !partials || !passed ||
      !min_selected ||
      !max_rejected || !mass || !mass_without_smallest || rows < 1 || rows > 65535 ||
      vocab < 1 || max_len < 1 || segments < 1 || segments > vocab ||
      segments > 0x7FFFFFFF || !(temperature > 0.0) || !(slack >= 0.0) ||
      (max_len + kThreads - 1) / kThreads > 0x7FFFFFFF ||
      reinterpret_cast<uintptr_t>(partials) % 8 != 0)
    return hipErrorInvalidValue;
  Args a{};
  a.logits = logits;
  a.sel = selected;
  a.len = lengths;
  a.rows = rows;
  a.vocab = vocab;
  a.max_len = max_len;
  a.k = k;
  a.top_p = top_p != 0;
  a.p = p;
  a.temperature = temperature;
  a.slack = slack;
  a.segments = segments;
  a.seg_len = seg_len;
  a.words = (vocab + 31) / 32;
  a.bitmap = scratch;
  a.flags = scratch ? scratch + rows * a.words : nullptr;
  a.partials = static_cast<Partial*>(partials);
  a.passed = passed;
  a.min_sel = min_selected;
  a.max_rej = max_rejected;
  a.mass = mass;
  a.without = mass_without_smallest;
  auto s = static_cast<hipStream_t>(stream);
  hipError_t err;
  if (lds_select) {
    err = launch_segments<true>(a, static_cast<size_t>((seg_len + 31) / 32) * sizeof(uint32_t), s);
  } else {
    const dim3 mark_grid(static_cast<unsigned>((max_len + kThreads - 1) / kThreads),
                         static_cast<unsigned>(rows));
    mark_kernel<<<mark_grid, dim3(kThreads), 0, s>>>(a);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
    err = launch_segments<false>(a, 0, s);
  }
  if (err != hipSuccess) return err;
  finish_kernel<<<dim3(static_cast<unsigned>((rows + kWaves - 1) / kWaves)), dim3(kThreads), 0,
                  s>>>(a, lds_select ? 1 : 0);
  return hipGetLastError();
}
