// GEMV y = W x for the decode hot path on gfx950: BF16 or OCP FP8 E4M3FN weights, BF16 x,
// FP32 accumulation and output.
//
// Numerics are defined by the summation tree, not by the hardware mapping.  The coalesced tree
// of `threads` = T virtual lanes (reference src/pck/cuda/csrc/gemv_kernel.cu:139-178, model
// src/pck/gemv.py:71-101): virtual lane t owns the 16-byte vectors t, t + T, t + 2T, ... of a
// row (8 BF16 or 16 FP8 columns each) and adds their products one at a time in column order,
// starting from its first product, with columns past n contributing +0; each virtual warp of
// 32 lanes is reduced by halving, then the T / 32 warp sums are reduced by halving.
//
// Hardware mapping (MI355X, wave64): one wave computes one row (two rows when T = 32).  Lane l
// of the wave runs the T / 64 chains l, l + 64, l + 128, ... so that for every vector index the
// wave reads 64 consecutive 16-byte vectors (1 KiB, fully coalesced), and all of a lane's loads
// for U vector positions are issued before any product is consumed, which keeps enough bytes in
// flight per CU to stream HBM.  The two halves of a wave are the two virtual warps 2j and
// 2j + 1 of chain slot j, so the in-warp halving is a width-32 xor butterfly (lane 0 of each
// half ends with exactly the halving order's value), and the warp sums are combined in the
// halving order from uniform registers.  No LDS and no barrier are needed.
//
// Products: BF16 x BF16 (8 + 8 significand bits) and E4M3 x BF16 (4 + 8) are exact in FP32
// except under underflow; they are formed with a separate v_mul_f32 and added with v_add_f32 (the
// library is built with -ffp-contract=off), exactly the reference's __fmul_rn / __fadd_rn.  The
// chain accumulator starts at -0.0, the additive identity of IEEE round-to-nearest, so
// "-0 + p0" equals "start from p0" bit for bit, signed zero included.
//
// The naive tree (reference model src/pck/gemv.py:14-57) fixes a different order: virtual lane
// t sums the contiguous chunk [t c, (t + 1) c) of a row, then neighbour pairs combine level by
// level.  Its kernel maps the levels of stride below 64 onto DPP / permlane moves inside a wave
// and meets only the wave sums in LDS (gemv_naive_kernel below).

#include <hip/hip_runtime.h>

#include <cstdint>

#include "check_pair.h"
#include "pck_hip.h"
#include "rowsum_check.h"

namespace pck {
namespace {

constexpr int kWave = 64;
constexpr int kWarp = 32;
constexpr int kWavesPerGroup = 4;
constexpr int kGroupThreads = kWave * kWavesPerGroup;

struct GemvItem {
  const void* W;
  const uint16_t* x;
  float* y;
  double* sums;  // (m, 2) FP64 row sums (d_i, s_i) of the in-pass path; unused otherwise
  int64_t m;
  int64_t n;
  int64_t per_lane;  // vectors per virtual lane: ceil(ceil(n / vec) / T)
  const float* scale = nullptr;  // (m,) FP32 row scales of an FP8 weight, with y_scaled
  float* y_scaled = nullptr;     // (m,) scale[i] * y[i], rounded to nearest; or null
};

// Writes row `row` of an item: the tree's sum, and the dequantised output `scale * value` when
// the item has row scales (one FP32 multiply, as y = s z would round it).
__device__ __forceinline__ void store_row(const GemvItem& it, int64_t row, float value,
                                          float scale) {
  it.y[row] = value;
  if (it.y_scaled != nullptr) it.y_scaled[row] = scale * value;
}

struct GemvBatch {
  GemvItem item[PCK_MAX_GROUP];
  int64_t first_group[PCK_MAX_GROUP + 1];  // workgroup prefix sums
  int count;
};

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

// Two E4M3FN codes (bytes 0-1, or 2-3 with kHigh) of `w` to FP32, exactly (hardware OCP decode).
template <bool kHigh>
__device__ __forceinline__ float2 fp8_pair(uint32_t w) {
  auto v = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(w), kHigh);
  return make_float2(v[0], v[1]);
}

__device__ __forceinline__ float fp8_one(uint8_t code) { return fp8_pair<false>(code).x; }

// Row sums of the in-pass path, from the FP32 products the tree already forms (exact: 8 + 8 or
// 4 + 8 significand bits, barring FP32 underflow).  Each pair of consecutive products is added
// in FP32 (rounding error at most u32 (|p0| + |p1|)), widened and added to d in FP64; |p| is
// added to s in FP32, one product at a time in column order.
struct RowSums {
  double d = 0.0;
  float s = 0.0f;
};

template <bool kSums>
__device__ __forceinline__ void add_pair(RowSums& rs, float p0, float p1) {
  if constexpr (kSums) {
    rs.d = rs.d + static_cast<double>(p0 + p1);
    rs.s = rs.s + __builtin_fabsf(p0);
    rs.s = rs.s + __builtin_fabsf(p1);
  }
}

// Adds the products of one vector to `acc` (and, with kSums, to the row sums), in column order.
template <bool kFp8, bool kSums = false>
__device__ __forceinline__ void add_products(float& acc, RowSums& rs, const uint4& w,
                                             const uint4& xa, const uint4& xb) {
  const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
  if constexpr (!kFp8) {
    const uint32_t xd[4] = {xa.x, xa.y, xa.z, xa.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float p0 = bf16_lo(wd[k]) * bf16_lo(xd[k]);
      const float p1 = bf16_hi(wd[k]) * bf16_hi(xd[k]);
      acc = acc + p0;
      acc = acc + p1;
      add_pair<kSums>(rs, p0, p1);
    }
  } else {
    const uint32_t xd[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float2 f01 = fp8_pair<false>(wd[k]);
      const float2 f23 = fp8_pair<true>(wd[k]);
      const float p0 = f01.x * bf16_lo(xd[2 * k]);
      const float p1 = f01.y * bf16_hi(xd[2 * k]);
      const float p2 = f23.x * bf16_lo(xd[2 * k + 1]);
      const float p3 = f23.y * bf16_hi(xd[2 * k + 1]);
      acc = acc + p0;
      acc = acc + p1;
      acc = acc + p2;
      acc = acc + p3;
      add_pair<kSums>(rs, p0, p1);
      add_pair<kSums>(rs, p2, p3);
    }
  }
}

// Element loads for rows that cannot take 16-byte vectors (n not a multiple of the vector width
// or a misaligned pointer): the same products in the same order, +0 past n.
template <bool kFp8, bool kSums = false>
__device__ __forceinline__ void add_products_scalar(float& acc, RowSums& rs, const void* w_row,
                                                    const uint16_t* x, int64_t col, int64_t n) {
  constexpr int V = kFp8 ? 16 : 8;
  float p[V];
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int64_t j = col + k;
    p[k] = 0.0f;
    if (j < n) {
      const float xv = __uint_as_float(static_cast<uint32_t>(x[j]) << 16);
      float wv;
      if constexpr (kFp8) {
        wv = fp8_one(static_cast<const uint8_t*>(w_row)[j]);
      } else {
        wv = __uint_as_float(static_cast<uint32_t>(static_cast<const uint16_t*>(w_row)[j]) << 16);
      }
      p[k] = wv * xv;
    }
    acc = acc + p[k];
  }
#pragma unroll
  for (int k = 0; k < V; k += 2) add_pair<kSums>(rs, p[k], p[k + 1]);
}

// a[i] += a[i + 16] ... a[0] += a[1] inside each 32-lane half of the wave, the halving order of
// the reference's 32-lane shuffle-down reduction, with lane 0 (and lane 32) ending on a[0].
// Step 16 moves whole rows of 16 lanes with gfx950's v_permlane16_swap (the second result holds
// each even row's partner row); steps 8 and 4 rotate inside a row (row_ror:8 gives lane i the
// value of lane i ^ 8, row_ror:12 that of lane i + 4 for the lanes i < 4 that matter); steps 2
// and 1 are quad permutes.  Everything stays in VALU instructions (DPP folds into the adds).
template <int kCtrl>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xF, 0xF, false));
}

__device__ __forceinline__ float halve32(float v) {
  const auto swapped = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false,
                                                        false);
  v = v + __int_as_float(swapped[1]);  // lanes 0-15 (32-47) receive lanes 16-31 (48-63)
  v = v + dpp_move<0x128>(v);          // row_ror:8
  v = v + dpp_move<0x12C>(v);          // row_ror:12
  v = v + dpp_move<0x4E>(v);           // quad_perm [2,3,0,1]
  v = v + dpp_move<0xB1>(v);           // quad_perm [1,0,3,2]
  return v;
}

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// How a launch reads W and x.
//   kAligned    16-byte loads at 16-byte addresses: n is a multiple of the vector width and every
//               pointer is aligned.
//   kUnaligned  16-byte loads at any byte address (every n of at least one vector): gfx950's
//               global loads take them, and a wave still reads contiguous kilobytes.  A row's
//               last, partial vector is read as the 16 bytes that end the row (nothing past the
//               row is touched) and moved into place in registers.
//   kElement    element loads: rows shorter than one vector.
enum class Load { kElement, kUnaligned, kAligned };

enum class Pad { kNone, kZeroed, kSkipped };

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_any __attribute__((aligned(1)));  // any byte address

template <bool kNt, bool kAny>
__device__ __forceinline__ uint4 load16(const void* p) {
  u32x4 v;
  if constexpr (kAny) {
    const auto* q = static_cast<const u32x4_any*>(p);
    v = kNt ? __builtin_nontemporal_load(q) : *q;
  } else {
    const auto* q = static_cast<const u32x4*>(p);
    v = kNt ? __builtin_nontemporal_load(q) : *q;
  }
  return make_uint4(v[0], v[1], v[2], v[3]);
}

typedef unsigned __int128 u128;

__device__ __forceinline__ u128 as_u128(const uint4& v) {
  return (static_cast<u128>((static_cast<uint64_t>(v.w) << 32) | v.z) << 64) |
         ((static_cast<uint64_t>(v.y) << 32) | v.x);
}
__device__ __forceinline__ uint4 as_uint4(u128 v) {
  const uint64_t lo = static_cast<uint64_t>(v), hi = static_cast<uint64_t>(v >> 64);
  return make_uint4(static_cast<uint32_t>(lo), static_cast<uint32_t>(lo >> 32),
                    static_cast<uint32_t>(hi), static_cast<uint32_t>(hi >> 32));
}

// Drops the first `skip` (0 .. V) of a vector's V elements, moves the rest to the front and
// fills with zeros: the partial vector of a row, read as the V elements that end the row.
template <bool kFp8>
__device__ __forceinline__ void drop_front(uint4& w, int skip) {
  const int bits = skip * (kFp8 ? 8 : 16);
  w = as_uint4(bits < 128 ? as_u128(w) >> bits : 0);
}
template <bool kFp8>
__device__ __forceinline__ void drop_front_x(uint4& xa, uint4& xb, int skip) {
  if constexpr (!kFp8) {
    drop_front<false>(xa, skip);
  } else {  // 16 activations in two registers of eight
    u128 lo = as_u128(skip >= 8 ? xb : xa), hi = skip >= 8 ? 0 : as_u128(xb);
    const int bits = (skip & 7) * 16;
    lo = bits ? (lo >> bits) | (hi << (128 - bits)) : lo;
    hi = hi >> bits;
    xa = as_uint4(skip < 16 ? lo : 0);
    xb = as_uint4(skip < 16 ? hi : 0);
  }
}

// T virtual lanes per row, R rows per wave slot, U vector positions loaded ahead, kNt:
// non-temporal weight loads (streamed once, so they need not displace x in the caches).
// kPad: what a launch does about vectors of a chain that lie past n (n is not a multiple of
// T * vec); their loads are redirected to column 0 (kUnaligned: to the row's last vector) and
// they add +0.
//   kNone     there are none.
//   kZeroed   they are zeroed in the registers they were loaded to.
//   kSkipped  a chain slot whose 64 vectors all lie past n adds +0 once instead of V products of
//             zeros (the same sum, sign of zero included), so a row's short last position costs
//             what its columns cost (FP8 4096 x 14336: 12.4 against 14.2 us).  Its branches cost
//             rows without such a slot 3 to 10%, so a launch takes this form only if it has one.
//
// kLive: chain slots per lane that hold any column, when every row of the launch ends inside the
// first kLive slots of its first position (n <= 64 kLive vec, one position).  The other slots'
// chains sum padding only, so they are +0 without being loaded or kept in registers: a tree of
// 512 or 1024 virtual lanes over a short row then costs what the row's own columns cost.
template <int T, int R, int U, bool kFp8, Load kLoad, Pad kPad, bool kNt, bool kSums = false,
          int kLive = (T >= kWave ? T / kWave : 1)>
__device__ __forceinline__ void gemv_rows(const GemvBatch& batch, int64_t group) {
  constexpr int V = kFp8 ? 16 : 8;
  constexpr int kLanesPerRow = T >= kWave ? kWave : T;
  constexpr int kSlots = kWave / kLanesPerRow;  // rows side by side in one wave (2 if T = 32)
  constexpr int kChains = T / kLanesPerRow;     // chains per lane
  constexpr int kElemBytes = kFp8 ? 1 : 2;

  int g = 0;
  while (g + 1 < batch.count && group >= batch.first_group[g + 1]) ++g;
  const GemvItem& it = batch.item[g];
  const int lane = static_cast<int>(threadIdx.x) & (kWave - 1);
  const int64_t first_group = batch.first_group[g];
  const int64_t m = it.m;
  const int64_t n = it.n;
  const int64_t P = it.per_lane;
  const void* W = it.W;
  const uint16_t* __restrict__ x = it.x;
  // BF16: everything ahead of the first load in one round trip to the scalar cache, not the three
  // that the scheduler forms (512 x 1024, T = 64: 2.69 against 2.95 us; the FP8 kernels, whose loads
  // it orders well, would lose 3%).
  if constexpr (!kFp8)
    __asm__ volatile("" ::"s"(first_group), "s"(m), "s"(n), "s"(P), "s"(W), "s"(x));
  const int64_t wave =
      (group - first_group) * kWavesPerGroup + (static_cast<int>(threadIdx.x) >> 6);
  const int slot = lane / kLanesPerRow;
  const int chain0 = lane % kLanesPerRow;

  // Rows past m compute on row m - 1 (a valid address) and are not stored.
  const unsigned char* w_rows[R];
  bool live[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t row = (wave * kSlots + slot) * R + r;
    live[r] = row < m;
    w_rows[r] = static_cast<const unsigned char*>(W) + (live[r] ? row : m - 1) * n * kElemBytes;
  }

  // Row scales of a scaled FP8 item, loaded ahead of the weight stream so that their latency
  // is hidden behind it instead of adding a dependent load to the launch's tail.
  float scale[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t row = (wave * kSlots + slot) * R + r;
    scale[r] = (kFp8 && it.y_scaled != nullptr) ? it.scale[live[r] ? row : m - 1] : 1.0f;
  }

  float acc[R][kLive];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int j = 0; j < kLive; ++j) acc[r][j] = -0.0f;
  RowSums rs[R][kLive];  // per row and chain: the lane's d and s (kSums only)

  constexpr bool kAny = kLoad == Load::kUnaligned;
  constexpr bool kZeroed = kPad == Pad::kZeroed && !kAny;
  for (int64_t v0 = 0; v0 < P; v0 += U) {
    if constexpr (kLoad != Load::kElement) {
      uint4 wb[U][R][kLive];
      uint4 xa[U][kLive];
      uint4 xb[U][kLive];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (U > 1 && v0 + u >= P) break;  // uniform: the tail of the last block
#pragma unroll
        for (int j = 0; j < kLive; ++j) {
          const int64_t col = ((v0 + u) * T + chain0 + kLanesPerRow * j) * V;
          const int64_t at = kPad == Pad::kNone ? col : kAny ? (col < n - V ? col : n - V) : (col < n ? col : 0);
          xa[u][j] = load16<false, kAny>(x + at);
          if constexpr (kFp8) xb[u][j] = load16<false, kAny>(x + at + 8);
#pragma unroll
          for (int r = 0; r < R; ++r)
            wb[u][r][j] = load16<kNt, kAny>(w_rows[r] + at * kElemBytes);
          if constexpr (kZeroed) {
            if (col >= n) {
              xa[u][j] = make_uint4(0, 0, 0, 0);
              xb[u][j] = make_uint4(0, 0, 0, 0);
#pragma unroll
              for (int r = 0; r < R; ++r) wb[u][r][j] = make_uint4(0, 0, 0, 0);
            }
          }
        }
      }
      auto products = [&](int u, int j) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          add_products<kFp8, kSums>(acc[r][j], rs[r][j], wb[u][r][j], xa[u][j],
                                    kFp8 ? xb[u][j] : xa[u][j]);
      };
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (U > 1 && v0 + u >= P) break;
        if (kPad == Pad::kNone || kZeroed || (v0 + u + 1) * T * V <= n) {  // nothing to drop
#pragma unroll
          for (int j = 0; j < kLive; ++j) products(u, j);
          continue;
        }
#pragma unroll
        for (int j = 0; j < kLive; ++j) {
          // the slot's first column, the same for every lane of the wave
          const int64_t first = ((v0 + u) * T + kLanesPerRow * j) * V;
          if (first >= n) {
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r][j] = acc[r][j] + 0.0f;
            continue;
          }
          if (first + kLanesPerRow * V > n) {  // some of the slot's columns lie past n
            const int64_t col = first + chain0 * V;
            if constexpr (kAny) {
              const int64_t over = col - (n - V);  // <= 0: a whole vector
              const int skip = over <= 0 ? 0 : over < V ? static_cast<int>(over) : V;
              drop_front_x<kFp8>(xa[u][j], xb[u][j], skip);
#pragma unroll
              for (int r = 0; r < R; ++r) drop_front<kFp8>(wb[u][r][j], skip);
            } else if (col >= n) {
              xa[u][j] = make_uint4(0, 0, 0, 0);
              xb[u][j] = make_uint4(0, 0, 0, 0);
#pragma unroll
              for (int r = 0; r < R; ++r) wb[u][r][j] = make_uint4(0, 0, 0, 0);
            }
          }
          products(u, j);
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int j = 0; j < kLive; ++j) {
          const int64_t col = (v0 * T + chain0 + kLanesPerRow * j) * V;
          add_products_scalar<kFp8, kSums>(acc[r][j], rs[r][j], w_rows[r], x, col, n);
        }
      }
    }
  }

  if constexpr (kSums) {
    // Each lane combines its chains' sums in halving order (chain i += chain i + half), then
    // the row's lanes combine theirs by an xor butterfly (symmetric, so every lane of the row
    // ends with the same pair); the row's first lane stores it as one 16-byte write.
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int half = kLive / 2; half > 0; half /= 2)
#pragma unroll
        for (int i = 0; i < half; ++i) {
          rs[r][i].d = rs[r][i].d + rs[r][i + half].d;
          rs[r][i].s = rs[r][i].s + rs[r][i + half].s;
        }
      RowSums t = rs[r][0];
#pragma unroll
      for (int off = kLanesPerRow / 2; off > 0; off /= 2) {
        const double od = __shfl_xor(t.d, off, kWave);
        const float os = __shfl_xor(t.s, off, kWave);
        t.d = t.d + od;
        t.s = t.s + os;
      }
      const int64_t row = (wave * kSlots + slot) * R + r;
      if (chain0 == 0 && live[r])
        reinterpret_cast<double2*>(it.sums)[row] = make_double2(t.d, static_cast<double>(t.s));
    }
  }

#pragma unroll
  for (int r = 0; r < R; ++r) {
    // Halving inside each 32-lane virtual warp.
#pragma unroll
    for (int j = 0; j < kLive; ++j) acc[r][j] = halve32(acc[r][j]);
    const int64_t row = (wave * kSlots + slot) * R + r;
    if constexpr (kSlots == 2) {
      // T = 32: one virtual warp per row; lanes 0 and 32 hold the two rows' sums.
      if (chain0 == 0 && live[r]) store_row(it, row, acc[r][0], scale[r]);
    } else {
      // Warp w = 2j + h is half h of chain slot j; reduce the T / 32 warp sums by halving.
      // The sums of slots past kLive are +0: adding them changes at most the sign of a zero.
      constexpr int kWarps = 2 * kLive;
      float ws[kWarps];
#pragma unroll
      for (int j = 0; j < kLive; ++j) {
        ws[2 * j] = lane_value(acc[r][j], 0);
        ws[2 * j + 1] = lane_value(acc[r][j], kWarp);
      }
      if constexpr (kLive < kChains) {
#pragma unroll
        for (int i = 0; i < kWarps; ++i) ws[i] = ws[i] + 0.0f;
      }
#pragma unroll
      for (int half = kWarps / 2; half > 0; half /= 2)
#pragma unroll
        for (int i = 0; i < half; ++i) ws[i] = ws[i] + ws[i + half];
      if (lane == 0 && live[r]) store_row(it, row, ws[0], scale[r]);
    }
  }
}

template <int T, int R, int U, bool kFp8, Load kLoad, Pad kPad, bool kNt, int kLive>
__global__ void __launch_bounds__(kGroupThreads) gemv_tree_kernel(const GemvBatch batch) {
  gemv_rows<T, R, U, kFp8, kLoad, kPad, kNt, false, kLive>(batch, blockIdx.x);
}

// A GEMV launch that also checks outputs of earlier launches: the first workgroups of the grid
// each run one (check, block) pair of `ride` (the standalone checker's code, so rho, tau and the
// verdicts are bit-identical to pck_blocked_check), the rest compute the GEMV rows.  The checked
// y were written by launches that finished before this one started (stream order), and the
// checker workgroups are separate wavefronts that read them from memory; their latency hides
// behind the GEMV's streaming, and the bank reads add about 2.3% (BF16, b = 128) to the bytes.
// Rows longer than 4,096 columns keep 8 quads per lane in flight (a 14,336-column row in two
// round trips instead of four); more would push the kernel past 128 VGPRs and halve the GEMV
// waves a SIMD holds.
template <int T, int R, int U, bool kFp8, Pad kPad, bool kNt>
__global__ void __launch_bounds__(kGroupThreads)
    gemv_ride_kernel(const GemvBatch batch, const PckCheckBatch ride) {
  __shared__ check::Quad lds[check::kWaves];
  const int64_t items = ride.start[ride.count];
  if (static_cast<int64_t>(blockIdx.x) < items) {
    const int g = check::owner(ride, blockIdx.x);
    if (ride.desc[g].n > 4 * 4 * check::kThreads)
      check::check_pair<8>(ride, blockIdx.x, g, lds);
    else
      check::check_pair<4>(ride, blockIdx.x, g, lds);
    return;
  }
  gemv_rows<T, R, U, kFp8, Load::kAligned, kPad, kNt>(batch,
                                                      static_cast<int64_t>(blockIdx.x) - items);
}

// The in-pass GEMV: the tree's outputs plus each row's sums (d_i, s_i), and in the first
// workgroups of the grid the row-sum checks of `ride` (outputs of earlier launches on the stream,
// read from memory; one wave per (check, block) pair, the code of pck_rowsum_check, so the
// results are bit-identical to it).  A check never reads anything this launch writes.
template <int T, int R, int U, bool kFp8, Load kLoad, Pad kPad, bool kNt, int kLive>
__global__ void __launch_bounds__(kGroupThreads)
    gemv_rowsum_kernel(const GemvBatch batch, const PckRowSumBatch ride) {
  const int64_t items = rowsum::items(ride);
  const int64_t ride_groups = (items + kWavesPerGroup - 1) / kWavesPerGroup;
  const int64_t group = static_cast<int64_t>(blockIdx.x);
  if (group < ride_groups) {
    const int64_t item = group * kWavesPerGroup + (static_cast<int>(threadIdx.x) >> 6);
    if (item < items) rowsum::check_item(ride, item);  // uniform per wave
    return;
  }
  gemv_rows<T, R, U, kFp8, kLoad, kPad, kNt, true, kLive>(batch, group - ride_groups);
}

// Naive tree (order of the reference model src/pck/gemv.py:14-57): `threads` = T virtual lanes
// per row, lane t owning the contiguous chunk [t c, (t + 1) c), c = ceil(n / T), summed in
// column order from its first product (columns past n add +0), then the T chain sums combined
// by neighbour pairs, stride 1, 2, 4, ...: a[t] += a[t + s] for t a multiple of 2s.
//
// One workgroup of max(T, 64) lanes takes R rows, lane t of the workgroup being virtual lane t
// (lanes t >= T, present only when T < 64, own chunks wholly past n and feed no level below T).
// The levels of stride 1 .. 32 run inside each wave: every lane adds the value of its partner lane
// t + s, moved by DPP (quad permutes for 1 and 2, row rotations for 4 and 8), permlane16_swap
// (16) or a read of lane 32 (32); the lanes that matter at a level read only lanes that
// mattered at the level before, so lane 0 ends with the wave's subtree.  The levels of stride 64
// and up combine the T / 64 wave sums, which meet in LDS behind one barrier, in the same pair
// order.  kLoad: kAligned, 16-byte loads of chunks that are whole aligned vectors, none past n (the
// chain's arithmetic bounds short rows, so a vector carries no bounds of its own); kUnaligned, the
// same at any 2-byte address (n >= 8), where a chunk's columns past its last whole vector, and
// vectors that cross n, are read as 16 bytes inside the row and moved into place, so no lane takes
// element loads; kElement, element loads, for chunks of fewer than four columns (a wave's lanes
// then read one contiguous piece) and rows shorter than a vector.
template <Load kLoad, int R>
__global__ void __launch_bounds__(1024)
    gemv_naive_kernel(const uint16_t* __restrict__ W, const uint16_t* __restrict__ x,
                      float* __restrict__ y, int64_t m, int64_t n, int64_t chunk, int threads) {
  __shared__ float wave_sum[R][1024 / kWave];
  const int t = static_cast<int>(threadIdx.x);
  const int lane = t & (kWave - 1);
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * R;
  const int64_t first = static_cast<int64_t>(t) * chunk;
  const uint16_t* rows[R];
#pragma unroll
  for (int r = 0; r < R; ++r)  // rows past m compute on row m - 1 and are not stored
    rows[r] = W + (R == 1 || row0 + r < m ? row0 + r : m - 1) * n;

  float acc[R];  // -0.0 + p0 is p0: the chain starts from its first product
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = -0.0f;
  auto add8 = [&](float& sum, const uint4& w, const uint4& xv) {
    const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
    const uint32_t xd[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      sum = sum + bf16_lo(wd[k]) * bf16_lo(xd[k]);
      sum = sum + bf16_hi(wd[k]) * bf16_hi(xd[k]);
    }
  };
  if constexpr (kLoad == Load::kAligned) {
    constexpr int A = R == 2 ? 2 : 1;  // vectors loaded ahead: a whole chunk of two
    for (int64_t v = 0; v < chunk; v += 8 * A) {
      uint4 wv[A][R], xv[A];
#pragma unroll
      for (int a = 0; a < A; ++a) {
        const int64_t col = first + v + 8 * a;
        xv[a] = make_uint4(0, 0, 0, 0);  // past n: +0 products
#pragma unroll
        for (int r = 0; r < R; ++r) wv[a][r] = make_uint4(0, 0, 0, 0);
        if (col < n && (a == 0 || v + 8 < chunk)) {
#pragma unroll
          for (int r = 0; r < R; ++r) wv[a][r] = load16<false, false>(rows[r] + col);
          xv[a] = load16<false, false>(x + col);
        }
      }
#pragma unroll
      for (int a = 0; a < A; ++a) {
        if (a == 1 && v + 8 >= chunk) break;  // uniform
#pragma unroll
        for (int r = 0; r < R; ++r) add8(acc[r], wv[a][r], xv[a]);
      }
    }
  } else if constexpr (kLoad == Load::kUnaligned) {
    // columns col .. col + 7 of x and of the rows (+0 past n)
    struct Vectors {
      uint4 x, w[R];
    };
    auto load = [&](int64_t col) {
      const int64_t at = col < n - 8 ? col : n - 8;
      Vectors v;
      v.x = load16<false, true>(x + at);
#pragma unroll
      for (int r = 0; r < R; ++r) v.w[r] = load16<false, true>(rows[r] + at);
      return v;
    };
    auto add = [&](Vectors& v, int64_t col, int count) {  // the first `count` columns
      if (col > n - 8) {
        const int skip = col < n ? static_cast<int>(col - (n - 8)) : 8;
        drop_front<false>(v.x, skip);
#pragma unroll
        for (int r = 0; r < R; ++r) drop_front<false>(v.w[r], skip);
      }
      const uint32_t xd[4] = {v.x.x, v.x.y, v.x.z, v.x.w};
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t wd[4] = {v.w[r].x, v.w[r].y, v.w[r].z, v.w[r].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (2 * k < count) acc[r] = acc[r] + bf16_lo(wd[k]) * bf16_lo(xd[k]);
          if (2 * k + 1 < count) acc[r] = acc[r] + bf16_hi(wd[k]) * bf16_hi(xd[k]);
        }
      }
    };
    int64_t c = 0;
    for (; c + 16 <= chunk; c += 16) {
      Vectors a = load(first + c), b = load(first + c + 8);
      add(a, first + c, 8);
      add(b, first + c + 8, 8);
    }
    for (; c < chunk; c += 8) {  // the last one or two vectors, the last perhaps partial
      Vectors a = load(first + c);
      if (c + 8 <= chunk) add(a, first + c, 8);
      else add(a, first + c, static_cast<int>(chunk - c));
    }
  } else {
    static_assert(R == 1);
    for (int64_t j = first; j < first + chunk; ++j) {
      float p = 0.0f;
      if (j < n) p = __uint_as_float(static_cast<uint32_t>(rows[0][j]) << 16) *
                     __uint_as_float(static_cast<uint32_t>(x[j]) << 16);
      acc[0] = j == first ? p : acc[0] + p;
    }
  }

#pragma unroll
  for (int r = 0; r < R; ++r) {
    float v = acc[r];
    // Levels inside the wave (uniform bounds: `threads` is the same for every lane).
    if (threads > 1) v = v + dpp_move<0xB1>(v);   // stride 1: quad_perm [1,0,3,2]
    if (threads > 2) v = v + dpp_move<0x4E>(v);   // stride 2: quad_perm [2,3,0,1]
    if (threads > 4) v = v + dpp_move<0x12C>(v);  // stride 4: row_ror:12, lane i <- i + 4
    if (threads > 8) v = v + dpp_move<0x128>(v);  // stride 8: row_ror:8, lane i <- i + 8
    if (threads > 16) {                            // stride 16: lanes 0-15 <- 16-31
      const auto swapped =
          __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
      v = v + __int_as_float(swapped[1]);
    }
    if (threads > 32) v = lane_value(v, 0) + lane_value(v, 32);  // stride 32
    acc[r] = v;
  }

  if (threads <= kWave) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (t == 0 && row0 + r < m) y[row0 + r] = acc[r];
    return;
  }
  // Levels across waves: wave w's subtree is a[64 w]; pairs of stride 64, 128, ...  Lane r of the
  // workgroup finishes row r.
  if (lane == 0) {
#pragma unroll
    for (int r = 0; r < R; ++r) wave_sum[r][t / kWave] = acc[r];
  }
  __syncthreads();
  if (t < R && row0 + t < m) {
    const int waves = threads / kWave;
    float a[1024 / kWave];
#pragma unroll
    for (int w = 0; w < 1024 / kWave; ++w) a[w] = w < waves ? wave_sum[t][w] : 0.0f;
#pragma unroll
    for (int s = 1; s < 1024 / kWave; s *= 2)
#pragma unroll
      for (int w = 0; w + s < 1024 / kWave; w += 2 * s)
        if (s < waves) a[w] = a[w] + a[w + s];
    y[row0 + t] = a[0];
  }
}

// Launch shape of the coalesced kernel: rows per wave slot, vector positions loaded ahead and
// non-temporal weight loads.  T = 256 with aligned rows (the reference's default tree) has every
// combination instantiated for tuning; every other route has only the shapes it uses (aligned rows
// of T != 256 with non-temporal or plain weight loads, kCachedBytes; the others non-temporal).
struct TreeShape {
  int rows;
  int unroll;
  int nt;
};

TreeShape g_shape_override = {0, 0, 0};

// Defaults from sweeps of every shape over Llama-3-8B decode launches and over 1024 .. 4096 rows of
// 4096 .. 14336 columns on MI355X.  Non-temporal weight loads won everywhere; the sweeps replay
// each launch over weight copies that do not fit the Infinity Cache (with four copies of FP8
// down, 235 MB, plain loads won from the cache; streamed from HBM, as in a decode pass,
// non-temporal loads take 12.4 against 14.6 us).  per_lane is the positions of the longest row.
//   BF16, one or two positions (n <= 4096): one row per wave, both positions ahead.
//   BF16, longer rows: two rows per wave above 3072 rows; fewer rows leave too few waves, so one
//     row, and below 1536 rows two positions ahead as well (2304 x 13824: 13.7 against 16.9 us
//     with two rows, 3573 x 13824: 20.2 against 19.2; 1024 x 14336: 8.5 against 11.4).
//   FP8 rows are half as long, so two rows per wave keep as many bytes in flight as one BF16 row;
//     one row per wave below 2048 rows (1024 x 14336: 6.8 against 8.6 us), for rows of one
//     position up to 4096 rows (o: 4.9 against 5.4 us) and of two up to 3072, these with both
//     positions ahead below 1536 rows (256 x 8192: 4.1 against 4.35).
TreeShape choose_shape(int64_t per_lane, int64_t rows, bool fp8) {
  if (g_shape_override.rows > 0) return g_shape_override;
  if (!fp8) {
    if (per_lane <= 2 || rows < 1536) return TreeShape{1, 2, 1};
    return rows <= 3072 ? TreeShape{1, 1, 1} : TreeShape{2, 1, 1};
  }
  if ((per_lane == 1 && rows <= 4096) || (per_lane == 2 && rows < 1536)) return TreeShape{1, 2, 1};
  if (rows < 2048 || (per_lane == 2 && rows <= 3072)) return TreeShape{1, 1, 1};
  return TreeShape{2, 1, 1};
}

// Trees of T != 256 lanes read aligned weights with plain loads below this size and with
// non-temporal ones (and more rows or positions per wave) from it on.  A launch cannot see whether
// its weights still lie in the 256 MB Infinity Cache, only what its own size allows: a pass that
// uses three or more such matrices in turn (a decode layer's launches are four) cannot keep them
// from a third of the cache on.  Below it either may be true, and there a wrong non-temporal load
// costs more than a wrong plain one.  Aligned launches of 64 .. 14336 rows and 512 .. 14336 columns
// at T = 32, 64 and 128, non-temporal against plain loads, time streamed from HBM / of one matrix
// again and again (geometric mean, range over launches):
//   below 85 MiB   0.95 (0.73 .. 1.37) / 1.14 (0.91 .. 1.63)
//   from 85 MiB    0.89 (0.77 .. 0.98) / 1.05 (0.98 .. 1.19)
// T = 256 is the decode path, which streams its weights: non-temporal.
constexpr int64_t kCachedBytes = int64_t{85} << 20;

// Fills the workgroup prefix sums for rows_per_group rows per workgroup; returns the total.
int64_t plan_groups(GemvBatch& batch, int64_t rows_per_group) {
  batch.first_group[0] = 0;
  for (int g = 0; g < batch.count; ++g) {
    batch.first_group[g + 1] =
        batch.first_group[g] + (batch.item[g].m + rows_per_group - 1) / rows_per_group;
  }
  return batch.first_group[batch.count];
}

// The launch plan of a group: validated items, how its rows are read, whether any chain has
// padding vectors, the longest row in vectors and per lane, the total rows and weight bytes.
struct GroupPlan {
  GemvBatch batch{};
  Load load = Load::kAligned;
  bool pad = false;
  int64_t dead_slots = 0;  // most chain slots of a last position that lie wholly past its row
  int64_t max_vectors = 1;
  int64_t max_per_lane = 1;
  int64_t rows = 0;
  int64_t bytes = 0;  // of weights
};

// kSums: the in-pass kernel, with `rs` the row-sum checks it carries; otherwise the plain tree.
template <int T, int R, int U, bool kFp8, Load kLoad, Pad kPad, bool kNt, bool kSums,
          int kLive = (T >= kWave ? T / kWave : 1)>
hipError_t launch_tree(GemvBatch& batch, const PckRowSumBatch* rs, hipStream_t stream) {
  constexpr int kLanesPerRow = T >= kWave ? kWave : T;
  const int64_t groups = plan_groups(batch, (kWave / kLanesPerRow) * R * kWavesPerGroup);
  if constexpr (kSums) {
    const int64_t total = groups + (rowsum::items(*rs) + kWavesPerGroup - 1) / kWavesPerGroup;
    if (total == 0) return hipSuccess;
    if (total * kGroupThreads > 0xFFFFFFFFll) return hipErrorInvalidValue;  // 32-bit dispatch
    gemv_rowsum_kernel<T, R, U, kFp8, kLoad, kPad, kNt, kLive>
        <<<dim3(static_cast<unsigned>(total)), dim3(kGroupThreads), 0, stream>>>(batch, *rs);
  } else {
    (void)rs;
    if (groups == 0) return hipSuccess;
    if (groups * kGroupThreads > 0xFFFFFFFFll) return hipErrorInvalidValue;  // 32-bit dispatch
    gemv_tree_kernel<T, R, U, kFp8, kLoad, kPad, kNt, kLive>
        <<<dim3(static_cast<unsigned>(groups)), dim3(kGroupThreads), 0, stream>>>(batch);
  }
  return hipGetLastError();
}

template <int T, int R, bool kFp8, Pad kPad, bool kNt, bool kSums>
hipError_t launch_unroll(GemvBatch& batch, int unroll, const PckRowSumBatch* rs, hipStream_t s) {
  constexpr Load L = Load::kAligned;
  if (unroll >= 4) return launch_tree<T, R, 4, kFp8, L, kPad, kNt, kSums>(batch, rs, s);
  if (unroll == 2) return launch_tree<T, R, 2, kFp8, L, kPad, kNt, kSums>(batch, rs, s);
  return launch_tree<T, R, 1, kFp8, L, kPad, kNt, kSums>(batch, rs, s);
}

// T = 256, aligned rows: every shape, and the default shapes with padding slots skipped.
template <bool kFp8, Pad kPad, bool kSums>
hipError_t launch_default(GemvBatch& batch, TreeShape shape, const PckRowSumBatch* rs,
                          hipStream_t s) {
  constexpr int T = 256;
  const bool nt = shape.nt != 0;
  const int u = shape.unroll;
  if constexpr (kPad == Pad::kSkipped) {
    constexpr Load L = Load::kAligned;
    if (shape.rows == 2) return launch_tree<T, 2, 1, kFp8, L, kPad, true, kSums>(batch, rs, s);
    return u == 2 ? launch_tree<T, 1, 2, kFp8, L, kPad, true, kSums>(batch, rs, s)
                  : launch_tree<T, 1, 1, kFp8, L, kPad, true, kSums>(batch, rs, s);
  } else {
    switch (shape.rows) {
      case 4:
        return nt ? launch_unroll<T, 4, kFp8, kPad, true, kSums>(batch, u, rs, s)
                  : launch_unroll<T, 4, kFp8, kPad, false, kSums>(batch, u, rs, s);
      case 2:
        return nt ? launch_unroll<T, 2, kFp8, kPad, true, kSums>(batch, u, rs, s)
                  : launch_unroll<T, 2, kFp8, kPad, false, kSums>(batch, u, rs, s);
      default:
        return nt ? launch_unroll<T, 1, kFp8, kPad, true, kSums>(batch, u, rs, s)
                  : launch_unroll<T, 1, kFp8, kPad, false, kSums>(batch, u, rs, s);
    }
  }
}

// Aligned rows in a tree of T != 256 lanes.  With non-temporal loads the shapes keep 8 to 16 vectors
// in flight per lane (chains x R x U), fewer chains per lane leaving room for more rows or positions;
// the best of R in {1, 2, 4}, U in {1 .. 4, 8} streamed from HBM.  Against R = 1, U = 2 with plain
// loads, which is what smaller launches take: BF16 14336 x 4096 T = 64 / 128 / 512 20.0 / 19.6 / 19.5
// against 23.2 / 21.9 / 21.5 us; FP8 14336 x 8192 23.0 / 23.0 / 23.0 against 24.9 / 24.7 / 32.2.
// T = 32 holds two rows side by side in a wave already: one such pair for BF16 (8192 x 8192 25.5
// against 30.6 us with two and 27.7 before).
template <int T, bool kFp8, Pad kPad, bool kNt, bool kSums>
hipError_t launch_other(GroupPlan& plan, const PckRowSumBatch* rs, hipStream_t s) {
  constexpr Load L = Load::kAligned;
  GemvBatch& b = plan.batch;
  if constexpr (T >= 1024) {
    return launch_tree<T, 1, 1, kFp8, L, kPad, kNt, kSums>(b, rs, s);
  } else if constexpr (T >= 512) {
    if (kFp8 && plan.rows >= 2048)
      return launch_tree<T, 2, 1, kFp8, L, kPad, kNt, kSums>(b, rs, s);
    return launch_tree<T, 1, 1, kFp8, L, kPad, kNt, kSums>(b, rs, s);
  } else {
    if constexpr (!kNt) {  // served from a cache, one row and two positions is the best shape
      return launch_tree<T, 1, 2, kFp8, L, kPad, kNt, kSums>(b, rs, s);
    } else {
      // one row per wave for BF16 rows of at most 4096 columns and for few rows
      if ((!kFp8 && plan.max_vectors <= 512) || plan.rows < 4096)
        return launch_tree<T, 1, 4, kFp8, L, kPad, kNt, kSums>(b, rs, s);
      if constexpr (T == 32 && !kFp8)
        return launch_tree<T, 1, 4, kFp8, L, kPad, kNt, kSums>(b, rs, s);
      else
        return launch_tree<T, 2, T >= 128 ? 2 : 4, kFp8, L, kPad, kNt, kSums>(b, rs, s);
    }
  }
}

template <int T, bool kFp8, Pad kPad, bool kSums>
hipError_t launch_aligned(GroupPlan& plan, const PckRowSumBatch* rs, hipStream_t s) {
  if constexpr (T == 256) {
    return launch_default<kFp8, kPad, kSums>(
        plan.batch, choose_shape(plan.max_per_lane, plan.rows, kFp8), rs, s);
  } else {
    return plan.bytes < kCachedBytes ? launch_other<T, kFp8, kPad, false, kSums>(plan, rs, s)
                                     : launch_other<T, kFp8, kPad, true, kSums>(plan, rs, s);
  }
}

// Rows read at any byte address.  Two rows per wave slot: the best shape of the same sweep for
// nearly every T and length.  Against element loads, at T = 256: BF16 14336 x 4100 20.6 against
// 118 us, 14337 x 4099 29.7 against 120; FP8 28672 x 4104 26.3 against 326 us, 28673 x 4099
// (addresses of any byte) 51 against 326.
template <int T, bool kFp8, bool kSums>
hipError_t launch_unaligned(GroupPlan& plan, const PckRowSumBatch* rs, hipStream_t s) {
  constexpr int R = T >= 1024 || (T >= 512 && !kFp8) ? 1 : 2;
  constexpr int U = T <= 64 ? 2 : 1;
  return launch_tree<T, R, U, kFp8, Load::kUnaligned, Pad::kSkipped, true, kSums>(plan.batch, rs, s);
}

// Rows that end inside the first kLive chain slots (at most 64 kLive vectors).
template <int T, int kLive, bool kFp8, bool kSums>
hipError_t launch_live(GroupPlan& plan, const PckRowSumBatch* rs, hipStream_t s) {
  constexpr Load A = Load::kAligned, X = Load::kUnaligned;
  constexpr int Ra = kFp8 || kLive == 2 ? 2 : 1;
  constexpr int Rx = kFp8 || kLive <= 4 ? 2 : 1;
  GemvBatch& b = plan.batch;
  return plan.load == A
             ? launch_tree<T, Ra, 1, kFp8, A, Pad::kZeroed, true, kSums, kLive>(b, rs, s)
             : launch_tree<T, Rx, 1, kFp8, X, Pad::kSkipped, true, kSums, kLive>(b, rs, s);
}

// The route of a launch: element loads for rows shorter than a vector; else the fewest live
// chain slots that hold the longest row (T = 1024, 14336 x 4096: BF16 8 slots of 16 20.3 against
// 36.6 us with all and 62 before, FP8 4 slots 19.9 against 69.5 and 139 us); else all slots, dead
// ones skipped where that pays for its branches: at T = 1024 for more than a quarter of the slots and
// from 2048 rows on (BF16 11264 columns, ten dead slots: 4096 rows 21.5 against 24.7 us zeroed; 14336
// columns, four: 512 rows 8.9 against 8.1), at T = 256 and 512 always (FP8 11264 columns at T = 512,
// five: 512 rows 5.6 against 6.2 us, 8192 rows 22.4 against 25.4).  pck_gemv_set_shape picks the shape
// of aligned T = 256 launches, which then keep all slots.
template <int T, bool kFp8, bool kSums = false>
hipError_t launch_for_threads(GroupPlan& plan, hipStream_t s, const PckRowSumBatch* rs = nullptr) {
  if (plan.load == Load::kElement)
    return launch_tree<T, 1, 1, kFp8, Load::kElement, Pad::kZeroed, false, kSums>(plan.batch, rs, s);
  const bool all =
      T == 256 && plan.load == Load::kAligned && g_shape_override.rows > 0;  // a chosen shape
  if constexpr (T >= 256) {
    if (!all && plan.max_vectors <= 2 * kWave) return launch_live<T, 2, kFp8, kSums>(plan, rs, s);
  }
  if constexpr (T >= 512) {
    if (plan.max_vectors <= 4 * kWave) return launch_live<T, 4, kFp8, kSums>(plan, rs, s);
  }
  if constexpr (T >= 1024) {
    if (plan.max_vectors <= 8 * kWave) return launch_live<T, 8, kFp8, kSums>(plan, rs, s);
  }
  if (plan.load == Load::kUnaligned) return launch_unaligned<T, kFp8, kSums>(plan, rs, s);
  if (!plan.pad) return launch_aligned<T, kFp8, Pad::kNone, kSums>(plan, rs, s);
  if constexpr (T >= 1024) {
    if (plan.dead_slots > 4 && plan.rows >= 2048)
      return launch_aligned<T, kFp8, Pad::kSkipped, kSums>(plan, rs, s);
  } else if constexpr (T >= 256) {
    if (plan.dead_slots > 0 && !all) return launch_aligned<T, kFp8, Pad::kSkipped, kSums>(plan, rs, s);
  }
  return launch_aligned<T, kFp8, Pad::kZeroed, kSums>(plan, rs, s);
}

template <int R, int U, bool kFp8, Pad kPad, bool kNt = true>
hipError_t launch_ride_shape(GemvBatch& batch, const PckCheckBatch& ride, hipStream_t stream) {
  const int64_t groups = plan_groups(batch, static_cast<int64_t>(R) * kWavesPerGroup);
  const int64_t total = groups + ride.start[ride.count];
  if (total * kGroupThreads > 0xFFFFFFFFll) return hipErrorInvalidValue;  // 32-bit dispatch size
  gemv_ride_kernel<256, R, U, kFp8, kPad, kNt>
      <<<dim3(static_cast<unsigned>(total)), dim3(kGroupThreads), 0, stream>>>(batch, ride);
  return hipGetLastError();
}

// The carried-check launch uses one shape per weight type and row length of the T = 256 aligned
// path, the launches a layer's checks ride in.
template <bool kFp8, Pad kPad>
hipError_t launch_ride_pad(GroupPlan& plan, const PckCheckBatch& ride, hipStream_t stream) {
  if constexpr (kFp8) {
    return launch_ride_shape<2, 1, true, kPad>(plan.batch, ride, stream);
  } else {
    return plan.max_per_lane > 2 ? launch_ride_shape<2, 2, false, kPad>(plan.batch, ride, stream)
                                 : launch_ride_shape<1, 2, false, kPad>(plan.batch, ride, stream);
  }
}

template <bool kFp8>
hipError_t launch_ride(GroupPlan& plan, const PckCheckBatch& ride, hipStream_t stream) {
  if (!plan.pad) return launch_ride_pad<kFp8, Pad::kNone>(plan, ride, stream);
  return plan.dead_slots > 0 ? launch_ride_pad<kFp8, Pad::kSkipped>(plan, ride, stream)
                        : launch_ride_pad<kFp8, Pad::kZeroed>(plan, ride, stream);
}

template <bool kFp8>
hipError_t plan_group(const PckGemv* gemvs, double* const* sums, int count, int threads,
                      GroupPlan& plan, const float* const* scales = nullptr,
                      float* const* scaled = nullptr) {
  constexpr int V = kFp8 ? 16 : 8;
  if (count < 1 || count > PCK_MAX_GROUP || gemvs == nullptr) return hipErrorInvalidValue;
  if (threads < kWarp || threads > 1024 || (threads & (threads - 1)) != 0)
    return hipErrorInvalidValue;
  plan.batch.count = count;
  for (int g = 0; g < count; ++g) {
    const PckGemv& d = gemvs[g];
    if (d.m < 0 || d.m > 0x7FFFFFFF || (d.m > 0 && (d.n < 1 || !d.W || !d.x || !d.y)))
      return hipErrorInvalidValue;
    double* rs = sums != nullptr ? sums[g] : nullptr;
    if (sums != nullptr && d.m > 0 && (rs == nullptr || reinterpret_cast<uintptr_t>(rs) % 16 != 0))
      return hipErrorInvalidValue;
    const int64_t n = d.m > 0 ? d.n : 1;
    const int64_t per_lane = ((n + V - 1) / V + threads - 1) / threads;
    plan.batch.item[g] =
        GemvItem{d.W, static_cast<const uint16_t*>(d.x), d.y, rs, d.m, n, per_lane};
    if (scaled != nullptr && d.m > 0) {
      if (scales == nullptr || scales[g] == nullptr || scaled[g] == nullptr)
        return hipErrorInvalidValue;
      plan.batch.item[g].scale = scales[g];
      plan.batch.item[g].y_scaled = scaled[g];
    }
    plan.rows += d.m;
    plan.bytes += d.m * n * (kFp8 ? 1 : 2);
    if (d.m > 0) {
      const bool aligned = n % V == 0 && reinterpret_cast<uintptr_t>(d.W) % 16 == 0 &&
                           reinterpret_cast<uintptr_t>(d.x) % 16 == 0;
      const Load load = n < V ? Load::kElement : aligned ? Load::kAligned : Load::kUnaligned;
      if (load < plan.load) plan.load = load;  // the narrowest loads any item needs
      const int64_t vectors = (n + V - 1) / V;
      plan.max_vectors = vectors > plan.max_vectors ? vectors : plan.max_vectors;
      plan.max_per_lane = per_lane > plan.max_per_lane ? per_lane : plan.max_per_lane;
      plan.pad = plan.pad || n % (static_cast<int64_t>(threads) * V) != 0;
      if (threads > kWave) {
        const int64_t slots = threads / kWave;
        const int64_t dead = (slots - (vectors + kWave - 1) / kWave % slots) % slots;
        plan.dead_slots = dead > plan.dead_slots ? dead : plan.dead_slots;
      }
    }
  }
  return hipSuccess;
}

template <bool kFp8>
hipError_t launch_group(const PckGemv* gemvs, int count, int threads, const PckCheckBatch* ride,
                        hipStream_t stream, const float* const* scales = nullptr,
                        float* const* scaled = nullptr) {
  GroupPlan plan;
  if (plan_group<kFp8>(gemvs, nullptr, count, threads, plan, scales, scaled) != hipSuccess)
    return hipErrorInvalidValue;
  if (ride != nullptr) {
    if (check::validate(*ride) != hipSuccess) return hipErrorInvalidValue;
    if (threads == 256 && plan.load == Load::kAligned && plan.rows > 0)
      return launch_ride<kFp8>(plan, *ride, stream);
    // Other configurations: the same check as its own launch first (identical results).
    const int64_t items = ride->start[ride->count];
    if (items * check::kThreads > 0xFFFFFFFFll) return hipErrorInvalidValue;
    const int err = pck_blocked_check(ride, stream);
    if (err != 0) return static_cast<hipError_t>(err);
  }
  switch (threads) {
    case 32: return launch_for_threads<32, kFp8>(plan, stream);
    case 64: return launch_for_threads<64, kFp8>(plan, stream);
    case 128: return launch_for_threads<128, kFp8>(plan, stream);
    case 256: return launch_for_threads<256, kFp8>(plan, stream);
    case 512: return launch_for_threads<512, kFp8>(plan, stream);
    default: return launch_for_threads<1024, kFp8>(plan, stream);
  }
}

template <bool kFp8>
hipError_t launch_group_rowsums(const PckGemv* gemvs, double* const* sums, int count, int threads,
                                const PckRowSumBatch* ride, hipStream_t stream) {
  if (sums == nullptr) return hipErrorInvalidValue;
  GroupPlan plan;
  if (plan_group<kFp8>(gemvs, sums, count, threads, plan) != hipSuccess)
    return hipErrorInvalidValue;
  PckRowSumBatch none{};
  const PckRowSumBatch* rs = ride != nullptr ? ride : &none;
  if (rowsum::validate(*rs) != hipSuccess) return hipErrorInvalidValue;
  switch (threads) {
    case 32: return launch_for_threads<32, kFp8, true>(plan, stream, rs);
    case 64: return launch_for_threads<64, kFp8, true>(plan, stream, rs);
    case 128: return launch_for_threads<128, kFp8, true>(plan, stream, rs);
    case 256: return launch_for_threads<256, kFp8, true>(plan, stream, rs);
    case 512: return launch_for_threads<512, kFp8, true>(plan, stream, rs);
    default: return launch_for_threads<1024, kFp8, true>(plan, stream, rs);
  }
}

}  // namespace
}  // namespace pck

extern "C" {

int pck_gemv_bf16_coalesced(const void* W, const void* x, float* y, int64_t m, int64_t n,
                            int threads, void* stream) {
  const PckGemv one{W, x, y, m, n};
  return pck::launch_group<false>(&one, 1, threads, nullptr, static_cast<hipStream_t>(stream));
}

int pck_gemv_fp8_coalesced(const void* Q, const void* x, float* z, int64_t m, int64_t n,
                           int threads, void* stream) {
  const PckGemv one{Q, x, z, m, n};
  return pck::launch_group<true>(&one, 1, threads, nullptr, static_cast<hipStream_t>(stream));
}

int pck_gemv_group_check(int weight_kind, const PckGemv* gemvs, int count, int threads,
                         const PckCheckBatch* ride, void* stream) {
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (weight_kind == 0) return pck::launch_group<false>(gemvs, count, threads, ride, s);
  if (weight_kind == 1) return pck::launch_group<true>(gemvs, count, threads, ride, s);
  return hipErrorInvalidValue;
}

int pck_gemv_group_rowsums(int weight_kind, const PckGemv* gemvs, double* const* sums, int count,
                           int threads, const PckRowSumBatch* ride, void* stream) {
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (weight_kind == 0) return pck::launch_group_rowsums<false>(gemvs, sums, count, threads, ride, s);
  if (weight_kind == 1) return pck::launch_group_rowsums<true>(gemvs, sums, count, threads, ride, s);
  return hipErrorInvalidValue;
}

int pck_gemv_group(int weight_kind, const PckGemv* gemvs, int count, int threads, void* stream) {
  return pck_gemv_group_check(weight_kind, gemvs, count, threads, nullptr, stream);
}

int pck_gemv_group_fp8_scaled(const PckGemv* gemvs, const float* const* scales,
                              float* const* scaled, int count, int threads,
                              const PckCheckBatch* ride, void* stream) {
  if (scales == nullptr || scaled == nullptr) return hipErrorInvalidValue;
  return pck::launch_group<true>(gemvs, count, threads, ride, static_cast<hipStream_t>(stream),
                                 scales, scaled);
}

int pck_gemv_bf16_naive(const void* W, const void* x, float* y, int64_t m, int64_t n, int threads,
                        void* stream) {
  if (threads < 1 || threads > 1024 || (threads & (threads - 1)) != 0) return hipErrorInvalidValue;
  const int64_t lanes = threads < 64 ? 64 : threads;  // workgroup size of the launch
  if (m < 0 || m > 0x7FFFFFFF || m * lanes > 0xFFFFFFFFll) return hipErrorInvalidValue;
  if (m == 0) return hipSuccess;
  if (n < 1 || !W || !x || !y) return hipErrorInvalidValue;
  const int64_t chunk = (n + threads - 1) / threads;
  using pck::Load;
  const bool aligned = chunk % 8 == 0 && n % 8 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(x) % 16 == 0;
  const Load load = n < 8 || chunk < 4 ? Load::kElement : aligned ? Load::kAligned : Load::kUnaligned;
  // Rows per workgroup, from 8192 rows on (fewer leave too few workgroups).  Aligned chunks of one
  // vector: four (14336 x 4096, T = 512: 22.4 against 25.3 us with one; 8192 x 2048, T = 256, from
  // the caches: 5.5 / 6.3).  Of two: two, both vectors ahead (14336 x 4096, T = 256, from HBM 25.1
  // us, one row 26.7, four 25.0; from the caches 18.6 / 18.8 / 19.3, as four rows' loads push each
  // other out of the L1).  Longer ones: one (4096 x 14336: 84 us with four, 58 with one).  Ragged
  // chunks: four (7182 x 8960, T = 256: 55 against 212 us with element loads), in fewer rows only
  // where those are long enough to be bound by their loads (3000 x 512, T = 128: equal; 2048 x 512:
  // 3.9 / 3.1).
  const bool many = load == Load::kUnaligned
                        ? m >= 8192 || (m >= 2048 && m * n >= 1500000)
                        : load == Load::kAligned && chunk <= 16 && m >= 8192 && threads >= 256;
  const int rows = !many ? 1 : load == Load::kAligned && chunk > 8 ? 2 : 4;
  const dim3 grid(static_cast<unsigned>((m + rows - 1) / rows)), group(static_cast<unsigned>(lanes));
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const auto* w16 = static_cast<const uint16_t*>(W);
  const auto* x16 = static_cast<const uint16_t*>(x);
  auto launch = [&](auto kernel) {
    kernel<<<grid, group, 0, s>>>(w16, x16, y, m, n, chunk, threads);
    return hipGetLastError();
  };
  if (load == Load::kElement) return launch(pck::gemv_naive_kernel<Load::kElement, 1>);
  if (load == Load::kAligned)
    return rows == 4   ? launch(pck::gemv_naive_kernel<Load::kAligned, 4>)
           : rows == 2 ? launch(pck::gemv_naive_kernel<Load::kAligned, 2>)
                       : launch(pck::gemv_naive_kernel<Load::kAligned, 1>);
  return many ? launch(pck::gemv_naive_kernel<Load::kUnaligned, 4>)
              : launch(pck::gemv_naive_kernel<Load::kUnaligned, 1>);
}

int pck_gemv_set_shape(int rows_per_wave, int unroll, int nontemporal) {
  if (rows_per_wave < 0 || rows_per_wave > 4 || rows_per_wave == 3 || unroll < 0 || unroll > 4 ||
      (rows_per_wave > 0 && unroll < 1))
    return hipErrorInvalidValue;
  pck::g_shape_override = pck::TreeShape{rows_per_wave, unroll, nontemporal != 0};
  return hipSuccess;
}

const char* pck_error_string(int err) { return hipGetErrorString(static_cast<hipError_t>(err)); }

}  // extern "C"
