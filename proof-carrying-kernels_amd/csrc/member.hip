// Sampled-token membership check (top-k / top-p / greedy) for a batch of rows, on gfx950.
//
// Semantics: reference src/pck/member.py:118-197 (`check_members`), per row with logits l,
// token t, k = top_k (vocab if none), p = top_p (1 if none):
//   above   = #{j : l_j > l_t}                                  exact FP32 compares
//   ok      = no NaN in l  and  0 <= t < vocab  and  above < (greedy ? 1 : k)
//   top-p   kept = {j : l_j >= kth} where kth is the k_eff-th largest logit, k_eff =
//           min(k, k_lim) (k_lim = largest host top-k below vocab: a stale host copy is
//           clamped, reference member.py:170,175); every logit is kept for a row without a
//           top-k, unless all_k (reference's top-(max k) path) says every row has one.
//           r = sum_{kept, l_j > l_t} e_j / sum_{kept} e_j with e_j the FP32 term
//           expf(hi) + expf(hi) lo of the exact split l_j - max = hi + lo (TwoSum), 0 when
//           hi < -128 (reference member.py:105-115), summed in FP64.
//           ok &= p >= 1 or greedy or r < next_up(p + slack); mass_above = p < 1 ? r : 0.
// The sums are order-free within member_eps32 (reference member.py:84-102); ok and above are
// exact.  For a token below kth (already rejected by the top-k test) r counts every kept
// logit above it, where the reference's top-(max k) path leaves out ties beyond max k; the
// verdict is the same (false).
//
// Kernel: one workgroup of 1024 lanes per row.
//   Prefix (the first kPrefix logits): count above, NaN flag and each lane's
//   maximum.  For a top-p row with a top-k, a 16-bit radix select over the 1024 lane maxima
//   gives L0, a value at or below the k_eff-th largest lane maximum, so at least k_eff logits of
//   the prefix are >= L0 and L0 is a lower bound of the row's kth (the k-th largest of a part
//   never exceeds that of the whole).
//   Stream (the rest of the row, read from HBM once, non-temporal): count above, NaN flag, row
//   maximum, and the logits >= L0 compacted into LDS, each wave into its own segment of kSeg
//   slots (a ballot per step; the wave's count is uniform, so no atomics); then the prefix,
//   held in registers (or re-read from L2 for unaligned or short rows), is compacted too.  For
//   LLM logits that is a few hundred values (a few dozen per wave); kth and both sums come from
//   LDS with no further pass over the row, each wave reading back its own segment (into
//   registers, one candidate per lane, when no wave holds more than 64).
//   Tail: one exchange for the counts, flags and maximum; kth by an exact radix select over the
//   candidates, four 8-bit rounds of one barrier each (every wave scans the histogram itself
//   and finds the digit in scalar registers); the two FP64 sums; the verdict.
//   Fallbacks: if more than kSeg values qualify in one wave (flat or adversarial rows), an
//   exact 4-pass radix select over the row and a summing pass take over.  Rows without a top-k
//   sum over the whole row in a second pass.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "pck_hip.h"
#include "rounding.h"

namespace pck {
namespace {

constexpr int kThreads = 1024;
constexpr int kWave = 64;
constexpr int kWaves = kThreads / kWave;
constexpr int kCap = 4096;  // candidates held in LDS
constexpr int kSeg = kCap / kWaves;  // candidates each wave holds, in its own segment
constexpr int64_t kPrefix = 16 * kThreads;  // logits that set the candidate threshold

using MemberArgs = PckMemberArgs;

// Order-preserving 64-bit key of an FP64 value (a larger value has a larger key), for the
// totals' running maximum of r - p, kept with an unsigned atomic maximum.
__device__ __forceinline__ unsigned long long order_key64(double v) {
  const unsigned long long u = static_cast<unsigned long long>(__double_as_longlong(v));
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}

// Order-preserving key: a larger float has a larger key; -0 and +0 share the key of +0.
__device__ __forceinline__ uint32_t order_key(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u << 1) == 0) u = 0;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// FP32 e^(x - m) from the exact split x - m = hi + lo (Knuth's TwoSum), 0 where hi < -128 or
// NaN; the operation order of reference member.py:110-115.
__device__ __forceinline__ float split_term(float x, float m) {
  const float nm = -m;
  const float hi = x + nm;
  const float bv = hi - x;
  const float lo = (x - (hi - bv)) + (nm - bv);
  const float eh = expf(hi);
  const float prod = eh * lo;
  return hi >= -128.0f ? eh + prod : 0.0f;
}

struct Scratch {
  alignas(16) float cand[kCap];
  alignas(16) uint32_t hist[3][256];
  double red_d[2][kWaves];
  int64_t red_i[kWaves];
  float red_f[kWaves];
  int red_flag[kWaves];
};

__device__ __forceinline__ int lane_id() { return static_cast<int>(threadIdx.x) & (kWave - 1); }
__device__ __forceinline__ int wave_id() { return static_cast<int>(threadIdx.x) / kWave; }

// The value of v in the lane kCtrl's DPP pattern names (every lane has a source here).
template <int kCtrl>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
  return static_cast<uint32_t>(
      __builtin_amdgcn_update_dpp(0, static_cast<int>(v), kCtrl, 0xF, 0xF, false));
}
template <int kCtrl>
__device__ __forceinline__ float dpp(float v) {
  return __uint_as_float(dpp<kCtrl>(__float_as_uint(v)));
}
template <int kCtrl>
__device__ __forceinline__ double dpp(double v) {
  const uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
  const uint64_t lo = dpp<kCtrl>(static_cast<uint32_t>(u));
  const uint64_t hi = dpp<kCtrl>(static_cast<uint32_t>(u >> 32));
  return __longlong_as_double(static_cast<long long>(lo | (hi << 32)));
}

__device__ __forceinline__ uint32_t read_lane(uint32_t v, int lane) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), lane));
}
__device__ __forceinline__ float read_lane(float v, int lane) {
  return __uint_as_float(read_lane(__float_as_uint(v), lane));
}
__device__ __forceinline__ double read_lane(double v, int lane) {
  const uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
  const uint64_t lo = read_lane(static_cast<uint32_t>(u), lane);
  const uint64_t hi = read_lane(static_cast<uint32_t>(u >> 32), lane);
  return __longlong_as_double(static_cast<long long>(lo | (hi << 32)));
}

// op over the wave's 64 lanes, returned in every lane, in a fixed order: inside each 16-lane
// row, partners at quad_perm [1,0,3,2] and [2,3,0,1], then row_ror 4 and row_ror 8 (every
// lane then holds its row's result; for a non-associative op the lanes may differ in how it
// was grouped, and only lanes 0, 16, 32 and 48 are read), then (r0 op r1) op (r2 op r3).
// Every lane must be active.
template <typename T, typename Op>
__device__ __forceinline__ T wave_reduce(T v, Op op) {
  v = op(v, dpp<0xB1>(v));
  v = op(v, dpp<0x4E>(v));
  v = op(v, dpp<0x124>(v));
  v = op(v, dpp<0x128>(v));
  return op(op(read_lane(v, 0), read_lane(v, 16)), op(read_lane(v, 32), read_lane(v, 48)));
}

// Workgroup sum of `count`, OR of `flag` and max of `v` (one barrier; the exchange slots are
// not reused afterwards).  A lane's count and the wave's sum fit in 32 bits.
__device__ void group_reduce(uint32_t lane_count, int64_t& count, int& flag, float& v,
                             Scratch& s) {
  const uint32_t c = wave_reduce(lane_count, [](uint32_t x, uint32_t y) { return x + y; });
  const uint32_t f =
      wave_reduce(static_cast<uint32_t>(flag), [](uint32_t x, uint32_t y) { return x | y; });
  const float mx = wave_reduce(v, [](float x, float y) { return fmaxf(x, y); });
  if (lane_id() == 0) {
    s.red_i[wave_id()] = c;
    s.red_flag[wave_id()] = static_cast<int>(f);
    s.red_f[wave_id()] = mx;
  }
  __syncthreads();
  count = 0;
  flag = 0;
  v = -__builtin_inff();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    count += s.red_i[w];
    flag |= s.red_flag[w];
    v = fmaxf(v, s.red_f[w]);
  }
}

// Two FP64 sums at once (the kept mass and the mass above the token), in a fixed order (one
// barrier; the exchange slots are not reused afterwards).
__device__ void group_sum2(double& a, double& b, Scratch& s) {
  const auto add = [](double x, double y) { return x + y; };
  a = wave_reduce(a, add);
  b = wave_reduce(b, add);
  if (lane_id() == 0) {
    s.red_d[0][wave_id()] = a;
    s.red_d[1][wave_id()] = b;
  }
  __syncthreads();
  a = 0.0;
  b = 0.0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    a += s.red_d[0][w];
    b += s.red_d[1][w];
  }
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <bool kNt>
__device__ __forceinline__ f32x4 load_quad(const f32x4* p) {
  if constexpr (kNt) return __builtin_nontemporal_load(p);
  else return *p;
}

// Calls f4(quad) for the 16-byte quads and f1(value) for the remaining logits of row[begin,
// end), each logit exactly once (begin % 4 == 0); four quads in flight per lane when the row is
// aligned, element loads otherwise.  kNt: non-temporal loads (data read once that need not stay
// in the caches).  pre() runs once, by every lane, after the first quads are requested and
// before any is used, so workgroup-wide work placed there overlaps their latency.
template <bool kNt, typename F4, typename F1, typename P>
__device__ __forceinline__ void for_each4(const float* __restrict__ row, int64_t begin,
                                          int64_t end, F4&& f4, F1&& f1, P&& pre) {
  const int t = static_cast<int>(threadIdx.x);
  int64_t done = begin;
  if ((reinterpret_cast<uintptr_t>(row) & 15) == 0) {
    const f32x4* quads = reinterpret_cast<const f32x4*>(row);
    const int64_t q1 = end / 4;
    int64_t q = begin / 4 + t;
    // four quads ahead where the wave's last lane has them all, so a wave's lanes go the same way
    const int64_t ahead = 3 * kThreads + (kWave - 1 - lane_id());
    const bool first = q + ahead < q1;
    f32x4 a, b, c, d;
    if (first) {
      a = load_quad<kNt>(quads + q);
      b = load_quad<kNt>(quads + q + kThreads);
      c = load_quad<kNt>(quads + q + 2 * kThreads);
      d = load_quad<kNt>(quads + q + 3 * kThreads);
    }
    pre();
    if (first) {
      f4(a), f4(b), f4(c), f4(d);
      q += 4 * kThreads;
    }
    for (; q + ahead < q1; q += 4 * kThreads) {
      a = load_quad<kNt>(quads + q);
      b = load_quad<kNt>(quads + q + kThreads);
      c = load_quad<kNt>(quads + q + 2 * kThreads);
      d = load_quad<kNt>(quads + q + 3 * kThreads);
      f4(a), f4(b), f4(c), f4(d);
    }
    for (; q < q1; q += kThreads) f4(load_quad<kNt>(quads + q));
    done = end > begin ? (q1 * 4 > begin ? q1 * 4 : begin) : end;
  } else {
    pre();
  }
  for (int64_t i = done + t; i < end; i += kThreads) f1(row[i]);
}

template <bool kNt, typename F4, typename F1>
__device__ __forceinline__ void for_each4(const float* __restrict__ row, int64_t begin,
                                          int64_t end, F4&& f4, F1&& f1) {
  for_each4<kNt>(row, begin, end, f4, f1, [] {});
}

// Calls f(value) for every logit of row[begin, end), each exactly once (begin % 4 == 0).
template <bool kNt, typename F>
__device__ __forceinline__ void for_each(const float* __restrict__ row, int64_t begin,
                                         int64_t end, F&& f) {
  for_each4<kNt>(row, begin, end, [&](const f32x4& v) { f(v[0]), f(v[1]), f(v[2]), f(v[3]); }, f);
}

// Inclusive prefix sum over the 64 lanes in VALU cross-lane moves: Hillis-Steele steps of
// 1, 2, 4 and 8 inside each 16-lane row (row_shr, lanes without a source read 0), then each
// row's total is carried into the next (row_bcast:15 into rows 1 and 3, row_bcast:31 into rows
// 2 and 3).
__device__ __forceinline__ uint32_t wave_inclusive_sum(uint32_t v) {
  const int x = static_cast<int>(v);
  int a = x + __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, true);  // row_shr:1
  a += __builtin_amdgcn_update_dpp(0, a, 0x112, 0xF, 0xF, true);         // row_shr:2
  a += __builtin_amdgcn_update_dpp(0, a, 0x114, 0xF, 0xF, true);         // row_shr:4
  a += __builtin_amdgcn_update_dpp(0, a, 0x118, 0xF, 0xF, true);         // row_shr:8
  a += __builtin_amdgcn_update_dpp(0, a, 0x142, 0xA, 0xF, false);        // row_bcast:15
  a += __builtin_amdgcn_update_dpp(0, a, 0x143, 0xC, 0xF, false);        // row_bcast:31
  return static_cast<uint32_t>(a);
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Adds the digits (k >> shift) & 255 of the keys with (k & mask) == prefix into hist.  Keys
// bunch into a few buckets (one exponent byte for every candidate): a wave whose counted lanes
// share one digit adds them with one atomic instead of serialising them.
__device__ __forceinline__ void radix_count(uint32_t k, uint32_t prefix, uint32_t mask,
                                            int shift, uint32_t* hist) {
  const bool hit = (k & mask) == prefix;
  const uint32_t digit = (k >> shift) & 255u;
  const uint64_t counted = __ballot(hit);
  const int first = counted ? __builtin_ctzll(counted) : 0;
  const uint32_t d0 = read_lane(digit, first);
  if (__ballot(hit && digit != d0) == 0) {
    if (counted != 0 && lane_id() == first)
      atomicAdd(&hist[d0], static_cast<uint32_t>(__builtin_popcountll(counted)));
  } else if (hit) {
    atomicAdd(&hist[digit], 1u);
  }
}

// The digit of a complete 256-bin histogram that holds the want-th largest key, with want
// turned into the rank within that digit; every wave computes it itself.  Lane l owns digits
// 255 - 4l ... 252 - 4l (descending; h[3] is digit 255 - 4l).  The first lane whose inclusive
// count reaches want owns the digit; its four counts and the count before them are read into
// scalar registers and the descent runs once per wave.
__device__ __forceinline__ uint32_t radix_find(const uint32_t* hist, uint32_t& want) {
  const u32x4 h = *reinterpret_cast<const u32x4*>(hist + 252 - 4 * lane_id());
  const uint32_t own = h[0] + h[1] + h[2] + h[3];
  const uint32_t incl = wave_inclusive_sum(own);
  const uint64_t reach = __ballot(incl >= want);
  const int src = reach ? __builtin_ctzll(reach) : kWave - 1;
  uint32_t rest = want - read_lane(incl - own, src);  // rank within the owner's four digits
  uint32_t digit = static_cast<uint32_t>(255 - 4 * src);
  const uint32_t c3 = read_lane(h[3], src);
  const uint32_t c2 = read_lane(h[2], src);
  const uint32_t c1 = read_lane(h[1], src);
  if (rest > c3) {
    rest -= c3, --digit;
    if (rest > c2) {
      rest -= c2, --digit;
      if (rest > c1) rest -= c1, --digit;
    }
  }
  want = rest;
  return digit;
}

// Key of the rank-th largest (1-based) of the workgroup's keys, by an exact radix select over
// 8-bit digits with LDS histograms.  visit(f) calls f(key) for each key a lane holds, the same
// way on every round (each key by one lane).  Every lane returns the same key.  With kRounds < 4
// only the top 8 kRounds bits are selected and the rest are zero: the result is the smallest key
// of the bucket that holds the rank-th largest.  The caller clears hist[0], with a barrier
// between that and the call.
template <int kRounds = 4, typename V>
__device__ uint32_t radix_select(int64_t rank, V&& visit, Scratch& s) {
  const int t = static_cast<int>(threadIdx.x);
  uint32_t prefix = 0;
  uint32_t mask = 0;
  uint32_t want = static_cast<uint32_t>(rank);  // counts fit in 32 bits (vocab < 2^31)
#pragma unroll
  for (int round = 0; round < kRounds; ++round) {
    const int shift = 24 - 8 * round;
    uint32_t* const hist = s.hist[round % 3];
    // Round r counts into hist[r % 3] and clears hist[(r + 1) % 3], last read by the scans of
    // round r - 2, which every wave finished before the barrier of round r - 1; every wave
    // scans the histogram itself, so a round takes one barrier.
    if (t < 256) s.hist[(round + 1) % 3][t] = 0;
    visit([&](uint32_t k) { radix_count(k, prefix, mask, shift, hist); });
    __syncthreads();
    prefix |= radix_find(hist, want) << shift;
    mask |= 255u << shift;
  }
  return prefix;
}

// One row's request, as the checks use it.
struct RowRequest {
  int64_t token;
  bool in_range;    // the token id lies in [0, vocab)
  int64_t k_row;    // top-k clamped to [1, vocab] (reference src/pck/member.py:153)
  bool request_ok;  // the request index lies inside the temperature array (or there is none)
  bool greedy;
  double p;
  bool want_mass;  // a top-p below 1
  bool use_kth;    // the kept set is cut at the k_eff-th largest logit
  int64_t k_eff;
};

// The token first, for the kernel that reads its logit ahead of the rest of the request.
__device__ __forceinline__ RowRequest row_token(const MemberArgs& A, int64_t r) {
  RowRequest q;
  q.token = A.tokens[r];
  q.in_range = q.token >= 0 && q.token < A.vocab;
  return q;
}

__device__ __forceinline__ RowRequest row_request(const MemberArgs& A, int64_t r, RowRequest q) {
  const int64_t k_req = A.top_k ? A.top_k[r] : A.vocab;
  q.k_row = k_req < 1 ? 1 : (k_req > A.vocab ? A.vocab : k_req);
  // Greedy rows: the caller's flags, or temperature 0 of the row's request (vLLM's sampling
  // state, read through the row's request index).  A request index outside the temperature
  // array rejects the row without reading it.
  const int64_t request = A.temperature ? A.temperature_index[r] : 0;
  q.request_ok = !A.temperature || (request >= 0 && request < A.temperature_count);
  q.greedy = A.temperature ? q.request_ok && A.temperature[q.request_ok ? request : 0] == 0.0f
                           : (A.greedy ? A.greedy[r] != 0 : false);
  const bool has_p = A.top_p != nullptr;
  q.p = !has_p ? 1.0
        : A.top_p_fp32 ? static_cast<double>(static_cast<const float*>(A.top_p)[r])
                       : static_cast<const double*>(A.top_p)[r];
  q.want_mass = has_p && q.p < 1.0;
  q.use_kth = A.all_k || (A.k_lim > 0 && q.k_row < A.vocab);
  q.k_eff = q.k_row < A.k_lim ? q.k_row : A.k_lim;
  return q;
}

// The row's verdict from its exact count above the token and its two masses (z kept, a kept and
// above the token; used when the row wants a mass), written by one lane.
__device__ __forceinline__ void write_verdict(const MemberArgs& A, int64_t r, const RowRequest& q,
                                              int64_t above, bool any_nan, double z, double a) {
  bool ok = q.request_ok && !any_nan && q.in_range && above < (q.greedy ? 1 : q.k_row);
  double mass = 0.0;
  if (q.want_mass) {
    const double ratio = a / z;
    mass = ratio;
    const double high = next_up(q.p + A.slack);  // the bound rounded outward
    ok = ok && (q.greedy || ratio < high);
  }
  if (A.ok) A.ok[r] = ok;
  if (A.above) A.above[r] = above;
  if (A.mass_above) A.mass_above[r] = mass;
  if (A.totals) {
    // Running totals (integer atomics, so the sums do not depend on the order of rows):
    // rows, rejected, injected, caught (rejected and injected), false alarms (rejected, not
    // injected), and the maximum of r - p over accepted top-p rows not greedy (the key of
    // -1 is the host's initial value: no such row yet).
    unsigned long long* tot = A.totals;
    const bool injected = A.injected ? A.injected[r] != 0 : false;
    atomicAdd(&tot[0], 1ull);
    if (!ok) atomicAdd(&tot[1], 1ull);
    if (injected) atomicAdd(&tot[2], 1ull);
    if (!ok && injected) atomicAdd(&tot[3], 1ull);
    if (!ok && !injected) atomicAdd(&tot[4], 1ull);
    if (ok && q.want_mass && !q.greedy) atomicMax(&tot[5], order_key64(mass - q.p));
  }
}

__global__ void __launch_bounds__(kThreads) member_kernel(const MemberArgs A) {
  __shared__ Scratch s;
  const int64_t r = blockIdx.x;
  const int t = static_cast<int>(threadIdx.x);
  const int64_t vocab = A.vocab;
  const float* __restrict__ row = A.logits + r * vocab;

  const RowRequest asked = row_token(A, r);
  const float lt = row[asked.in_range ? asked.token : (asked.token < 0 ? 0 : vocab - 1)];
  const RowRequest q = row_request(A, r, asked);
  const bool want_mass = q.want_mass, use_kth = q.use_kth;
  const int64_t k_eff = q.k_eff;
  const bool fused = want_mass && use_kth && k_eff <= kThreads;
  const int64_t prefix = vocab < kPrefix ? vocab : kPrefix;

  // Exact count above the token, NaN flag and lane maxima over the prefix (kept in L2).
  uint32_t above_lane = 0;
  int nan = 0;
  float lane_max = -__builtin_inff();
  auto scan = [&](float l) {
    above_lane += l > lt;
    nan |= l != l;
    lane_max = fmaxf(lane_max, l);
  };
  // An aligned row with a full prefix keeps its prefix quads in registers for the compaction.
  const bool held = (reinterpret_cast<uintptr_t>(row) & 15) == 0 && prefix == kPrefix;
  constexpr int kHeld = kPrefix / (4 * kThreads);
  f32x4 pq[kHeld];
  if (held) {
    const f32x4* quads = reinterpret_cast<const f32x4*>(row);
#pragma unroll
    for (int j = 0; j < kHeld; ++j) pq[j] = quads[t + j * kThreads];
#pragma unroll
    for (int j = 0; j < kHeld; ++j) scan(pq[j][0]), scan(pq[j][1]), scan(pq[j][2]), scan(pq[j][3]);
  } else {
    for_each<false>(row, 0, prefix, scan);
  }

  // Candidate threshold: the smallest value of the 16-bit key bucket that holds the k_eff-th
  // largest lane maximum of the prefix (a NaN bit pattern there means -inf: keep everything).
  // It is selected while the stream's first loads are in flight.
  float low = -__builtin_inff();
  auto threshold = [&] {
    const uint32_t key = order_key(lane_max);
    if (t < 256) s.hist[0][t] = 0;
    __syncthreads();
    low = key_value(radix_select<2>(k_eff, [&](auto&& f) { f(key); }, s));
    if (low != low) low = -__builtin_inff();
  };
  // Compacts every logit >= low into the wave's LDS segment.  The wave's count follows the
  // ballots, so no atomic is needed.  Lanes may diverge at the end of a range: the lanes that
  // run a step are then always a prefix of the wave from its lane 0 (for_each4 unrolls by whole
  // waves, and a lane's trip count never exceeds that of a lower lane), so lane 0 runs every step
  // and holds the wave's count, and each step takes the count from the first active lane.
  float* const seg = s.cand + wave_id() * kSeg;
  int wcount = 0;
  auto compact = [&](float l) {
    const bool take = l >= low;
    const uint64_t want = __ballot(take);
    if (want != 0) {
      const int first = __builtin_amdgcn_readfirstlane(wcount);
      if (take) {
        const uint64_t below = lane_id() ? want & (~0ull >> (kWave - lane_id())) : 0ull;
        const int at = first + __builtin_popcountll(below);
        if (at < kSeg) seg[at] = l;
      }
      wcount = first + __builtin_popcountll(want);
    }
  };
  // Most quads hold no candidate: one ballot per quad decides whether any lane needs compact.
  auto compact4 = [&](const f32x4& v) {
    const bool any = (v[0] >= low) | (v[1] >= low) | (v[2] >= low) | (v[3] >= low);
    if (__ballot(any) != 0) compact(v[0]), compact(v[1]), compact(v[2]), compact(v[3]);
  };
  // The rest of the row, streamed from HBM once.
  if (fused) {
    for_each4<true>(
        row, prefix, vocab,
        [&](const f32x4& v) {
          scan(v[0]), scan(v[1]), scan(v[2]), scan(v[3]);
          compact4(v);
        },
        [&](float l) {
          scan(l);
          compact(l);
        },
        threshold);
    if (held) {
#pragma unroll
      for (int j = 0; j < kHeld; ++j) compact4(pq[j]);
    } else {
      for_each4<false>(row, 0, prefix, compact4, compact);
    }
  } else {
    for_each<true>(row, prefix, vocab, scan);
  }
  // bit 0: a NaN in the row; bit 1: a wave's segment overflowed; bit 2: a wave holds more
  // candidates than lanes (every lane runs here, so the first active lane is lane 0)
  wcount = __builtin_amdgcn_readfirstlane(wcount);
  int64_t above = 0;
  int flags = nan | (wcount > kSeg ? 2 : 0) | (wcount > kWave ? 4 : 0);
  float m = lane_max;
  // hist[0] is cleared for the select below; its last readers (the threshold's first round)
  // are done, and the barrier of group_reduce orders the clear before the select
  if (t < 256) s.hist[0][t] = 0;
  group_reduce(above_lane, above, flags, m, s);
  const bool any_nan = flags & 1;
  const bool overflow = flags & 2;

  double z = 0.0;
  double a = 0.0;
  if (want_mass) {
    if (!use_kth) {
      for_each<false>(row, 0, vocab, [&](float l) {
        const float e = split_term(l, m);
        z += e;
        a += l > lt ? e : 0.0;
      });
    } else if (fused && !(flags & 4)) {
      // At most one candidate per lane (the common case): each lane keeps its candidate, key
      // and term in registers for every round of the select.
      const bool have = lane_id() < wcount;
      const float c = have ? seg[lane_id()] : 0.0f;
      const uint32_t key = order_key(c);
      const float e = have ? split_term(c, m) : 0.0f;
      const float kth = key_value(radix_select(k_eff, [&](auto&& f) {
        if (have) f(key);
      }, s));
      if (have && c >= kth) {
        z = e;
        a = c > lt ? e : 0.0;
      }
    } else if (fused && !overflow) {
      // each wave reads back its own segment (LDS is in order within a wave)
      const float kth = key_value(radix_select(k_eff, [&](auto&& f) {
        for (int j = lane_id(); j < wcount; j += kWave) f(order_key(seg[j]));
      }, s));
      for (int j = lane_id(); j < wcount; j += kWave) {
        const float l = seg[j];
        if (l >= kth) {
          const float e = split_term(l, m);
          z += e;
          a += l > lt ? e : 0.0;
        }
      }
    } else {
      const float kth = key_value(radix_select(k_eff, [&](auto&& f) {
        for (int64_t i = t; i < vocab; i += kThreads) f(order_key(row[i]));
      }, s));
      for_each<false>(row, 0, vocab, [&](float l) {
        if (l >= kth) {
          const float e = split_term(l, m);
          z += e;
          a += l > lt ? e : 0.0;
        }
      });
    }
    group_sum2(z, a, s);
  }
  if (t == 0) write_verdict(A, r, q, above, any_nan, z, a);
}

// ---- rows split over workgroups ----------------------------------------------------------------
//
// One workgroup per row leaves most of the GPU idle for a small batch, reads a row without a
// top-k twice, and needs FP32 logits.  The split check gives every (row, segment of L logits) a
// 256-lane workgroup that reads its segment once, in the logits' own type, and keeps it in
// registers:
//   segment  count above the token, NaN flag, maximum; then, for a row cut at its k_eff-th
//            largest logit, `low`: each wave finds the ceil(k_eff / 4)-th largest of its 64 lane
//            maxima (its top 16 key bits, by ballots), and low is the smallest of the four, so at
//            least k_eff of the segment's logits are >= low and the row's kth is >= low.  Every
//            logit > low goes into the segment's slots, those equal to it are counted.  For a
//            row that keeps everything: the FP64 sums of its terms relative to the segment's own
//            maximum.
//   finish   a workgroup per row.  Lower bounds of kth are every segment's low and, in the same
//            way as low, the smallest over the four waves of the ceil(k_eff / 4)-th largest of
//            the wave's lane maxima over the slots; G is the largest of them.  Only slots > G
//            matter, one or two hundred values: kth is the k_eff-th largest of them, or G itself
//            when fewer than k_eff exceed it (the logits equal to G then enter as one term times
//            their count, so ties, such as the -inf of masked logits, take no slots).  A row
//            without a top-k adds the segments' sums scaled by exp(m_s - max) in FP64.
// Orders are fixed (lane, wave, segment), nothing depends on scheduling.  A segment with more
// logits above its low than slots, or more than kCap of them above G, sends the row to an exact
// radix select over the row by the finish workgroup (130 us at 50,257 logits), so both are kept
// rare.  A segment has a slot for each logit of one load of the workgroup (16 bytes a lane): finite
// logits in a run no longer than that fit whatever their low is (-inf where a wave holds none of
// them), a longer run reaches every lane, and in a row sorted by token id the logits above low lie
// within one load.  The logits of a row's last, partial segment are dealt to the lanes one by one,
// so 256 of them are enough for a low above -inf.
constexpr int kSegThreads = 256;
constexpr int kSegWaves = kSegThreads / kWave;
constexpr int kFinishThreads = 256;
constexpr int kFinishWaves = kFinishThreads / kWave;
constexpr int64_t kSplitMaxK = 128;  // top-k values the lane maxima of a segment can bound

// The largest float of 16 key bits that at least `want` of the wave's lanes hold a value >= of
// (-inf if fewer do): the key's top 16 bits, from the highest down, each kept if enough lanes
// still reach it.
__device__ __forceinline__ float wave_bound(float v, int want) {
  const uint32_t key = order_key(v);
  uint32_t bound = 0;
#pragma unroll
  for (int bit = 31; bit >= 16; --bit) {
    const uint32_t trial = bound | (1u << bit);
    if (__builtin_popcountll(__ballot(key >= trial)) >= want) bound = trial;
  }
  const float low = key_value(bound);
  return low == low ? low : -__builtin_inff();  // below the finite values
}

enum class Logits { kF32, kBf16, kF16 };

template <Logits kType>
struct LogitType;  // slots: one 16-byte load of the workgroup
template <>
struct LogitType<Logits::kF32> {
  typedef float type;
  static constexpr int kSlots = kSegThreads * 4;
  static __device__ __forceinline__ float widen(float v) { return v; }
};
template <>
struct LogitType<Logits::kBf16> {
  typedef uint16_t type;
  static constexpr int kSlots = kSegThreads * 8;
  static __device__ __forceinline__ float widen(uint16_t v) {
    return __uint_as_float(static_cast<uint32_t>(v) << 16);
  }
};
template <>
struct LogitType<Logits::kF16> {
  typedef _Float16 type;
  static constexpr int kSlots = kSegThreads * 8;
  static __device__ __forceinline__ float widen(_Float16 v) { return static_cast<float>(v); }
};

struct alignas(16) SegmentHeader {
  float max, low;
  uint32_t above, ties;  // logits above the token's; logits equal to low
  uint32_t count;        // logits above low (the first kSlots are in the slots)
  int flags;             // bit 0: a NaN
  double z, a;           // kept mass and mass above the token, relative to max (no top-k)
  uint64_t unused;
};
static_assert(sizeof(SegmentHeader) == 48, "three 16-byte words");

struct SplitArgs {
  MemberArgs m;
  SegmentHeader* headers;  // (rows, segments)
  float* slots;            // (rows, segments, kSlots), when any row has a top-k
  int64_t segments;
  int64_t length;  // logits per segment
};

struct SegmentScratch {
  uint32_t above[kSegWaves], ties[kSegWaves], count[kSegWaves];
  int flags[kSegWaves];
  float max[kSegWaves], low[kSegWaves];
  double z[kSegWaves], a[kSegWaves];
};

template <Logits kType, int kLoads>
__global__ void __launch_bounds__(kSegThreads) member_segment_kernel(const SplitArgs S) {
  using L = LogitType<kType>;
  using T = typename L::type;
  constexpr int kVec = 16 / static_cast<int>(sizeof(T));
  constexpr int kElems = kLoads * kVec;
  typedef T vec __attribute__((ext_vector_type(kVec)));
  typedef vec vec_any __attribute__((aligned(sizeof(T))));  // a row may start at any logit
  __shared__ SegmentScratch s;

  const MemberArgs& A = S.m;
  const int t = static_cast<int>(threadIdx.x);
  const uint32_t item = blockIdx.x;  // row * segments + segment
  const uint32_t segments = static_cast<uint32_t>(S.segments);
  const int64_t r = item / segments;
  const int64_t j0 = static_cast<int64_t>(item % segments) * S.length;
  const int64_t vocab = A.vocab;
  const T* __restrict__ row = reinterpret_cast<const T*>(A.logits) + r * vocab;
  const float inf = __builtin_inff();

  // The segment in registers; slots past the row hold -inf, which no count, sum or candidate
  // sees.
  float x[kElems];
  if (j0 + S.length <= vocab) {
    vec v[kLoads];
#pragma unroll
    for (int q = 0; q < kLoads; ++q)
      v[q] = __builtin_nontemporal_load(
          reinterpret_cast<const vec_any*>(row + j0 + (q * kSegThreads + t) * kVec));
#pragma unroll
    for (int i = 0; i < kElems; ++i) x[i] = L::widen(v[i / kVec][i % kVec]);
  } else {
#pragma unroll
    for (int i = 0; i < kElems; ++i) {
      const int64_t j = j0 + i * kSegThreads + t;
      const float v = L::widen(row[j < vocab ? j : vocab - 1]);
      x[i] = j < vocab ? v : -inf;
    }
  }
  const RowRequest q = row_request(A, r, row_token(A, r));
  const float lt = L::widen(row[q.in_range ? q.token : (q.token < 0 ? 0 : vocab - 1)]);

  uint32_t above = 0;
  int nan = 0;
  float top = -inf;
#pragma unroll
  for (int i = 0; i < kElems; ++i) {
    above += x[i] > lt;
    nan |= x[i] != x[i];
    top = fmaxf(top, x[i]);
  }
  const uint32_t wave_above = wave_reduce(above, [](uint32_t a, uint32_t b) { return a + b; });
  const uint32_t wave_nan =
      wave_reduce(static_cast<uint32_t>(nan), [](uint32_t a, uint32_t b) { return a | b; });
  const float wave_max = wave_reduce(top, [](float a, float b) { return fmaxf(a, b); });
  const int wave = t / kWave;
  const bool cut = q.want_mass && q.use_kth;  // uniform over the workgroup
  float wave_low = -inf;
  if (cut) wave_low = wave_bound(top, static_cast<int>((q.k_eff + kSegWaves - 1) / kSegWaves));
  if (lane_id() == 0) {
    s.above[wave] = wave_above;
    s.flags[wave] = static_cast<int>(wave_nan);
    s.max[wave] = wave_max;
    s.low[wave] = wave_low;
  }
  __syncthreads();
  SegmentHeader h{};
  h.above = (s.above[0] + s.above[1]) + (s.above[2] + s.above[3]);
  h.flags = (s.flags[0] | s.flags[1]) | (s.flags[2] | s.flags[3]);
  h.max = fmaxf(fmaxf(s.max[0], s.max[1]), fmaxf(s.max[2], s.max[3]));
  h.low = -inf;

  if (cut) {
    const float low = fminf(fminf(s.low[0], s.low[1]), fminf(s.low[2], s.low[3]));
    uint32_t mine = 0, ties = 0;
#pragma unroll
    for (int i = 0; i < kElems; ++i) {
      mine += x[i] > low;
      ties += x[i] == low;
    }
    const uint32_t incl = wave_inclusive_sum(mine);
    const uint32_t wave_ties = wave_reduce(ties, [](uint32_t a, uint32_t b) { return a + b; });
    if (lane_id() == kWave - 1) s.count[wave] = incl;
    if (lane_id() == 0) s.ties[wave] = wave_ties;
    __syncthreads();
    uint32_t at = incl - mine;
    for (int w = 0; w < wave; ++w) at += s.count[w];
    float* slots = S.slots + static_cast<int64_t>(item) * L::kSlots;
    if (mine != 0) {
#pragma unroll
      for (int i = 0; i < kElems; ++i) {
        if (x[i] > low) {
          if (at < L::kSlots) slots[at] = x[i];
          ++at;
        }
      }
    }
    h.low = low;
    h.count = (s.count[0] + s.count[1]) + (s.count[2] + s.count[3]);
    h.ties = (s.ties[0] + s.ties[1]) + (s.ties[2] + s.ties[3]);
  } else if (q.want_mass) {
    double z = 0.0, a = 0.0;
#pragma unroll
    for (int i = 0; i < kElems; ++i) {
      const float e = split_term(x[i], h.max);
      z += e;
      a += x[i] > lt ? e : 0.0;
    }
    const auto add = [](double u, double v) { return u + v; };
    z = wave_reduce(z, add);
    a = wave_reduce(a, add);
    if (lane_id() == 0) {
      s.z[wave] = z;
      s.a[wave] = a;
    }
    __syncthreads();
    h.z = (s.z[0] + s.z[1]) + (s.z[2] + s.z[3]);
    h.a = (s.a[0] + s.a[1]) + (s.a[2] + s.a[3]);
  }
  if (t == 0) S.headers[item] = h;
}

struct FinishScratch : Scratch {
  float low[kFinishWaves], kth[kFinishWaves], max[kFinishWaves];
  uint32_t above[kFinishWaves], count[kFinishWaves], ties[kFinishWaves];
  int flags[kFinishWaves];
  double z[kFinishWaves], a[kFinishWaves];
};

// 256 lanes: the exchanges between waves are short chains of LDS reads, and a row of 152 K logits
// has 19 segments, one round of early slots (64 rows with a top-k and a top-p: 5.8 us).
template <Logits kType>
__global__ void __launch_bounds__(kFinishThreads) member_finish_kernel(const SplitArgs S) {
  using L = LogitType<kType>;
  using T = typename L::type;
  constexpr int kEarly = 5;  // segments per wave whose first slots are read ahead,
  constexpr int kDeep = 2;   // this many 64-slot rows of each
  constexpr int kHeld = 4;   // candidates per lane when one wave selects
  __shared__ FinishScratch s;

  const MemberArgs& A = S.m;
  const int64_t r = blockIdx.x;
  const int t = static_cast<int>(threadIdx.x);
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int64_t n = S.segments;
  const SegmentHeader* hs = S.headers + r * n;
  const float* slots = S.slots + r * n * L::kSlots;
  const float inf = __builtin_inff();
  // Lane i of wave w holds the header of segment w + 4 i; the first slots of the wave's first
  // segments are requested with the headers (what they hold past a segment's count is not used).
  const int64_t own = wave + static_cast<int64_t>(lane) * kFinishWaves;
  SegmentHeader mine_h{};
  mine_h.max = mine_h.low = -inf;
  if (own < n) mine_h = hs[own];
  float early[kEarly][kDeep];
  const bool any_cut = A.top_p != nullptr && A.k_lim > 0;  // there are slots
  if (any_cut) {
#pragma unroll
    for (int i = 0; i < kEarly; ++i) {
      const int64_t seg = wave + static_cast<int64_t>(i) * kFinishWaves;
#pragma unroll
      for (int d = 0; d < kDeep; ++d)
        early[i][d] = slots[(seg < n ? seg : 0) * L::kSlots + d * kWave + lane];
    }
  }
  const RowRequest q = row_request(A, r, row_token(A, r));
  const int64_t vocab = A.vocab;
  const T* __restrict__ row = reinterpret_cast<const T*>(A.logits) + r * vocab;
  const float lt = L::widen(row[q.in_range ? q.token : (q.token < 0 ? 0 : vocab - 1)]);
  const bool cut = q.want_mass && q.use_kth;  // uniform

  // f(header) for each of this lane's segments
  auto headers = [&](auto&& f) {
    if (own < n) f(mine_h);
    for (int64_t i = own + kFinishThreads; i < n; i += kFinishThreads) f(hs[i]);
  };
  uint32_t above32 = 0;  // at most vocab in all, below 2^31
  int flags = 0;
  float m = -inf, low = -inf;
  headers([&](const SegmentHeader& h) {
    above32 += h.above;
    flags |= h.flags | (h.count > L::kSlots ? 2 : 0) | (h.count > kDeep * kWave ? 4 : 0);
    m = fmaxf(m, h.max);
    low = fmaxf(low, h.low);
  });
  const auto add = [](uint32_t u, uint32_t v) { return u + v; };
  const auto larger = [](float u, float v) { return fmaxf(u, v); };
  float wave_kth = -inf;
  if (cut) {
    float top = -inf;
#pragma unroll
    for (int i = 0; i < kEarly; ++i) {
      const int count = static_cast<int>(read_lane(mine_h.count, i));  // 0 past the row
#pragma unroll
      for (int d = 0; d < kDeep; ++d) {
        if (d * kWave + lane >= count) early[i][d] = -inf;
        top = fmaxf(top, early[i][d]);
      }
    }
    wave_kth = wave_bound(top, static_cast<int>((q.k_eff + kFinishWaves - 1) / kFinishWaves));
  }
  {
    const uint32_t wave_above = wave_reduce(above32, add);
    const uint32_t wave_flags =
        wave_reduce(static_cast<uint32_t>(flags), [](uint32_t u, uint32_t v) { return u | v; });
    const float wave_max = wave_reduce(m, larger);
    const float wave_low = wave_reduce(low, larger);
    if (lane == 0) {
      s.above[wave] = wave_above;
      s.flags[wave] = static_cast<int>(wave_flags);
      s.max[wave] = wave_max;
      s.low[wave] = wave_low;
      s.kth[wave] = wave_kth;
    }
  }
  s.hist[0][t] = 0;  // for a radix select below, behind the barriers between
  __syncthreads();
  int64_t above = 0;
  flags = 0;
  m = -inf;
  float floor_value = -inf, every_wave = inf;
#pragma unroll
  for (int w = 0; w < kFinishWaves; ++w) {
    above += s.above[w];
    flags |= s.flags[w];
    m = fmaxf(m, s.max[w]);
    floor_value = fmaxf(floor_value, s.low[w]);
    every_wave = fminf(every_wave, s.kth[w]);
  }
  floor_value = fmaxf(floor_value, every_wave);  // G

  double z = 0.0, a = 0.0;
  auto term = [&](float l, float kth) {
    if (l >= kth) {
      const float e = split_term(l, m);
      z += e;
      a += l > lt ? e : 0.0;
    }
  };
  bool one_wave = !q.want_mass;  // wave 0 holds the row's sums
  if (cut) {
    bool whole_row = flags & 2;
    if (!whole_row) {
      // This wave's slots above G and its logits equal to G (ties): counted, then compacted at
      // the wave's offset, in segment and slot order.  A segment whose low is G has its ties in
      // its header (its slots are all above G); one whose low is below G has them in its slots.
      const bool more = (flags & 4) || n > static_cast<int64_t>(kEarly) * kFinishWaves;
      auto each = [&](auto&& f) {  // f(value) by whole waves, -inf where there is no slot
#pragma unroll
        for (int i = 0; i < kEarly; ++i)
#pragma unroll
          for (int d = 0; d < kDeep; ++d) f(early[i][d]);
        if (more) {
          for (int64_t seg = wave, i = 0; seg < n; seg += kFinishWaves, ++i) {
            const int count = static_cast<int>(
                i < kWave ? read_lane(mine_h.count, static_cast<int>(i)) : hs[seg].count);
            for (int j = i < kEarly ? kDeep * kWave : 0; j < count; j += kWave) {
              const float v = slots[seg * L::kSlots + (j + lane < count ? j + lane : count - 1)];
              f(j + lane < count ? v : -inf);
            }
          }
        }
      };
      uint32_t mine = 0, ties = 0;
      each([&](float v) {
        mine += v > floor_value;
        ties += v == floor_value;
      });
      headers([&](const SegmentHeader& h) { ties += h.low == floor_value ? h.ties : 0u; });
      const uint32_t wave_n = wave_reduce(mine, add);
      const uint32_t wave_ties = wave_reduce(ties, add);
      if (lane == 0) {
        s.count[wave] = wave_n;
        s.ties[wave] = wave_ties;
      }
      __syncthreads();
      uint32_t total = 0, tied = 0, at = 0;
#pragma unroll
      for (int w = 0; w < kFinishWaves; ++w) {
        at = w == wave ? total : at;
        total += s.count[w];
        tied += s.ties[w];
      }
      whole_row = total > static_cast<uint32_t>(kCap);
      if (!whole_row) {
        each([&](float v) {
          const bool take = v > floor_value;
          const uint64_t want = __ballot(take);
          if (take) {
            const uint64_t below = lane ? want & (~0ull >> (kWave - lane)) : 0ull;
            s.cand[at + __builtin_popcountll(below)] = v;
          }
          at += __builtin_popcountll(want);
        });
        __syncthreads();
        const bool select = static_cast<int64_t>(total) >= q.k_eff;  // kth exceeds G
        if (!select && t == 0) {
          z = static_cast<double>(split_term(floor_value, m)) * tied;
          a = floor_value > lt ? z : 0.0;
        }
        if (total <= kHeld * kWave) {
          // Wave 0 alone, with no further barrier: the candidates in its registers, kth bit by
          // bit from the first bit in which G and the maximum differ, until exactly k_eff of
          // them reach the bound (kth is then the smallest of those) or no bit is left.
          if (wave != 0) return;
          one_wave = true;
          float c[kHeld];
          uint32_t key[kHeld];
#pragma unroll
          for (int i = 0; i < kHeld; ++i) {
            const uint32_t j = lane + i * kWave;
            const float v = s.cand[j < total ? j : 0];
            c[i] = j < total ? v : -inf;
            key[i] = j < total ? order_key(v) : 0u;
          }
          float kth = floor_value;
          if (select) {
            const uint32_t hi = order_key(m), lo = order_key(floor_value);
            const uint32_t diff = hi ^ lo;  // hi > lo: some logit exceeds G
            int bit = 31 - __builtin_clz(diff | 1u);
            uint32_t bound = bit == 31 ? 0u : (hi >> (bit + 1)) << (bit + 1);
            for (; bit >= 0; --bit) {
              const uint32_t trial = bound | (1u << bit);
              int count = 0;
#pragma unroll
              for (int i = 0; i < kHeld; ++i)
                count += __builtin_popcountll(__ballot(key[i] >= trial));
              if (count >= q.k_eff) bound = trial;
              if (count == q.k_eff) break;
            }
            uint32_t least = 0xFFFFFFFFu;
#pragma unroll
            for (int i = 0; i < kHeld; ++i)
              if (key[i] >= bound && key[i] < least) least = key[i];
            kth = key_value(wave_reduce(least, [](uint32_t u, uint32_t v) { return u < v ? u : v; }));
          }
#pragma unroll
          for (int i = 0; i < kHeld; ++i)
            if (c[i] > floor_value) term(c[i], kth);
        } else {
          float kth = floor_value;
          if (select) {
            kth = key_value(radix_select(q.k_eff, [&](auto&& f) {
              for (uint32_t i = t; i < total; i += kFinishThreads) f(order_key(s.cand[i]));
            }, s));
          }
          for (uint32_t i = t; i < total; i += kFinishThreads) term(s.cand[i], kth);
        }
      }
    }
    if (whole_row) {
      // f(logit) for the row's logits, kAhead in flight per lane
      constexpr int kAhead = 8;
      auto logits = [&](auto&& f) {
        for (int64_t i = t; i < vocab; i += kAhead * kFinishThreads) {
          float v[kAhead];
#pragma unroll
          for (int e = 0; e < kAhead; ++e) {
            const int64_t j = i + e * kFinishThreads;
            v[e] = L::widen(row[j < vocab ? j : vocab - 1]);
          }
#pragma unroll
          for (int e = 0; e < kAhead; ++e)
            if (i + e * kFinishThreads < vocab) f(v[e]);
        }
      };
      const float kth = key_value(radix_select(
          q.k_eff, [&](auto&& f) { logits([&](float l) { f(order_key(l)); }); }, s));
      logits([&](float l) { term(l, kth); });
    }
  } else if (q.want_mass) {
    headers([&](const SegmentHeader& h) {
      if (h.max > -inf) {
        const double scale = exp(static_cast<double>(h.max) - static_cast<double>(m));
        z += h.z * scale;
        a += h.a * scale;
      }
    });
  }
  if (q.want_mass) {
    const auto sum = [](double u, double v) { return u + v; };
    z = wave_reduce(z, sum);
    a = wave_reduce(a, sum);
    if (!one_wave) {
      if (lane == 0) {
        s.z[wave] = z;
        s.a[wave] = a;
      }
      __syncthreads();
      z = (s.z[0] + s.z[1]) + (s.z[2] + s.z[3]);
      a = (s.a[0] + s.a[1]) + (s.a[2] + s.a[3]);
    }
  }
  if (t == 0) write_verdict(A, r, q, above, flags & 1, z, a);
}

}  // namespace
}  // namespace pck

namespace pck {
namespace {

hipError_t validate(const PckMemberArgs* args) {
  if (args == nullptr) return hipErrorInvalidValue;
  const PckMemberArgs& a = *args;
  if (a.rows < 0 || a.rows * kThreads > 0xFFFFFFFFll || a.vocab < 1 || a.vocab > 0x7FFFFFFF ||
      a.k_lim < 0 || a.k_lim > a.vocab)
    return hipErrorInvalidValue;
  if (a.rows == 0) return hipSuccess;
  if (!a.logits || !a.tokens ||
      (a.temperature && (!a.temperature_index || a.temperature_count < 1)) ||
      (a.all_k && a.k_lim < 1))
    return hipErrorInvalidValue;
  return hipSuccess;
}

// The split of a batch: logits per segment, segments per row and the workspace (0 bytes: the
// one-workgroup kernel).  Each line of splits() is where the split stops being the faster one, by
// both routes timed at 24 vocabularies from 100 to 262,144 and 1 to 384 rows.  Time of the split
// relative to one workgroup per row, FP32 rows at 16-byte addresses:
//                     4 rows   64 rows   128 rows   256 rows
//   top-k alone
//     32,000          1.08      1.11      1.18       1.13
//     65,536          0.88      1.01      1.12       1.07
//     151,936         0.58      0.75      0.96       1.02
//   top-k and top-p
//     24,576          1.00      1.04      1.09       1.06
//     32,000          0.97      0.98      1.04       1.05
//     151,936         0.54      0.67      0.91       1.11
//   top-p alone
//     12,000          0.91      0.96      1.01       1.11
//     16,384          0.89      0.94      1.06       1.09
//     24,576          0.69      0.82      0.85       0.94
//   top-p, a top-k in some rows
//     24,576          1.03      1.09      1.14       1.15
//     32,000          0.95      1.00      1.01       1.09
//     40,000          0.82      0.86      0.94       0.99
// Rows at other addresses make the one-workgroup kernel two to four times slower from 20,000
// logits, the segments hardly at all (20,001: 0.75 to 1.05, 151,937: 0.18 to 0.40).  16-bit logits
// cost that kernel a conversion first; the split is faster but for cut rows too short to fill a
// segment, up to a workgroup per compute unit (1,000 logits 1.10, 4,096 0.98).
// Segments are 8,192 logits (their candidates are what the finish reads), shorter ones only
// where no row is cut and the batch would not fill the GPU.
struct SplitPlan {
  int64_t length = 0, segments = 0, header_bytes = 0, bytes = 0;
};

bool splits(const PckMemberArgs& a, int kind, bool cut, bool keeps_all) {
  if (kind != 0) return !cut || a.vocab >= 4096 || a.rows > 256;
  if (reinterpret_cast<uintptr_t>(a.logits) % 16 != 0 || (a.vocab % 4 != 0 && a.rows > 1)) {
    if (keeps_all) return a.vocab >= (cut ? 20000 : 16384);
    return a.vocab >= 20000 && a.rows < 192;
  }
  if (keeps_all)
    return cut ? a.vocab >= 40000 || (a.vocab >= 32000 && a.rows <= 96)
               : a.vocab >= 24576 || (a.vocab >= 16384 && a.rows <= 96);
  if (cut) return a.vocab >= 32000 && a.rows <= 160 && a.rows <= a.vocab / 512;
  return a.vocab >= 65536 && a.rows <= 128 && a.rows <= (a.vocab - 32768) / 1024;
}

SplitPlan split_plan(const PckMemberArgs& a, int kind) {
  SplitPlan p;
  if (a.rows < 1) return p;
  const bool cut = a.top_p != nullptr && a.k_lim > 0;     // a row may be cut at its k-th logit
  const bool keeps_all = a.top_p != nullptr && !a.all_k;  // a row may keep every logit
  if (!splits(a, kind, cut, keeps_all)) return p;
  int64_t length = 8192;
  while (!cut && length > 2048 && a.rows * ((a.vocab + length - 1) / length) < 1024) length /= 2;
  const int64_t segments = (a.vocab + length - 1) / length;
  // about 1.4 k candidates of each segment reach the finish workgroup, which holds kCap
  if (cut && (a.k_lim > kSplitMaxK || segments * a.k_lim > kCap * 5 / 8)) return p;
  if (a.rows * segments > 0x7FFFFFFF / kSegThreads) return p;
  p.length = length;
  p.segments = segments;
  const int64_t slots =
      kind == 0 ? LogitType<Logits::kF32>::kSlots : LogitType<Logits::kBf16>::kSlots;
  p.header_bytes = a.rows * segments * static_cast<int64_t>(sizeof(SegmentHeader));
  p.bytes = p.header_bytes +
            (cut ? a.rows * segments * slots * static_cast<int64_t>(sizeof(float)) : 0);
  return p;
}

template <Logits kType>
hipError_t launch_split(const SplitArgs& s, hipStream_t stream) {
  constexpr int kVec = kType == Logits::kF32 ? 4 : 8;
  constexpr int kUnit = kSegThreads * kVec;  // logits per load of the workgroup
  const dim3 grid(static_cast<unsigned>(s.m.rows * s.segments)), group(kSegThreads);
  if (s.length == 8192)
    member_segment_kernel<kType, 8192 / kUnit><<<grid, group, 0, stream>>>(s);
  else if (s.length == 4096)
    member_segment_kernel<kType, 4096 / kUnit><<<grid, group, 0, stream>>>(s);
  else
    member_segment_kernel<kType, 2048 / kUnit><<<grid, group, 0, stream>>>(s);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  member_finish_kernel<kType>
      <<<dim3(static_cast<unsigned>(s.m.rows)), dim3(kFinishThreads), 0, stream>>>(s);
  return hipGetLastError();
}

}  // namespace
}  // namespace pck

extern "C" int pck_check_members_workspace(const PckMemberArgs* args, int logits_kind,
                                           int64_t* bytes) {
  if (pck::validate(args) != hipSuccess || logits_kind < 0 || logits_kind > 2 || bytes == nullptr)
    return hipErrorInvalidValue;
  *bytes = pck::split_plan(*args, logits_kind).bytes;
  return hipSuccess;
}

extern "C" int pck_check_members_split(const PckMemberArgs* args, int logits_kind, void* workspace,
                                       int64_t workspace_bytes, void* stream) {
  using namespace pck;
  if (validate(args) != hipSuccess || logits_kind < 0 || logits_kind > 2)
    return hipErrorInvalidValue;
  if (args->rows == 0) return hipSuccess;
  const SplitPlan p = split_plan(*args, logits_kind);
  if (p.bytes == 0 || workspace == nullptr || workspace_bytes < p.bytes ||
      reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
    return hipErrorInvalidValue;
  const SplitArgs s{*args, static_cast<SegmentHeader*>(workspace),
                    reinterpret_cast<float*>(static_cast<char*>(workspace) + p.header_bytes),
                    p.segments, p.length};
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (logits_kind == 0) return launch_split<Logits::kF32>(s, st);
  if (logits_kind == 1) return launch_split<Logits::kBf16>(s, st);
  return launch_split<Logits::kF16>(s, st);
}

extern "C" int pck_check_members_ex(const PckMemberArgs* args, void* stream) {
  if (pck::validate(args) != hipSuccess) return hipErrorInvalidValue;
  const PckMemberArgs& a = *args;
  if (a.rows == 0) return hipSuccess;
  pck::member_kernel<<<dim3(static_cast<unsigned>(a.rows)), dim3(pck::kThreads), 0,
                       static_cast<hipStream_t>(stream)>>>(a);
  return hipGetLastError();
}

extern "C" int pck_check_members(const float* logits, int64_t rows, int64_t vocab,
                                 const int64_t* tokens, const int64_t* top_k, const double* top_p,
                                 const uint8_t* greedy, double slack, int64_t k_lim, int all_k,
                                 uint8_t* ok, int64_t* above, double* mass_above, void* stream) {
  if (rows > 0 && (!ok || !above || !mass_above)) return hipErrorInvalidValue;
  PckMemberArgs a{};
  a.logits = logits;
  a.rows = rows;
  a.vocab = vocab;
  a.tokens = tokens;
  a.top_k = top_k;
  a.top_p = top_p;
  a.greedy = greedy;
  a.slack = slack;
  a.k_lim = k_lim;
  a.all_k = all_k;
  a.ok = ok;
  a.above = above;
  a.mass_above = mass_above;
  return pck_check_members_ex(&a, stream);
}
