// score_reduce.hpp -- what the generalized scorers (score.hip, digit_score.hip)
// share: the reducers' per-column state and the sum over a batch row's query
// tokens.
#pragma once

#include "common.hpp"
#include "internal.hpp"

namespace msim {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kLowest = -3.402823466e+38f;

template <int RED>
struct ReducerState;

// kRedMax: running maximum.
template <>
struct ReducerState<kRedMax> {
  float m;
  __device__ void init() { m = kNegInf; }
  // Two three-way maxima (v_max3_f32) for four values: exact, any order.
  __device__ void add4(const float (&z)[4]) { m = max5_op(m, z[0], z[1], z[2], z[3]); }
  __device__ float finish(int len, float mul, float colmul, float, float weight, float doc_scale) const {
    return len == 0 ? 0.0f : m * mul * colmul * weight * doc_scale;
  }
};

// kRedTop2 / kRedTop4: the K largest values, sorted descending.
template <int K>
struct TopState {
  float t[K];
  __device__ void init() {
#pragma unroll
    for (int i = 0; i < K; ++i) t[i] = kNegInf;
  }
  // With t sorted descending, the new i-th largest of t and v is the median
  // of t[i - 1], t[i] and v (the maximum for i = 0): one v_med3_f32 each,
  // all from the old values.  Only selections, so the result is exact.
  __device__ void insert(float v) {
    float n[K];
    n[0] = fmaxf(t[0], v);
#pragma unroll
    for (int i = 1; i < K; ++i) n[i] = __builtin_amdgcn_fmed3f(t[i - 1], t[i], v);
#pragma unroll
    for (int i = 0; i < K; ++i) t[i] = n[i];
  }
  __device__ void add4(const float (&z)[4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) insert(z[r]);
  }
  __device__ float finish(int len, float mul, float colmul, float, float, float doc_scale) const {
    const int kept = len < K ? len : K;
    if (kept == 0) return 0.0f;
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < K; ++i)
      if (i < kept) total += t[i];
    return total / (float)kept * mul * colmul * doc_scale;
  }
};
template <>
struct ReducerState<kRedTop2> : TopState<2> {};
template <>
struct ReducerState<kRedTop4> : TopState<4> {};

// kRedLse: online log-sum-exp in base 2 over u = z * k with k = colmul *
// doc_scale * log2(e) / tau, i.e. u = x log2(e) / tau for the scaled
// similarity x = z * colmul * doc_scale: m = running maximum of u (starts at
// the lowest finite float so that masked -inf values never form inf - inf),
// s = sum 2^(u - m).  Every exponent is <= 0 and the maximum's term is 1, so
// v_exp_f32 itself serves (exp2f adds a rescaling path for results below
// 2^-126, which are negligible next to that 1).  The score, max x + tau ln
// sum e^((x - max x) / tau), is then (m + log2 s) * tau * ln 2.  (Folding
// log2(e) / tau into k saves a multiply per similarity.)
__device__ __forceinline__ float exp2_nonpos(float x) { return __builtin_amdgcn_exp2f(x); }
template <>
struct ReducerState<kRedLse> {
  float m, s, k;  // k = colmul * doc_scale * log2(e) / tau for the current target
  __device__ void init() {
    m = kLowest;
    s = 0.0f;
  }
  // mask: -inf for rows that do not count, else -0, joined after the product
  // with k (-inf times a k of 0 would be NaN, times a negative one +inf).
  __device__ void add4(const float (&z)[4], const float (&mask)[4]) {
    float u[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = fmaf(z[r], k, mask[r]);
    const float mn = max3_op(max3_op(m, u[0], u[1]), u[2], u[3]);
    float acc = s * exp2_nonpos(m - mn);
#pragma unroll
    for (int r = 0; r < 4; ++r) acc += exp2_nonpos(u[r] - mn);
    s = acc;
    m = mn;
  }
  // Merge with another (m, s).
  __device__ void merge(float mo, float so) {
    const float mn = fmaxf(m, mo);
    s = s * exp2_nonpos(m - mn) + so * exp2_nonpos(mo - mn);
    m = mn;
  }
  __device__ float finish(int len, float, float, float temperature, float, float) const {
    return len == 0 ? 0.0f : (m + log2f(s)) * (temperature * kLn2);
  }
};

// Sum of a batch row's `n` per-token values x[0 .. n) (LDS): lane l of each 16
// adds x[l], x[l + 16], ..., then a butterfly over the 16 lanes.  Every scorer
// and pool_sum_kernel use this order, so a row's score does not depend on how
// the query rows are split into passes.  16 partial sums instead of one chain:
// a chain of 32 dependent LDS reads and adds took about 1 us at each document
// end.  The result is in every lane of the 16.
__device__ __forceinline__ float row_butterfly16(float p) {
  auto dpp = [](float x, auto ctrl) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), decltype(ctrl)::value, 0xF, 0xF, true));
  };
  p += dpp(p, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
  p += dpp(p, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  p += dpp(p, std::integral_constant<int, 0x141>{});  // row_half_mirror: the other quad of the eight
  p += dpp(p, std::integral_constant<int, 0x140>{});  // row_mirror: the other eight
  return p;
}
__device__ __forceinline__ float token_sum16(const float* x, int n) {
  float p = 0.0f;
  for (int q = lane_id() & 15; q < n; q += 16) p += x[q];
  return row_butterfly16(p);
}
// The scores of the nb batch rows whose n per-token values each lie in
// x[0 .. nb * n) (LDS, visible): four rows at a time, put(row, score) from one
// lane per row.
template <typename Put>
__device__ __forceinline__ void sum_batch_rows(const float* x, int nb, int n, Put put) {
  const int g = lane_id() >> 4;
  for (int b0 = 0; b0 < nb; b0 += 4) {
    const int b = b0 + g;
    const float s = token_sum16(x + min(b, nb - 1) * n, n);
    if (b < nb && (lane_id() & 15) == 0) put(b, s);
  }
}

// A wave's tiles from its workgroup's list of work units (ScoreArgs::
// group_units): it starts with units `wave` and wave + WAVES and takes the following
// ones from the counter `taken` in LDS (set to 2 WAVES, visible), the unit after the
// current one known ahead.  next() is called once per tile, ahead of its use;
// past the list's end it returns the table's padding entry (token 0), which
// tiles_ended() recognises.  The waves of a SIMD do not share it evenly (the older
// wave issues first); taking units as they go, all finish with the list.
template <int WAVES>
struct TileStream {
  using TilePtr = const __attribute__((address_space(4))) uint64_t*;
  TilePtr pad, cur, after;
  const __attribute__((address_space(4))) int64_t* info;
  int left, count, units, lane;
  int* taken;
  __device__ __forceinline__ TileStream(const ScoreArgs& p, int wave, int lane_, int& counter) {
    pad = cur = after = as_constant(p.tiles);
    units = wave < 0 ? 0 : p.group_units;  // (wave -1: no list)
    info = as_constant(p.wave_info) + (int64_t)blockIdx.x * units * kScoreInfoWords;
    lane = lane_;
    taken = &counter;
    unit(wave, cur, left);
    unit(wave + WAVES, after, count);
  }
  __device__ __forceinline__ void unit(int k, TilePtr& tp, int& n) const {
    n = 0;
    tp = pad;
    if (k < units) {
      n = (int)info[(int64_t)k * kScoreInfoWords + 2];
      tp = pad + info[(int64_t)k * kScoreInfoWords + 3];
    }
  }
  __device__ __forceinline__ uint64_t next() {
    if (left == 0) {
      cur = after;
      left = max(count, 1);  // past the end: the padding entry, again and again
      if (count > 0) {
        int k = 0;
        if (lane == 0) k = atomicAdd(taken, 1);
        unit(__builtin_amdgcn_readfirstlane(k), after, count);
      }
    }
    --left;
    return *cur++;
  }
};
__device__ __forceinline__ bool tiles_ended(uint64_t e) {
  return ((e >> kTileLastShift) & 3) == 2;  // empty, and no target's last tile
}

// 32 sign bits of one lane (dims 32g .. 32g + 31, bit b = dim 32g + b; set =
// +1) as the fp4 (e2m1) operand of v_mfma_scale_f32_16x16x128_f8f6f4: dword
// q holds dims 32g + 4i + q in nibble i, +1 as 0x2 and -1 as 0xA: operand
// element s (of the lane's 32) is dim 32g + 4 (s % 8) + s / 8.
__device__ __forceinline__ v4i fp4_signs(unsigned w) {
  // 0x2 | (not sign ? 0x8) of every nibble: one v_bitop3_b32 (c | (~a & b)).
  auto dword = [](unsigned x) __attribute__((always_inline)) {
    return (int)__builtin_amdgcn_bitop3_b32(x, 0x88888888u, 0x22222222u, 0xAE);
  };
  return (v4i){dword(w << 3), dword(w << 2), dword(w << 1), dword(w)};
}

}  // namespace msim
