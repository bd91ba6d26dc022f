// hamming.hip -- MaxSim of sign-bit queries against sign documents, Hamming
// form: the +-1 dot q . d = 128 - 2 popcount(q ^ d) of each (query row, token),
// its maximum over a document's tokens, summed over the query tokens of a
// batch row (the sum cpu_extension.cpp:82-126 computes for +-1 queries; every
// value an integer below 2^24, so float sums and maxima are exact).
//
// One v_mfma_scale_f32_16x16x128_f8f6f4 on fp4 +-1 operands covers 16 tokens x
// 16 query rows x 128 dims (twice the K of the int8 MFMA at the same issue
// rate).  What bounds it: with many query rows the SIMD's issue of MFMAs (16
// cycles) and of the VALU beside them (two maxima per block and the tile's
// unpacking, 11 cycles), with few the work per tile around them.
//
// Layout: a pass holds NT blocks of 16 query rows in registers (4 VGPRs each, up
// to 256 rows; 2 to 16 blocks, so that few query rows do not pay for 256); two
// workgroups per CU (four waves per SIMD), each wave taking work units
// (documents) from its workgroup's list.  A tile's sign words (one dword per
// lane) are loaded kRing - 1 tiles ahead by buffer loads; rows past a short
// document read its last token again, which leaves every maximum unchanged.
// Each block's maxima (two v_max3_f32) follow kLag MFMAs later, across tiles
// and documents too, so neither a fence nor a second set of accumulators per
// block is needed.
//
// Measured, 10,240 documents of 256..1,024 tokens, queries of 32 tokens (before:
// passes of always 256 rows, a tile's maxima behind a fence, tables of one
// list per wave): 1 query 115 -> 33 us, 4 queries 115 -> 54, 8: 115 -> 84 (kernel);
// 256: 3,380 -> 2,137 (10.3 ns per block and SIMD; MFMAs alone 8.7 at two waves per
// SIMD, with two maxima after each 10.9: microbench/rates.hip).  One workgroup
// per CU instead of two: 15 % slower; units followed by position instead of
// TileStream's running pointer: another 8 %.
#include <algorithm>

#include "common.hpp"
#include "internal.hpp"
#include "score_reduce.hpp"

namespace msim {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4f mfma_fp4(const v4i& a, const v4i& b) {
  typedef int v8i __attribute__((ext_vector_type(8)));
  const v8i a8 = {a[0], a[1], a[2], a[3], 0, 0, 0, 0}, b8 = {b[0], b[1], b[2], b[3], 0, 0, 0, 0};
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  // Formats 4 / 4: fp4 A and B; E8M0 scales 127 = 2^0.
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a8, b8, zero, 4, 4, 0, 127, 0, 127);
}

constexpr int kWaves = 8, kGroupThreads = kWaves * kWave;

template <int NT>
__global__ __launch_bounds__(kGroupThreads, 4) void hamming_kernel(ScoreArgs p) {
  constexpr int kRing = NT > 8 ? 4 : 8;
  constexpr int kLag = NT > 2 ? 3 : 2;  // MFMAs between a block's and its maxima
  static_assert(NT == 2 || NT % 4 == 0, "accumulator slots");
  constexpr float kNone = -1.0e30f;
  __shared__ float s_pool[kWaves][16 * NT];
  __shared__ int s_next;
  if (threadIdx.x == 0) s_next = 2 * kWaves;
  __syncthreads();
  const int lane = lane_id();
  const int wave = wave_uniform(threadIdx.x / kWave);
  const int g = lane >> 4, c = lane & 15;
  const int lr0 = ((int)blockIdx.y + p.first_pass) * p.pass_rows;  // first query row of the pass

  // The tile stream (see digit_score_kernel).
  TileStream<kWaves> stream(p, wave, lane, s_next);

  // Query operands: rows lr0 + 16 j + c (rows past the query read 0 bits).
  const __amdgpu_buffer_rsrc_t rq = make_rsrc(p.qbits, (uint32_t)p.grp_rows * 16u);
  unsigned qw[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) qw[j] = load_b32(rq, (lr0 + 16 * j + c) * 16 + 4 * g);
  __builtin_amdgcn_sched_barrier(0);

  struct Tile {
    uint64_t e;
    unsigned w;
  };
  auto load = [&](uint64_t e, Tile& t) __attribute__((always_inline)) {
    t.e = e;
    const int rows1 = (int)((e >> kTileRowsShift) & 15);
    t.w = load_b32(make_rsrc(p.codes + (int64_t)(e & kTileStartMask) * 16, 256u), min(c, rows1) * 16 + 4 * g);
  };
  Tile ring[kRing];
#pragma unroll
  for (int u = 0; u < kRing - 1; ++u) load(stream.next(), ring[u]);
  uint64_t next = stream.next();
  if (tiles_ended(ring[0].e)) return;  // no barriers below

  v4i bq[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) bq[j] = fp4_signs(qw[j]);
  float m[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) m[j] = kNone;

  const int pass_rows = min(p.pass_rows, p.grp_rows - lr0);
  // Sums go out as float or as int32 (launch_hamming: not both): the lane
  // group's batch row of the first four.
  const bool sums = p.out || p.iout, as_int = p.iout != nullptr;
  const int64_t stride = as_int ? p.iout_stride : p.out_stride;
  uint32_t* const out_row =
      (as_int ? reinterpret_cast<uint32_t*>(p.iout) : reinterpret_cast<uint32_t*>(p.out)) +
      (lr0 / p.query_tokens + g) * stride;
  const bool sum_regs = NT >= 4 && p.query_tokens == 32 && sums;
  // End of the target whose last tile is e.
  auto finish_target = [&](uint64_t e) __attribute__((always_inline)) {
    const int64_t tg = (int64_t)(e >> kTileLocalShift);
    const float scale = ((e >> kTileEmptyShift) & 1) != 0 ? 0.0f : p.scale;
    auto max32 = [](float a, float b) __attribute__((always_inline)) {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
      return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    };
    auto max16 = [](float a, float b) __attribute__((always_inline)) {
      const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
      return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    };
    // Blocks 4 i .. 4 i + 3: lane group g holds block 4 i + (g >> 1) + 2 (g & 1).
    // (An empty document: 0 x the start value, + 0 for the sign.)
    constexpr int kQuads = (NT + 3) / 4;
    float v[kQuads];
#pragma unroll
    for (int i = 0; i < kQuads; ++i) {
      const float x = max32(m[4 * i], m[4 * i + 1]);
      const float y = NT > 2 ? max32(m[NT > 2 ? 4 * i + 2 : 0], m[NT > 2 ? 4 * i + 3 : 0]) : kNone;
      v[i] = fmaf(max16(x, y), scale, 0.0f);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) m[j] = kNone;
    // Batch row first + g of the pass.
    auto put = [&](int first, float sum) __attribute__((always_inline)) {
      out_row[first * stride + tg] = as_int ? (uint32_t)(int32_t)sum : __float_as_uint(sum);
    };
    if (sum_regs) {
      // 32-token queries: tokens l and l + 16 of a batch row are 32 lanes
      // apart; two quads' sums (batch rows 4 i .. 4 i + 3) in one register,
      // one batch row per lane group.  Of no other length do two whole 16-row
      // blocks make a batch row; those go through LDS, about 1 % slower (31 / 32
      // tokens, the call: 4 queries 52.8 / 52.5 us, 8 84.3 / 83.5, 32 288 / 285).
#pragma unroll
      for (int i = 0; i < kQuads; i += 2) {
        const auto r = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(v[i]), __float_as_uint(i + 1 < kQuads ? v[i + 1 < kQuads ? i + 1 : 0] : 0.0f), false, false);
        const float sum = row_butterfly16(__uint_as_float(r[0]) + __uint_as_float(r[1]));
        if (c == 0 && 32 * (2 * i + g) < pass_rows) put(2 * i, sum);
      }
      return;
    }
    const int blk = (g >> 1) | ((g & 1) << 1);
    if (sums) {
#pragma unroll
      for (int i = 0; i < kQuads; ++i)
        if (4 * i + blk < NT) s_pool[wave][16 * (4 * i + blk) + c] = v[i];
      wave_sync_lds();
      const int nb = pass_rows / p.query_tokens;
      for (int b = 0; b < nb; b += 4) {
        const float sum = token_sum16(s_pool[wave] + min(b + g, nb - 1) * p.query_tokens, p.query_tokens);
        if (b + g < nb && c == 0) put(b, sum);
      }
      wave_sync_lds();
    } else {
      float* out = p.pooled + tg * p.grp_rows + lr0;
#pragma unroll
      for (int i = 0; i < kQuads; ++i) {
        const int r = 16 * (4 * i + blk) + c;
        if (4 * i + blk < NT && r < pass_rows) out[r] = v[i];
      }
    }
  };

  v4f acc[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x] = (v4f){kNone, kNone, kNone, kNone};
  uint64_t before = score_tile_entry(0, 1, false, false, 0);  // the tile before
  // An MFMA stays before its pin and the reads of its result behind the next
  // one: the compiler otherwise sinks the tile's last MFMAs to their maxima in
  // the next tile, where max3_op reads them too early (its inline asm operands
  // get no wait states).
  auto pin = [](v4f& x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); };
  auto fold = [&](int j, int slot) __attribute__((always_inline)) {
    pin(acc[slot]);
    const v4f& x = acc[slot];
    m[j] = max5_op(m[j], x[0], x[1], x[2], x[3]);
  };
  // The tile in slot U: its MFMAs, behind each the maxima of the block kLag
  // before it (of the previous tile first).
  auto tile_steps = [&](auto u_c) __attribute__((always_inline)) {
    constexpr int U = decltype(u_c)::value, kPrev = (U + kRing - 1) % kRing;
    constexpr int kSlot0 = NT == 2 ? 2 * (U & 1) : 0;
    const v4i a = fp4_signs(ring[U].w);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      acc[(kSlot0 + j) & 3] = mfma_fp4(a, bq[j]);
      pin(acc[(kSlot0 + j) & 3]);
      if (j == 0) load(next, ring[kPrev]);
      if (j == 1) next = stream.next();
      fold(j >= kLag ? j - kLag : NT + j - kLag, (kSlot0 + j - kLag) & 3);
      __builtin_amdgcn_sched_barrier(0);
      if (j == kLag - 1) {
        if ((before >> kTileLastShift) & 1) finish_target(before);
        before = ring[U].e;
      }
    }
  };
  // The tiles of slots k .. kRing - 1; false at the stream's end.
  int last_slot0 = 0;
  auto round = [&](auto self, auto u_c) __attribute__((always_inline)) -> bool {
    constexpr int k = decltype(u_c)::value;
    if constexpr (k == kRing) {
      return true;
    } else {
      if (tiles_ended(ring[k].e)) {
        last_slot0 = NT == 2 ? 2 * ((k + 1) & 1) : 0;  // of slot k - 1
        return false;
      }
      tile_steps(u_c);
      return self(self, std::integral_constant<int, k + 1>{});
    }
  };
  while (round(round, std::integral_constant<int, 0>{})) {
  }
  // The last kLag blocks.
  mfma_results_fence();
#pragma unroll
  for (int j = 0; j < kLag; ++j) {
    const int blk = NT - kLag + j;
    if (NT == 2 && last_slot0 != 0) fold(blk, 2 + blk);
    else fold(blk, blk & 3);
  }
  finish_target(before);
}

}  // namespace

HammingPlan hamming_plan(int64_t batch, int64_t query_tokens) {
  // Whole batch rows per pass where one fits, spread evenly over the passes.
  HammingPlan h;
  h.whole = query_tokens <= kHammingRowsPerPass;
  const int64_t rows = batch * query_tokens;
  if (h.whole) {
    const int64_t per = kHammingRowsPerPass / query_tokens, passes = (batch + per - 1) / per;
    h.pass_rows = (batch + passes - 1) / passes * query_tokens;
  } else {
    h.pass_rows = kHammingRowsPerPass;
  }
  h.subs = (rows + h.pass_rows - 1) / h.pass_rows;
  return h;
}

hipError_t launch_hamming(const ScoreArgs& a, hipStream_t stream) {
  if (a.group_units <= 0 || a.num_waves <= 0 || a.num_waves % a.group_units != 0 || a.subs <= 0 ||
      a.pass_rows <= 0 || a.pass_rows > kHammingRowsPerPass || (a.out && a.iout) || a.qbits == nullptr || a.wave_info == nullptr ||
      a.tiles == nullptr)
    return hipErrorInvalidValue;
  ScoreArgs part = a;
  for (int64_t first = 0; first < a.subs; first += kMaxGridRows) {
    const dim3 grid((unsigned)(a.num_waves / a.group_units), (unsigned)std::min(kMaxGridRows, a.subs - first));
    part.first_pass = (int32_t)first;
    if (a.pass_rows <= 32) hamming_kernel<2><<<grid, kGroupThreads, 0, stream>>>(part);
    else if (a.pass_rows <= 64) hamming_kernel<4><<<grid, kGroupThreads, 0, stream>>>(part);
    else if (a.pass_rows <= 128) hamming_kernel<8><<<grid, kGroupThreads, 0, stream>>>(part);
    else if (a.pass_rows <= 192) hamming_kernel<12><<<grid, kGroupThreads, 0, stream>>>(part);
    else hamming_kernel<16><<<grid, kGroupThreads, 0, stream>>>(part);
  }
  return hipGetLastError();
}

}  // namespace msim
