// digit_kernel.hpp -- MaxSim scoring of fp32 queries on gfx950's fp6/fp4 MFMA:
// int4 or sign-bit documents (optionally with an int4 residual stream), the
// reference's five reducers, every document or given candidates.  Semantics:
// score.hip's header (the same restated lines of the reference).
//
// Query rows as digits.  A row q is fixed-point on a power-of-two grid: with
// colmul = 2^(E-1), max|q| <= 2^E, each q / colmul in [-2, 2] is rounded to a
// multiple of 2^-23 and written as five balanced digits of base 32,
//   q = colmul * sum_i d_i 2^-3 32^-i,  i = 0..4,  |d_0| <= 16, -16 <= d_i <= 15,
// every digit exact as fp6 (e2m3 holds the integers to 16 in units of 1/8).
// The grid keeps every bit of the row's largest elements and resolves the
// row to 2^-25..2^-24 of max|q|.
//
// Documents.  int4 codes are integers up to 8, exact in e2m3 too.  A handle in
// steady use keeps a copy of its codes as fp6 rows (96 bytes per token and 128
// dims, encode_fp6_kernel), because decoding nibbles to 6-bit fields in registers
// takes 37 VALU instructions per tile and chunk (decode_fp6: first calls,
// candidates, no memory for the copy).  Sign documents become
// fp4 +-1 with two instructions per dword (fp4_signs).  The MFMA's E8M0 scales
// hold the digits' weights 32^-i, so one v_mfma_scale_f32_16x16x128_f8f6f4
// per digit and 128 dims adds all digits into one fp32 accumulator, lowest
// digit first, so that the smaller digits keep their bits until the last steps.
// Each MFMA rounds: it cuts the accumulator at about 2^-25 of its largest
// product's power of two, downwards, and rounds its partial sums.  Similarities
// of unit queries against float64, int4 of 64..512 dims: 8.5e-8..1.1e-7 (2-norm,
// relative), of queries whose elements spread widely 1.5e-7..3.7e-7; three int8
// limbs 1.0e-7..1.2e-7 and 2.2e-7..5.5e-7.  A similarity is then one fma (times
// the token scale, the row mask as addend), or nothing for sign documents
// without token scales.
//
// Why digits rather than int8 limbs: three exact int8 limb dots need six MFMAs
// of 64 dims per 16 x 16 block and 4.5 VALU instructions per similarity to
// recombine (9 for sign documents); five MFMAs of 128 dims and one (or no)
// VALU instruction do the same.  Rates per MFMA and SIMD, two waves
// (microbench/rates.hip): i8 16x16x64 9.1 ns, fp6 x fp6 16x16x128 10.0, fp4 x fp6
// 9.4; with two fmas after each 10.0, 12.4 and 11.7.  MaxSim launches with three
// limbs and now, 32 query tokens:
//   int4, 16,384 documents of 64..192 tokens, 4 queries   117.6 -> 79.3 us
//   int4,  4,096 of the same, 2 queries                    20.8 -> 17.4 us
//   signs, 10,240 documents of 256..1,024 tokens, 1 / 2    125 / 206 -> 62 / 96 us
// (73 ns per 16 x 16 block of int4 at four blocks, 59 of signs, against 50 and 47
// of the MFMAs alone; one int4 query, 35.8 us, is bound by memory.)
//
// Work split: the waves of a workgroup (group_waves) share one pass of
// query rows; its digits are staged once in LDS and held in registers (NT
// blocks of 16 rows, 30 VGPRs each per 128 dims).  A wave walks 16-token tiles
// (the MFMA's A operand), held in a ring of registers filled by buffer loads
// (an address is a descriptor in SGPRs and a constant offset: 64-bit VGPR
// addresses would share registers with pending loads and make the compiler wait
// for them, 9 % slower; filling the ring in LDS by DMA took 29 % longer), from
// work units its workgroup's waves take from a counter in LDS (every document),
// or of one candidate document per wave.
// Step j of a tile issues row block j's MFMAs; the epilogue of the block one
// step back (the previous tile's last block for j = 0) is spread between them
// from the third MFMA on, so that its accumulators are at least two further
// MFMAs (32 cycles) old: no MFMA-result fence, and the matrix core and the
// VALU work at once.
#pragma once

#include "common.hpp"
#include "internal.hpp"
#include "score_reduce.hpp"

namespace msim {
namespace digit {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v8i __attribute__((ext_vector_type(8)));

constexpr int kDigits = kScoreDigits;
// Waves per workgroup: two per SIMD; one at four chunks, so that a pass holds
// 32 query rows (240 VGPRs of digits) and three tiles in flight (28 each).  With
// two waves a pass held 16 rows and one tile was in flight, and the calls waited
// for memory: 4,096 documents of 512 dims, queries of 32 tokens, the call: 1 / 4
// queries 101 / 287 us, now 73 / 164; with a residual stream 161 / 525, now
// 113 / 297; signs 113 / 318, now 85 / 193.
constexpr int group_waves(int kc) { return kc == 4 ? 4 : 8; }
constexpr int kFormatFp6 = 2, kFormatFp4 = 4;  // cbsz / blgp: e2m3, e2m1

// E8M0 scale bytes: 2^-5i of digit i, and of the document operand (int4 codes
// are held as code / 8: 2^3).
constexpr int kDigitScales = 127 | (122 << 8) | (117 << 16) | (112 << 24);
constexpr int kDigitScale4 = 107;

// Six dwords of a lane: 16 bytes at 16 g of a 96-byte row, 8 at 64 + 8 g.
struct Six {
  int w[6];
};
__device__ __forceinline__ Six load_six(const void* row, uint32_t byte_lo, uint32_t byte_hi) {
  const v4i lo = *reinterpret_cast<const v4i*>(static_cast<const char*>(row) + byte_lo);
  const v2i hi = *reinterpret_cast<const v2i*>(static_cast<const char*>(row) + byte_hi);
  return {{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1]}};
}
__device__ __forceinline__ Six load_six(__amdgpu_buffer_rsrc_t r, int byte_lo, int byte_hi) {
  const v4u lo = load_b128(r, byte_lo);
  const uint64_t hi = load_b64(r, byte_hi);
  return {{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)(uint32_t)hi, (int)(uint32_t)(hi >> 32)}};
}
__device__ __forceinline__ v8i operand(const Six& x) {
  return (v8i){x.w[0], x.w[1], x.w[2], x.w[3], x.w[4], x.w[5], 0, 0};
}
__device__ __forceinline__ v8i operand(const v4i& x) { return (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0}; }

// One lane's 32 nibbles of int4 codes as the fp6 fields the copy of the corpus
// holds (encode_fp6_kernel): 37 VALU instructions.  Nibbles q and q + 4 of a dword
// lie 16 bits apart and are elements 8 q + 2 d and the next one of the operand:
// with bit 3 flipped under the exponent of 1024 they are the halves 1024 + v + 8 (or,
// in bits 4..7, 1024 + 16 (v + 8)), one fma makes them v / 8, exactly, and one
// conversion packs all 32.  Against decode_fp6_lean, calls over 3,000 documents, 4
// queries of 32 tokens / one of 8: 128 dims 62.6 -> 59.6 / 35.1 -> 33.7 us, residual
// 82.8 -> 75.9 / 43.1 -> 40.1, 256 dims 97 -> 91 / 42.9 -> 40.2, residual 151 -> 125 /
// 58.0 -> 51.8, 512 dims 173 -> 149 / 71.5 -> 55.1 (and a kernel of 16 rows), residual
// 280 -> 231 / 103 -> 77.
__device__ __forceinline__ Six decode_fp6(const v4i& nibbles) {
  typedef _Float16 v2h __attribute__((ext_vector_type(2)));
  typedef _Float16 v32h __attribute__((ext_vector_type(32)));
  union {
    v2h pair[16];
    v32h all;
  } h;
  uint32_t flip_lo = 0x64086408u, flip_hi = 0x64806480u;
  asm("" : "+v"(flip_lo), "+v"(flip_hi));  // in VGPRs: and + xor is one v_bitop3_b32
  auto eighths = [&](uint32_t w, bool hi) __attribute__((always_inline)) -> v2h {
    const _Float16 unit = hi ? (_Float16)0.0078125f : (_Float16)0.125f, bias = hi ? (_Float16)-9.0f : (_Float16)-129.0f;
    const uint32_t x = hi ? (w & 0x00F000F0u) ^ flip_hi : (w & 0x000F000Fu) ^ flip_lo;
    return __builtin_elementwise_fma(__builtin_bit_cast(v2h, x), (v2h){unit, unit}, (v2h){bias, bias});
  };
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const uint32_t w = (uint32_t)nibbles[d], w8 = w >> 8;
    h.pair[d] = eighths(w, false);
    h.pair[4 + d] = eighths(w, true);
    h.pair[8 + d] = eighths(w8, false);
    h.pair[12 + d] = eighths(w8, true);
  }
  const auto f = __builtin_amdgcn_cvt_scalef32_pk32_fp6_f16(h.all, 1.0f);
  return {{(int)f[0], (int)f[1], (int)f[2], (int)f[3], (int)f[4], (int)f[5]}};
}

// The same in 82 instructions, sign and magnitude by bit operations, fields joined
// by dot products, without the 16 registers of halves: for the kernels that would
// spill 30 registers for them (residual, two chunks, TopK4 and SmoothSim: 60 us
// where those take 74, of 4 queries 158 against 186).
__device__ __forceinline__ Six decode_fp6_lean(const v4i& nibbles) {
  uint32_t pair[4][4];  // [8 fields][field 2 d and 2 d + 1 as 12 bits]
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const uint32_t w = (uint32_t)nibbles[d], neg = w & 0x88888888u, one = neg >> 3;
    const uint32_t mag = (w ^ (neg | (neg - one))) + one;  // |v| of each nibble
    // Fields as bytes: sign bit 5, magnitude below it.
    const uint32_t even = (mag & 0x0F0F0F0Fu) | ((neg & 0x08080808u) << 2);
    const uint32_t odd = ((mag >> 4) & 0x0F0F0F0Fu) | ((neg & 0x80808080u) >> 2);
    pair[0][d] = __builtin_amdgcn_udot4(even, 0x00400001u, 0u, false);
    pair[1][d] = __builtin_amdgcn_udot4(odd, 0x00400001u, 0u, false);
    pair[2][d] = __builtin_amdgcn_udot4(even, 0x40000100u, 0u, false);
    pair[3][d] = __builtin_amdgcn_udot4(odd, 0x40000100u, 0u, false);
  }
  Six x;
#pragma unroll
  for (int h = 0; h < 2; ++h) {  // 16 fields, three dwords
    const uint32_t(&a)[4] = pair[2 * h], (&b)[4] = pair[2 * h + 1];
    x.w[3 * h] = (int)(a[0] | (a[1] << 12) | (a[2] << 24));
    x.w[3 * h + 1] = (int)((a[2] >> 8) | (a[3] << 4) | (b[0] << 16) | (b[1] << 28));
    x.w[3 * h + 2] = (int)((b[1] >> 4) | (b[2] << 8) | (b[3] << 20));
  }
  return x;
}

// acc + documents (A) x digit D of the query (B).
template <int DOC, int D>
__device__ __forceinline__ v4f mfma_digit(const v8i& a, const v8i& b, const v4f& c, int sa, int s03, int s4) {
  constexpr int kA = DOC == kDocInt4 ? kFormatFp6 : kFormatFp4;
  if constexpr (D < 4) return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kA, kFormatFp6, 0, sa, D, s03);
  else return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kA, kFormatFp6, 0, sa, 0, s4);
}

// Tiles held per wave (one computed, the rest in flight): what the registers
// left by the query digits take (rings of eight at four chunks were no faster).
// Signs are small (256 bytes per tile), so only many of them in flight cover the
// memory latency.
constexpr int ring_size(int doc, bool res, int nt, int kc, bool unit) {
  if (doc == kDocSign && !res && kc == 1) return unit ? 8 : nt == 4 ? 4 : 8;
  if (kc == 4) return res && nt == 2 ? 2 : 4;
  if (res) return nt * kc >= 4 ? 2 : 4;
  return kc == 1 ? 4 : nt * kc >= 4 ? 2 : 4;
}

// State of row block a in lanes 0 .. 31 and of b in lanes 32 .. 63, each merged
// over the wave's two halves (row 0 / 1 or 2 / 3 of 16 lanes for swap16).
template <int RED, typename Swap>
__device__ __forceinline__ ReducerState<RED> swap_merge(const ReducerState<RED>& a, const ReducerState<RED>& b, Swap swap) {
  ReducerState<RED> x = a, y = b;
  auto sw = [&](float& u, float& v) __attribute__((always_inline)) {
    const auto r = swap(__float_as_uint(u), __float_as_uint(v));
    u = __uint_as_float(r[0]);
    v = __uint_as_float(r[1]);
  };
  if constexpr (RED == kRedMax) {
    sw(x.m, y.m);
    x.m = fmaxf(x.m, y.m);
  } else if constexpr (RED == kRedLse) {
    sw(x.m, y.m);
    sw(x.s, y.s);
    x.merge(y.m, y.s);
  } else {
    constexpr int K = RED == kRedTop2 ? 2 : 4;
#pragma unroll
    for (int i = 0; i < K; ++i) sw(x.t[i], y.t[i]);
#pragma unroll
    for (int i = 0; i < K; ++i) x.insert(y.t[i]);
  }
  return x;
}

// UNIT: sign documents without token scales, MaxSim: the similarity is the
// accumulator itself.  DIRECT: one target per wave, its document's token range
// from p.direct_offsets; else work units.  RAW: int4 streams as nibbles
// (p.code_bytes a token), decoded tile by tile: handles without the fp6 copy.
template <int DOC, bool RES, int NT, int RED, int KC, bool UNIT, bool DIRECT, bool RAW>
__global__ __launch_bounds__(kWave * group_waves(KC), group_waves(KC) / 4) void digit_score_kernel(
    ScoreArgs p) {
  constexpr int kWavesPerGroup = group_waves(KC), kThreads = kWavesPerGroup * kWave;
  static_assert(!UNIT || (DOC == kDocSign && !RES && RED == kRedMax), "accumulators as similarities");
  static_assert(!(DOC == kDocSign && RES) || KC == 1, "sign prefix + residual: 128 dims");
  constexpr int kRing = ring_size(DOC, RES, NT, KC, UNIT);
  static_assert(kRing % 2 == 0, "accumulator sets alternate over an even ring");
  constexpr int kSets = NT == 1 ? 2 : NT;  // accumulators of a step and of the step before it
  constexpr int kCodeBytes = 16 * KC, kResBytes = 96 * KC, kRowBytes = 96 * KC;
  constexpr float kStart = UNIT ? kNegInf : 0.0f;  // accumulators before the first tile
  constexpr int kChain = kDigits * KC, kSteps = RES ? 2 * kChain : kChain;  // MFMAs of a step

  // The pass's query digits: [row][digit][96 KC], rows 16 j + c.
  constexpr int kVecs = kDigits * 16 * NT * kRowBytes / 16;
  __shared__ __attribute__((aligned(16))) v4i s_q[kVecs];
  __shared__ float s_pool[kWavesPerGroup][16 * NT];
  __shared__ int s_next;
  if constexpr (!DIRECT) {
    if (threadIdx.x == 0) s_next = 2 * kWavesPerGroup;
    __syncthreads();
  }
  const int lane = lane_id();
  const int wave = wave_uniform(threadIdx.x / kWave);
  const int g = lane >> 4, c = lane & 15;
  const int pass = (int)blockIdx.y + p.first_pass, grp = pass / p.subs, sub = pass % p.subs;
  const int lr0 = sub * p.pass_rows;                      // first local row of the pass
  const int64_t grow0 = (int64_t)grp * p.grp_rows + lr0;  // its global query row

  // The wave's tiles: work units, or (DIRECT) the tiles of one target.  Either
  // way the end is an entry that tiles_ended() recognises, of token 0, again and
  // again.
  const int64_t gw = (int64_t)wave * gridDim.x + blockIdx.x;  // DIRECT: the target
  int64_t ds = 0, doc0 = 0;
  int ntok = 0, na = 0, q = 0;
  if constexpr (DIRECT) {
    if (gw < p.direct_count) {
      doc0 = as_constant(p.targets)[grp * p.targets_grp_stride + gw];
      ds = as_constant(p.direct_offsets)[doc0];
      ntok = (int)(as_constant(p.direct_offsets)[doc0 + 1] - ds);
      na = ntok == 0 ? 1 : (ntok + 15) / 16;  // an empty document: one tile, not scored
    }
  }
  TileStream<kWavesPerGroup> stream(p, DIRECT ? -1 : wave, lane, s_next);
  auto next_entry = [&]() __attribute__((always_inline)) -> uint64_t {
    if constexpr (DIRECT) {
      const int left = ntok - 16 * q;
      const bool in = left > 0;
      const uint64_t e =
          score_tile_entry(in ? ds + 16 * (int64_t)q : 0, in ? min(16, left) : 1, q + 1 == na, left <= 0, 0);
      q = min(q + 1, na);
      return e;
    } else {
      return stream.next();
    }
  };

  // The query digits: global loads first, the first tiles behind them, then
  // to LDS.
  constexpr int kStage = (kVecs + kThreads - 1) / kThreads;
  v4i stage[kStage];
#pragma unroll
  for (int x = 0; x < kStage; ++x)
    stage[x] = reinterpret_cast<const v4i*>(p.qpack + grow0 * (kDigits * kRowBytes))[min((int)threadIdx.x + x * kThreads, kVecs - 1)];
  // At a target's end lane group g holds row block (g >> 1) + 2 (g & 1).
  const int blk = (g >> 1) | ((g & 1) << 1);
  const int64_t my_row = grow0 + 16 * min(blk, NT - 1) + c;
  const float colmul_row = p.colmul[my_row], weight = p.weights ? p.weights[my_row] : 1.0f;
  float lse_mul[RED == kRedLse ? NT : 1];
  if constexpr (RED == kRedLse) {
#pragma unroll
    for (int j = 0; j < NT; ++j) lse_mul[j] = p.colmul[grow0 + 16 * j + c];
  }
  __builtin_amdgcn_sched_barrier(0);

  using Codes = std::conditional_t<RAW, v4i, Six>;  // one chunk of an int4 stream
  struct Tile {
    uint64_t e;
    Codes code[DOC == kDocInt4 ? KC : 1];
    unsigned sign[DOC == kDocSign ? KC : 1];
    Codes res[RES ? KC : 1];
    float s[UNIT ? 1 : 4], sr[RES ? 4 : 1];
  };
  // A tile's loads: one buffer per stream at the tile's first token, the lane's
  // part a constant offset.  Rows past a short document hold the next tokens'
  // codes (or those of the kScanPadTokens zero tokens after the last one) and a
  // scale of 0 (the buffers end there: a product with the next document's scale
  // may not be finite, and -inf then does not mask it).
  const int va = c * kCodeBytes + 4 * g;  // sign documents
  const int vr = c * kResBytes + 16 * g, vs = 16 * g, vn = RAW ? c * p.code_bytes + 16 * g : 0;
  // (Nibbles past a token's row are the next token's, or 0 past the tile's last
  // row: they meet zero query digits.)
  auto load_codes = [&](const uint8_t* codes, int64_t start, int rows, Codes (&out)[KC]) __attribute__((always_inline)) {
    if constexpr (RAW) {
      const __amdgpu_buffer_rsrc_t r = make_rsrc(codes + start * p.code_bytes, (uint32_t)(rows * p.code_bytes));
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        const v4u w = load_b128(r, vn + 64 * kc);
        out[kc] = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
      }
    } else {
      const __amdgpu_buffer_rsrc_t r = make_rsrc(codes + start * kResBytes, 16 * kResBytes);
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) out[kc] = load_six(r, vr + 96 * kc, vr + 96 * kc + 64 - 8 * g);
    }
  };
  auto load = [&](uint64_t e, Tile& t) __attribute__((always_inline)) {
    t.e = e;
    const int64_t start = (int64_t)(e & kTileStartMask);
    const int rows = (int)((e >> kTileRowsShift) & 15) + 1;
    if constexpr (DOC == kDocInt4) {
      load_codes(p.codes, start, rows, t.code);
    } else {
      const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.codes + start * kCodeBytes, 16 * kCodeBytes);
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) t.sign[kc] = load_b32(ra, va + 16 * kc);
    }
    if constexpr (RES) load_codes(p.rcodes, start, rows, t.res);
    if constexpr (!UNIT) {
      const uint32_t scale_bytes = 4u * (uint32_t)rows;
      const v4u sv = load_b128(make_rsrc(p.tscale + start, scale_bytes), vs);
#pragma unroll
      for (int k = 0; k < 4; ++k) t.s[k] = __uint_as_float(sv[k]);
      if constexpr (RES) {
        const v4u rv = load_b128(make_rsrc(p.rtscale + start, scale_bytes), vs);
#pragma unroll
        for (int k = 0; k < 4; ++k) t.sr[k] = __uint_as_float(rv[k]);
      }
    }
  };
  Tile ring[kRing];
#pragma unroll
  for (int u = 0; u < kRing - 1; ++u) load(next_entry(), ring[u]);
  uint64_t next = next_entry();  // the entry of the tile loaded next
  __builtin_amdgcn_sched_barrier(0);

#pragma unroll
  for (int x = 0; x < kStage; ++x) s_q[min((int)threadIdx.x + x * kThreads, kVecs - 1)] = stage[x];
  __syncthreads();
  if (tiles_ended(ring[0].e)) return;  // no barriers below
  Six bq[NT][kDigits][KC];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
#pragma unroll
    for (int d = 0; d < kDigits; ++d)
#pragma unroll
      for (int kc = 0; kc < KC; ++kc)
        bq[j][d][kc] = load_six(reinterpret_cast<const char*>(s_q) + ((16 * j + c) * kDigits + d) * kRowBytes + 96 * kc,
                                16u * g, 64u + 8u * g);
  }
  // Factors of a similarity before (int4 token scales are stored / 16) and
  // after the reduction; one stream takes its constant factor after it, before
  // colmul (the two alone may leave the floats' range).
  const float mul = DOC == kDocInt4 ? 16.0f * p.tmul : p.tmul;
  const float after_mul = RES ? 1.0f : mul;
  const float k2 = kLog2e / p.temperature;
  int sa = DOC == kDocInt4 ? 130 : 127, sr = 130, s03 = kDigitScales, s4 = kDigitScale4;
  asm volatile("" : "+v"(sa), "+v"(sr), "+v"(s03), "+v"(s4));  // kept in VGPRs
  const auto doc_scale = p.doc_scale ? as_constant(p.doc_scale) : nullptr;

  ReducerState<RED> st[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    st[j].init();
    if constexpr (RED == kRedLse) st[j].k = 0.0f;  // of the masked tile before the first
  }
  v4f acc[kSets], accr[RES ? kSets : 1];
  int len = 0;  // tokens of the current target so far
  auto rows_of = [](uint64_t e) -> int { return (int)((e >> kTileRowsShift) & 15) + 1; };
  auto target_of = [&](uint64_t e) -> int64_t { return DIRECT ? gw : (int64_t)(e >> kTileLocalShift); };
  auto scale_of = [&](int64_t target) -> float { return doc_scale ? doc_scale[DIRECT ? doc0 : target] : p.scale; };
  auto begin_target = [&](uint64_t e) __attribute__((always_inline)) {
    if constexpr (RED == kRedLse) {
      const float f = scale_of(target_of(e)) * k2;
#pragma unroll
      for (int j = 0; j < NT; ++j) st[j].k = lse_mul[j] * after_mul * f;
    }
  };
  const int pass_rows = min(p.pass_rows, p.grp_rows - lr0);
  const bool sum_regs = NT > 1 && p.out && p.query_tokens == 32;
  // End of the target whose last tile is e.
  auto finish_target = [&](uint64_t e) __attribute__((always_inline)) {
    const int64_t tg = target_of(e);
    auto sw32 = [](uint32_t a, uint32_t b) { return __builtin_amdgcn_permlane32_swap(a, b, false, false); };
    auto sw16 = [](uint32_t a, uint32_t b) { return __builtin_amdgcn_permlane16_swap(a, b, false, false); };
    ReducerState<RED> none;
    none.init();
    const ReducerState<RED> x = swap_merge<RED>(st[0], NT > 1 ? st[NT > 1 ? 1 : 0] : none, sw32);
    const ReducerState<RED> y = NT > 2 ? swap_merge<RED>(st[NT > 2 ? 2 : 0], st[NT > 3 ? 3 : 0], sw32) : none;
    const ReducerState<RED> all = swap_merge<RED>(x, y, sw16);
    const bool empty = ((e >> kTileEmptyShift) & 1) != 0;
    const float v = all.finish(empty ? 0 : len, after_mul, colmul_row, p.temperature, weight, scale_of(tg));
#pragma unroll
    for (int j = 0; j < NT; ++j) st[j].init();
    len = 0;
    const int64_t b0 = grow0 / p.query_tokens;
    if (sum_regs) {
      // 32-token queries: a batch row's token l and l + 16 are 32 lanes apart
      // (lane groups g and g + 2), summed in token_sum16's order.  Of no other
      // length do two whole 16-row blocks make a batch row; those go through LDS,
      // at most 3 % slower (16,384 documents, 31 / 32 tokens, the call: 1 query
      // 38.7 / 38.3 us, 2 49.1 / 47.7, 4 85.1 / 83.5).
      float w = v, o = 0.0f;
      const auto r = sw32(__float_as_uint(w), __float_as_uint(o));  // upper half of w over the lower of o
      w = row_butterfly16(__uint_as_float(r[0]) + __uint_as_float(r[1]));
      if (c == 0 && 32 * g < pass_rows && g < NT / 2) p.out[(b0 + g) * p.out_stride + tg] = w;
    } else if (p.out) {
      // Whole batch rows in this pass: their query tokens summed here.
      if (blk < NT) s_pool[wave][16 * blk + c] = v;
      wave_sync_lds();
      sum_batch_rows(s_pool[wave], pass_rows / p.query_tokens, p.query_tokens,
                     [&](int b, float s) { p.out[(b0 + b) * p.out_stride + tg] = s; });
      wave_sync_lds();
    } else {
      float* out = p.pooled + grp * p.pooled_grp_stride + tg * p.grp_rows + lr0;
      if (blk < NT && 16 * blk + c < pass_rows) out[16 * blk + c] = v;
    }
  };

  // What the epilogue of a tile needs once its ring slot is reused.  mask: -inf
  // for rows past the tile's, else -0 (x + -0 = x for every x), which joins
  // the similarity's fma (SmoothSim: that of its scaled form).
  struct Pend {
    float s[UNIT ? 1 : 4], sr[RES ? 4 : 1], mask[UNIT ? 1 : 4];
    uint64_t e;
  };
  // Row k of an accumulator set as similarities, and a row block's four into
  // its reducer.
  auto zval = [&](const Pend& P, const v4f& x, const v4f& y, int k) __attribute__((always_inline)) -> float {
    if constexpr (UNIT) return x[k];
    const float z = RED == kRedLse ? x[k] * P.s[k] : fmaf(x[k], P.s[k], P.mask[k]);
    if constexpr (RES) return fmaf(y[k], P.sr[k], z);
    return z;
  };
  auto fold = [&](const Pend& P, float (&z)[4], int j) __attribute__((always_inline)) {
    if constexpr (UNIT) {
      const int rows = rows_of(P.e);
      if (rows < 16) {
#pragma unroll
        for (int k = 0; k < 4; ++k) z[k] = 4 * g + k >= rows ? kNegInf : z[k];
      }
    }
    if constexpr (RED == kRedLse) st[j].add4(z, P.mask);
    else st[j].add4(z);
  };
  // MFMAs stay before the pins of their result, and its reads behind the next
  // one: the compiler otherwise sinks a chain to its epilogue in a later
  // step, or hoists the row mask up to the chain, and the epilogue stands
  // right behind the MFMAs (too early for max3_op, whose inline asm operands
  // get no wait states, and with nothing to overlap).
  auto pin = [](v4f& x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); };
  // One step: the MFMAs of row block j of tile t into accumulator set `set`.
  // Between them, from the third MFMA on, the epilogue of the step before
  // (tile P, its block jp and set), and what extra(m) puts after MFMA m.
  struct Fp6 {  // decoded streams of a tile (RAW)
    Six code[RAW && DOC == kDocInt4 ? KC : 1], res[RAW && RES ? KC : 1];
  };
  auto decode = [&](const Tile& t, Fp6& f) __attribute__((always_inline)) {
    if constexpr (RAW) {
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        constexpr bool kLean = RES && KC == 2 && (RED == kRedTop4 || RED == kRedLse);
        if constexpr (DOC == kDocInt4) f.code[kc] = kLean ? decode_fp6_lean(t.code[kc]) : decode_fp6(t.code[kc]);
        if constexpr (RES) f.res[kc] = kLean ? decode_fp6_lean(t.res[kc]) : decode_fp6(t.res[kc]);
      }
    }
  };
  auto step = [&](const Tile& t, const Fp6& f, int j, int set, const Pend& P, int jp, int setp, auto extra)
                  __attribute__((always_inline)) {
    constexpr int kWait = 2, kSpan = kSteps - kWait;  // >= 3 slots
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    float z[4];
    int m = 0;
    auto after = [&](int m) __attribute__((always_inline)) {
      extra(m);
      if (m >= kWait) {
        if (m == kWait) {
          pin(acc[setp]);
          if constexpr (RES) pin(accr[setp]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (kWait + k * kSpan / 4 == m) z[k] = zval(P, acc[setp], accr[RES ? setp : 0], k);
        if (m == kSteps - 1) fold(P, z, jp);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    v8i a[KC];
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      if constexpr (DOC == kDocSign) a[kc] = operand(fp4_signs(t.sign[kc]));
      else if constexpr (RAW) a[kc] = operand(f.code[kc]);
      else a[kc] = operand(t.code[kc]);
    }
    auto digits = [&](auto digit_c, v4f& dst, const v8i (&ops)[KC], auto doc_c, int scale)
                      __attribute__((always_inline)) {
      constexpr int d = decltype(digit_c)::value;
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        const v4f& from = d == kDigits - 1 && kc == 0 ? zero : dst;
        dst = mfma_digit<decltype(doc_c)::value, d>(ops[kc], operand(bq[j][d][kc]), from, scale, s03, s4);
        if (m == kWait) pin(dst);
        after(m++);
      }
    };
    auto chain = [&](v4f& dst, const v8i (&ops)[KC], auto doc_c, int scale) __attribute__((always_inline)) {
      digits(std::integral_constant<int, 4>{}, dst, ops, doc_c, scale);
      digits(std::integral_constant<int, 3>{}, dst, ops, doc_c, scale);
      digits(std::integral_constant<int, 2>{}, dst, ops, doc_c, scale);
      digits(std::integral_constant<int, 1>{}, dst, ops, doc_c, scale);
      digits(std::integral_constant<int, 0>{}, dst, ops, doc_c, scale);
      pin(dst);
    };
    chain(acc[set], a, std::integral_constant<int, DOC>{}, sa);
    if constexpr (RES) {
      v8i r[KC];
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        if constexpr (RAW) r[kc] = operand(f.res[kc]);
        else r[kc] = operand(t.res[kc]);
      }
      chain(accr[set], r, std::integral_constant<int, kDocInt4>{}, sr);
    }
  };

  // All steps of the tile in slot U, the previous tile's last epilogue in its
  // first step.  The loads of the tile kRing - 1 ahead go to the previous
  // tile's slot; their address arithmetic and the entry after them lie between
  // the MFMAs.
  Pend P;
  bool masked = true;  // P.mask has rows past its tile
  int last_set = 0;    // accumulator set of the last tile (one row block)
  auto set_masks = [&](int rows) __attribute__((always_inline)) {
    if constexpr (!UNIT) {
      if (rows < 16 || masked) {
#pragma unroll
        for (int k = 0; k < 4; ++k) P.mask[k] = 4 * g + k >= rows ? kNegInf : -0.0f;
        masked = rows < 16;
      }
    }
  };
  auto tile_steps = [&](auto u_c) __attribute__((always_inline)) {
    constexpr int U = decltype(u_c)::value, kPrev = (U + kRing - 1) % kRing;
    const Tile& t = ring[U];
    auto fetch = [&](int m) __attribute__((always_inline)) {
      if (m == 0) load(next, ring[kPrev]);
      if (m == 1) next = next_entry();
    };
    auto none = [](int) {};
    Fp6 f;
    decode(t, f);
    step(t, f, 0, NT == 1 ? U & 1 : 0, P, NT - 1, NT == 1 ? (U + 1) & 1 : NT - 1, fetch);
    const bool fresh = ((P.e >> kTileLastShift) & 1) != 0;
    len += rows_of(P.e);
    if (fresh) finish_target(P.e);
    P.e = t.e;
    last_set = U & 1;
    if constexpr (!UNIT) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        P.s[k] = RES ? t.s[k] * mul : t.s[k];
        if constexpr (RES) P.sr[k] = t.sr[k] * (16.0f * p.rmul);
      }
      set_masks(rows_of(P.e));
    }
    if (len == 0) begin_target(P.e);  // (after the start's masked tile too)
#pragma unroll
    for (int j = 1; j < NT; ++j) step(t, f, j, j, P, j - 1, j - 1, none);
  };
  // Before the first tile: zero accumulators and every row masked, whose
  // epilogue changes nothing (no copy of the loop's body for the first tile:
  // the compiler would wait for every load in flight to move it into the
  // loop's registers).
  P.e = score_tile_entry(0, 1, false, false, 0);
#pragma unroll
  for (int k = 0; k < (UNIT ? 1 : 4); ++k) {
    P.s[k] = 0.0f;
    P.mask[k] = kNegInf;
  }
#pragma unroll
  for (int k = 0; k < (RES ? 4 : 1); ++k) P.sr[k] = 0.0f;
#pragma unroll
  for (int x = 0; x < kSets; ++x) acc[x] = (v4f){kStart, kStart, kStart, kStart};
#pragma unroll
  for (int x = 0; x < (RES ? kSets : 1); ++x) accr[x] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
  len = -1;  // that tile's row count
  // The tiles of slots k .. kRing - 1; false at the stream's end.
  auto round = [&](auto self, auto u_c) __attribute__((always_inline)) -> bool {
    constexpr int k = decltype(u_c)::value;
    if constexpr (k == kRing) {
      return true;
    } else {
      if (tiles_ended(ring[k].e)) return false;
      tile_steps(u_c);
      return self(self, std::integral_constant<int, k + 1>{});
    }
  };
  while (round(round, std::integral_constant<int, 0>{})) {
  }
  // The last block of the last tile, right after its MFMAs.
  mfma_results_fence();
  {
    float z[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v4f x = acc[NT == 1 ? 0 : NT - 1], y = accr[RES && NT > 1 ? NT - 1 : 0];
      if constexpr (NT == 1) {
        x[k] = last_set ? acc[kSets - 1][k] : acc[0][k];
        if constexpr (RES) y[k] = last_set ? accr[kSets - 1][k] : accr[0][k];
      }
      z[k] = zval(P, x, y, k);
    }
    fold(P, z, NT - 1);
  }
  len += rows_of(P.e);
  finish_target(P.e);
}

template <int DOC, bool RES, int NT, int RED, int KC, bool UNIT = false, bool RAW = false>
hipError_t launch_mode(const ScoreArgs& a, dim3 grid, hipStream_t s) {
  constexpr int kThreads = kWave * group_waves(KC);
  if (a.direct_offsets) digit_score_kernel<DOC, RES, NT, RED, KC, UNIT, true, RAW><<<grid, kThreads, 0, s>>>(a);
  else digit_score_kernel<DOC, RES, NT, RED, KC, UNIT, false, RAW><<<grid, kThreads, 0, s>>>(a);
  return hipGetLastError();
}
template <int DOC, bool RES, int NT, int KC, bool RAW = false>
hipError_t launch_reducer(const ScoreArgs& a, int reducer, dim3 grid, hipStream_t s) {
  switch (reducer) {
    case kRedMax: return launch_mode<DOC, RES, NT, kRedMax, KC, false, RAW>(a, grid, s);
    case kRedTop2: return launch_mode<DOC, RES, NT, kRedTop2, KC, false, RAW>(a, grid, s);
    case kRedTop4: return launch_mode<DOC, RES, NT, kRedTop4, KC, false, RAW>(a, grid, s);
    case kRedLse: return launch_mode<DOC, RES, NT, kRedLse, KC, false, RAW>(a, grid, s);
    default: return hipErrorInvalidValue;
  }
}

// The instantiations by document format (one source file each).
hipError_t launch_int4(const ScoreArgs& a, bool residual, int nt, int reducer, dim3 grid, hipStream_t s);
hipError_t launch_sign(const ScoreArgs& a, bool residual, int nt, int reducer, dim3 grid, hipStream_t s);
hipError_t launch_wide2(const ScoreArgs& a, int doc, bool residual, int nt, int reducer, dim3 grid, hipStream_t s);
hipError_t launch_wide4(const ScoreArgs& a, int doc, bool residual, int nt, int reducer, dim3 grid, hipStream_t s);
hipError_t launch_wide4_residual(const ScoreArgs& a, int nt, int reducer, dim3 grid, hipStream_t s);
// ScoreArgs::code_bytes set.
hipError_t launch_raw(const ScoreArgs& a, int doc, bool residual, int nt, int reducer, dim3 grid, hipStream_t s);
hipError_t launch_raw_wide(const ScoreArgs& a, bool residual, int nt, int reducer, dim3 grid, hipStream_t s);

}  // namespace digit
}  // namespace msim
