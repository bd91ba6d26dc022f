// digit_score.hip -- launches of the fp32-query scorer (digit_kernel.hpp): the
// query's digits, the documents' fp6 copies, and which kernel scores a call.
#include <algorithm>

#include "digit_kernel.hpp"

namespace msim {

namespace {

// Tiles times passes that pay for pool_sum_kernel (2 us beside the scores it
// reads); half of it at four chunks, whose tiles take twice as long.  Whole
// rows / packed, the call in us: 8,200 tiles, 4 queries of 40 tokens (four
// passes / three) 39.6 / 40.0; 12,000: 43.8 / 43.3; 16,400: 49.1 / 47.1; 33,000:
// 69 / 63, 8 queries 103 / 83, 16 of 33 tokens 177 / 121; 256 dims, 3 of 20:
// 74.6 / 54.4.
constexpr int64_t kPackTiles = 12288;

// Six-bit fields of one lane's 32 operand elements: element s is bits 6 s ..
// 6 s + 5 of 192 (six dwords).
struct Fields {
  uint32_t w[6];
  __device__ __forceinline__ void put(int s, uint32_t code) {
    const int bit = 6 * s, word = bit / 32, at = bit % 32;
    w[word] |= code << at;
    if (at > 26) w[word + 1] |= code >> (32 - at);
  }
};
// Operand element s of lane group g is dim 32 g + 4 (s % 8) + s / 8 of a
// chunk: the order in which sign bits become fp4 elements (fp4_signs).
__device__ __forceinline__ constexpr int element_dim(int s) { return 4 * (s % 8) + s / 8; }
// Integer |v| <= 16 as e2m3 in units of 1 / 8: the magnitude is its code up to
// 16 (8 + m mantissa steps above 7, then exponent 2), the sign bit above it.
__device__ __forceinline__ uint32_t e2m3_int(int v) { return (uint32_t)abs(v) | (v < 0 ? 32u : 0u); }

__device__ __forceinline__ void store_fields(uint8_t* row, int g, const Fields& f) {
  *reinterpret_cast<v4u*>(row + 16 * g) = (v4u){f.w[0], f.w[1], f.w[2], f.w[3]};
  *reinterpret_cast<uint2*>(row + 64 + 8 * g) = make_uint2(f.w[4], f.w[5]);
}

// One thread per (token, 128-dim chunk, lane group): 16 bytes of nibbles to 24
// of fp6 (a read of 64 and a write of 96 bytes per token and chunk: bound by
// memory, once per corpus).  Bytes past the token's row count as zero codes.
__global__ __launch_bounds__(256) void encode_fp6_kernel(const uint8_t* __restrict__ codes, int64_t groups,
                                                         int64_t row_bytes, int64_t token_groups,
                                                         uint8_t* __restrict__ out) {
  const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (x >= groups) return;
  const int64_t first = 16 * (x % token_groups);
  const uint8_t* src = codes + (x / token_groups) * row_bytes + first;
  v4u in = {0u, 0u, 0u, 0u};
  if (row_bytes % 16 == 0) {
    if (first < row_bytes) in = *reinterpret_cast<const v4u*>(src);
  } else {
#pragma unroll
    for (int b = 0; b < 16; ++b)
      if (first + b < row_bytes) in[b / 4] |= (uint32_t)src[b] << (8 * (b % 4));
  }
  Fields f = {{0u, 0u, 0u, 0u, 0u, 0u}};
#pragma unroll
  for (int s = 0; s < 32; ++s) {
    const int n = element_dim(s);  // nibble n of the 32
    f.put(s, e2m3_int((int)(in[n / 8] << (28 - 4 * (n % 8))) >> 28));
  }
  store_fields(out + (x >> 2) * 96, (int)(x & 3), f);
}

// One wave per query row of 128 * chunks floats.  colmul = 2^(E-1) with
// 2^(E-1) < max|q| <= 2^E, clamped to the normal floats (1 for a zero row):
// Y = q / colmul in units of 2^-23, rounded to the integer (|Y| <= 2^24); with
// the bias 16 (1 + 32 + 32^2 + 32^3) the balanced digits of Y are its plain
// base-32 digits.  NaN elements count as 0; a row with an infinity gets
// colmul = inf, so its scores are not finite.  The workgroups past the rows
// copy src to dst.
__global__ __launch_bounds__(256) void quantize_digits_kernel(const float* __restrict__ query, int64_t rows,
                                                              int64_t rows_padded, uint8_t* __restrict__ qpack,
                                                              float* __restrict__ colmul, int chunks,
                                                              const int64_t* __restrict__ src,
                                                              int64_t* __restrict__ dst, int64_t count) {
  constexpr int kDigits = kScoreDigits, kMaxDims = 512;
  __shared__ int s_y[4][kMaxDims];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= rows_padded) {  // whole waves, no barrier below
    const int64_t i = (int64_t)(blockIdx.x - (rows_padded + 3) / 4) * 256 + threadIdx.x;
    if (i >= 0 && i < count) dst[i] = src[i];
    return;
  }
  const int width = 128 * chunks;
  float v[8];
  float m = 0.0f;
#pragma unroll
  for (int kc = 0; kc < 4; ++kc) {
    float2 x = make_float2(0.0f, 0.0f);
    if (kc < chunks && row < rows) x = reinterpret_cast<const float2*>(query + row * width + 128 * kc)[lane];
    v[2 * kc] = x.x;
    v[2 * kc + 1] = x.y;
    m = fmaxf(m, fmaxf(fabsf(x.x), fabsf(x.y)));
  }
  const uint32_t mb = __float_as_uint(wave_reduce(m, [](float x, float y) { return fmaxf(x, y); }));
  // max = f 2^x with 1 <= f < 2 (x = exponent field - 127): E = x for a power
  // of two, else x + 1; the exponent field of colmul is that of 2^(E-1).
  const bool infinite = mb >= 0x7F800000u;
  int field = (int)(mb >> 23) - ((mb & 0x7FFFFFu) == 0u ? 1 : 0);
  field = mb == 0u ? 127 : max(field, 1);
#pragma unroll
  for (int kc = 0; kc < 4; ++kc)
    if (kc < chunks) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        // Digit i counts 2^-3 32^-i, so the last one 2^-23; colmul = 2^(field - 127).
        const float y = rintf(__builtin_amdgcn_ldexpf(v[2 * kc + e], 150 - field));
        s_y[wave][128 * kc + 2 * lane + e] = infinite ? 0 : (int)y;
      }
    }
  wave_sync_lds();
  // Lane (chunk, digit, group): its 32 elements' digit as fp6 fields.
  constexpr int kBias = 16 * (1 + 32 + 32 * 32 + 32 * 32 * 32);
  for (int t = lane; t < chunks * kDigits * 4; t += kWave) {
    const int g = t & 3, d = (t >> 2) % kDigits, kc = (t >> 2) / kDigits;
    const int shift = 5 * (kDigits - 1 - d);
    Fields f = {{0u, 0u, 0u, 0u, 0u, 0u}};
#pragma unroll
    for (int s = 0; s < 32; ++s) {
      const int y = (s_y[wave][128 * kc + 32 * g + element_dim(s)] + kBias) >> shift;
      f.put(s, e2m3_int(d == 0 ? y : (y & 31) - 16));
    }
    store_fields(qpack + (row * kDigits + d) * (96 * (int64_t)chunks) + 96 * kc, g, f);
  }
  if (lane == 0)
    colmul[row] = row >= rows ? 0.0f : infinite ? __builtin_huge_valf() : __uint_as_float((uint32_t)field << 23);
}

}  // namespace

hipError_t launch_encode_fp6(const uint8_t* codes, int64_t tokens, int64_t row_bytes, int chunks, uint8_t* out,
                             hipStream_t stream) {
  if (row_bytes <= 0 || row_bytes > 64 * (int64_t)chunks) return hipErrorInvalidValue;
  // (A launch has fewer than 2^32 threads.)
  constexpr int64_t kMost = int64_t(1) << 26;
  for (int64_t first = 0; first < tokens; first += kMost) {
    const int64_t groups = std::min(kMost, tokens - first) * chunks * 4;
    encode_fp6_kernel<<<dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, stream>>>(
        codes + first * row_bytes, groups, row_bytes, 4 * (int64_t)chunks, out + first * 96 * chunks);
  }
  return hipGetLastError();
}

hipError_t launch_quantize_digits(const float* d_query, int64_t rows, int64_t rows_padded, uint8_t* qpack,
                                  float* colmul, int chunks, const int64_t* src, int64_t* dst, int64_t count,
                                  hipStream_t stream) {
  if (rows_padded <= 0) return hipSuccess;
  if (chunks != 1 && chunks != 2 && chunks != 4) return hipErrorInvalidValue;
  const int64_t blocks = (rows_padded + 3) / 4 + (count + 255) / 256;
  quantize_digits_kernel<<<dim3((unsigned)blocks), dim3(256), 0, stream>>>(d_query, rows, rows_padded, qpack, colmul,
                                                                         chunks, src, dst, count);
  return hipGetLastError();
}

DigitPlan digit_plan(int64_t batch, int64_t query_tokens, int chunks, int64_t tiles) {
  // The most rows a pass holds in registers: 64, or 32 of more than 128 dims.
  // Whole batch rows per pass where one fits (the kernel then sums their
  // tokens), spread evenly over the passes; blocks of 1, 2 or 4.  Batch rows
  // that fill their passes badly (33 of 64) are cut at the passes' ends where
  // that saves kPackTiles tiles: pool_sum_kernel then sums their tokens.
  const int64_t most = chunks == 1 ? 64 : 32;
  const int64_t packed = (batch * query_tokens + most - 1) / most;
  DigitPlan d;
  d.pass_rows = most;
  d.subs = packed;
  d.whole = false;
  if (query_tokens <= most) {
    const int64_t per = most / query_tokens, passes = (batch + per - 1) / per;
    if ((passes - packed) * tiles * (chunks == 4 ? 2 : 1) < kPackTiles) {
      d.pass_rows = (batch + passes - 1) / passes * query_tokens;
      d.subs = (batch * query_tokens + d.pass_rows - 1) / d.pass_rows;
      d.whole = true;
    }
  }
  d.nt = d.pass_rows <= 16 ? 1 : d.pass_rows <= 32 ? 2 : 4;
  return d;
}

hipError_t launch_digit_score(const ScoreArgs& a, int doc, bool residual, int nt, int reducer, int64_t groups,
                              hipStream_t stream) {
  using namespace digit;
  if (a.subs <= 0 || groups <= 0 || a.pass_rows <= 0 || a.pass_rows > 16 * nt || a.tscale == nullptr ||
      (residual && (a.rcodes == nullptr || a.rtscale == nullptr)) || a.code_bytes % 4 != 0 || a.code_bytes < 0 ||
      a.code_bytes > 64 * a.chunks)
    return hipErrorInvalidValue;
  const int64_t waves = group_waves(a.chunks);
  int64_t blocks;
  if (a.direct_offsets != nullptr) {
    if (a.targets == nullptr) return hipErrorInvalidValue;
    // As many workgroups as CUs before a workgroup gets a second document:
    // a wave alone on its SIMD runs faster than one of two.
    const int64_t spread = std::max<int64_t>(1, device_cu_count() / (groups * a.subs));
    blocks = std::max<int64_t>((a.direct_count + waves - 1) / waves, std::min(a.direct_count, spread));
  } else {
    if (a.group_units <= 0 || a.num_waves <= 0 || a.num_waves % a.group_units != 0) return hipErrorInvalidValue;
    blocks = a.num_waves / a.group_units;
  }
  if (blocks <= 0) return hipErrorInvalidValue;
  ScoreArgs part = a;
  for (int64_t first = 0; first < groups * a.subs; first += kMaxGridRows) {
    const dim3 grid((unsigned)blocks, (unsigned)std::min(kMaxGridRows, groups * a.subs - first));
    part.first_pass = (int32_t)first;
    hipError_t e;
    if (a.code_bytes != 0) e = launch_raw(part, doc, residual, nt, reducer, grid, stream);
    else if (a.chunks == 4) e = launch_wide4(part, doc, residual, nt, reducer, grid, stream);
    else if (a.chunks == 2) e = launch_wide2(part, doc, residual, nt, reducer, grid, stream);
    else if (doc == kDocInt4) e = launch_int4(part, residual, nt, reducer, grid, stream);
    else e = launch_sign(part, residual, nt, reducer, grid, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace msim
