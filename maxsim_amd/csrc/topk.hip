// topk.hip -- stand-alone block top-k: one workgroup per score row.  Order and
// the radix form: topk_block.hpp (reference order cu:1629-1692,
// _api.py:732-735); the threshold forms below.
#include <algorithm>

#include "common.hpp"
#include "internal.hpp"
#include "topk_block.hpp"

namespace msim {

constexpr int kTopkThreads = 1024;

__global__ __launch_bounds__(kTopkThreads) void topk_kernel(const float* __restrict__ scores,
                                                           int64_t n, int64_t row_stride, int32_t k,
                                                           const int64_t* __restrict__ id_map,
                                                           float* __restrict__ out_scores,
                                                           int64_t* __restrict__ out_ids) {
  __shared__ TopkSmem<kTopkThreads, kTopkMaxK> sm;
  const int64_t b = blockIdx.x;
  block_topk<kTopkThreads, 16, kTopkMaxK>(scores + b * row_stride, n, k,
                                          id_map ? id_map + b * n : nullptr, out_scores + b * k,
                                          out_ids + b * k, sm);
}

constexpr int kSmallTopkMaxK = 32;

// -------------------------------------------------------- row threshold
// k <= min(n, kTopkThreads), any n: one 1024-thread workgroup per row.  T =
// the k-th largest of the threads' maximum scores (order-preserving 32-bit
// integers), by radix rounds of eight bits over 1,024 values in LDS: k
// threads hold a score >= T, so every score of the row's top k is >= T, and
// only those threads and ties of T hold such scores (k to a few k of them,
// the threads' elements being spread over the row).  They are compacted into
// LDS as distinct 64-bit keys (score key above 2^32 - 1 - position: a larger
// key is a better element) and ranked by counting, or sorted when many.
// Per element that is four VALU instructions in each of the two passes (64-bit
// keys from the start took 22 us for 65,536 scores, one CU's VALU busy).
//
// What bounds it: one CU reads the row (twice when it is longer than the
// registers hold), so the time is the launch, one or two passes at what a CU
// draws from the caches, and about 2 us of selection.  The radix form reads
// the row once per digit, with two block scans and a histogram atomic per
// element: 224 us for 65,536 scores and k = 100, and k rounds of wave maxima
// took 23 us for 10,240 and k = 10 (kernel times); now 13 us in two launches
// and 5 us (event time over back-to-back launches 7.9 us).
//
// Longer rows are cut into chunks of about kRowChunk scores, a workgroup
// each, and the chunks' top k (in order, so that position order is still the
// order of ties) are selected from in the same way: one CU alone draws a
// 65,536-score row in about 10 us.
//
// GROUPS > 0: the row in registers (n <= 1024 * (VEC ? 4 : 1) * GROUPS);
// 0: streamed twice.  VEC: four consecutive elements per thread and load
// (16-byte buffer loads, which need dword alignment only).  gridDim.y = chunks:
// chunk y of row x is its elements [n y / chunks, n (y + 1) / chunks), its k
// best go to out[(x * chunks + y) * k ...].
constexpr int64_t kRowChunk = 8192;
constexpr int64_t kRowRegs = kTopkThreads * 16;  // a row of at most this stays in registers
constexpr int kRowCap = 4096;       // candidates at most; more fall back to the radix form
constexpr int kRowRankMax = 512;    // ranked by counting up to here, sorted beyond
template <int GROUPS, bool VEC>
__global__ __launch_bounds__(kTopkThreads) void topk_row_kernel(const float* __restrict__ scores, int64_t n_row,
                                                               int64_t row_stride, int32_t k,
                                                               const int64_t* __restrict__ id_map,
                                                               float* __restrict__ out_scores,
                                                               int64_t* __restrict__ out_ids) {
  constexpr int kWaves = kTopkThreads / kWave, kPer = VEC ? 4 : 1, kRounds = 4;
  constexpr int64_t kStep = (int64_t)kTopkThreads * kPer;
  static_assert(GROUPS == 0 || VEC || GROUPS <= 4, "row in registers");
  struct Select {
    uint32_t hist[kRounds][256];
    uint64_t key[kRowCap];
    uint32_t raw[kRowCap];
  };
  __shared__ union {
    Select s;
    TopkSmem<kTopkThreads, kTopkMaxK> radix;
  } sm;
  __shared__ uint32_t s_or[kWaves], s_and[kWaves];
  __shared__ uint32_t s_count;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int64_t b = blockIdx.x, chunk = blockIdx.y, chunks = gridDim.y;
  const int64_t first = n_row * chunk / chunks, n = n_row * (chunk + 1) / chunks - first;
  const float* row = scores + b * row_stride + first;
  // Group j of the row: elements j * kStep + tid * kPer + e of this thread.
  auto load = [&](int64_t j) -> v4u {
    const int64_t base = j * kStep;
    const __amdgpu_buffer_rsrc_t r = make_rsrc(row + base, (uint32_t)(min(max(n - base, (int64_t)0), kStep) * 4));
    if constexpr (VEC) return load_b128(r, tid * 16);
    else return (v4u){load_b32(r, tid * 4), 0u, 0u, 0u};
  };
  auto key_of = [&](uint32_t bits, int64_t i) -> uint64_t {
    return ((uint64_t)score_key(__uint_as_float(bits)) << 32) | (0xFFFFFFFFu - (uint32_t)i);
  };
  const int64_t groups = (n + kStep - 1) / kStep;
  v4u held[GROUPS > 0 ? GROUPS : 1];
  // f(group j, its bits), every group of the row; `again`: the second pass.
  auto each_group = [&](auto f, bool again) {
    if constexpr (GROUPS > 0) {
      if (!again) {
#pragma unroll
        for (int j = 0; j < GROUPS; ++j) held[j] = load(j);
      }
#pragma unroll
      for (int j = 0; j < GROUPS; ++j) f((int64_t)j, held[j]);
    } else {
      constexpr int kAhead = 4;
      for (int64_t j = 0; j < groups; j += kAhead) {
        v4u v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = load(j + u);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) f(j + u, v[u]);
      }
    }
  };
  for (int i = tid; i < kRounds * 256; i += kTopkThreads) (&sm.s.hist[0][0])[i] = 0u;
  if (tid == 0) s_count = 0;
  // Signed integers in the order of the scores (-0 directly below +0).
  auto ordered = [](uint32_t u) -> int { return (int)(u ^ (uint32_t)(((int)u >> 31) & 0x7FFFFFFF)); };
  int mine = INT32_MIN;
  each_group(
      [&](int64_t j, const v4u& v) {
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
          const int x = ordered(v[e]);
          // Positions past n (loads give 0 there) count as the lowest value.
          mine = max(mine, j * kStep + kStep <= n || j * kStep + tid * kPer + e < n ? x : INT32_MIN);
        }
      },
      false);
  // T's digits from the highest bit in which the threads' maxima differ.
  const uint32_t hi = (uint32_t)mine ^ 0x80000000u;
  const bool valid = tid * kPer < n;  // this thread holds an element
  const uint32_t wor = wave_reduce(valid ? hi : 0u, [](uint32_t x, uint32_t y) { return x | y; });
  const uint32_t wand = wave_reduce(valid ? hi : ~0u, [](uint32_t x, uint32_t y) { return x & y; });
  if (lane == 0) {
    s_or[wave] = wor;
    s_and[wave] = wand;
  }
  __syncthreads();
  uint32_t kor = 0u, kand = ~0u;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    kor |= s_or[w];
    kand &= s_and[w];
  }
  const uint32_t diff = kor ^ kand;
  int top = diff != 0u ? 31 - __clz((int)diff) : -1;
  uint32_t mask = top == 31 ? 0u : ~0u << (top + 1);
  uint32_t prefix = kand & mask;
  uint32_t need = (uint32_t)k;
  for (int r = 0; r < kRounds && top >= 0; ++r, top -= 8) {
    const int shift = top >= 7 ? top - 7 : 0;
    const uint32_t dbits = (2u << (top - shift)) - 1u;
    uint32_t* hist = sm.s.hist[r];
    if (valid && (hi & mask) == prefix) atomicAdd(&hist[255u - ((hi >> shift) & dbits)], 1u);
    __syncthreads();
    // Every wave finds the digit: bins 4 lane .. 4 lane + 3 (larger digits first).
    const v4u c = *reinterpret_cast<const v4u*>(&hist[4 * lane]);
    const uint32_t incl = wave_inclusive_scan(c[0] + c[1] + c[2] + c[3]);
    const int src = min((int)__builtin_ctzll(__ballot(incl >= need)), kWave - 1);
    uint32_t above = incl - (c[0] + c[1] + c[2] + c[3]), bin = 0, cnt = 0, over = 0;
    bool found = false;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const bool here = !found && above + c[x] >= need;
      bin = here ? (uint32_t)(4 * lane + x) : bin;
      cnt = here ? c[x] : cnt;
      over = here ? above : over;
      found = found || here;
      above += c[x];
    }
    bin = (uint32_t)__builtin_amdgcn_readlane((int)bin, src);
    cnt = (uint32_t)__builtin_amdgcn_readlane((int)cnt, src);
    over = (uint32_t)__builtin_amdgcn_readlane((int)over, src);
    prefix |= (255u - bin) << shift;
    mask |= dbits << shift;
    need -= over;
    if (cnt == need || shift == 0) break;
  }
  // Scores whose ordered value reaches T (the prefix, zeros below it); +0's
  // threshold takes -0 as well.
  int t = (int)(prefix ^ 0x80000000u);
  t = t == 0 ? -1 : t;
  each_group(
      [&](int64_t j, const v4u& v) {
        uint64_t m[kPer];
        uint32_t total = 0;
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
          m[e] = __ballot(ordered(v[e]) >= t && (j * kStep + kStep <= n || j * kStep + tid * kPer + e < n));
          total += (uint32_t)__popcll(m[e]);
        }
        if (total == 0) return;
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(&s_count, total);
        at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
          if ((m[e] >> lane) & 1ull) {
            const uint32_t slot = at + __builtin_amdgcn_mbcnt_hi((uint32_t)(m[e] >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)m[e], 0u));
            if (slot < (uint32_t)kRowCap) {
              sm.s.key[slot] = key_of(v[e], j * kStep + tid * kPer + e);
              sm.s.raw[slot] = v[e];
            }
          }
          at += (uint32_t)__popcll(m[e]);
        }
      },
      true);
  __syncthreads();
  const int c = (int)s_count;
  const int64_t* ids = id_map ? id_map + b * n_row + first : nullptr;
  float* os = out_scores + (b * chunks + chunk) * k;
  int64_t* oi = out_ids + (b * chunks + chunk) * k;
  if (c > kRowCap) {  // most of the best elements in a few threads, or tied with the k-th
    __syncthreads();
    block_topk<kTopkThreads, 16, kTopkMaxK>(row, n, k, ids, os, oi, sm.radix);
    if (ids == nullptr && first != 0) {
      for (int r = tid; r < k; r += kTopkThreads) oi[r] += first;
    }
    return;
  }
  auto write = [&](int r, uint64_t x, float v) {
    const int64_t pos = (int64_t)(0xFFFFFFFFu - (uint32_t)x);
    os[r] = v;
    oi[r] = ids ? ids[pos] : first + pos;
  };
  int padded = 8;
  if (c <= kRowRankMax) {
    padded = (c + 7) & ~7;
  } else {
    while (padded < c) padded <<= 1;
  }
  for (int i = c + tid; i < padded; i += kTopkThreads) sm.s.key[i] = 0u;
  __syncthreads();
  if (c <= kRowRankMax) {
    if (tid >= c) return;
    const uint64_t x = sm.s.key[tid];
    int r = 0;
    for (int j = 0; j < padded; j += 8) {
      uint64_t y[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) y[u] = sm.s.key[j + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) r += y[u] > x ? 1 : 0;
    }
    if (r < k) write(r, x, __uint_as_float(sm.s.raw[tid]));
    return;
  }
  // Descending bitonic sort; the scores are read again by position.
  for (int size = 2; size <= padded; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = tid; i < padded / 2; i += kTopkThreads) {
        const int lo = 2 * i - (i & (stride - 1)), hi2 = lo + stride;
        const uint64_t x = sm.s.key[lo], y = sm.s.key[hi2];
        if ((x < y) == ((lo & size) == 0)) {
          sm.s.key[lo] = y;
          sm.s.key[hi2] = x;
        }
      }
      __syncthreads();
    }
  }
  for (int r = tid; r < k; r += kTopkThreads) {
    const uint64_t x = sm.s.key[r];
    write(r, x, row[(int64_t)(0xFFFFFFFFu - (uint32_t)x)]);
  }
}

// ------------------------------------------------------ threshold filter
// k <= kSmallTopkMaxK and n <= kFilterThreads * EPT: four waves, element i of
// the row in thread i % 256 (coalesced loads; the id map, when given, loaded
// beside the scores).  Keys are 64-bit, order-preserving score bits above
// 2^32 - 1 - position, so every key is distinct and a larger key is a higher
// score or, on a tie, a lower position.  In each wave, T_w = the k-th largest
// of the 64 lanes' maximum keys (a radix selection by ballot counts, no
// shuffles): k lanes of the wave hold a key >= T_w, so every key of the row's
// top k is >= T = max_w T_w.  At most k lanes per wave have a maximum >= T,
// so at most 4 * k * EPT keys pass the filter; they go to a list in LDS
// (one atomic per wave for its range, ballot offsets inside it) with their
// float bits and ids, and each one's rank is counted against the list.
// kCap is a multiple of eight.  The key of rank r < k is written to slot r.
constexpr int kFilterThreads = 256;
constexpr int kFilterWaves = kFilterThreads / kWave;

// The k-th largest of the wave's nonzero keys (wave-uniform), 0 when fewer
// than k lanes hold one.  The low 32 bits of every nonzero key are >= 2^32 -
// 4096 (positions below 4096), so those 20 bits of the result need no step.
__device__ __forceinline__ uint64_t wave_kth_largest_key(uint64_t x, int k) {
  if (__popcll(__ballot(x != 0)) < k) return 0;
  uint64_t t = 0;
#pragma unroll
  for (int bit = 63; bit >= 32; --bit) {
    const uint64_t c = t | (1ull << bit);
    t = __popcll(__ballot(x >= c)) >= k ? c : t;
  }
  t |= 0xFFFFF000ull;
#pragma unroll
  for (int bit = 11; bit >= 0; --bit) {
    const uint64_t c = t | (1ull << bit);
    t = __popcll(__ballot(x >= c)) >= k ? c : t;
  }
  return t;
}

template <int EPT>
__global__ __launch_bounds__(kFilterThreads) void topk_filter_kernel(const float* __restrict__ scores, int64_t n,
                                                                     int64_t row_stride, int32_t k,
                                                                     const int64_t* __restrict__ id_map,
                                                                     float* __restrict__ out_scores,
                                                                     int64_t* __restrict__ out_ids) {
  constexpr int kCap = kFilterWaves * kSmallTopkMaxK * EPT;
  static_assert(kCap % 8 == 0, "rank steps of eight keys");
  __shared__ uint64_t s_key[kCap];
  __shared__ int64_t s_id[kCap];
  __shared__ uint32_t s_raw[kCap];
  __shared__ uint64_t s_thr[kFilterWaves];
  __shared__ uint32_t s_count;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int64_t b = blockIdx.x;
  const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(scores + b * row_stride, (uint32_t)(n * 4));
  const __amdgpu_buffer_rsrc_t rid = make_rsrc(id_map ? id_map + b * n : nullptr, id_map ? (uint32_t)(n * 8) : 0u);
  uint32_t v[EPT];
  int64_t id[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) v[e] = load_b32(rsrc, (e * kFilterThreads + tid) * 4);
  if (id_map) {
#pragma unroll
    for (int e = 0; e < EPT; ++e) id[e] = (int64_t)load_b64(rid, (e * kFilterThreads + tid) * 8);
  }
  if (tid == 0) s_count = 0;
  for (int i = tid; i < kCap; i += kFilterThreads) s_key[i] = 0u;
  uint64_t key[EPT], lmax = 0;
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const int i = e * kFilterThreads + tid;
    key[e] = i < n ? ((uint64_t)score_key(__uint_as_float(v[e])) << 32) | (0xFFFFFFFFu - (uint32_t)i) : 0u;
    lmax = key[e] > lmax ? key[e] : lmax;
  }
  const uint64_t tw = wave_kth_largest_key(lmax, k);
  if (lane == 0) s_thr[wave] = tw;
  __syncthreads();
  uint64_t t = 0;
#pragma unroll
  for (int w = 0; w < kFilterWaves; ++w) t = s_thr[w] > t ? s_thr[w] : t;
  uint64_t mask[EPT];
  uint32_t cnt = 0;
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    mask[e] = __ballot(key[e] != 0 && key[e] >= t);
    cnt += (uint32_t)__popcll(mask[e]);
  }
  uint32_t base = 0;
  if (lane == 0 && cnt != 0) base = atomicAdd(&s_count, cnt);
  base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    if ((mask[e] >> lane) & 1ull) {
      const uint32_t at =
          base + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask[e] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask[e], 0u));
      s_key[at] = key[e];
      s_raw[at] = v[e];
      if (id_map) s_id[at] = id[e];
    }
    base += (uint32_t)__popcll(mask[e]);
  }
  __syncthreads();
  // Ranks, counted against the whole list (broadcast LDS reads, eight keys
  // per step; the zeroed tail pads the list to a multiple of eight).
  const int c = (int)s_count, c8 = (c + 7) & ~7;
  for (int i = tid; i < c; i += kFilterThreads) {
    const uint64_t x = s_key[i];
    int r = 0;
    for (int j = 0; j < c8; j += 8) {
      uint64_t y[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) y[u] = s_key[j + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) r += y[u] > x ? 1 : 0;
    }
    if (r < k) {
      out_scores[b * k + r] = __uint_as_float(s_raw[i]);
      out_ids[b * k + r] = id_map ? s_id[i] : (int64_t)(0xFFFFFFFFu - (uint32_t)x);
    }
  }
}

namespace {

// Chunks a row of n scores is cut into (1: none): rows longer than a
// workgroup's registers, when the chunks' k best are at most half of it.
int64_t topk_chunks(int64_t n, int64_t k) {
  if (n <= kRowRegs || k > kTopkThreads) return 1;
  const int64_t chunks = (n + kRowChunk - 1) / kRowChunk;
  return chunks * k * 2 <= n ? std::min<int64_t>(chunks, 65535) : 1;
}

void launch_row(const float* d_scores, int64_t batch, int64_t n, int64_t row_stride, int64_t k, int64_t chunks,
                const int64_t* d_id_map, float* d_out_scores, int64_t* d_out_ids, hipStream_t stream) {
  const dim3 grid((unsigned)batch, (unsigned)chunks), block(kTopkThreads);
  const int64_t len = (n + chunks - 1) / chunks;  // the longest chunk
  // A thread needs an element for its maximum to count: one element per
  // thread and group up to 4,096.
  if (len <= kTopkThreads * 4 && chunks == 1)
    topk_row_kernel<4, false><<<grid, block, 0, stream>>>(d_scores, n, row_stride, (int32_t)k, d_id_map, d_out_scores,
                                                          d_out_ids);
  else if (len <= kRowRegs)
    topk_row_kernel<4, true><<<grid, block, 0, stream>>>(d_scores, n, row_stride, (int32_t)k, d_id_map, d_out_scores,
                                                         d_out_ids);
  else
    topk_row_kernel<0, true><<<grid, block, 0, stream>>>(d_scores, n, row_stride, (int32_t)k, d_id_map, d_out_scores,
                                                         d_out_ids);
}

}  // namespace

size_t topk_scratch_bytes(int64_t batch, int64_t n, int64_t k) {
  size_t bytes = 0;
  for (int64_t chunks = topk_chunks(n, k); chunks > 1; n = chunks * k, chunks = topk_chunks(n, k))
    bytes += (size_t)(batch * chunks * k) * (sizeof(float) + sizeof(int64_t)) + 8;
  return bytes;
}

hipError_t launch_topk(const float* d_scores, int64_t batch, int64_t n, int64_t row_stride,
                       int64_t k, const int64_t* d_id_map, float* d_out_scores,
                       int64_t* d_out_ids, hipStream_t stream, void* scratch) {
  if (batch == 0 || k == 0) return hipSuccess;
  if (k > kTopkMaxK || k > n) return hipErrorInvalidValue;
  // Long rows, chunk by chunk: each level's candidates (ids, then scores) in
  // the scratch memory.
  char* free_scratch = reinterpret_cast<char*>(scratch);
  for (int64_t chunks = scratch ? topk_chunks(n, k) : 1; chunks > 1; chunks = topk_chunks(n, k)) {
    const int64_t count = batch * chunks * k;
    int64_t* ids = reinterpret_cast<int64_t*>(free_scratch);
    float* best = reinterpret_cast<float*>(ids + count);
    free_scratch += (sizeof(int64_t) + sizeof(float)) * (size_t)count;
    free_scratch += (8 - (uintptr_t)free_scratch % 8) % 8;
    launch_row(d_scores, batch, n, row_stride, k, chunks, d_id_map, best, ids, stream);
    d_scores = best;
    d_id_map = ids;
    n = row_stride = chunks * k;
  }
  if (k <= kSmallTopkMaxK && n <= kFilterThreads * 16) {
    const dim3 grid((unsigned)batch), block(kFilterThreads);
    if (n <= kFilterThreads * 2)
      topk_filter_kernel<2><<<grid, block, 0, stream>>>(d_scores, n, row_stride, (int32_t)k, d_id_map, d_out_scores,
                                                        d_out_ids);
    else if (n <= kFilterThreads * 4)
      topk_filter_kernel<4><<<grid, block, 0, stream>>>(d_scores, n, row_stride, (int32_t)k, d_id_map, d_out_scores,
                                                        d_out_ids);
    else if (n <= kFilterThreads * 8)
      topk_filter_kernel<8><<<grid, block, 0, stream>>>(d_scores, n, row_stride, (int32_t)k, d_id_map, d_out_scores,
                                                        d_out_ids);
    else
      topk_filter_kernel<16><<<grid, block, 0, stream>>>(d_scores, n, row_stride, (int32_t)k, d_id_map, d_out_scores,
                                                         d_out_ids);
  } else if (k <= kTopkThreads) {
    launch_row(d_scores, batch, n, row_stride, k, 1, d_id_map, d_out_scores, d_out_ids, stream);
  } else {
    topk_kernel<<<dim3((unsigned)batch), dim3(kTopkThreads), 0, stream>>>(
        d_scores, n, row_stride, (int32_t)k, d_id_map, d_out_scores, d_out_ids);
  }
  return hipGetLastError();
}

}  // namespace msim
