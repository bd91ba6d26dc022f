// score.hip -- int8-query and sign-bit-query MaxSim over sign-bit documents
// (optionally with an int4 residual stream) on gfx950 MFMA, over every
// document or per-row candidates.  fp32 queries, the other reducers and int4
// documents: digit_score.hip.
//
// Semantics restated from the reference:
//  * MaxSim: cu:477-653, CPU closed form _api.py:558-585; an empty document
//    scores 0; the document scale is applied after the reduction;
//  * residual fused similarity p s^p_t (q . v^p_t) + r s^r_t (q . v^r_t) reduced
//    once (cu:967-1266, cascade.py:272-291);
//  * sign documents: q . sign(d_t) times the token scale (cu:297-352), the
//    int8-query form 2 (q8 . bits) - sum(q8) (cu:1368-1447).
//
// Design (MI355X): the dot products run on v_mfma_i32_16x16x64_i8 (exact int32
// dots of the int8 query).
//
// Work split: a wave owns a range of targets (documents, or candidate
// positions) and walks their 16-token tiles from a table (or, in direct
// mode, one candidate per wave, the tiles of its document's token range); a
// tile is the MFMA A operand (16 tokens x 128 dims), the query rows of the pass
// are B operands held in registers.  Each lane keeps the running maximum of
// its query column over its four token rows; at a target's last tile the
// four lane groups are merged and the per-row pooled values are summed over
// each batch row's query tokens, or written to pooled[target][row] for
// pool_sum_kernel.
#include <algorithm>

#include "common.hpp"
#include "internal.hpp"
#include "score_reduce.hpp"

namespace msim {

namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerGroup = kThreads / kWave;

// A operands (two MFMAs of 64 dims) from the tile bytes of one chunk.
__device__ __forceinline__ void unpack_a(const v4u& w, v4i& a0, v4i& a1) {
  // Nibbles moved to the high half of each byte: the int8 value is 16 v.
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    a0[x] = (int)((w[x] << 4) & 0xF0F0F0F0u);  // even dims
    a1[x] = (int)(w[x] & 0xF0F0F0F0u);         // odd dims
  }
}
__device__ __forceinline__ void unpack_a(unsigned w, v4i& a0, v4i& a1) {
  // Dword i holds bits i, i + 8, i + 16, i + 24 as bytes 0/1 (dims 32g + 8j + i).
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a0[i] = (int)((w >> i) & 0x01010101u);
    a1[i] = (int)((w >> (i + 4)) & 0x01010101u);
  }
}
// Sign bits in the int4 lane order (a0: even dims, a1: odd dims), for a sign
// stream that shares its query operands with an int4 stream.  Bits 0, 2, 4, 6
// of a byte move to bits 0, 8, 16, 24 by one multiply with 0x41041 (shifts
// 0, 6, 12, 18): the partial products overlap only at bits 6, 12 and 18,
// whose carries stop at bits 7, 13 and 19, away from the kept bits.
__device__ __forceinline__ void unpack_a_int4_order(unsigned w, v4i& a0, v4i& a1) {
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const unsigned b = w >> (8 * x);
    a0[x] = (int)(((b & 0x55u) * 0x41041u) & 0x01010101u);
    a1[x] = (int)((((b >> 1) & 0x55u) * 0x41041u) & 0x01010101u);
  }
}

// INTMAX (no residual, no token scale): the +-1 dot 2 (q8 . bits) - sum(q8) is
// increasing in the MFMA result, so the running maximum is kept on the int32
// accumulators and converted once per document.
template <bool RES, int NT, bool INTMAX>
__global__ __launch_bounds__(kThreads, NT == 8 ? 2 : 1) void score_kernel(ScoreArgs p) {
  static_assert(!INTMAX || !RES, "integer maximum form");
  constexpr int kCodeBytes = 16, kResBytes = 64, kQueryBytes = 128;  // per token and per query row
  __shared__ float s_pool[kWavesPerGroup][16 * NT];
  const int lane = lane_id();
  const int wave = wave_uniform(threadIdx.x / kWave);
  const int g = lane >> 4, c = lane & 15;
  const int pass = (int)blockIdx.y + p.first_pass, grp = pass / p.subs, sub = pass % p.subs;
  const int64_t gw = (int64_t)blockIdx.x * kWavesPerGroup + wave;
  const auto targets = p.targets ? as_constant(p.targets) + grp * p.targets_grp_stride : nullptr;
  const int lr0 = sub * 16 * NT;                           // first local row of the pass
  const int64_t grow0 = (int64_t)grp * p.grp_rows + lr0;  // its global query row

  // Table mode: the wave's first target, tile count and tiles from the
  // tables.  Direct mode: target gw of the group, its tiles from the token
  // range of its document.
  const bool direct = p.direct_offsets != nullptr;
  int64_t t0, ds = 0, de = 0;
  int ntiles;
  const __attribute__((address_space(4))) uint64_t* tt = nullptr;
  if (direct) {
    if (gw >= p.direct_count) return;  // no barriers below: a wave may leave early
    t0 = gw;
    const int64_t doc = targets[gw];
    ds = as_constant(p.direct_offsets)[doc];
    de = as_constant(p.direct_offsets)[doc + 1];
    ntiles = ds == de ? 1 : (int)((de - ds + 15) / 16);
  } else {
    if (gw >= p.num_waves) return;  // the last workgroup's waves past the table
    const auto info = as_constant(p.wave_info) + grp * p.info_grp_stride + gw * kScoreInfoWords;
    t0 = info[0];
    ntiles = (int)info[2];
    if (ntiles == 0) return;
    tt = as_constant(p.tiles) + info[3];
  }
  // Tile i of the wave's table (i >= ntiles: a padding entry at token 0).
  auto entry = [&](int i) -> uint64_t { return i < ntiles ? tt[i] : score_tile_entry(0, 1, false, false, 0); };
  const auto doc_scale = p.doc_scale ? as_constant(p.doc_scale) : nullptr;

  // Query B operands and per-column constants.
  v4i bq[NT][2];
  float colmul[NT];
  int qsum[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int64_t r = grow0 + 16 * j + c;
    const v4i* src = reinterpret_cast<const v4i*>(p.qpack + r * kQueryBytes + 32 * g);
    bq[j][0] = src[0];
    bq[j][1] = src[1];
    qsum[j] = p.qsum[r];
    colmul[j] = p.colmul[r];
  }

  float mx[NT];
  int imax[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    mx[j] = kNegInf;
    imax[j] = INT32_MIN;
  }

  // One tile as loaded: lane (g, c) holds token c's bytes of lane group g and
  // the scales of token rows 4g .. 4g + 3.
  struct Tile {
    uint64_t e;  // its table entry (table mode)
    unsigned a;  // 32 sign bits: dims 32g .. + 31
    v4u r;       // 16 bytes: the same dims as nibbles
    float s[4], sr[4];
  };
  // Every load is unconditional: rows past a short document read its last
  // token again (masked below); table padding entries point at token 0.
  auto load = [&](uint64_t e, Tile& t) {
    t.e = e;
    const int64_t start = (int64_t)(e & kTileStartMask);
    const int rows1 = (int)((e >> kTileRowsShift) & 15);
    const int64_t tok = start + min(c, rows1);
    t.a = *reinterpret_cast<const unsigned*>(p.codes + tok * kCodeBytes + 4 * g);
    if constexpr (RES) t.r = *reinterpret_cast<const v4u*>(p.rcodes + tok * kResBytes + 16 * g);
    if constexpr (!INTMAX) {
      // Token rows 4g .. 4g + 3 in one load; rows past the tile read 0
      // (buffer bounds at the tile's last row; they are masked below).
      const uint32_t nbytes = (uint32_t)(rows1 + 1) * 4u;
      const v4u sv = load_b128(make_rsrc(p.tscale + start, nbytes), 16 * g);
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) t.s[rr] = __uint_as_float(sv[rr]);
      if constexpr (RES) {
        const v4u rv = load_b128(make_rsrc(p.rtscale + start, nbytes), 16 * g);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) t.sr[rr] = __uint_as_float(rv[rr]);
      }
    }
  };

  int len = 0;  // tokens of the current target seen so far (wave-uniform)
  float dscale = 1.0f;
  bool fresh = true;

  // Accumulators of one tile, and what its epilogue needs once its ring slot
  // is reused.
  struct Acc {
    v4i s[NT];
    v4i r[RES ? NT : 1];
  };
  struct Pend {
    uint64_t e;
    float s[4], sr[4];
  };
  auto pend_of = [&](const Tile& t) {
    Pend q;
    q.e = t.e;
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      q.s[rr] = t.s[rr];
      q.sr[rr] = RES ? t.sr[rr] : 0.0f;
    }
    return q;
  };
  struct Ops {
    v4i a0, a1, r0, r1;
  };
  auto unpack = [&](const Tile& t) {
    Ops o;
    if constexpr (RES) unpack_a_int4_order(t.a, o.a0, o.a1);
    else unpack_a(t.a, o.a0, o.a1);
    if constexpr (RES) unpack_a(t.r, o.r0, o.r1);
    return o;
  };
  // MFMAs of K half h of row block j (h = 0 starts from zero).
  auto mfma_half = [&](Acc& A, const Ops& o, int h, int j) __attribute__((always_inline)) {
    const v4i zero = {0, 0, 0, 0};
    A.s[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(h ? o.a1 : o.a0, bq[j][h], h ? A.s[j] : zero, 0, 0, 0);
    if constexpr (RES)
      A.r[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(h ? o.r1 : o.r0, bq[j][h], h ? A.r[j] : zero, 0, 0, 0);
  };
  // Start of a tile's epilogue: its row count, and the document's scale when
  // it is its target's first tile.
  auto begin_tile = [&](const Pend& P) __attribute__((always_inline)) {
    const uint64_t e = P.e;
    if (fresh) {
      const int64_t tg = t0 + (int)(e >> kTileLocalShift);
      const int64_t doc = targets ? targets[tg] : tg;
      dscale = doc_scale ? doc_scale[doc] : p.scale;
    }
    return ((e >> kTileEmptyShift) & 1) ? 0 : (int)((e >> kTileRowsShift) & 15) + 1;
  };
  // Epilogue of row block j of a tile.  The +-1 dot 2 (q8 . bits) - sum(q8) is
  // one fma on the converted accumulator (every term an integer below 2^24:
  // exact).
  auto epi_j = [&](const Acc& A, const Pend& P, int rows, int j) __attribute__((always_inline)) {
    if constexpr (INTMAX) {
      v4i a = A.s[j];
      if (rows < 16) {
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          if (4 * g + rr >= rows) a[rr] = INT32_MIN;
      }
      imax[j] = max(max(imax[j], max(a[0], a[1])), max(a[2], a[3]));
    } else {
      float z[4];
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const float y = fmaf((float)A.s[j][rr], 2.0f, (float)-qsum[j]);
        z[rr] = y * (P.s[rr] * p.tmul);
        if constexpr (RES) z[rr] = z[rr] + (float)A.r[j][rr] * (P.sr[rr] * p.rmul);
      }
      if (rows < 16) {
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          if (4 * g + rr >= rows) z[rr] = kNegInf;
      }
      // Two three-way maxima (v_max3_f32) for four values: exact, any order.
      mx[j] = max3_op(max3_op(mx[j], z[0], z[1]), z[2], z[3]);
    }
  };
  // Score of target tg from the maxima over its `len` tokens.
  auto finish_target = [&](int64_t tg) __attribute__((always_inline)) {
    float v[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if constexpr (INTMAX) {
        int m = max(imax[j], __shfl_xor(imax[j], 16));
        m = max(m, __shfl_xor(m, 32));
        v[j] = len == 0 ? 0.0f : (float)(2 * m - qsum[j]) * colmul[j] * dscale;
        imax[j] = INT32_MIN;
      } else {
        float m = fmaxf(mx[j], __shfl_xor(mx[j], 16));
        m = fmaxf(m, __shfl_xor(m, 32));
        v[j] = len == 0 ? 0.0f : m * colmul[j] * dscale;
        mx[j] = kNegInf;
      }
    }
    if (p.out || p.iout) {
      // Whole batch rows in this pass: sum each row's query tokens here and
      // write the score.
      if (g == 0) {
#pragma unroll
        for (int j = 0; j < NT; ++j) s_pool[wave][16 * j + c] = v[j];
      }
      wave_sync_lds();
      const int nb = min(16 * NT, p.grp_rows - lr0) / p.query_tokens;
      const int64_t b0 = grow0 / p.query_tokens;
      sum_batch_rows(s_pool[wave], nb, p.query_tokens, [&](int b, float sum) {
        if (p.out) p.out[(b0 + b) * p.out_stride + tg] = sum;
        if (p.iout) p.iout[(b0 + b) * p.iout_stride + tg] = (int32_t)sum;
      });
      wave_sync_lds();
    } else {
      float* out = p.pooled + grp * p.pooled_grp_stride + tg * p.grp_rows;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int lr = lr0 + 16 * j + c;
        if (g == 0 && lr < p.grp_rows) out[lr] = v[j];
      }
    }
    len = 0;
  };
  // End of a tile's epilogue: at its target's last tile, the target's score.
  auto end_tile = [&](const Pend& P, int rows) __attribute__((always_inline)) {
    const uint64_t e = P.e;
    const bool last = ((e >> kTileLastShift) & 1) != 0;
    len += rows;
    if (last) finish_target(t0 + (int)(e >> kTileLocalShift));
    fresh = last;
  };
  // The epilogue of a tile whose MFMAs were issued just before.
  auto consume_now = [&](const Acc& A, const Pend& P, int rows) __attribute__((always_inline)) {
    mfma_results_fence();
#pragma unroll
    for (int j = 0; j < NT; ++j) epi_j(A, P, rows, j);
  };
  // Pipelined form: the MFMAs of tile q, the epilogue of the previous tile p
  // (its accumulators a whole tile old) interleaved with q's second halves.
  auto issue_consume = [&](Acc& Q, const Tile& tq, const Acc& A, const Pend& P, int rows)
                           __attribute__((always_inline)) {
    const Ops o = unpack(tq);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NT; ++j) mfma_half(Q, o, 0, j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      mfma_half(Q, o, 1, j);
      epi_j(A, P, rows, j);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // All MFMAs of a tile: the sign stream's halves, then the residual's (its
  // operands unpacked only then, so fewer registers are live).
  auto issue = [&](Acc& Q, const Tile& tq) __attribute__((always_inline)) {
    const v4i zero = {0, 0, 0, 0};
    v4i a0, a1;
    if constexpr (RES) unpack_a_int4_order(tq.a, a0, a1);
    else unpack_a(tq.a, a0, a1);
#pragma unroll
    for (int j = 0; j < NT; ++j) Q.s[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, bq[j][0], zero, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < NT; ++j) Q.s[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, bq[j][1], Q.s[j], 0, 0, 0);
    if constexpr (RES) {
      v4i r0, r1;
      unpack_a(tq.r, r0, r1);
#pragma unroll
      for (int j = 0; j < NT; ++j) Q.r[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(r0, bq[j][0], zero, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NT; ++j) Q.r[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(r1, bq[j][1], Q.r[j], 0, 0, 0);
    }
  };

  // Two-block passes (candidate rescoring: few waves per SIMD, short
  // documents): a ring of kAhead + 1 tiles, tile i in slot i % (kAhead + 1),
  // the loads of tile i + kAhead issued before tile i is computed; each
  // tile's epilogue interleaved with the next tile's MFMAs (two accumulator
  // sets).  fetch(i, Tile&) issues tile i's loads (i >= n allowed), meta(i,
  // Pend&) returns its row count after starting its epilogue, done(Pend&,
  // rows) ends it.
  constexpr int kAhead = 3;
  static_assert((kAhead + 1) % 2 == 0, "tiles alternate between two accumulator sets");
  auto run_ring = [&](int n, auto fetch, auto meta, auto done) __attribute__((always_inline)) {
    Tile ring[kAhead + 1];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) fetch(u, ring[u]);
    Acc acc[2];
    Pend pend[2];
    fetch(kAhead, ring[kAhead]);
    issue(acc[0], ring[0]);
    pend[0] = pend_of(ring[0]);
    int rows_p = meta(0, pend[0]);
    // Tile i (i >= 1) is in slot (u + 1) % (kAhead + 1) and set (u + 1) % 2;
    // its loads reuse the slot of tile i - 1, whose epilogue data is in pend.
    for (int i0 = 1; i0 < n; i0 += kAhead + 1) {
#pragma unroll
      for (int u = 0; u <= kAhead; ++u) {
        if (i0 + u >= n) break;
        const int sl = (u + 1) % (kAhead + 1), so = u % (kAhead + 1);
        const int sq = (u + 1) % 2, sp = u % 2;
        fetch(i0 + u + kAhead, ring[so]);
        pend[sq] = pend_of(ring[sl]);
        issue_consume(acc[sq], ring[sl], acc[sp], pend[sp], rows_p);
        done(pend[sp], rows_p);
        rows_p = meta(i0 + u, pend[sq]);
      }
    }
    if ((n - 1) % 2 == 0) {
      consume_now(acc[0], pend[0], rows_p);
      done(pend[0], rows_p);
    } else {
      consume_now(acc[1], pend[1], rows_p);
      done(pend[1], rows_p);
    }
  };

  // One document per wave (tokens [ds, de)): one buffer per stream over the
  // document, a tile's loads at offsets from it (rows past the end read 0
  // and are masked), the document's scale once before its tiles and its
  // score once after them.
  auto run_direct = [&](auto run) __attribute__((always_inline)) {
    const int ntok = (int)(de - ds);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.codes + ds * kCodeBytes, (uint32_t)ntok * kCodeBytes);
    const __amdgpu_buffer_rsrc_t rr =
        make_rsrc(RES ? p.rcodes + ds * kResBytes : p.codes, RES ? (uint32_t)ntok * (uint32_t)kResBytes : 0u);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.tscale + ds, (uint32_t)ntok * 4u);
    const __amdgpu_buffer_rsrc_t rsr = make_rsrc(RES ? p.rtscale + ds : p.tscale, RES ? (uint32_t)ntok * 4u : 0u);
    dscale = doc_scale ? doc_scale[targets[gw]] : p.scale;
    auto fetch = [&](int i, Tile& t) __attribute__((always_inline)) {
      t.e = 0;
      const int row = 16 * i + c;
      t.a = load_b32(ra, row * kCodeBytes + 4 * g);
      if constexpr (RES) t.r = load_b128(rr, row * kResBytes + 16 * g);
      if constexpr (!INTMAX) {
        const v4u sv = load_b128(rs, (16 * i + 4 * g) * 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) t.s[q] = __uint_as_float(sv[q]);
        if constexpr (RES) {
          const v4u rv = load_b128(rsr, (16 * i + 4 * g) * 4);
#pragma unroll
          for (int q = 0; q < 4; ++q) t.sr[q] = __uint_as_float(rv[q]);
        }
      }
    };
    auto meta = [&](int i, Pend&) { return max(0, min(16, ntok - 16 * i)); };
    auto done = [&](Pend&, int) {};
    run(ntiles, fetch, meta, done);
    len = ntok;
    finish_target(t0);
  };

  if constexpr (NT > 2) {
    // Eight row blocks: a tight loop, one tile in flight, each tile's epilogue
    // behind the fence.
    auto run_plain = [&](int n, auto fetch, auto meta, auto done) __attribute__((always_inline)) {
      Tile cur, nxt;
      fetch(0, cur);
      for (int i = 0; i < n; ++i) {
        fetch(i + 1, nxt);
        Acc a;
        issue(a, cur);
        Pend P = pend_of(cur);
        const int rows = meta(i, P);
        consume_now(a, P, rows);
        done(P, rows);
        cur = nxt;
      }
    };
    if (direct) {
      run_direct(run_plain);
    } else {
      auto fetch = [&](int i, Tile& t) __attribute__((always_inline)) { load(entry(i), t); };
      auto meta = [&](int, Pend& P) { return begin_tile(P); };
      run_plain(ntiles, fetch, meta, end_tile);
    }
  } else if (direct) {
    run_direct(run_ring);
  } else {
    auto fetch = [&](int i, Tile& t) __attribute__((always_inline)) { load(entry(i), t); };
    auto meta = [&](int, Pend& P) { return begin_tile(P); };
    run_ring(ntiles, fetch, meta, end_tile);
  }
}

// ------------------------------------------------------------ quantisation

// Byte position of dim d in a 128-byte query row for the MFMA B operands.
// int4 documents: lane group g = d / 32 holds the even dims of its 32 in
// bytes [32g, 32g + 16) and the odd dims in [32g + 16, 32g + 32) (the order
// of the low / high nibbles).  Sign documents: byte 32g + 16 (i / 4) +
// 4 (i % 4) + j holds dim 32g + 8j + i (the order of the unpacked bits).
__device__ __forceinline__ int query_byte(int d, int layout) {
  const int g = d >> 5, e = d & 31;
  if (layout == kDocInt4) return 32 * g + (e & 1) * 16 + (e >> 1);
  const int j = e >> 3, i = e & 7;
  return 32 * g + 16 * (i >> 2) + 4 * (i & 3) + j;
}

// One wave per query row of 128 dims (lane l holds dims 2l, 2l + 1).  sigma =
// f32(max|q| / 127) (0 -> 1), code = clip(rint(q / sigma), -127, 127); with
// `recip` the quotient is q * (1 / sigma), the binary int8 query rounding of
// cu:1328-1366.  colmul = sigma; qsum = sum of the codes.  With qpack2, the
// same codes also in layout2 (a cascade's two passes).
__global__ __launch_bounds__(256) void quantize_limbs_kernel(const float* __restrict__ query, int64_t rows,
                                                             int64_t rows_padded, int layout, int recip,
                                                             int8_t* __restrict__ qpack,
                                                             float* __restrict__ colmul,
                                                             int32_t* __restrict__ qsum, int layout2,
                                                             int8_t* __restrict__ qpack2) {
  const int lane = lane_id();
  const int64_t row = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (row >= rows_padded) return;
  const int d0 = 2 * lane, d1 = 2 * lane + 1;
  int8_t* dst = qpack + row * 128;
  int8_t* dst2 = qpack2 ? qpack2 + row * 128 : nullptr;
  auto put = [&](int a, int b) {
    dst[query_byte(d0, layout)] = (int8_t)a;
    dst[query_byte(d1, layout)] = (int8_t)b;
    if (dst2) {
      dst2[query_byte(d0, layout2)] = (int8_t)a;
      dst2[query_byte(d1, layout2)] = (int8_t)b;
    }
  };
  if (row >= rows) {
    put(0, 0);
    if (lane == 0) {
      qsum[row] = 0;
      colmul[row] = 0.0f;
    }
    return;
  }
  const float2 v = reinterpret_cast<const float2*>(query + row * 128)[lane];
  const float m = wave_reduce(fmaxf(fabsf(v.x), fabsf(v.y)), [](float x, float y) { return fmaxf(x, y); });
  const float sigma = m == 0.0f ? 1.0f : __fdiv_rn(m, 127.0f);
  const float inv = recip ? __fdiv_rn(1.0f, sigma) : 0.0f;
  const float qx = recip ? v.x * inv : __fdiv_rn(v.x, sigma);
  const float qy = recip ? v.y * inv : __fdiv_rn(v.y, sigma);
  const int a = max(-127, min(127, (int)rintf(qx)));
  const int b = max(-127, min(127, (int)rintf(qy)));
  put(a, b);
  const int sum = wave_reduce(a + b, [](int x, int y) { return x + y; });
  if (lane == 0) {
    qsum[row] = sum;
    colmul[row] = sigma;
  }
}

// Sign-binarised query rows (pack_signs bit order, 16 bytes per row) as
// +-1 int8 codes in the sign-document layout; colmul = 1.
__global__ __launch_bounds__(256) void quantize_bits_kernel(const uint8_t* __restrict__ qbits, int64_t rows,
                                                            int64_t rows_padded, int8_t* __restrict__ qpack,
                                                            float* __restrict__ colmul,
                                                            int32_t* __restrict__ qsum) {
  const int lane = lane_id();
  const int64_t row = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (row >= rows_padded) return;
  const int d0 = 2 * lane, d1 = 2 * lane + 1;
  int8_t* dst = qpack + row * 128;
  int a = 0, b = 0;
  if (row < rows) {
    const unsigned byte = qbits[row * 16 + (d0 >> 3)];
    a = ((byte >> (d0 & 7)) & 1) ? 1 : -1;
    b = ((byte >> (d1 & 7)) & 1) ? 1 : -1;
  }
  dst[query_byte(d0, kDocSign)] = (int8_t)a;
  dst[query_byte(d1, kDocSign)] = (int8_t)b;
  const int sum = wave_reduce(a + b, [](int x, int y) { return x + y; });
  if (lane == 0) {
    qsum[row] = sum;
    colmul[row] = row < rows ? 1.0f : 0.0f;
  }
}

// out[b, t] = sum over q < Q of pooled[b * bs + t * ts + q], in token_sum16's
// order: sixteen lanes per output (a chain of one lane per output waited for
// its loads one by one: 5 us for 24 tokens and 4,000 outputs).
__global__ __launch_bounds__(256) void pool_sum_kernel(const float* __restrict__ pooled, int64_t batch,
                                                       int64_t query_tokens, int64_t targets, int64_t bs,
                                                       int64_t ts, float* __restrict__ out, int64_t out_stride,
                                                       int32_t* __restrict__ iout, int64_t iout_stride) {
  for (int64_t idx = (int64_t)blockIdx.x * (blockDim.x / 16) + threadIdx.x / 16; idx < batch * targets;
       idx += (int64_t)gridDim.x * (blockDim.x / 16)) {
    const int64_t b = idx / targets, t = idx % targets;
    const float sum = token_sum16(pooled + b * bs + t * ts, (int)query_tokens);
    if ((threadIdx.x & 15) != 0) continue;
    if (out) out[b * out_stride + t] = sum;
    if (iout) iout[b * iout_stride + t] = (int32_t)sum;
  }
}

}  // namespace

// Passes of 32 query rows, or 128 beyond.
int score_rows_per_pass(int64_t rows) { return rows <= 32 ? 32 : 128; }

hipError_t launch_score(const ScoreArgs& a, bool residual, int64_t groups, hipStream_t stream) {
  if (a.num_waves <= 0 || a.num_waves % kWavesPerGroup != 0 || a.subs <= 0 || groups <= 0) return hipErrorInvalidValue;
  if (a.tscale == nullptr || (residual && (a.rcodes == nullptr || a.rtscale == nullptr))) return hipErrorInvalidValue;
  const bool narrow = score_rows_per_pass(a.grp_rows) == 32;
  ScoreArgs part = a;
  for (int64_t first = 0; first < groups * a.subs; first += kMaxGridRows) {
    const dim3 grid((unsigned)(a.num_waves / kWavesPerGroup), (unsigned)std::min(kMaxGridRows, groups * a.subs - first));
    part.first_pass = (int32_t)first;
    if (residual) {
      if (narrow) score_kernel<true, 2, false><<<grid, kThreads, 0, stream>>>(part);
      else score_kernel<true, 8, false><<<grid, kThreads, 0, stream>>>(part);
    } else if (a.unit_tscale) {
      if (narrow) score_kernel<false, 2, true><<<grid, kThreads, 0, stream>>>(part);
      else score_kernel<false, 8, true><<<grid, kThreads, 0, stream>>>(part);
    } else {
      if (narrow) score_kernel<false, 2, false><<<grid, kThreads, 0, stream>>>(part);
      else score_kernel<false, 8, false><<<grid, kThreads, 0, stream>>>(part);
    }
  }
  return hipGetLastError();
}

hipError_t launch_quantize_limbs(const float* d_query, int64_t rows, int64_t rows_padded, int layout, bool recip,
                                 int8_t* qpack, float* colmul, int32_t* qsum, hipStream_t stream, int layout2,
                                 int8_t* qpack2) {
  if (rows_padded <= 0) return hipSuccess;
  quantize_limbs_kernel<<<dim3((unsigned)((rows_padded + 3) / 4)), dim3(256), 0, stream>>>(
      d_query, rows, rows_padded, layout, recip ? 1 : 0, qpack, colmul, qsum, layout2, qpack2);
  return hipGetLastError();
}

hipError_t launch_quantize_bits(const uint8_t* d_qbits, int64_t rows, int64_t rows_padded, int8_t* qpack,
                                float* colmul, int32_t* qsum, hipStream_t stream) {
  if (rows_padded <= 0) return hipSuccess;
  const int64_t blocks = (rows_padded + 3) / 4;
  quantize_bits_kernel<<<dim3((unsigned)blocks), dim3(256), 0, stream>>>(d_qbits, rows, rows_padded, qpack, colmul,
                                                                       qsum);
  return hipGetLastError();
}

hipError_t launch_pool_sum(const float* pooled, int64_t batch, int64_t query_tokens, int64_t targets, int64_t bs,
                           int64_t ts, float* out, int64_t out_stride, int32_t* iout, int64_t iout_stride,
                           hipStream_t stream) {
  const int64_t n = batch * targets;
  if (n <= 0) return hipSuccess;
  // (A launch has fewer than 2^32 threads: large outputs are walked.)
  const int64_t blocks = std::min<int64_t>((n + 15) / 16, 1 << 18);
  pool_sum_kernel<<<dim3((unsigned)blocks), dim3(256), 0, stream>>>(pooled, batch, query_tokens, targets, bs, ts, out,
                                                                  out_stride, iout, iout_stride);
  return hipGetLastError();
}

}  // namespace msim
