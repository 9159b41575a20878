// Device helpers of the buff-major layout shared by its kernels
// (buff_major.hip) and the batched query kernels (buff_batch.hip).
//
// A sparse column's bytes for a lane are the majority byte replicated, with the
// outlier bytes patched in: the lane's 16-bit slice of the outlier bitmap says
// which rows, the tile's prefix count plus an exclusive scan of the lanes'
// popcounts says where their bytes start in the compacted array.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <type_traits>

#include "buff_common.h"
#include "buff_device.h"
#include "buff_major.h"

namespace buffgpu {

// The first S sparse columns of a MajorView (the same layout as its prefix):
// what a kernel reading the view from memory needs in registers for S columns.
template <int S>
struct MajorPrefix {
  ChunkView dense;
  SparseDev col[S];
};
static_assert(sizeof(MajorPrefix<3>) == offsetof(MajorView, col) + 3 * sizeof(SparseDev), "MajorView prefix layout");

// The lane's packed outlier bytes (k-th outlier of the lane = byte k) as four
// dwords, from a 20-byte window of aligned loads at its compacted position.
struct Packed16 {
  uint32_t d0, d1, d2, d3;
};
__device__ __forceinline__ Packed16 load_packed(const uint8_t* outl, uint64_t pos) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(outl + (pos & ~3ull));
  const uint32_t sh = (uint32_t)(pos & 3);
  const uint32_t a = w[0], b = w[1], c = w[2], d = w[3], e = w[4];
  Packed16 p;
  p.d0 = __builtin_amdgcn_alignbyte(b, a, sh);
  p.d1 = __builtin_amdgcn_alignbyte(c, b, sh);
  p.d2 = __builtin_amdgcn_alignbyte(d, c, sh);
  p.d3 = __builtin_amdgcn_alignbyte(e, d, sh);
  return p;
}
// Row masks (bit b <-> row 16*lane + b) of one sparse column against target byte
// t: majority rows all at once, outlier rows from the packed bytes. The lane's
// k-th outlier (k-th set bit of m16, ascending rows) is byte k of its packed
// window; k runs with a wave-uniform bound in an unrolled loop, so every step
// reads a fixed register and byte (no per-lane select of the byte). Only the
// rows in `want` keep their results.
__device__ __forceinline__ void sparse_cmp(const Packed16& pk, uint32_t m16, uint32_t want, uint32_t major, uint32_t t,
                                           uint32_t& gt, uint32_t& eq) {
  const uint32_t nm = ~m16 & 0xFFFFu;
  const uint32_t d[4] = {pk.d0, pk.d1, pk.d2, pk.d3};
  uint32_t go = 0, eo = 0, rem = m16;
#pragma unroll
  for (uint32_t k = 0; k < 16; ++k) {
    if (!__ballot((rem & want) != 0)) break;
    const uint32_t pos = (uint32_t)__builtin_ctz(rem | 0x10000u);   // 16 once the lane has no outlier left
    rem &= rem - 1u;
    const uint32_t v = (d[k >> 2] >> (8 * (k & 3))) & 0xFFu;
    go |= (uint32_t)(v > t) << pos;
    eo |= (uint32_t)(v == t) << pos;
  }
  gt = (major > t ? nm : 0u) | (go & want);
  eq = (major == t ? nm : 0u) | (eo & want);
}

// Replaces byte b (row 16*lane + b: dword b%4, byte b/4) of a lane's 16 bytes
// when `on` (written with selects: every lane runs the same instructions).
__device__ __forceinline__ void set_byte(uint32_t& d0, uint32_t& d1, uint32_t& d2, uint32_t& d3, uint32_t b,
                                         uint32_t v, bool on) {
  const uint32_t sh = 8 * ((b >> 2) & 3);
  const uint32_t keep = ~(0xFFu << sh), val = v << sh;
  const uint32_t i = b & 3;
  d0 = on && i == 0 ? (d0 & keep) | val : d0;
  d1 = on && i == 1 ? (d1 & keep) | val : d1;
  d2 = on && i == 2 ? (d2 & keep) | val : d2;
  d3 = on && i == 3 ? (d3 & keep) | val : d3;
}

// The lane's 16 bytes of a sparse column: the majority byte, with the outlier
// bytes of the rows in `want` (a subset of m16) patched in. The outliers are
// walked by rank as in sparse_cmp.
__device__ __forceinline__ uint4 patch_outliers(const Packed16& pk, uint32_t m16, uint32_t want, uint32_t major) {
  const uint32_t M = 0x01010101u * major;
  uint32_t o0 = M, o1 = M, o2 = M, o3 = M;
  const uint32_t d[4] = {pk.d0, pk.d1, pk.d2, pk.d3};
  uint32_t rem = m16;
#pragma unroll
  for (uint32_t k = 0; k < 16; ++k) {
    if (!__ballot((rem & want) != 0)) break;
    const uint32_t pos = (uint32_t)__builtin_ctz(rem | 0x10000u);
    rem &= rem - 1u;
    const uint32_t v = (d[k >> 2] >> (8 * (k & 3))) & 0xFFu;
    set_byte(o0, o1, o2, o3, pos, v, (want >> pos) & 1u);
  }
  return make_uint4(o0, o1, o2, o3);
}

// max over the outlier rows in `want` of (byte + 1); 0 when there is none.
__device__ __forceinline__ uint32_t sparse_max_plus1(const Packed16& pk, uint32_t m16, uint32_t want) {
  const uint32_t d[4] = {pk.d0, pk.d1, pk.d2, pk.d3};
  uint32_t rem = m16, best = 0;
#pragma unroll
  for (uint32_t k = 0; k < 16; ++k) {
    if (!__ballot((rem & want) != 0)) break;
    const uint32_t pos = (uint32_t)__builtin_ctz(rem | 0x10000u);
    rem &= rem - 1u;
    const uint32_t v = (d[k >> 2] >> (8 * (k & 3))) & 0xFFu;
    best = (want >> pos) & 1u ? max(best, v + 1u) : best;
  }
  return best;
}

// The outlier window of column sd for the lane in tile c (every lane of the
// wave calls it together: the exclusive scan).
__device__ __forceinline__ Packed16 lane_outliers(const SparseDev& sd, uint64_t c, uint32_t lane, uint32_t m16) {
  const uint32_t excl = wave_excl_scan_u32(__popc(m16), lane);
  return m16 ? load_packed(sd.outl, (uint64_t)sd.prefix[c] + excl) : Packed16{0, 0, 0, 0};
}

// Masks and outlier windows of every sparse column of tile c, with all their
// loads issued before any is consumed (the columns are independent).
struct SparseLanes {
  uint32_t m[kMaxSparse];
  Packed16 pk[kMaxSparse];
};

__device__ __forceinline__ void load_sparse(const MajorView& mv, uint64_t c, uint32_t lane, SparseLanes& sl) {
  uint32_t pre[kMaxSparse];
#pragma unroll
  for (uint32_t j = 0; j < kMaxSparse; ++j) {
    sl.m[j] = j < mv.S ? (uint32_t)mv.col[j].mask16[c * 64 + lane] : 0u;
    pre[j] = j < mv.S ? mv.col[j].prefix[c] : 0u;
  }
#pragma unroll
  for (uint32_t j = 0; j < kMaxSparse; ++j) {
    sl.pk[j] = Packed16{0, 0, 0, 0};
    if (j < mv.S) {
      const uint32_t excl = wave_excl_scan_u32(__popc(sl.m[j]), lane);
      if (sl.m[j]) sl.pk[j] = load_packed(mv.col[j].outl, (uint64_t)pre[j] + excl);
    }
  }
}

// One sparse column's outliers of a tile against target byte t, deposited in
// row order. Outlier k of the tile (k = 0..cnt-1, in row order) goes to lane
// k % 64, which ORs (1 << b) | (byte > t) << (16 + b) | (byte == t) << (32 + b)
// into dep[L] for its row 16L + b. Lane L then reads its word: the outlier rows
// of its 16 (bits 0-15), those above t (16-31) and those equal (32-47). The
// first outlier of each lane arrives preloaded (row0 / byte0); further ones (a
// tile with more than 64) are loaded here. dep is clear before.
__device__ __forceinline__ void deposit_outliers(unsigned long long* dep, const SparseDev& sd, uint32_t p0,
                                                 uint32_t cnt, uint32_t lane, uint32_t row0, uint32_t byte0,
                                                 uint32_t t) {
  auto put = [&](uint32_t row, uint32_t byte) {
    const uint32_t one = 1u << (row & 15u);
    const uint32_t lo = one | (byte > t ? one << 16 : 0u), hi = byte == t ? one : 0u;
    atomicOr(&dep[row >> 4], ((unsigned long long)hi << 32) | lo);
  };
  if (lane < cnt) put(row0, byte0);
  for (uint32_t k = lane + 64; k < cnt; k += 64) put(sd.pos[p0 + k], sd.outl[p0 + k]);
}

// LDS words a wave needs for major_filter_group: one per lane, column (of the
// kDepCols columns of a phase) and tile.
constexpr int kDepCols = 3;
constexpr uint32_t dep_words(int S, int U) { return 64u * (S < kDepCols ? S : kDepCols) * U; }

// The rules of a filter's sparse columns as 16-row masks, so that a tile's
// columns take a few bitwise operations without a branch. Per column, with cand
// the rows equal to the target so far, out the outlier rows, G / E those above /
// equal to its target byte t:
//   res |= (G | out & zero) & (cand | any) | cand & ~out & gtm
//   cand &= (~out & eqm | E) & keep
// gtm / eqm: the majority byte is above / equal to t; any: outliers count for
// every row and not only candidates (the reference's range filter, columns after
// the first); zero, and keep = none: its rule for t = 0 = majority byte (the
// candidate outliers qualify, nothing stays a candidate).
template <int S>
struct MajorRules {
  uint32_t gtm[S], eqm[S], any[S], zero[S], keep[S];
};
template <int MODE, int S, typename MV>
__device__ __forceinline__ MajorRules<S> major_rules(const MV& mv, const MajorTarget& tg, bool sem) {
  MajorRules<S> r;
#pragma unroll
  for (int j = 0; j < S; ++j) {
    const uint32_t major = mv.col[j].major, t = tg.digit[j];
    const bool ref = MODE == 0 && !sem && j > 0, z = ref && t == 0 && major == 0;
    r.gtm[j] = major > t ? 0xFFFFu : 0u;
    r.eqm[j] = major == t ? 0xFFFFu : 0u;
    r.any[j] = ref && !z ? 0xFFFFu : 0u;
    r.zero[j] = z ? 0xFFFFu : 0u;
    r.keep[j] = z ? 0u : 0xFFFFu;
  }
  return r;
}

// Tiles [c0, c0 + U) of a buff-major filter (buff_simd.rs:863-1277 range,
// 1916-2292 equality; rules with sem: the intended answer on the true offsets):
// res[u] is the lane's 16-row result mask of tile c0 + u (tiles past the
// chunk's last are computed empty and are not meant to be stored). dep: the
// wave's dep_words(S, U) LDS words: the outliers of up to kDepCols columns and
// all tiles are deposited in one phase. Every load of the first round (tile
// prefixes, the first dense plane, each lane's first outlier row and byte of
// every column) is in flight together; with 258 vector instructions a range tile
// (300 with the rules as branches and a deposit phase per column and tile) the
// filter of 33,554,432 rows takes 26.8 us (28.9), equality 23.0 (25.5), the
// reads alone 16.
//
// PF (the target's sparse bytes are the majority bytes, so most rows stay
// candidates into the dense planes): the second dense plane and a tail of at
// most kPfTail bits are loaded in the first round as well, in full, instead of
// for the candidates' lines in later dependent rounds.
//
// STEP (equality with a target of which some sparse byte is not the majority
// byte): one column a phase, ending with the first that leaves no candidate,
// since only outliers match such a byte. 67,108,864 rows of three sparse columns
// with 5% outliers: 40.4 us, 43.2 with the columns in one phase (38.4 and 43 for
// the rarest first byte); with 9%, where a tile's further outliers are loaded per
// phase, 51.5 and 63.2.
constexpr uint32_t kPfTail = 2;

template <int MODE, int S, int U, bool PF = false, bool STEP = false, typename MV>
__device__ __forceinline__ void major_filter_group(const MV& mv, const MajorTarget& tg, const MajorRules<S>& ru,
                                                   uint64_t c0, uint32_t lane, unsigned long long* dep,
                                                   uint32_t (&res)[U]) {
  const ChunkView& dv = mv.dense;
  uint32_t p0[U][S], cnt[U][S], row0[U][S], byte0[U][S];
  uint4 w0[U], w1[U];
  uint32_t hp[U][kPfTail];
  const bool pf_tail = PF && dv.r <= kPfTail;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const bool in = c0 + u < dv.ntiles;
    const uint64_t c = in ? c0 + u : dv.ntiles - 1;
#pragma unroll
    for (int j = 0; j < S; ++j) {
      p0[u][j] = mv.col[j].prefix[c];
      cnt[u][j] = in ? mv.col[j].prefix[c + 1] - p0[u][j] : 0u;
    }
    w0[u] = dv.P ? load_plane(dv, 0, c, lane) : make_uint4(0, 0, 0, 0);
    w1[u] = PF && dv.P > 1 ? load_plane(dv, 1, c, lane) : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (uint32_t j = 0; j < kPfTail; ++j) hp[u][j] = pf_tail && j < dv.r ? load_tail(dv, j, c, lane) : 0u;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int j = 0; j < S; ++j) {
      const bool has = lane < cnt[u][j];
      row0[u][j] = has ? mv.col[j].pos[p0[u][j] + lane] : 0u;
      byte0[u][j] = has ? mv.col[j].outl[p0[u][j] + lane] : 0u;
    }
  }
  uint32_t cand[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    res[u] = 0;
    cand[u] = tile_full(dv.n, c0 + u) ? 0xFFFFu : lane_valid16(dv.n, c0 + u, lane);
  }
  constexpr int N = STEP ? 1 : S < kDepCols ? S : kDepCols;   // words per lane and tile
#pragma unroll
  for (int jp = 0; jp < S; jp += N) {
#pragma unroll
    for (int i = 0; i < N * U; ++i) dep[64 * i + lane] = 0;
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int j = jp; j < S && j < jp + N; ++j)
        deposit_outliers(dep + 64 * (u * N + j - jp), mv.col[j], p0[u][j], cnt[u][j], lane, row0[u][j], byte0[u][j],
                         tg.digit[j]);
    }
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int j = jp; j < S && j < jp + N; ++j) {
        const uint64_t w = dep[64 * (u * N + j - jp) + lane];
        const uint32_t out = (uint32_t)w & 0xFFFFu, G = (uint32_t)w >> 16, E = (uint32_t)(w >> 32);
        if (MODE == 0)
          res[u] |= ((G | (out & ru.zero[j])) & (cand[u] | ru.any[j])) | (cand[u] & ~out & ru.gtm[j]);
        cand[u] &= ((~out & ru.eqm[j]) | E) & ru.keep[j];
      }
    }
    wave_lds_sync();   // every lane has read its words before they are cleared again
    if (STEP) {
      uint32_t live = 0;
#pragma unroll
      for (int u = 0; u < U; ++u) live |= cand[u];
      if (__ballot(live != 0) == 0) return;   // res is 0 still
    }
  }
  auto any_live = [&]() {
    uint32_t live = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) live |= cand[u];
    return __ballot(live != 0) != 0;
  };
  auto plane = [&](uint32_t p, const uint4 (&wp)[U]) {
    const Digit dg = make_digit(tg.digit[S + p]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (MODE == 0) res[u] |= cand[u] & mask_gt(wp[u], dg);
      cand[u] &= mask_eq(wp[u], dg);
    }
  };
  bool live = any_live();
  if (live && dv.P > 0) {
    plane(0, w0);
    if (PF && dv.P > 1) plane(1, w1);
    live = any_live();
    for (uint32_t p = PF ? 2 : 1; live && p < dv.P; ++p) {
      uint4 wp[U];
#pragma unroll
      for (int u = 0; u < U; ++u) wp[u] = load_plane(dv, p, min(c0 + u, dv.ntiles - 1), refine_src(cand[u], lane));
      plane(p, wp);
      live = any_live();
    }
  }
  if (live && dv.r) {
    if (pf_tail) {   // the prefetched bit-planes, most significant first (absent ones are 0 with target 0)
#pragma unroll
      for (int j = (int)kPfTail - 1; j >= 0; --j) {
        const uint32_t t = (uint32_t)j < dv.r && ((tg.tail >> j) & 1) ? 0xFFFFu : 0u;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (MODE == 0) res[u] |= cand[u] & hp[u][j] & ~t;
          cand[u] &= ~(hp[u][j] ^ t);
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (c0 + u < dv.ntiles) refine_tail<MODE>(dv, c0 + u, tg.tail, lane, res[u], cand[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
    res[u] = MODE == 0 ? (tile_full(dv.n, c0 + u) ? res[u] : res[u] & lane_valid16(dv.n, c0 + u, lane)) : cand[u];
}

// Sum of the lane's outlier bytes of one sparse column (its k = popc(m16)
// outliers are the first k bytes of its packed window).
__device__ __forceinline__ uint32_t packed_sum(const Packed16& pk, uint32_t m16) {
  const uint32_t k = (uint32_t)__popc(m16);
  auto keep = [k](uint32_t i) -> uint32_t {   // bytes of dword i below k
    return k >= 4 * (i + 1) ? 0xFFFFFFFFu : (k > 4 * i ? (1u << (8 * (k - 4 * i))) - 1u : 0u);
  };
  uint32_t a = __builtin_amdgcn_sad_u8(pk.d0 & keep(0), 0u, 0u);
  a = __builtin_amdgcn_sad_u8(pk.d1 & keep(1), 0u, a);
  a = __builtin_amdgcn_sad_u8(pk.d2 & keep(2), 0u, a);
  return __builtin_amdgcn_sad_u8(pk.d3 & keep(3), 0u, a);
}

// LDS bytes a wave needs for major_tile_offsets' column images.
constexpr uint32_t kImageBytes = kMaxSparse * kTileRows;

// The lane's 16 stored offsets of tile c of a buff-major chunk
// (buff_decode_majority, buff_simd.rs:633-861): column 0 places its byte; a
// later sparse column ORs its outlier bytes at its shift and the majority byte
// at twice its shift, and only for rows up to its last outlier (SEM: every row
// gets its byte once, the true offset). Then the dense planes and tail.
//
// A sparse column's 16 bytes per lane come from an image of the tile in `img`
// (S * 1024 bytes of the wave's LDS, the plane layout of buff_common.h): every
// lane writes the fill byte of its rows, then outlier k of the tile goes to
// lane k % 64, which writes its byte over it. The offsets are assembled by byte
// permutes from the images and planes (the dense value from its lowest byte, so
// that the positions do not depend on the number of dense planes). The kernels
// that call this are bound by their vector instructions: walking every lane's
// outliers by rank and shifting each plane's byte into 64 bits took 91 us
// (compat 106) for 33,554,432 rows of three sparse columns, two planes and two
// tail bits, now 66 (71); the values' write and the bytes' read take 62 at the
// copy rate.
template <int SEM, int S, typename MV>
__device__ __forceinline__ void major_tile_offsets(const MV& mv, uint64_t c, uint32_t lane, uint8_t* img,
                                                   uint64_t (&v)[16]) {
  constexpr int SS = S > 0 ? S : 1;
  constexpr int NPM = (int)kMaxPlanes - S > 0 ? (int)kMaxPlanes - S : 1;   // dense planes at most (F <= 64)
  const ChunkView& dv = mv.dense;
  const uint32_t P = dv.P, r = dv.r;
  // every load of the tile first: each lane's first outlier of every column,
  // the dense planes (w[q]: the q-th from the lowest) and the tail
  uint32_t p0[SS], cnt[SS], row0[SS], byte0[SS], m[SS];
#pragma unroll
  for (int j = 0; j < S; ++j) {
    p0[j] = mv.col[j].prefix[c];
    cnt[j] = mv.col[j].prefix[c + 1] - p0[j];
    m[j] = SEM || j == 0 ? 0u : (uint32_t)mv.col[j].mask16[c * 64 + lane];
  }
  uint4 w[NPM];
#pragma unroll
  for (int q = 0; q < NPM; ++q) w[q] = (uint32_t)q < P ? load_plane(dv, P - 1 - q, c, lane) : make_uint4(0, 0, 0, 0);
  uint32_t h[7];
#pragma unroll
  for (uint32_t j = 0; j < 7; ++j) h[j] = j < r ? load_tail(dv, j, c, lane) : 0u;
#pragma unroll
  for (int j = 0; j < S; ++j) {
    const bool has = lane < cnt[j];
    row0[j] = has ? mv.col[j].pos[p0[j] + lane] : 0u;
    byte0[j] = has ? mv.col[j].outl[p0[j] + lane] : 0u;
  }
  uint4 ws[SS];
  if constexpr (S > 0) {
#pragma unroll
    for (int j = 0; j < S; ++j) {
      const uint32_t M = SEM || j == 0 ? 0x01010101u * mv.col[j].major : 0u;
      reinterpret_cast<uint4*>(img + j * kTileRows)[lane] = make_uint4(M, M, M, M);
    }
    wave_lds_sync();
    auto put = [&](int j, uint32_t row, uint32_t byte) {
      img[j * kTileRows + (row & ~15u) + 4 * (row & 3u) + ((row >> 2) & 3u)] = (uint8_t)byte;
    };
#pragma unroll
    for (int j = 0; j < S; ++j) {
      if (lane < cnt[j]) put(j, row0[j], byte0[j]);
      for (uint32_t k = lane + 64; k < cnt[j]; k += 64) put(j, mv.col[j].pos[p0[j] + k], mv.col[j].outl[p0[j] + k]);
    }
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < S; ++j) ws[j] = reinterpret_cast<const uint4*>(img + j * kTileRows)[lane];
    wave_lds_sync();   // the images may be overwritten from here on
  }
  // tail byte of row 4k + i in byte k of T[i], its bits at the top
  uint32_t T[4];
  tail_bytes<7>(h, r, T);
  auto dword = [](const uint4& q, uint32_t i) -> uint32_t { return i == 0 ? q.x : i == 1 ? q.y : i == 2 ? q.z : q.w; };
  // byte m of the dense value of rows b % 4 == i: the tail byte, then the planes from the lowest
  auto dense_src = [&](int k, uint32_t i) -> uint32_t { return k == 0 ? T[i] : k - 1 < NPM ? dword(w[k - 1 < NPM ? k - 1 : 0], i) : 0u; };
  auto dense_rows = [&](auto npairs) {
#pragma unroll
    for (uint32_t b = 0; b < 16; ++b) {
      const uint32_t i = b & 3, sel = (b >> 2) | (((b >> 2) + 4) << 8) | 0x0C0C0000u;
      uint64_t X = 0;
#pragma unroll
      for (int k = 0; k < decltype(npairs)::value; ++k)
        X |= (uint64_t)__builtin_amdgcn_perm(dense_src(2 * k + 1, i), dense_src(2 * k, i), sel) << (16 * k);
      v[b] = X >> (8u - r);
    }
  };
  if (P <= 1) dense_rows(std::integral_constant<int, 1>{});
  else if (P <= 3 || NPM <= 3) dense_rows(std::integral_constant<int, 2>{});
  else dense_rows(std::integral_constant<int, 4>{});
  if constexpr (S > 0) {
    // the sparse bytes above them, column 0 the highest
    auto sparse_src = [&](int k, uint32_t i) -> uint32_t { return k < S ? dword(ws[k < S ? S - 1 - k : 0], i) : 0u; };
#pragma unroll
    for (uint32_t b = 0; b < 16; ++b) {
      const uint32_t i = b & 3, sel = (b >> 2) | (((b >> 2) + 4) << 8) | 0x0C0C0000u;
      uint64_t X = 0;
#pragma unroll
      for (int k = 0; 2 * k < S; ++k)
        X |= (uint64_t)__builtin_amdgcn_perm(sparse_src(2 * k + 1, i), sparse_src(2 * k, i), sel) << (16 * k);
      v[b] |= X << dv.F;
    }
    if (!SEM) {
      const uint64_t row0 = c * kTileRows + 16ull * lane;
#pragma unroll
      for (int j = 1; j < S; ++j) {
        const uint32_t sh = mv.col[j].shift;
        const uint64_t twice = ((uint64_t)mv.col[j].major << sh) << sh;
        if (!twice) continue;
        const uint64_t last = mv.col[j].last;   // ~0 without outliers: every row
        const uint32_t in = last >= row0 + 15 ? 0xFFFFu : (last >= row0 ? (2u << (uint32_t)(last - row0)) - 1u : 0u);
        const uint32_t nm = ~m[j] & in;
#pragma unroll
        for (uint32_t b = 0; b < 16; ++b) v[b] |= (nm >> b) & 1u ? twice : 0ull;
      }
    }
  }
}

}  // namespace buffgpu
