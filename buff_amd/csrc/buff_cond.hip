// Filter -> project: the values of the rows set in a condition bitmap,
// compacted in row order (buff_decode_condition, buff_simd.rs:1528-1712).
//
// The condition has the layout every filter here writes: ceil(n/64) u64 words,
// bit i = row i, so the lane owning rows 16t..16t+15 of tile c reads u16 word
// c*64 + t. Three or four launches:
//   k_cond_count   per-tile and per-workgroup counts of condition rows and of
//                  tiles holding any (workgroup w owns 64 consecutive tiles);
//   k_cond_scan    one workgroup: exclusive prefixes of the per-workgroup
//                  counts and the totals (columns above kCondSelf ranges);
//   k_cond_index   the tiles holding condition rows, compacted in tile order,
//                  each with its first output row;
//   k_cond_gather  per compacted tile, the waves of the grid in turn: the
//                  planes and tail bits of the
//                  lanes that hold such rows (idle lanes load a live lane's
//                  bytes), the values built per row, compacted through LDS and
//                  written with contiguous stores at the tile's output offset.
#include <algorithm>
#include <type_traits>

#include "buff_cond.h"
#include "buff_device.h"
#include "buff_launch.h"

namespace buffgpu {

// The lane's condition rows of tile c. Lanes past the last row read word 0
// instead (the bitmap holds ceil(n/64) words, fewer than a full last tile).
__device__ __forceinline__ uint32_t cond_lane(const uint16_t* cond, uint64_t n, uint64_t c, uint32_t lane) {
  const uint32_t valid = lane_valid16(n, c, lane);
  const uint64_t idx = valid ? c * 64 + lane : 0;
  return (uint32_t)cond[idx] & valid;
}

// Sum of v over each row of 16 lanes, in the row's last lane.
__device__ __forceinline__ uint32_t row16_sum(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);   // row_shr:1
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);   // row_shr:2
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);   // row_shr:4
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);   // row_shr:8
  return v;
}

// Workgroup w owns tiles [64w, 64w + 64): 1024 bitmap words, four per thread
// (coalesced, all in flight together). A tile's 16 words sit in one row of 16
// lanes, whose last lane writes the tile's count.
__global__ __launch_bounds__(256) void k_cond_count(const uint64_t* __restrict__ cond, uint64_t n, uint64_t ntiles,
                                                    uint16_t* __restrict__ tile_cnt, uint32_t* __restrict__ wg_rows,
                                                    uint32_t* __restrict__ wg_tiles) {
  const uint32_t t = threadIdx.x, lane = __lane_id(), wave = wave_in_wg();
  const uint64_t nw = (n + 63) / 64;
  const uint64_t w0 = (uint64_t)blockIdx.x * kCondTilesPerWg * 16;
  uint32_t pc[4];
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) {
    const uint64_t i = w0 + t + 256 * j;
    uint64_t v = cond[i < nw ? i : 0];
    if (i >= nw) v = 0;
    else if (i == nw - 1 && (n & 63)) v &= (1ull << (n & 63)) - 1;
    pc[j] = (uint32_t)__popcll(v);
  }
  uint32_t rows = 0, tiles = 0;
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) {
    const uint32_t tc = row16_sum(pc[j]);
    const uint64_t c = (uint64_t)blockIdx.x * kCondTilesPerWg + 16 * j + t / 16;
    if ((t & 15) == 15 && c < ntiles) {
      tile_cnt[c] = (uint16_t)tc;   // at most 1024
      rows += tc;
      tiles += tc ? 1u : 0u;
    }
  }
  rows = wave_sum_u32(rows);
  tiles = wave_sum_u32(tiles);
  __shared__ uint32_t part[8];
  if (lane == 0) {
    part[wave] = rows;
    part[4 + wave] = tiles;
  }
  __syncthreads();
  if (t == 0) {
    wg_rows[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
    wg_tiles[blockIdx.x] = part[4] + part[5] + part[6] + part[7];
  }
}

// One workgroup: exclusive prefixes of the per-workgroup row and tile counts
// (their totals land at index nwg), 4096 entries per round.
__global__ __launch_bounds__(256) void k_cond_scan(const uint32_t* __restrict__ wg_rows,
                                                   const uint32_t* __restrict__ wg_tiles, uint32_t nwg,
                                                   unsigned long long* __restrict__ off_rows,
                                                   uint32_t* __restrict__ off_tiles) {
  __shared__ unsigned long long sr[256];
  __shared__ uint32_t st[256];
  const uint32_t t = threadIdx.x;
  unsigned long long carry_r = 0;
  uint32_t carry_t = 0;
  for (uint32_t base = 0; base < nwg; base += 4096) {
    uint32_t vr[16], vt[16];
    unsigned long long lr = 0;
    uint32_t lt = 0;
#pragma unroll
    for (uint32_t j = 0; j < 16; ++j) {
      const uint32_t i = base + t * 16 + j;
      vr[j] = i < nwg ? wg_rows[i] : 0u;
      vt[j] = i < nwg ? wg_tiles[i] : 0u;
      lr += vr[j];
      lt += vt[j];
    }
    sr[t] = lr;
    st[t] = lt;
    __syncthreads();
    for (uint32_t o = 1; o < 256; o <<= 1) {
      const unsigned long long a = t >= o ? sr[t - o] : 0ull;
      const uint32_t b = t >= o ? st[t - o] : 0u;
      __syncthreads();
      sr[t] += a;
      st[t] += b;
      __syncthreads();
    }
    unsigned long long rr = carry_r + sr[t] - lr;
    uint32_t rt = carry_t + st[t] - lt;
#pragma unroll
    for (uint32_t j = 0; j < 16; ++j) {
      const uint32_t i = base + t * 16 + j;
      if (i < nwg) {
        off_rows[i] = rr;
        off_tiles[i] = rt;
      }
      rr += vr[j];
      rt += vt[j];
    }
    carry_r += sr[255];
    carry_t += st[255];
    __syncthreads();
  }
  if (t == 0) {
    off_rows[nwg] = carry_r;
    off_tiles[nwg] = carry_t;
  }
}

// Scratch layout (each region 256-byte aligned): off_rows (nwg + 1 u64),
// row_off (ntiles u64), off_tiles (nwg + 1 u32), wg_rows, wg_tiles (nwg u32
// each), list (ntiles u32), tile_cnt (ntiles u16).
struct CondLayout {
  uint32_t nwg;
  uint64_t off_rows, row_off, off_tiles, wg_rows, wg_tiles, list, tile_cnt, bytes;
};

static CondLayout cond_layout(uint64_t ntiles) {
  CondLayout L;
  L.nwg = (uint32_t)((ntiles + kCondTilesPerWg - 1) / kCondTilesPerWg);
  if (L.nwg < 1) L.nwg = 1;
  uint64_t at = 0;
  auto take = [&](uint64_t bytes) {
    const uint64_t here = at;
    at += (bytes + 255) & ~255ull;
    return here;
  };
  L.off_rows = take(8ull * (L.nwg + 1));
  L.row_off = take(8ull * ntiles);
  L.off_tiles = take(4ull * (L.nwg + 1));
  L.wg_rows = take(4ull * L.nwg);
  L.wg_tiles = take(4ull * L.nwg);
  L.list = take(4ull * ntiles);
  L.tile_cnt = take(2ull * ntiles);
  L.bytes = at;
  return L;
}

// One wave per workgroup range (one tile per lane): the tiles holding
// condition rows, compacted in tile order, each with its first output row. Up
// to kCondSelf ranges (SELF) a wave adds up the counts of the ranges before its
// own, eight loads in flight together, and the last one writes the totals: a
// scan launch less (a call with next to no hits, 16M / 67M / 134M / 268M rows:
// 16.7 / 17.9 / 20.4 / 25.5 us, with the scan 19.7 / 20.6 / 23.4 / 29.9 us).
// Beyond, the reads grow with the square of the ranges and the scan takes over.
constexpr uint32_t kCondSelf = 4096;

template <bool SELF>
__global__ __launch_bounds__(64) void k_cond_index(const uint16_t* __restrict__ tile_cnt, uint64_t ntiles,
                                                   const uint32_t* __restrict__ wg_rows,
                                                   const uint32_t* __restrict__ wg_tiles,
                                                   unsigned long long* __restrict__ off_rows,
                                                   uint32_t* __restrict__ off_tiles,
                                                   uint32_t* __restrict__ list,
                                                   unsigned long long* __restrict__ row_off) {
  const uint32_t lane = __lane_id();
  const uint64_t c = (uint64_t)blockIdx.x * kCondTilesPerWg + lane;
  const uint32_t cnt = c < ntiles ? (uint32_t)tile_cnt[c] : 0u;
  unsigned long long r0;
  uint32_t t0;
  if (SELF) {
    uint32_t rows = 0, tiles = 0;   // at most kCondSelf * 64 * 1024 rows
    for (uint32_t i = lane; i < blockIdx.x; i += 256) {
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t k = i + 64 * j;
        const uint32_t a = wg_rows[k < blockIdx.x ? k : 0], b = wg_tiles[k < blockIdx.x ? k : 0];
        rows += k < blockIdx.x ? a : 0u;
        tiles += k < blockIdx.x ? b : 0u;
      }
    }
    r0 = wave_sum_u32(rows);
    t0 = wave_sum_u32(tiles);
    if (blockIdx.x == gridDim.x - 1 && lane == 0) {
      off_rows[gridDim.x] = r0 + wg_rows[blockIdx.x];
      off_tiles[gridDim.x] = t0 + wg_tiles[blockIdx.x];
    }
  } else {
    r0 = off_rows[blockIdx.x];
    t0 = off_tiles[blockIdx.x];
  }
  const uint32_t rp = wave_excl_scan_u32(cnt, lane);
  const uint32_t tp = wave_excl_scan_u32(cnt ? 1u : 0u, lane);
  if (cnt) {
    const uint32_t k = t0 + tp;
    list[k] = (uint32_t)c;
    row_off[k] = r0 + rp;
  }
}

// The tile list and row offsets of a condition (k_cond_count .. k_cond_index).
static void launch_cond_list(const uint64_t* cond, uint64_t n, uint64_t ntiles, uint8_t* scratch, const CondLayout& L,
                             hipStream_t s) {
  unsigned long long* off_rows = reinterpret_cast<unsigned long long*>(scratch + L.off_rows);
  unsigned long long* row_off = reinterpret_cast<unsigned long long*>(scratch + L.row_off);
  uint32_t* off_tiles = reinterpret_cast<uint32_t*>(scratch + L.off_tiles);
  uint32_t* wg_rows = reinterpret_cast<uint32_t*>(scratch + L.wg_rows);
  uint32_t* wg_tiles = reinterpret_cast<uint32_t*>(scratch + L.wg_tiles);
  uint32_t* list = reinterpret_cast<uint32_t*>(scratch + L.list);
  uint16_t* tile_cnt = reinterpret_cast<uint16_t*>(scratch + L.tile_cnt);
  const uint16_t* tc = tile_cnt;
  const uint32_t *wr = wg_rows, *wt = wg_tiles;
  launch_k(k_cond_count, dim3(L.nwg), dim3(256), 0, s, cond, n, ntiles, tile_cnt, wg_rows, wg_tiles);
  if (L.nwg <= kCondSelf) {
    launch_k(k_cond_index<true>, dim3(L.nwg), dim3(64), 0, s, tc, ntiles, wr, wt, off_rows, off_tiles, list, row_off);
  } else {
    launch_k(k_cond_scan, dim3(1), dim3(256), 0, s, wr, wt, L.nwg, off_rows, off_tiles);
    launch_k(k_cond_index<false>, dim3(L.nwg), dim3(64), 0, s, tc, ntiles, wr, wt, off_rows, off_tiles, list, row_off);
  }
}

// Offset of row b (lane's rows) from NP planes and r tail bits. compat: when
// F >= 8 and r > 0 the tail field is OR-ed in shifted left by r, as the
// reference does (buff_simd.rs:1693, 1701); otherwise in place.
template <int NP>
__device__ __forceinline__ uint64_t cond_offset(const RowBytes<NP>& rb, uint32_t r, uint32_t b, bool compat) {
  const uint64_t X = row_bytes_x<NP>(rb, b);
  if (NP == 0 || !compat) return X >> (8u - r);
  const uint64_t v = X >> 8, t = (X & 0xFFu) >> (8u - r);
  return (v | t) << r;
}

// Waves take the compacted tiles in turn, so clustered condition rows spread
// over the whole grid. A tile is a chain of three loads (its list entry, its
// condition words, its planes); the list entry is read two tiles ahead and the
// condition words one tile ahead, which leaves one load's latency a tile. The
// offsets are staged in 32 bits where they fit (SV): half the LDS, so the CU's
// 32 waves are resident; the values are built from the compacted rows. 67M rows of 19 bits, a tenth of them set (0.22 GB read and
// written): 34 us, 6.5 TB/s; tile by tile with 64-bit staging 47 us.
template <int NP, typename SV>
__global__ __launch_bounds__(64) void k_cond_gather(ChunkView cv, double inv_scale, uint32_t compat,
                                                     const uint16_t* __restrict__ cond,
                                                     const uint32_t* __restrict__ ntiles_live,
                                                     const uint32_t* __restrict__ list,
                                                     const unsigned long long* __restrict__ row_off,
                                                     double* __restrict__ out, uint64_t cap) {
  __shared__ SV sv[kTileRows];
  const uint32_t lane = __lane_id();
  const uint32_t total = *cmem(ntiles_live);
  const uint64_t step = waves_in_grid();
  uint64_t i = wave_global();
  if (i >= total) return;
  const uint64_t last = total - 1;
  uint64_t c = cmem(list)[i], o = cmem(row_off)[i];
  uint32_t live = cond_lane(cond, cv.n, c, lane);
  uint64_t c1 = cmem(list)[min(i + step, last)], o1 = cmem(row_off)[min(i + step, last)];
  while (true) {
    const uint32_t src = refine_src(live, lane);
    RowBytes<NP> rb;
    load_row_bytes<NP>(cv, c, src, rb);
    const uint32_t live1 = cond_lane(cond, cv.n, c1, lane);   // past the end: the last tile's, not used
    const uint64_t i2 = min(i + 2 * step, last);
    const uint64_t c2 = cmem(list)[i2], o2 = cmem(row_off)[i2];
    const uint32_t cntl = (uint32_t)__popc(live);
    uint32_t pos = wave_excl_scan_u32(cntl, lane);
    const uint32_t tot = wave_total_u32(cntl);
#pragma unroll
    for (uint32_t b = 0; b < 16; ++b)
      if ((live >> b) & 1u) sv[pos++] = (SV)cond_offset<NP>(rb, cv.r, b, compat != 0);
    wave_lds_sync();
    for (uint32_t k = lane; k < tot; k += 64)
      if (o + k < cap)
        __builtin_nontemporal_store((double)(int64_t)((uint64_t)cv.base + (uint64_t)sv[k]) * inv_scale,
                                    gmem_w(out) + o + k);
    wave_lds_sync();
    i += step;
    if (i >= total) return;
    c = c1, o = o1, live = live1;
    c1 = c2, o1 = o2;
  }
}

// The condition rows of an already decoded column `vals` (n doubles), in row
// order: the same tile list and row offsets as k_cond_gather.
__global__ __launch_bounds__(64) void k_cond_gather_values(const double* __restrict__ vals, uint64_t n,
                                                            const uint16_t* __restrict__ cond,
                                                            const uint32_t* __restrict__ ntiles_live,
                                                            const uint32_t* __restrict__ list,
                                                            const unsigned long long* __restrict__ row_off,
                                                            double* __restrict__ out, uint64_t cap) {
  __shared__ double sv[kTileRows];
  const uint32_t lane = __lane_id();
  const uint32_t total = *cmem(ntiles_live);
  for (uint64_t i = wave_global(); i < total; i += waves_in_grid()) {
    const uint64_t c = cmem(list)[i];
    const unsigned long long o = cmem(row_off)[i];
    const uint32_t live = cond_lane(cond, n, c, lane);
    const uint32_t cntl = (uint32_t)__popc(live);
    uint32_t pos = wave_excl_scan_u32(cntl, lane);
    const uint32_t tot = wave_total_u32(cntl);
    const uint64_t r0 = c * kTileRows + 16ull * lane;
#pragma unroll
    for (uint32_t b = 0; b < 16; ++b)
      if ((live >> b) & 1u) sv[pos++] = vals[r0 + b];
    wave_lds_sync();
    for (uint32_t k = lane; k < tot; k += 64)
      if (o + k < cap) __builtin_nontemporal_store(sv[k], gmem_w(out) + o + k);
    wave_lds_sync();
  }
}

uint64_t cond_scratch_bytes(uint64_t ntiles) { return cond_layout(ntiles).bytes; }

uint64_t cond_total_offset(uint64_t ntiles) {
  const CondLayout L = cond_layout(ntiles);
  return L.off_rows + 8ull * L.nwg;
}

hipError_t launch_cond_values(const double* vals, uint64_t n, const uint64_t* cond, double* out, uint64_t cap,
                              uint8_t* scratch, hipStream_t s) {
  const uint64_t ntiles = (n + kTileRows - 1) / kTileRows;
  if (ntiles == 0) return hipSuccess;
  const CondLayout L = cond_layout(ntiles);
  launch_cond_list(cond, n, ntiles, scratch, L, s);
  const uint32_t* nlive = reinterpret_cast<const uint32_t*>(scratch + L.off_tiles) + L.nwg;
  const uint32_t* lst = reinterpret_cast<const uint32_t*>(scratch + L.list);
  const unsigned long long* ro = reinterpret_cast<const unsigned long long*>(scratch + L.row_off);
  const uint32_t grid = (uint32_t)std::min<uint64_t>(ntiles, 5120);
  launch_k(k_cond_gather_values, dim3(grid), dim3(64), 0, s, vals, n, reinterpret_cast<const uint16_t*>(cond),
           nlive, lst, ro, out, cap);
  return hipGetLastError();
}

hipError_t launch_cond_decode(const ChunkView& cv, double inv_scale, bool compat, const uint64_t* cond, double* out,
                              uint64_t cap, uint8_t* scratch, hipStream_t s) {
  if (cv.ntiles == 0) return hipSuccess;
  const CondLayout L = cond_layout(cv.ntiles);
  launch_cond_list(cond, cv.n, cv.ntiles, scratch, L, s);
  const uint32_t* nlive = reinterpret_cast<const uint32_t*>(scratch + L.off_tiles) + L.nwg;
  const uint32_t* lst = reinterpret_cast<const uint32_t*>(scratch + L.list);
  const unsigned long long* ro = reinterpret_cast<const unsigned long long*>(scratch + L.row_off);
  const uint16_t* c16 = reinterpret_cast<const uint16_t*>(cond);
  const uint32_t cm = compat ? 1u : 0u;
  // one wave per workgroup, 4 or 8 KB of LDS staging each: the waves that fit the CUs
#define BUFF_GATHER(NP)                                                                                           \
  do {                                                                                                            \
    constexpr bool narrow = NP <= 3;   /* at most 31 bits */                                                      \
    using SV = std::conditional_t<narrow, uint32_t, uint64_t>;                                                    \
    const uint32_t grid = (uint32_t)std::min<uint64_t>(cv.ntiles, narrow ? 8192 : 5120);                          \
    launch_k(k_cond_gather<NP, SV>, dim3(grid), dim3(64), 0, s, cv, inv_scale, cm, c16, nlive, lst, ro, out, cap); \
  } while (0)
  switch (cv.P) {
    case 0: BUFF_GATHER(0); break;
    case 1: BUFF_GATHER(1); break;
    case 2: BUFF_GATHER(2); break;
    case 3: BUFF_GATHER(3); break;
    case 4: BUFF_GATHER(4); break;
    case 5: BUFF_GATHER(5); break;
    case 6: BUFF_GATHER(6); break;
    case 7: BUFF_GATHER(7); break;
    default: BUFF_GATHER(8); break;
  }
#undef BUFF_GATHER
  return hipGetLastError();
}

}  // namespace buffgpu
