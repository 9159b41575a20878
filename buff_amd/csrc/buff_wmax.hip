// Windowed max (buff_max_range, buff_simd.rs:5096-5334): the max stored offset
// of every window of W rows of [s, e), and the rows holding their window's max.
//
// The reference walks plane 0 of [s, e) keeping, per window, the rows tied on
// the running max byte, then narrows them plane by plane; the result is each
// window's max offset. Here every tile of [s, e) is read once and every window
// segment it holds reduced. Windows of kWmaxBlockMin .. kWmaxBlockMax rows take
// one launch (but for the longest on large columns, wmax_block_form):
//   k_wmax_block   a workgroup holds consecutive tiles in registers, completes
//                  their windows' maxima in LDS (the rows of its first and last
//                  window outside its tiles are read too), then compares its
//                  rows with them and writes bitmap and values.
// Other windows:
//   k_wmax_tiles   (short windows) windows that lie inside one tile are final;
//                  every tile also emits (window, max) for its first and last
//                  window segment;
//   k_wmax_tiles_wide   the same for long windows, in registers;
//   k_wmax_reduce  the emitted pairs are sorted by window: a reduce-by-key per
//                  block of 256 pairs writes the windows that end inside the
//                  block and passes on the two boundary runs, until one block
//                  remains (three levels for 134M rows at any window size);
//   k_wmax_argmax  each row of [s, e) against its window's max -> bitmap;
//   k_wmax_values  max offsets -> the reference's f64 (x + base) / 2^dlen.
#include <algorithm>
#include <type_traits>

#include "buff_device.h"
#include "buff_launch.h"
#include "buff_wmax.h"

namespace buffgpu {

// Offsets of the lane's 16 rows of tile c: NP planes, then r tail bits.
template <int NP>
__device__ __forceinline__ void lane_offsets(const ChunkView& cv, uint64_t c, uint32_t lane, uint64_t (&off)[16]) {
  RowBytes<NP> rb;
  load_row_bytes<NP>(cv, c, lane, rb);
#pragma unroll
  for (uint32_t b = 0; b < 16; ++b) off[b] = row_offset<NP>(rb, b, cv.r);
}

// One wave per tile of [s, e): tiles t_first + blockIdx.x (W < kWmaxBlockMin).
template <int NP>
__global__ __launch_bounds__(64) void k_wmax_tiles(ChunkView cv, uint64_t s, uint64_t e, uint64_t W, uint64_t t_first,
                                                   unsigned long long* __restrict__ wmax, uint32_t* __restrict__ ekey,
                                                   unsigned long long* __restrict__ eval) {
  __shared__ uint64_t so[kLdsRow * 64];
  const uint32_t lane = __lane_id();
  const uint64_t c = t_first + blockIdx.x;
  const uint64_t r0 = c * kTileRows;
  uint64_t off[16];
  lane_offsets<NP>(cv, c, lane, off);
#pragma unroll
  for (uint32_t b = 0; b < 16; ++b) so[kLdsRow * lane + b] = off[b];
  wave_lds_sync();
  // this tile's rows of [s, e): tile-local [a, b); its windows fw .. lw
  const uint64_t a = (s > r0 ? s : r0) - r0;
  const uint64_t b = (e < r0 + kTileRows ? e : r0 + kTileRows) - r0;
  const uint64_t fw = (r0 + a - s) / W, lw = (r0 + b - 1 - s) / W;
  const uint64_t nwin = lw - fw + 1;
  const uint32_t e0 = 2 * blockIdx.x, e1 = 2 * blockIdx.x + 1;
  // many short windows: one lane per window
  for (uint64_t wi = lane; wi < nwin; wi += 64) {
    const uint64_t w = fw + wi;
    const uint64_t ws = s + w * W, we = ws + W < e ? ws + W : e;
    const uint64_t x0 = (ws > r0 + a ? ws : r0 + a) - r0, x1 = (we < r0 + b ? we : r0 + b) - r0;
    uint64_t m = 0;
    for (uint64_t q = x0; q < x1; ++q) m = max(m, so[lds_slot((uint32_t)q)]);
    if (ws >= r0 && we <= r0 + kTileRows) wmax[w] = m;
    if (wi == 0) {
      ekey[e0] = (uint32_t)w;
      eval[e0] = m;
    }
    if (wi == nwin - 1) {
      ekey[e1] = (uint32_t)w;
      eval[e1] = m;
    }
  }
}

// Windows of at least one tile (W >= 1024): a tile holds at most two window
// segments, so each lane keeps its rows' max for both and the wave reduces
// them; no LDS. One wave per tile, four per workgroup.
template <int NP>
__global__ __launch_bounds__(256) void k_wmax_tiles_wide(ChunkView cv, uint64_t s, uint64_t e, uint64_t W,
                                                         uint64_t t_first, uint64_t ntiles,
                                                         unsigned long long* __restrict__ wmax,
                                                         uint32_t* __restrict__ ekey,
                                                         unsigned long long* __restrict__ eval) {
  const uint32_t lane = __lane_id();
  const uint64_t k = wave_global();
  if (k >= ntiles) return;
  const uint64_t c = t_first + k;
  const uint64_t r0 = c * kTileRows, lr0 = r0 + 16ull * lane;
  uint64_t off[16];
  lane_offsets<NP>(cv, c, lane, off);
  const uint64_t a = (s > r0 ? s : r0), b = (e < r0 + kTileRows ? e : r0 + kTileRows);   // rows [a, b)
  const uint64_t fw = (a - s) / W, lw = (b - 1 - s) / W;
  const uint64_t split = s + (fw + 1) * W;   // first row of window fw + 1
  uint64_t m0 = 0, m1 = 0;
#pragma unroll
  for (uint32_t j = 0; j < 16; ++j) {
    const uint64_t row = lr0 + j;
    if (row < a || row >= b) continue;
    if (row < split) m0 = max(m0, off[j]);
    else m1 = max(m1, off[j]);
  }
  m0 = wave_max_u64(m0);
  m1 = wave_max_u64(m1);
  if (lane == 0) {
    const uint64_t ws0 = s + fw * W, we0 = ws0 + W < e ? ws0 + W : e;
    if (ws0 >= r0 && we0 <= r0 + kTileRows) wmax[fw] = m0;
    ekey[2 * k] = (uint32_t)fw;
    eval[2 * k] = m0;
    ekey[2 * k + 1] = (uint32_t)lw;
    eval[2 * k + 1] = lw == fw ? m0 : m1;
    if (lw != fw) {
      const uint64_t ws1 = s + lw * W, we1 = ws1 + W < e ? ws1 + W : e;
      if (ws1 >= r0 && we1 <= r0 + kTileRows) wmax[lw] = m1;
    }
  }
}

// Windows of kWmaxBlockMin .. kWmaxBlockMax rows in one launch. A workgroup owns
// 4U consecutive tiles (wave w: tiles w, w + 4, ...), whose plane and tail bytes
// stay in registers: the maxima need one pass over them and the argmax rows a
// second, so nothing is read twice from memory except the rows of the first and
// last window that lie in a neighbour's tiles (on average W rows a workgroup,
// 6% at W = 1000). Offsets are compared as row_bytes_x gives them (the offset
// shifted left by 8 - r, the same order), in 32 bits up to three planes. Per
// tile: every lane reduces its 16 rows to at most two window segments (W >= 16),
// a segmented max over the lanes completes each window's part, and the lane
// where a window leaves the tile folds it into the window's LDS word. Bound by
// the read of planes and tail (and about 340 vector instructions a tile):
// 33,554,432 rows of 3 planes and 5 tail bits at W = 1000 took 83 us in six
// launches that read everything twice, 38 in this one (the read alone: 21).
constexpr uint32_t kWmaxWaves = 4;

template <int NP>
using WmaxKey = std::conditional_t<(NP <= 3), unsigned int, unsigned long long>;

__device__ __forceinline__ unsigned int wave_max_key(unsigned int v) { return wave_max_u32_dpp(v); }
__device__ __forceinline__ unsigned long long wave_max_key(unsigned long long v) { return wave_max_u64(v); }

template <int NP, int U>
__global__ __launch_bounds__(64 * kWmaxWaves) void k_wmax_block(ChunkView cv, uint64_t s, uint64_t e, uint32_t W,
                                                                uint32_t magic, uint64_t first_tile, uint64_t k,
                                                                double inv_scale, double* __restrict__ vals,
                                                                uint32_t want, uint16_t* __restrict__ out16,
                                                                uint64_t nout16) {
  using K = WmaxKey<NP>;
  constexpr uint32_t kTiles = kWmaxWaves * U;
  __shared__ K win[kTiles * kTileRows / kWmaxBlockMin + 2];
  const uint32_t lane = __lane_id(), wave = wave_in_wg();
  const uint64_t g0 = first_tile + (uint64_t)blockIdx.x * kTiles, g1 = min(g0 + kTiles, cv.ntiles);
  const uint64_t R0 = g0 * kTileRows, R1 = g1 * kTileRows;
  const uint64_t a = max(s, R0), b = min(e, R1);   // this workgroup's rows of [s, e)
  if (a >= b) {
    if (out16)
      for (uint64_t c = g0 + wave; c < g1; c += kWmaxWaves)
        if (c * 64 + lane < nout16) out16[c * 64 + lane] = 0;
    return;
  }
  // its windows w0 .. w0 + nw - 1; window i of them starts at row ws0 + i * W
  const uint64_t w0 = (a - s) / W;
  const uint64_t ws0 = s + w0 * W;
  const uint32_t nw = __umulhi((uint32_t)(b - 1 - ws0), magic) + 1;
  for (uint32_t i = threadIdx.x; i < nw; i += blockDim.x) win[i] = 0;
  RowBytes<NP> rb[U];
#pragma unroll
  for (int u = 0; u < U; ++u) load_row_bytes<NP>(cv, min(g0 + kWmaxWaves * u + wave, cv.ntiles - 1), lane, rb[u]);
  __syncthreads();
  // rows [lo, hi) outside the own tiles, all of window i; wave `first` takes the first tile
  auto halo = [&](uint64_t lo, uint64_t hi, uint32_t i, uint32_t first) {
    for (uint64_t c = lo / kTileRows + (wave + kWmaxWaves - first) % kWmaxWaves; c * kTileRows < hi; c += kWmaxWaves) {
      const uint64_t lr0 = c * kTileRows + 16ull * lane;
      K m = 0;
      if (lr0 < hi && lr0 + 16 > lo) {
        RowBytes<NP> hb;
        load_row_bytes<NP>(cv, c, lane, hb);
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j) {
          const K x = (K)row_bytes_x<NP>(hb, j);
          m = lr0 + j >= lo && lr0 + j < hi && x > m ? x : m;
        }
      }
      m = wave_max_key(m);
      if (lane == 0) atomicMax(&win[i], m);
    }
  };
  if (ws0 < R0) halo(ws0, R0, 0, 0);
  const uint64_t wend = min(ws0 + (uint64_t)nw * W, e);
  if (wend > R1) halo(R1, wend, nw - 1, kWmaxWaves / 2);
  // the lane's rows of [s, e) in tile g0 + 4u + wave: mask `in`, windows iA
  // (first row) and iB (last row), rows from `split` on in iB
  struct Seg {
    uint32_t in, iA, iB;
    int32_t split;
  };
  auto segments = [&](uint64_t c) {
    Seg q;
    const uint64_t lr0 = c * kTileRows + 16ull * lane;
    const uint32_t lo = lr0 >= a ? 0u : (a - lr0 < 16 ? (uint32_t)(a - lr0) : 16u);
    const uint32_t hi = lr0 >= b ? 0u : (b - lr0 < 16 ? (uint32_t)(b - lr0) : 16u);
    q.in = lo < hi ? ((1u << hi) - 1u) & ~((1u << lo) - 1u) : 0u;
    const uint32_t rel = (uint32_t)(lr0 - ws0);   // of a row >= ws0 whenever q.in != 0
    q.iA = q.in ? __umulhi(rel + lo, magic) : (lr0 < a ? 0u : nw - 1);
    q.iB = q.in ? __umulhi(rel + hi - 1, magic) : q.iA;
    q.split = (int32_t)(q.iB * W - rel);
    return q;
  };
  K x[U][16];
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (uint32_t j = 0; j < 16; ++j) x[u][j] = (K)row_bytes_x<NP>(rb[u], j);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint64_t c = g0 + kWmaxWaves * u + wave;
    if (c >= g1) break;
    const Seg q = segments(c);
    K mA = 0, mB = 0;
    if (__ballot(q.in != 0xFFFFu)) {   // the ends of [s, e)
#pragma unroll
      for (uint32_t j = 0; j < 16; ++j)
        if (!((q.in >> j) & 1u)) x[u][j] = 0;
    }
#pragma unroll
    for (uint32_t j = 0; j < 16; ++j) {
      if ((int32_t)j >= q.split) mB = x[u][j] > mB ? x[u][j] : mB;
      else mA = x[u][j] > mA ? x[u][j] : mA;
    }
    // mB of every lane of the run of lanes that end in the same window, from its first lane on
    K v = mB;
#pragma unroll
    for (uint32_t o = 1; o < 64; o <<= 1) {
      const K up = __shfl_up(v, o, 64);
      const uint32_t ku = (uint32_t)__shfl_up((int)q.iB, o, 64);
      if (lane >= o && ku == q.iB) v = up > v ? up : v;
    }
    const K prev = __shfl_up(v, 1, 64);
    const uint32_t kprev = (uint32_t)__shfl_up((int)q.iB, 1, 64);
    const uint32_t anext = (uint32_t)__shfl_down((int)q.iA, 1, 64);
    if (q.iA != q.iB) {   // window iA ends among this lane's rows
      const K t = lane > 0 && kprev == q.iA && prev > mA ? prev : mA;
      atomicMax(&win[q.iA], t);
    }
    if (lane == 63 || anext != q.iB) atomicMax(&win[q.iB], v);
  }
  __syncthreads();
  // the windows that start here (the others are a neighbour's to write)
  for (uint32_t i = threadIdx.x; i < nw; i += blockDim.x)
    if (ws0 + (uint64_t)i * W >= R0 && w0 + i < k)
      vals[w0 + i] = (double)(int64_t)((uint64_t)cv.base + ((uint64_t)win[i] >> (8u - cv.r))) * inv_scale;
  if (!out16) return;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint64_t c = g0 + kWmaxWaves * u + wave;
    if (c >= g1) break;
    uint32_t bits = 0;
    if (want) {
      const Seg q = segments(c);
      const K A = win[q.iA], B = win[q.iB];
#pragma unroll
      for (uint32_t j = 0; j < 16; ++j)
        bits |= (uint32_t)(x[u][j] == ((int32_t)j >= q.split ? B : A)) << j;
      bits &= q.in;
    }
    const uint64_t idx = c * 64 + lane;
    if (idx < nout16) out16[idx] = (uint16_t)bits;
  }
}

// Reduce-by-key over pairs sorted by window (one block of 256 pairs per
// workgroup). A run of equal windows that touches neither end of its block is
// complete: its max is written. The runs at the block's ends go to the next
// level as its pairs 2b and 2b+1 (the same run twice when it fills the block).
// last: one block holds every pair, so every run is complete.
__global__ __launch_bounds__(256) void k_wmax_reduce(const uint32_t* __restrict__ kin,
                                                     const unsigned long long* __restrict__ vin, uint64_t nin,
                                                     uint32_t* __restrict__ kout, unsigned long long* __restrict__ vout,
                                                     unsigned long long* __restrict__ wmax, uint32_t last) {
  __shared__ uint32_t sk[256];
  __shared__ unsigned long long sv[256];
  const uint32_t t = threadIdx.x;
  const uint64_t i = (uint64_t)blockIdx.x * 256 + t;
  const bool valid = i < nin;
  const uint32_t key = valid ? kin[i] : 0xFFFFFFFFu;
  sk[t] = key;
  sv[t] = valid ? vin[i] : 0ull;
  __syncthreads();
  // segmented inclusive max: keys are sorted, so sk[t-o] == key means the
  // whole span t-o .. t belongs to the run
  for (uint32_t o = 1; o < 256; o <<= 1) {
    const unsigned long long v = (t >= o && sk[t - o] == key) ? sv[t - o] : 0ull;
    __syncthreads();
    sv[t] = sv[t] > v ? sv[t] : v;
    __syncthreads();
  }
  if (!valid) return;
  const bool at_end = t == 255 || i == nin - 1;
  const bool run_end = at_end || sk[t + 1] != key;
  if (!run_end) return;
  const bool at_start = sk[0] == key;
  const unsigned long long m = sv[t];
  if (last || (!at_start && !at_end)) wmax[key] = m;
  if (!last) {
    if (at_start) {
      kout[2 * blockIdx.x] = key;
      vout[2 * blockIdx.x] = m;
    }
    if (at_end) {
      kout[2 * blockIdx.x + 1] = key;
      vout[2 * blockIdx.x + 1] = m;
    }
  }
}

// Every tile of the chunk: the rows of [s, e) equal to their window's max
// (want = 0: none), as the lane's 16 bits of the bitmap.
template <int NP>
__global__ __launch_bounds__(256) void k_wmax_argmax(ChunkView cv, uint64_t s, uint64_t e, uint64_t W, uint32_t want,
                                                     const unsigned long long* __restrict__ wmax,
                                                     uint16_t* __restrict__ out16, uint64_t nout16) {
  const uint32_t lane = __lane_id();
  {
    const uint64_t c = wave_global();   // one tile per wave
    if (c >= cv.ntiles) return;
    const uint64_t idx = c * 64 + lane;
    const uint64_t r0 = c * kTileRows, lr0 = r0 + 16ull * lane;
    uint32_t bits = 0;
    const bool tile_in = want && r0 < e && r0 + kTileRows > s;
    if (tile_in) {
      uint64_t off[16];
      lane_offsets<NP>(cv, c, lane, off);
      const bool lane_in = lr0 < e && lr0 + 16 > s;
      if (lane_in) {
        const uint64_t first = lr0 > s ? lr0 : s;
        uint64_t w = (first - s) / W;
        uint64_t next = s + (w + 1) * W;   // first row of the following window
        unsigned long long m = wmax[w];
#pragma unroll
        for (uint32_t b = 0; b < 16; ++b) {
          const uint64_t row = lr0 + b;
          if (row < s || row >= e) continue;
          if (row >= next) {
            w = (row - s) / W;
            next = s + (w + 1) * W;
            m = wmax[w];
          }
          bits |= (uint32_t)(off[b] == m) << b;
        }
      }
    }
    if (idx < nout16) out16[idx] = (uint16_t)bits;
  }
}

__global__ void k_wmax_values(const unsigned long long* __restrict__ wmax, uint64_t k, int64_t base, double inv_scale,
                              double* __restrict__ vals) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < k; i += (uint64_t)gridDim.x * blockDim.x)
    vals[i] = (double)(int64_t)((uint64_t)base + wmax[i]) * inv_scale;
}

// ---------------------------------------------------------------------------

WmaxLayout wmax_layout(uint64_t s, uint64_t e, uint64_t W) {
  WmaxLayout L;
  const uint64_t rows = e - s;
  L.nwin = rows ? (rows + W - 1) / W : 0;
  L.t_first = rows ? s / kTileRows : 0;
  L.ntiles = rows ? (e - 1) / kTileRows - L.t_first + 1 : 0;
  uint64_t at = 0;
  auto take = [&](uint64_t bytes) {
    const uint64_t here = at;
    at += (bytes + 255) & ~255ull;
    return here;
  };
  L.wmax = take(8 * (L.nwin ? L.nwin : 1));
  const uint64_t np = 2 * (L.ntiles ? L.ntiles : 1);
  L.k[0] = take(4 * np);
  L.v[0] = take(8 * np);
  const uint64_t np2 = 2 * ((np + 255) / 256);
  L.k[1] = take(4 * np2);
  L.v[1] = take(8 * np2);
  L.bytes = at;
  return L;
}

template <int NP>
static hipError_t launch_wmax_np(const ChunkView& cv, uint64_t s, uint64_t e, uint64_t W, const WmaxLayout& L,
                                 uint8_t* scratch, hipStream_t st) {
  unsigned long long* wmax = reinterpret_cast<unsigned long long*>(scratch + L.wmax);
  uint32_t* kb[2] = {reinterpret_cast<uint32_t*>(scratch + L.k[0]), reinterpret_cast<uint32_t*>(scratch + L.k[1])};
  unsigned long long* vb[2] = {reinterpret_cast<unsigned long long*>(scratch + L.v[0]),
                               reinterpret_cast<unsigned long long*>(scratch + L.v[1])};
  if (W >= kTileRows)
    launch_k(k_wmax_tiles_wide<NP>, dim3((uint32_t)((L.ntiles + 3) / 4)), dim3(256), 0, st, cv, s, e, W, L.t_first,
             L.ntiles, wmax, kb[0], vb[0]);
  else
    launch_k(k_wmax_tiles<NP>, dim3((uint32_t)L.ntiles), dim3(64), 0, st, cv, s, e, W, L.t_first, wmax, kb[0], vb[0]);
  uint64_t nin = 2 * L.ntiles;
  uint32_t cur = 0;
  while (true) {
    const uint64_t nb = (nin + 255) / 256;
    const uint32_t last = nb == 1 ? 1u : 0u;
    launch_k(k_wmax_reduce, dim3((uint32_t)nb), dim3(256), 0, st, static_cast<const uint32_t*>(kb[cur]),
             static_cast<const unsigned long long*>(vb[cur]), nin, kb[cur ^ 1], vb[cur ^ 1], wmax, last);
    if (last) break;
    nin = 2 * nb;
    cur ^= 1;
  }
  return hipGetLastError();
}

template <int NP>
static void launch_wmax_block_np(const ChunkView& cv, uint64_t s, uint64_t e, uint32_t W, uint64_t k, double inv_scale,
                                 double* vals, bool want, uint64_t* argmax, hipStream_t st) {
  const uint32_t magic = (uint32_t)(((1ull << 32) + W - 1) / W);   // x / W = mulhi(x, magic) while x * W < 2^32
  // with a bitmap every tile of the chunk is written, else only [s, e) is visited
  const uint64_t t0 = argmax ? 0 : s / kTileRows;
  const uint64_t nt = (argmax ? cv.ntiles : (e + kTileRows - 1) / kTileRows) - t0;
  const uint64_t nout16 = 4 * ((cv.n + 63) / 64);
  uint16_t* o16 = reinterpret_cast<uint16_t*>(argmax);
  const uint32_t w = want ? 1u : 0u;
  // few tiles: one per wave, so that they spread over the CUs
  if (nt <= kWmaxSmallTiles)
    launch_k((k_wmax_block<NP, 1>), dim3((uint32_t)((nt + kWmaxWaves - 1) / kWmaxWaves)), dim3(64 * kWmaxWaves), 0, st,
             cv, s, e, W, magic, t0, k, inv_scale, vals, w, o16, nout16);
  else
    launch_k((k_wmax_block<NP, 4>), dim3((uint32_t)((nt + 4 * kWmaxWaves - 1) / (4 * kWmaxWaves))),
             dim3(64 * kWmaxWaves), 0, st, cv, s, e, W, magic, t0, k, inv_scale, vals, w, o16, nout16);
}

// The rows read beyond a workgroup's own tiles (W on average; none where the
// windows' starts divide its 16 tiles) are further dependent loads, and with
// 64-bit keys (four planes and more) a CU holds half the waves to hide them: the
// launches that read everything twice, but stream, catch up the sooner the larger
// the column and the fewer its planes. 134,217,728 rows of four planes, us in one
// launch and in six: W = 1000 227 and 259, 2047 234 and 234, 7001 291 and 230, 4096
// 185 and 228; 16,777,216 rows at 7001 42 and 45; 134,217,728 rows of six planes at
// 7001 284 and 298. Three planes and fewer: at most 0.77 of the six everywhere.
// Columns of one tile a wave (four in a workgroup, so that at W = 8192 they read
// three times their rows): 7 us and 23 for 2,097,152 rows of four planes.
bool wmax_block_form(const ChunkView& cv, uint64_t s, uint64_t e, uint64_t W) {
  if (W < kWmaxBlockMin || W > kWmaxBlockMax) return false;
  constexpr uint64_t kOwnRows = 16 * kTileRows;
  if (cv.P <= 3 || (s % kOwnRows == 0 && kOwnRows % W == 0)) return true;
  uint64_t most = cv.P == 4 ? 1536 : cv.P == 5 ? 2560 : 5120;
  for (uint64_t tiles = (e - s + kTileRows - 1) / kTileRows; tiles <= 65536 && most < kWmaxBlockMax; tiles *= 2) most *= 2;
  return W <= most;
}

hipError_t launch_wmax_block(const ChunkView& cv, uint64_t s, uint64_t e, uint64_t W, uint64_t k, double inv_scale,
                             double* vals, bool want, uint64_t* argmax, hipStream_t st) {
  if (W < kWmaxBlockMin || W > kWmaxBlockMax || s >= e || e > cv.n) return hipErrorInvalidValue;
#define BUFF_WB(NP) launch_wmax_block_np<NP>(cv, s, e, (uint32_t)W, k, inv_scale, vals, want, argmax, st)
  switch (cv.P) {
    case 0: BUFF_WB(0); break;
    case 1: BUFF_WB(1); break;
    case 2: BUFF_WB(2); break;
    case 3: BUFF_WB(3); break;
    case 4: BUFF_WB(4); break;
    case 5: BUFF_WB(5); break;
    case 6: BUFF_WB(6); break;
    case 7: BUFF_WB(7); break;
    default: return hipErrorInvalidValue;
  }
#undef BUFF_WB
  return hipGetLastError();
}

hipError_t launch_wmax(const ChunkView& cv, uint64_t s, uint64_t e, uint64_t W, const WmaxLayout& L,
                       uint8_t* scratch, hipStream_t st) {
  if (L.ntiles == 0) return hipSuccess;
  switch (cv.P) {
    case 0: return launch_wmax_np<0>(cv, s, e, W, L, scratch, st);
    case 1: return launch_wmax_np<1>(cv, s, e, W, L, scratch, st);
    case 2: return launch_wmax_np<2>(cv, s, e, W, L, scratch, st);
    case 3: return launch_wmax_np<3>(cv, s, e, W, L, scratch, st);
    case 4: return launch_wmax_np<4>(cv, s, e, W, L, scratch, st);
    case 5: return launch_wmax_np<5>(cv, s, e, W, L, scratch, st);
    case 6: return launch_wmax_np<6>(cv, s, e, W, L, scratch, st);
    case 7: return launch_wmax_np<7>(cv, s, e, W, L, scratch, st);
    default: return launch_wmax_np<8>(cv, s, e, W, L, scratch, st);
  }
}

hipError_t launch_wmax_argmax(const ChunkView& cv, uint64_t s, uint64_t e, uint64_t W, bool want,
                              const uint8_t* scratch, const WmaxLayout& L, uint64_t* out, hipStream_t st) {
  if (cv.ntiles == 0) return hipSuccess;
  const unsigned long long* wmax = reinterpret_cast<const unsigned long long*>(scratch + L.wmax);
  uint16_t* o16 = reinterpret_cast<uint16_t*>(out);
  const uint64_t nout16 = 4 * ((cv.n + 63) / 64);
  const uint32_t wg = (uint32_t)((cv.ntiles + 3) / 4);
  const uint32_t w = want && L.nwin ? 1u : 0u;
#define BUFF_ARG(NP) launch_k(k_wmax_argmax<NP>, dim3(wg), dim3(256), 0, st, cv, s, e, W, w, wmax, o16, nout16)
  switch (cv.P) {
    case 0: BUFF_ARG(0); break;
    case 1: BUFF_ARG(1); break;
    case 2: BUFF_ARG(2); break;
    case 3: BUFF_ARG(3); break;
    case 4: BUFF_ARG(4); break;
    case 5: BUFF_ARG(5); break;
    case 6: BUFF_ARG(6); break;
    case 7: BUFF_ARG(7); break;
    default: BUFF_ARG(8); break;
  }
#undef BUFF_ARG
  return hipGetLastError();
}

hipError_t launch_wmax_values(const uint8_t* scratch, const WmaxLayout& L, uint64_t k, int64_t base, double inv_scale,
                              double* vals, hipStream_t st) {
  if (k == 0) return hipSuccess;
  const unsigned long long* wmax = reinterpret_cast<const unsigned long long*>(scratch + L.wmax);
  const uint32_t wg = (uint32_t)std::min<uint64_t>((k + 255) / 256, 1024);
  launch_k(k_wmax_values, dim3(wg), dim3(256), 0, st, wmax, k, base, inv_scale, vals);
  return hipGetLastError();
}

}  // namespace buffgpu
