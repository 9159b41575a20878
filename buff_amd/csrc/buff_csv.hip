// CSV -> f64 ingest on the device: construct_file_iterator_skip_newline::<f64>
// (database/src/client.rs:163-182) over a file's bytes resident in HBM.
//
// The reference reads lines (split on '\n', a trailing "\r" removed), splits
// each line on `delim`, skips the first skip_val items of the line, and keeps
// every item `f64::from_str` accepts, in file order. Here:
//   k_csv_blocks  one workgroup per 4 KiB block: items ending in the block,
//                 items after its last newline, its last delimiter;
//   k_csv_scan    one workgroup: prefixes over the blocks (item base, index of
//                 the block's first item within its line, previous delimiter);
//   k_csv_parse   one workgroup per block: the items ending in it are listed in
//                 LDS and parsed one per lane in turn; each value goes to its
//                 item's slot, an item that is none leaves kCsvNone there;
//   k_csv_okscan, k_csv_compact  only when some item was rejected: the values
//                 moved to their final place.
// Parsing is exact: Rust's grammar (optional sign; digits with an optional
// point and at least one digit; optional exponent; or inf / infinity / nan in
// any case), the value correctly rounded (ties to even) by the exact fast path
// (at most 2^53 for the digits and |exponent| <= 22: one IEEE multiply or
// divide by an exact power of ten) or else by the 192-bit product of the
// normalized digits with 5^q truncated to 128 bits, whose rounding is decided
// unless a carry from the truncated part could reach the rounding bit (then
// the item is reported undecided). More than 19 significant digits: both
// 19-digit bounds must round alike.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "buff_csv.h"
#include "buff_device.h"
#include "buff_launch.h"

namespace buffgpu {

// ---- host: the table of 5^q ------------------------------------------------------

namespace {

struct Big {  // little-endian base-2^32 magnitude
  std::vector<uint32_t> d;
  uint32_t bits() const {
    for (size_t i = d.size(); i-- > 0;)
      if (d[i]) return (uint32_t)(32 * i + 32 - __builtin_clz(d[i]));
    return 0;
  }
  void mul_small(uint32_t m) {
    uint64_t c = 0;
    for (uint32_t& x : d) {
      const uint64_t v = (uint64_t)x * m + c;
      x = (uint32_t)v;
      c = v >> 32;
    }
    if (c) d.push_back((uint32_t)c);
  }
  void div_small(uint32_t m) {  // floor division
    uint64_t r = 0;
    for (size_t i = d.size(); i-- > 0;) {
      const uint64_t v = (r << 32) | d[i];
      d[i] = (uint32_t)(v / m);
      r = v % m;
    }
  }
  bool bit(uint32_t k) const { return k / 32 < d.size() && ((d[k / 32] >> (k % 32)) & 1u); }
  // bits [k, k+64) as an integer
  uint64_t window64(int64_t k) const {
    uint64_t v = 0;
    for (int j = 63; j >= 0; --j) v = (v << 1) | (k + j >= 0 && bit((uint32_t)(k + j)) ? 1u : 0u);
    return v;
  }
};

}  // namespace

void csv_pow5_table(Pow5* out) {
  for (int q = kPow5Min; q <= kPow5Max; ++q) {
    Pow5& t = out[q - kPow5Min];
    const uint32_t k = (uint32_t)(q < 0 ? -q : q);
    Big p5{{1u}};
    for (uint32_t i = 0; i < k; ++i) p5.mul_small(5);
    const uint32_t L = p5.bits();
    if (q >= 0) {
      // 5^q = (5^q << (128 - L)) * 2^(L - 128); exact while it fits 128 bits
      const int64_t sh = (int64_t)L - 128;
      t.hi = p5.window64(sh + 64);
      t.lo = p5.window64(sh);
      t.e = (int32_t)sh;
      t.exact = L <= 128 ? 1u : 0u;
    } else {
      // 5^q = 2^(127+L) / 5^k * 2^-(127+L); floor of the quotient by repeated /5
      Big a;
      a.d.assign((127 + L) / 32 + 1, 0u);
      a.d[(127 + L) / 32] = 1u << ((127 + L) % 32);
      for (uint32_t i = 0; i < k; ++i) a.div_small(5);
      t.hi = a.window64(64);
      t.lo = a.window64(0);
      t.e = -(int32_t)(127 + L);
      t.exact = 0;
    }
  }
}

// ---- device: one item -> f64 -------------------------------------------------------

namespace {

__host__ __device__ __forceinline__ bool csv_digit(uint32_t c) { return c - '0' < 10u; }

// The correctly rounded f64 bits of w * 10^q (w >= 1), or false when the
// truncated power leaves the rounding open.
__device__ bool round_w10q(uint64_t w, int64_t q, const Pow5* __restrict__ tab, uint64_t* bits) {
  if (q < kPow5Min) {  // below half the smallest subnormal
    *bits = 0;
    return true;
  }
  if (q > kPow5Max) {
    *bits = 0x7FF0000000000000ull;
    return true;
  }
  const Pow5 t = tab[q - kPow5Min];
  const int lz = __clzll((long long)w);
  const uint64_t wn = w << lz;
  const uint64_t a_lo = wn * t.hi, a_hi = __umul64hi(wn, t.hi);
  const uint64_t b_lo = wn * t.lo, b_hi = __umul64hi(wn, t.lo);
  const uint64_t lo = b_lo;
  const uint64_t mid = a_lo + b_hi;
  const uint64_t hi = a_hi + (mid < a_lo ? 1u : 0u);
  const int m = (hi >> 63) ? 191 : 190;  // msb of the 192-bit product
  const int64_t ex = (int64_t)m + t.e + q - lz;
  if (ex > 1023) {
    *bits = 0x7FF0000000000000ull;
    return true;
  }
  const int64_t K = ex >= -1022 ? 53 : ex + 1075;  // mantissa bits kept
  if (K < 0) {
    *bits = 0;
    return true;
  }
  const int hs = (int)(m - K + 1 - 128);  // lsb of the kept bits within hi
  const int hr = hs - 1;                   // rounding bit within hi (>= 9)
  uint64_t mant = hs >= 64 ? 0 : (hi >> hs);
  const uint64_t round = (hi >> hr) & 1u;
  const uint64_t below_mask = (1ull << hr) - 1;
  const uint64_t below = hi & below_mask;
  bool sticky;
  if (t.exact) {
    sticky = below || mid || lo;
  } else {
    if (below == below_mask && mid == ~0ull) return false;
    sticky = true;  // the true product exceeds the truncated one
  }
  if (round && (sticky || (mant & 1u))) mant += 1;
  uint64_t b = ex >= -1022 ? ((uint64_t)(ex + 1022) << 52) + mant : mant;
  if (b >= 0x7FF0000000000000ull) b = 0x7FF0000000000000ull;
  *bits = b;
  return true;
}

__constant__ double kPow10Exact[23] = {1e0,  1e1,  1e2,  1e3,  1e4,  1e5,  1e6,  1e7,  1e8,  1e9,  1e10, 1e11,
                                       1e12, 1e13, 1e14, 1e15, 1e16, 1e17, 1e18, 1e19, 1e20, 1e21, 1e22};

// The correctly rounded bits of w * 10^q (w >= 1), or false when undecided:
// the exact fast path; then, for q < 0 with 5^-q dividing w (the only way the
// value can be a dyadic rational, so sit exactly on a double or a tie),
// (w / 5^-q) * 2^q from one correctly rounded u64 -> f64 conversion and an
// exact scaling; otherwise the 192-bit product, where the value cannot sit on
// a boundary and only a carry out of the truncated part is left open.
__device__ bool w10q_bits(uint64_t w, int64_t q, const Pow5* __restrict__ tab, uint64_t* bits) {
  if (q >= -22 && q <= 22 && w <= (1ull << 53)) {
    const double v = (double)w;
    *bits = (uint64_t)__double_as_longlong(q >= 0 ? v * kPow10Exact[q] : v / kPow10Exact[-q]);
    return true;
  }
  if (q < 0 && q >= -27) {
    uint64_t p5 = 1;
    for (int64_t j = 0; j < -q; ++j) p5 *= 5;
    if (w % p5 == 0) {
      *bits = (uint64_t)__double_as_longlong(ldexp((double)(w / p5), (int)q));
      return true;
    }
  }
  return round_w10q(w, q, tab, bits);
}

__device__ __forceinline__ bool ci_eq(const uint8_t* p, const char* word, uint64_t n) {
  for (uint64_t j = 0; j < n; ++j)
    if ((uint32_t)(p[j] | 0x20u) != (uint32_t)word[j]) return false;
  return true;
}

// 0: not an f64 in Rust's grammar; 1: *out holds the value; 2: undecided.
__device__ int parse_item(const uint8_t* __restrict__ p, uint64_t n, const Pow5* __restrict__ tab, double* out) {
  if (n == 0) return 0;
  uint64_t i = 0;
  bool neg = false;
  if (p[0] == '+' || p[0] == '-') {
    neg = p[0] == '-';
    i = 1;
  }
  const uint64_t sign = neg ? 0x8000000000000000ull : 0ull;
  const uint64_t rest = n - i;
  if ((rest == 3 && ci_eq(p + i, "inf", 3)) || (rest == 8 && ci_eq(p + i, "infinity", 8))) {
    *out = __longlong_as_double((long long)(sign | 0x7FF0000000000000ull));
    return 1;
  }
  if (rest == 3 && ci_eq(p + i, "nan", 3)) {
    *out = __longlong_as_double((long long)(sign | 0x7FF8000000000000ull));
    return 1;
  }
  uint64_t w = 0;
  int nsig = 0;
  int64_t q = 0;
  bool trunc = false;
  uint64_t ndig = 0;
  while (i < n && csv_digit(p[i])) {
    const uint32_t d = p[i] - '0';
    ++ndig;
    if (w == 0 && d == 0) {
    } else if (nsig < 19) {
      w = w * 10 + d;
      ++nsig;
    } else {
      ++q;
      trunc |= d != 0;
    }
    ++i;
  }
  if (i < n && p[i] == '.') {
    ++i;
    while (i < n && csv_digit(p[i])) {
      const uint32_t d = p[i] - '0';
      ++ndig;
      if (w == 0 && d == 0) {
        --q;
      } else if (nsig < 19) {
        w = w * 10 + d;
        ++nsig;
        --q;
      } else {
        trunc |= d != 0;
      }
      ++i;
    }
  }
  if (ndig == 0) return 0;
  if (i < n && (p[i] | 0x20u) == 'e') {
    ++i;
    bool eneg = false;
    if (i < n && (p[i] == '+' || p[i] == '-')) {
      eneg = p[i] == '-';
      ++i;
    }
    if (i >= n || !csv_digit(p[i])) return 0;
    int64_t ev = 0;
    while (i < n && csv_digit(p[i])) {
      if (ev < 100000000) ev = ev * 10 + (p[i] - '0');
      ++i;
    }
    q += eneg ? -ev : ev;
  }
  if (i != n) return 0;
  uint64_t bits = 0;
  if (w != 0) {
    if (!w10q_bits(w, q, tab, &bits)) return 2;
    if (trunc) {  // the digits past the 19th put the value strictly between w and w + 1 units
      uint64_t b2 = 0;
      if (!w10q_bits(w + 1, q, tab, &b2) || b2 != bits) return 2;
    }
  }
  *out = __longlong_as_double((long long)(sign | bits));
  return 1;
}

__device__ __forceinline__ bool csv_delim(uint32_t c, uint32_t delim) { return c == delim || c == '\n'; }

// The 16 bytes at `at` (zero past the end).
__device__ __forceinline__ uint4 load16(const uint8_t* __restrict__ text, uint64_t len, uint64_t at) {
  if (at + 16 <= len) return *reinterpret_cast<const uint4*>(text + at);
  uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < 16; ++j) w[j / 4] |= (at + j < len ? (uint32_t)text[at + j] : 0u) << (8 * (j % 4));
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// bit 0 of each byte of four dwords -> 16 bits, in byte order
__device__ __forceinline__ uint32_t byte_bits(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  const uint32_t lo = __builtin_amdgcn_udot4(b, 0x80402010u, __builtin_amdgcn_udot4(a, 0x08040201u, 0u, false), false);
  const uint32_t hi = __builtin_amdgcn_udot4(d, 0x80402010u, __builtin_amdgcn_udot4(c, 0x08040201u, 0u, false), false);
  return lo | (hi << 8);
}
__device__ __forceinline__ uint32_t eq_bytes(const uint4& w, uint32_t c) {
  const uint32_t D = 0x01010101u * c;
  return byte_bits(swar_eq(w.x, D) >> 7, swar_eq(w.y, D) >> 7, swar_eq(w.z, D) >> 7, swar_eq(w.w, D) >> 7);
}

// A lane's 16 bytes as masks (bit j: byte j): newlines, delimiters (newlines
// among them), and the bytes that end an item: delimiters, and the last byte of
// the text after any other byte.
struct LaneMasks {
  uint32_t nl, dl, ends;
};
__device__ __forceinline__ LaneMasks lane_masks(const uint4& w, uint64_t at, uint64_t len, uint32_t delim) {
  const uint32_t valid = at + 16 <= len ? 0xFFFFu : (at < len ? (1u << (uint32_t)(len - at)) - 1u : 0u);
  LaneMasks m;
  m.nl = eq_bytes(w, '\n') & valid;
  m.dl = (eq_bytes(w, delim) & valid) | m.nl;
  m.ends = m.dl | (valid && at + 16 >= len ? 1u << (uint32_t)(len - 1 - at) : 0u);
  return m;
}
// 1 + the position in the block of the highest bit of a lane's mask (0: none)
__device__ __forceinline__ uint32_t last_of(uint32_t m, uint32_t base) { return m ? base + 32u - (uint32_t)__clz(m) : 0u; }

// Inclusive max over the lanes up to this one.
__device__ __forceinline__ uint32_t wave_incl_max_u32(uint32_t v) {
  uint32_t s = v;
  s = max(s, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)s, 0x111, 0xf, 0xf, false));   // row_shr:1
  s = max(s, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)s, 0x112, 0xf, 0xf, false));   // row_shr:2
  s = max(s, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)s, 0x114, 0xf, 0xf, false));   // row_shr:4
  s = max(s, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)s, 0x118, 0xf, 0xf, false));   // row_shr:8
  s = max(s, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)s, 0x142, 0xa, 0xf, false));   // row_bcast:15
  s = max(s, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)s, 0x143, 0xc, 0xf, false));   // row_bcast:31
  return s;
}

// Exclusive sum / max over the lanes of a workgroup of NW waves in lane order;
// *total gets the workgroup's. lds: NW words of its own.
template <uint32_t NW>
__device__ __forceinline__ uint32_t wg_excl_sum(uint32_t v, uint32_t* lds, uint32_t* total) {
  const uint32_t lane = __lane_id(), wave = wave_in_wg();
  const uint32_t ex = wave_excl_scan_u32(v, lane);
  if (lane == 63) lds[wave] = ex + v;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (uint32_t w = 0; w < NW; ++w) {
    before += w < wave ? lds[w] : 0u;
    all += lds[w];
  }
  *total = all;
  return before + ex;
}
template <uint32_t NW>
__device__ __forceinline__ uint32_t wg_excl_max(uint32_t v, uint32_t* lds, uint32_t* total) {
  const uint32_t lane = __lane_id(), wave = wave_in_wg();
  const uint32_t in = wave_incl_max_u32(v);
  uint32_t ex = (uint32_t)__shfl_up((int)in, 1, 64);
  if (lane == 0) ex = 0;
  if (lane == 63) lds[wave] = in;
  __syncthreads();
  uint32_t all = 0;
#pragma unroll
  for (uint32_t w = 0; w < NW; ++w) {
    ex = max(ex, w < wave ? lds[w] : 0u);
    all = max(all, lds[w]);
  }
  *total = all;
  return ex;
}

// An item of up to 8 digits, a point and up to 8 digits behind an optional sign
// (what a data file holds), by byte-parallel steps: `end` is one past its last
// byte in LDS (16 readable bytes before it), n its length. false: not of this
// form (parse_item decides). The digits make w <= 2^53 and the value is w / 10^f,
// the exact fast path of w10q_bits. Four digits take two dot products.
__device__ __forceinline__ uint32_t unaligned_u32(const uint8_t* p) {
  const uint32_t a = (uint32_t)(uintptr_t)p & 3u;
  const uint32_t* w = reinterpret_cast<const uint32_t*>(p - a);
  return __builtin_amdgcn_alignbyte(w[1], w[0], a);
}
__device__ __forceinline__ uint32_t four_digits(uint32_t d) {   // byte 0 the first digit
  return __builtin_amdgcn_udot4(d, 0x0000010Au, 0u, false) * 100u + __builtin_amdgcn_udot4(d, 0x010A0000u, 0u, false);
}
// The n <= 8 digits before `end` as a number (their characters checked before).
__device__ __forceinline__ uint32_t eight_digits(const uint8_t* end, uint32_t n) {
  // the first dword holds the digits before the last four
  const uint32_t hi = unaligned_u32(end - 8) ^ 0x30303030u, lo = unaligned_u32(end - 4) ^ 0x30303030u;
  const uint32_t kh = n > 4 ? n - 4 : 0u, kl = n < 4 ? n : 4u;
  const uint32_t mh = kh ? 0xFFFFFFFFu << (8 * (4 - kh)) : 0u, ml = kl ? 0xFFFFFFFFu << (8 * (4 - kl)) : 0u;
  return four_digits(hi & mh) * 10000u + four_digits(lo & ml);
}
// bits of the bytes that are no digit
__device__ __forceinline__ uint32_t non_digits(uint32_t w) {
  const uint32_t d = w ^ 0x30303030u;
  return ((((d & 0x7F7F7F7Fu) + 0x76767676u) | d) >> 7) & 0x01010101u;
}
__device__ __forceinline__ bool parse_short(const uint8_t* end, uint32_t n, const double* p10, double* out) {
  const uint32_t c0 = end[-(int)n];
  const bool neg = c0 == '-';
  const uint32_t m = n - (neg || c0 == '+' ? 1u : 0u);   // bytes after the sign
  if (n > 16 || m == 0) return false;
  const uint32_t nd = byte_bits(non_digits(unaligned_u32(end - 16)), non_digits(unaligned_u32(end - 12)),
                                non_digits(unaligned_u32(end - 8)), non_digits(unaligned_u32(end - 4))) &
                      (0xFFFFu << (16 - m));
  // at most one other byte, the point: bit 15 - f
  const uint32_t f = nd ? __clz(nd) - 16u : 0u;
  const uint32_t point = nd ? 1u : 0u;
  const uint32_t ni = m - f - point;
  if ((nd & (nd - 1u)) || (nd && end[-(int)f - 1] != '.') || f > 8 || ni > 8 || f + ni == 0) return false;
  const double p = p10[f];
  const uint64_t w = (uint64_t)eight_digits(end - f - point, ni) * (uint32_t)p + eight_digits(end, f);
  if (w > (1ull << 53)) return false;
  const double v = (double)w / p;
  *out = neg ? -v : v;
  return true;
}

}  // namespace

__global__ __launch_bounds__(256) void k_csv_blocks(const uint8_t* __restrict__ text, uint64_t len, uint32_t delim,
                                                    CsvBlock* __restrict__ blk) {
  __shared__ uint32_t s_nl[4], s_dl[4], s_hi[4], s_tok[4], s_since[4];
  const uint64_t b = blockIdx.x;
  const uint32_t lane = __lane_id(), wave = wave_in_wg(), base = 16 * threadIdx.x;
  const uint64_t at = b * kCsvBlock + base;
  const uint4 w = load16(text, len, at);
  const LaneMasks m = lane_masks(w, at, len, delim);
  const uint32_t ntok = wave_total_u32(__popc(m.ends));
  const uint32_t nl = wave_max_u32_dpp(last_of(m.nl, base)), dl = wave_max_u32_dpp(last_of(m.dl, base));
  const bool hi = __ballot(((w.x | w.y | w.z | w.w) & 0x80808080u) != 0) != 0;
  if (lane == 0) {
    s_nl[wave] = nl;
    s_dl[wave] = dl;
    s_hi[wave] = hi ? 1u : 0u;
    s_tok[wave] = ntok;
  }
  __syncthreads();
  // items after the block's last newline: their bytes lie at or after `last`
  const uint32_t last = max(max(s_nl[0], s_nl[1]), max(s_nl[2], s_nl[3]));
  const uint32_t after = last <= base ? m.ends : (last >= base + 16 ? 0u : m.ends >> (last - base));
  const uint32_t since = wave_total_u32(__popc(after));
  if (lane == 0) s_since[wave] = since;
  __syncthreads();
  if (threadIdx.x == 0) {
    CsvBlock o;
    o.ntok = (uint16_t)(s_tok[0] + s_tok[1] + s_tok[2] + s_tok[3]);
    o.since = (uint16_t)(s_since[0] + s_since[1] + s_since[2] + s_since[3]);
    o.last_delim = (uint16_t)max(max(s_dl[0], s_dl[1]), max(s_dl[2], s_dl[3]));
    o.flags = (uint16_t)((last ? kCsvHasNewline : 0u) | (s_hi[0] | s_hi[1] | s_hi[2] | s_hi[3] ? kCsvNonAscii : 0u));
    blk[b] = o;
  }
}

// One workgroup of 1024 threads, each taking 8 consecutive blocks (two dwordx4
// pairs of 8-byte facts), 8192 blocks a round: item base, line index and
// previous delimiter of every block, totals[0..1], and the parse's counters
// cleared. A block's line index is its item base less the items up to the last
// newline before it, whose count only grows: a max scan.
__global__ __launch_bounds__(1024) void k_csv_scan(const CsvBlock* __restrict__ blk, CsvPre* __restrict__ pre,
                                                   uint64_t nblocks, unsigned long long* __restrict__ totals) {
  constexpr uint32_t kPer = 8, kRound = 1024 * kPer;
  __shared__ uint32_t s_sum[2][16], s_nl[2][16], s_dl[2][16];
  if (threadIdx.x >= 2 && threadIdx.x < kCsvWords) totals[threadIdx.x] = threadIdx.x == 5 ? ~0ull : 0ull;
  uint64_t carry_tok = 0;     // items of earlier rounds
  uint64_t carry_line = 0;    // their items up to the last newline
  int64_t carry_delim = -1;
  uint32_t nonascii = 0, par = 0;
  for (uint64_t base = 0; base < nblocks; base += kRound, par ^= 1u) {
    const uint64_t i0 = base + (uint64_t)threadIdx.x * kPer;
    CsvBlock c[kPer];
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) c[q] = i0 + q < nblocks ? blk[i0 + q] : CsvBlock{0, 0, 0, 0};
    uint32_t tok = 0;
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
      tok += c[q].ntok;
      nonascii |= c[q].flags & kCsvNonAscii;
    }
    // one LDS set per round parity: a wave can be a round ahead of the slowest
    uint32_t sum = 0, nl_all = 0, dl_all = 0;
    const uint32_t ex = wg_excl_sum<16>(tok, s_sum[par], &sum);
    // 1 + items of this round up to the newline; 1 + position in this round of the delimiter
    uint32_t nl = 0, dl = 0, at = ex;
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
      at += c[q].ntok;
      if (c[q].flags & kCsvHasNewline) nl = at - c[q].since + 1;
      if (c[q].last_delim) dl = (threadIdx.x * kPer + q) * kCsvBlock + c[q].last_delim;
    }
    uint32_t nl_ex = wg_excl_max<16>(nl, s_nl[par], &nl_all);
    uint32_t dl_ex = wg_excl_max<16>(dl, s_dl[par], &dl_all);
    at = ex;
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
      if (i0 + q < nblocks) {
        CsvPre p;
        p.tok_base = carry_tok + at;
        p.ok_base = 0;
        p.line_idx = (uint32_t)(p.tok_base - (nl_ex ? carry_tok + (nl_ex - 1) : carry_line));
        p.ok = 0;
        p.prev_delim = dl_ex ? (int64_t)(base * kCsvBlock + dl_ex - 1) : carry_delim;
        pre[i0 + q] = p;
      }
      at += c[q].ntok;
      if (c[q].flags & kCsvHasNewline) nl_ex = at - c[q].since + 1;
      if (c[q].last_delim) dl_ex = (threadIdx.x * kPer + q) * kCsvBlock + c[q].last_delim;
    }
    if (nl_all) carry_line = carry_tok + (nl_all - 1);
    if (dl_all) carry_delim = (int64_t)(base * kCsvBlock + dl_all - 1);
    carry_tok += sum;
  }
  const bool any = __syncthreads_or(nonascii != 0) != 0;
  if (threadIdx.x == 0) {
    totals[0] = carry_tok;
    totals[1] = any ? 1 : 0;
  }
}

// The parsed-item base of every block (only when some item was rejected), each
// lane 16 consecutive blocks, 4096 per step.
__global__ __launch_bounds__(256) void k_csv_okscan(CsvPre* __restrict__ pre, uint64_t nblocks) {
  constexpr uint32_t kPer = 16;
  __shared__ uint32_t s_sum[2][4];
  uint64_t carry = 0;
  uint32_t par = 0;
  for (uint64_t base = 0; base < nblocks; base += 256ull * kPer, par ^= 1u) {
    const uint64_t i0 = base + (uint64_t)threadIdx.x * kPer;
    uint32_t oks[kPer], ok = 0, sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) oks[q] = i0 + q < nblocks ? pre[i0 + q].ok : 0u;
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) ok += oks[q];
    uint64_t acc = carry + wg_excl_sum<4>(ok, s_sum[par], &sum);
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
      if (i0 + q < nblocks) pre[i0 + q].ok_base = acc;
      acc += oks[q];
    }
    carry += sum;
  }
}

// Bound by its vector instructions: the items are listed in LDS first, so that
// lane t parses item t, t + 256, ... (a lane that parsed the items of its own 16
// bytes left others idle and scattered the values), and a short decimal takes
// about 100 instructions instead of a loop over its bytes. 3,000,000 values of
// 9 bytes: 88.7 -> 30.5 us, the block facts 22.0 -> 9.8, the scan 20.9 -> 12.9.
__global__ __launch_bounds__(256) void k_csv_parse(const uint8_t* __restrict__ text, uint64_t len, uint32_t delim,
                                                   uint32_t skip, const Pow5* __restrict__ tab,
                                                   CsvPre* __restrict__ pre, double* __restrict__ dst, uint64_t cap,
                                                   CsvSlow* __restrict__ slow, uint64_t slow_cap,
                                                   unsigned long long* __restrict__ totals) {
  // the block and the 512 bytes before it in LDS: items are parsed from there
  constexpr uint32_t kHalo = 512;
  __shared__ __align__(16) uint8_t txt[kHalo + kCsvBlock + 16];   // unaligned_u32 reads a dword further
  __shared__ uint16_t s_end[kCsvBlock];   // per item: the position in the block of the byte that ends it
  __shared__ uint32_t s_skip[kCsvBlock / 32];   // bit per item: among the first `skip` of its line
  __shared__ double s_p10[9];
  __shared__ uint32_t lds_t[4], lds_n[4], lds_ok[4];
  // non-ASCII text, or more items than dst holds: the caller answers it otherwise
  if (cmem(totals)[1] || cmem(totals)[0] > cap) return;
  const uint64_t b = blockIdx.x;
  const CsvPre bp = cload(pre, b);
  const uint32_t lane = __lane_id(), wave = wave_in_wg(), base = 16 * threadIdx.x;
  const uint64_t blk0 = b * kCsvBlock, at = blk0 + base;
  const uint4 w = load16(text, len, at);
  *reinterpret_cast<uint4*>(txt + kHalo + base) = w;
  if (b > 0 && threadIdx.x < kHalo / 16)
    *reinterpret_cast<uint4*>(txt + base) = *reinterpret_cast<const uint4*>(text + blk0 - kHalo + base);
  if (threadIdx.x < 9) s_p10[threadIdx.x] = kPow10Exact[threadIdx.x];
  if (skip && threadIdx.x < kCsvBlock / 32) s_skip[threadIdx.x] = 0;
  const LaneMasks m = lane_masks(w, at, len, delim);
  uint32_t ntok = 0;
  const uint32_t ex = wg_excl_sum<4>(__popc(m.ends), lds_t, &ntok);
  {
    uint32_t k = ex;
    for (uint32_t e = m.ends; e; e &= e - 1u) s_end[k++] = (uint16_t)(base + (uint32_t)__builtin_ctz(e));
  }
  if (skip) {   // the lane's items, counted from the last newline before each
    const uint32_t last = m.nl ? 32u - (uint32_t)__clz(m.nl) : 0u;   // bytes up to the lane's last newline
    uint32_t all = 0;
    const uint32_t nl = wg_excl_max<4>(m.nl ? ex + __popc(m.ends & ((1u << last) - 1u)) + 1 : 0u, lds_n, &all);
    uint32_t li = nl ? ex - (nl - 1) : bp.line_idx + ex, k = ex;
    for (uint32_t e = m.ends; e; e &= e - 1u, ++k) {
      if (li < skip) atomicOr(&s_skip[k / 32], 1u << (k % 32));
      li = (m.nl >> __builtin_ctz(e)) & 1u ? 0u : li + 1;
    }
  }
  __syncthreads();
  const uint64_t staged = b > 0 ? blk0 - kHalo : 0;  // first byte held in LDS
  const uint8_t* lds_at = txt + kHalo;                 // LDS address of byte blk0
  uint32_t nok = 0;
  for (uint32_t k = threadIdx.x; k < ntok; k += blockDim.x) {
    uint64_t bits = kCsvNone;
    if (!skip || !((s_skip[k / 32] >> (k % 32)) & 1u)) {
      const uint32_t pe = s_end[k];
      const uint64_t pos = blk0 + pe;
      const uint64_t start = (uint64_t)((k ? (int64_t)(blk0 + s_end[k - 1]) : bp.prev_delim) + 1);
      const uint32_t c = lds_at[pe];
      const bool eof = pos + 1 == len && !csv_delim(c, delim);
      uint64_t end = eof ? len : pos;
      if (c == '\n' && end > start && lds_at[(int64_t)(end - 1) - (int64_t)blk0] == '\r') end -= 1;  // "\r\n"
      const uint64_t n = end - start;
      const uint8_t* lend = lds_at + ((int64_t)end - (int64_t)blk0);
      double v = 0.0;
      int r = 0;
      if (n) {
        if (start >= staged && n <= 16 && parse_short(lend, (uint32_t)n, s_p10, &v)) r = 1;
        else r = parse_item(start >= staged ? lend - n : text + start, n, tab, &v);
      }
      if (r) bits = (uint64_t)__double_as_longlong(v);
      if (r == 2) {  // a valid item: its exact value is filled in by k_csv_slow
        bits = 0;
        const unsigned long long e = atomicAdd(&totals[3], 1ull);
        if (e < slow_cap) {
          slow[e] = CsvSlow{start, end, bp.tok_base + k};
        } else {
          atomicAdd(&totals[4], 1ull);
          atomicMin(&totals[5], (unsigned long long)start);
        }
      }
    }
    nok += bits != kCsvNone ? 1u : 0u;
    dst[bp.tok_base + k] = __longlong_as_double((long long)bits);
  }
  nok = wave_total_u32(nok);
  if (lane == 0) lds_ok[wave] = nok;
  __syncthreads();
  if (threadIdx.x == 0) {
    nok = lds_ok[0] + lds_ok[1] + lds_ok[2] + lds_ok[3];
    pre[b].ok = nok;
    // rejected items: device atomics on one address serialize, so one of 32
    // slots (and none at all for a block without any)
    if (nok != ntok) atomicAdd(&totals[kCsvTotals + b % kCsvSlots], (unsigned long long)(ntok - nok));
  }
}

// ---- the exact slow path: a per-thread big integer ---------------------------------

namespace {

constexpr int kBigLimbs = 72;  // 2304 bits: 300 significant digits at any exponent
constexpr int kMaxSigDigits = 300;

struct DevBig {
  uint32_t d[kBigLimbs];
  int n;  // limbs in use (top limb nonzero)
};

__host__ __device__ void big_mul_add(DevBig& b, uint32_t m, uint32_t a) {
  uint64_t c = a;
  for (int i = 0; i < b.n; ++i) {
    const uint64_t v = (uint64_t)b.d[i] * m + c;
    b.d[i] = (uint32_t)v;
    c = v >> 32;
  }
  if (c && b.n < kBigLimbs) b.d[b.n++] = (uint32_t)c;
}

__host__ __device__ uint32_t big_div_small(DevBig& b, uint32_t m) {
  uint64_t r = 0;
  for (int i = b.n - 1; i >= 0; --i) {
    const uint64_t v = (r << 32) | b.d[i];
    b.d[i] = (uint32_t)(v / m);
    r = v % m;
  }
  while (b.n > 0 && b.d[b.n - 1] == 0) --b.n;
  return (uint32_t)r;
}

__host__ __device__ int big_bits(const DevBig& b) { return b.n ? 32 * (b.n - 1) + 32 - __builtin_clz(b.d[b.n - 1]) : 0; }

__host__ __device__ void big_shl(DevBig& b, int s) {
  const int ls = s / 32, bs = s % 32;
  if (b.n == 0 || s == 0) return;
  int nn = b.n + ls + 1;
  if (nn > kBigLimbs) nn = kBigLimbs;
  for (int i = nn - 1; i >= 0; --i) {
    const int src = i - ls;
    const uint32_t hi = src >= 0 && src < b.n ? b.d[src] : 0u;
    const uint32_t lo = src - 1 >= 0 && src - 1 < b.n ? b.d[src - 1] : 0u;
    b.d[i] = bs ? (hi << bs) | (lo >> (32 - bs)) : hi;
  }
  b.n = nn;
  while (b.n > 0 && b.d[b.n - 1] == 0) --b.n;
}

__host__ __device__ uint32_t big_bit(const DevBig& b, int k) { return k >= 0 && k / 32 < b.n ? (b.d[k / 32] >> (k % 32)) & 1u : 0u; }

__host__ __device__ bool big_any_below(const DevBig& b, int k) {  // any bit < k
  for (int i = 0; i < b.n && 32 * i < k; ++i) {
    const int top = k - 32 * i;
    const uint32_t mask = top >= 32 ? ~0u : ((1u << top) - 1u);
    if (b.d[i] & mask) return true;
  }
  return false;
}

// The f64 bits nearest to (A + f) * 2^E2, where 0 <= f < 1 is nonzero iff
// `extra` (A has at least 55 bits whenever extra is set).
__host__ __device__ uint64_t big_round(const DevBig& A, int64_t E2, bool extra) {
  const int L = big_bits(A);
  const int64_t ex = (int64_t)L - 1 + E2;
  if (ex > 1023) return 0x7FF0000000000000ull;
  const int64_t K = ex >= -1022 ? 53 : ex + 1075;
  if (K < 0) return 0;
  const int64_t lsb = L - K;
  uint64_t mant = 0;
  for (int64_t j = K - 1; j >= 0; --j) mant = (mant << 1) | big_bit(A, (int)(lsb + j));
  const uint32_t round = lsb >= 1 ? big_bit(A, (int)(lsb - 1)) : 0u;
  const bool sticky = (lsb >= 2 && big_any_below(A, (int)(lsb - 1))) || extra;
  if (round && (sticky || (mant & 1u))) mant += 1;
  uint64_t b = ex >= -1022 ? ((uint64_t)(ex + 1022) << 52) + mant : mant;
  if (b >= 0x7FF0000000000000ull) b = 0x7FF0000000000000ull;
  return b;
}

// The exact value of a valid item (the grammar was checked by parse_item).
__host__ __device__ bool exact_item(const uint8_t* __restrict__ p, uint64_t n, uint64_t* out) {
  uint64_t i = 0;
  uint64_t sign = 0;
  if (p[0] == '+' || p[0] == '-') {
    sign = p[0] == '-' ? 0x8000000000000000ull : 0ull;
    i = 1;
  }
  DevBig D;
  D.n = 0;
  int nsd = 0;
  int64_t Q = 0;
  while (i < n && csv_digit(p[i])) {
    const uint32_t d = p[i] - '0';
    if (D.n || d) {
      if (++nsd > kMaxSigDigits) return false;
      if (D.n == 0) {
        D.d[0] = d;
        D.n = 1;
      } else {
        big_mul_add(D, 10, d);
      }
    }
    ++i;
  }
  if (i < n && p[i] == '.') {
    ++i;
    while (i < n && csv_digit(p[i])) {
      const uint32_t d = p[i] - '0';
      if (D.n || d) {
        if (++nsd > kMaxSigDigits) return false;
        if (D.n == 0) {
          D.d[0] = d;
          D.n = 1;
        } else {
          big_mul_add(D, 10, d);
        }
      }
      --Q;
      ++i;
    }
  }
  if (i < n && (p[i] | 0x20u) == 'e') {
    ++i;
    bool eneg = false;
    if (i < n && (p[i] == '+' || p[i] == '-')) {
      eneg = p[i] == '-';
      ++i;
    }
    int64_t ev = 0;
    while (i < n && csv_digit(p[i])) {
      if (ev < 100000000) ev = ev * 10 + (p[i] - '0');
      ++i;
    }
    Q += eneg ? -ev : ev;
  }
  uint64_t bits;
  if (D.n == 0) {
    bits = 0;
  } else if (Q >= 0) {
    if (Q + nsd > 310) {
      bits = 0x7FF0000000000000ull;
    } else {
      for (int64_t j = 0; j < Q; ++j) big_mul_add(D, 10, 0);
      bits = big_round(D, 0, false);
    }
  } else {
    const int64_t k = -Q;
    if (k - nsd > 345) {
      bits = 0;
    } else {
      const int64_t need = 56 + (k * 3322 + 999) / 1000 - big_bits(D);  // >= 55 quotient bits
      big_shl(D, need > 0 ? (int)need : 0);
      bool rem = false;
      for (int64_t j = 0; j < k; ++j) rem |= big_div_small(D, 10) != 0;
      bits = big_round(D, -(need > 0 ? need : 0), rem);
    }
  }
  *out = sign | bits;
  return true;
}

}  // namespace

__global__ __launch_bounds__(64) void k_csv_slow(const uint8_t* __restrict__ text, const CsvSlow* __restrict__ slow,
                                                 uint64_t count, double* __restrict__ dst,
                                                 unsigned long long* __restrict__ totals) {
  const uint64_t e = (uint64_t)blockIdx.x * 64 + threadIdx.x;
  if (e >= count) return;
  const CsvSlow it = slow[e];
  uint64_t bits = 0;
  if (exact_item(text + it.start, it.end - it.start, &bits)) {
    dst[it.slot] = __longlong_as_double((long long)bits);
  } else {
    atomicAdd(&totals[4], 1ull);
    atomicMin(&totals[5], (unsigned long long)it.start);
  }
}

// Moves block b's parsed values (items [tok_base, tok_base + ntok) that are not
// kCsvNone) to out[ok_base ...] in item order: each lane takes 16 consecutive
// items.
__global__ __launch_bounds__(256) void k_csv_compact(const CsvBlock* __restrict__ blk, const CsvPre* __restrict__ pre,
                                                     const double* __restrict__ src, double* __restrict__ out) {
  __shared__ uint32_t lds[4];
  constexpr uint32_t kPer = kCsvBlock / 256;  // at most kCsvBlock items end in a block
  const CsvPre bp = cload(pre, blockIdx.x);
  const uint32_t ntok = blk[blockIdx.x].ntok;
  const uint32_t i0 = threadIdx.x * kPer;
  double v[kPer];
  uint32_t cnt = 0, tot = 0;
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i) {
    v[i] = i0 + i < ntok ? src[bp.tok_base + i0 + i] : __longlong_as_double((long long)kCsvNone);
    cnt += (uint64_t)__double_as_longlong(v[i]) != kCsvNone ? 1u : 0u;
  }
  uint64_t r = bp.ok_base + wg_excl_sum<4>(cnt, lds, &tot);
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i)
    if ((uint64_t)__double_as_longlong(v[i]) != kCsvNone) out[r++] = v[i];
}

// ---- launchers ------------------------------------------------------------------------

static inline uint64_t rup256(uint64_t x) { return (x + 255) / 256 * 256; }

uint64_t csv_totals_offset(uint64_t nblocks) {
  return rup256(nblocks * sizeof(CsvBlock)) + rup256(nblocks * sizeof(CsvPre));
}
uint64_t csv_scratch_bytes(uint64_t nblocks) { return csv_totals_offset(nblocks) + rup256(8 * kCsvWords); }

static inline CsvBlock* blk_of(uint8_t* s) { return reinterpret_cast<CsvBlock*>(s); }
static inline CsvPre* pre_of(uint8_t* s, uint64_t nb) {
  return reinterpret_cast<CsvPre*>(s + rup256(nb * sizeof(CsvBlock)));
}

hipError_t launch_csv_count(const uint8_t* text, uint64_t len, uint8_t delim, uint8_t* scratch, uint64_t nblocks,
                            hipStream_t s) {
  launch_k(k_csv_blocks, dim3((uint32_t)nblocks), dim3(256), 0, s, text, len, (uint32_t)delim, blk_of(scratch));
  return hipGetLastError();
}

hipError_t launch_csv_parse(const uint8_t* text, uint64_t len, uint8_t delim, uint32_t skip, const Pow5* tab,
                            uint8_t* scratch, uint64_t nblocks, double* dst, uint64_t cap, CsvSlow* slow,
                            uint64_t slow_cap, hipStream_t s) {
  unsigned long long* totals = reinterpret_cast<unsigned long long*>(scratch + csv_totals_offset(nblocks));
  launch_k(k_csv_scan, dim3(1), dim3(1024), 0, s, (const CsvBlock*)blk_of(scratch), pre_of(scratch, nblocks), nblocks,
           totals);
  launch_k(k_csv_parse, dim3((uint32_t)nblocks), dim3(256), 0, s, text, len, (uint32_t)delim, skip, tab,
           pre_of(scratch, nblocks), dst, cap, slow, slow_cap, totals);
  return hipGetLastError();
}

hipError_t launch_csv_slow(const uint8_t* text, const CsvSlow* slow, uint64_t count, uint8_t* scratch,
                           uint64_t nblocks, double* dst, hipStream_t s) {
  unsigned long long* totals = reinterpret_cast<unsigned long long*>(scratch + csv_totals_offset(nblocks));
  if (count) launch_k(k_csv_slow, dim3((uint32_t)((count + 63) / 64)), dim3(64), 0, s, text, slow, count, dst, totals);
  return hipGetLastError();
}

hipError_t launch_csv_compact(const uint8_t* scratch, uint64_t nblocks, const double* src, double* out,
                              hipStream_t s) {
  uint8_t* sc = const_cast<uint8_t*>(scratch);
  launch_k(k_csv_okscan, dim3(1), dim3(256), 0, s, pre_of(sc, nblocks), nblocks);
  launch_k(k_csv_compact, dim3((uint32_t)nblocks), dim3(256), 0, s, (const CsvBlock*)blk_of(sc),
           (const CsvPre*)pre_of(sc, nblocks), src, out);
  return hipGetLastError();
}

}  // namespace buffgpu

// ---- host entry points ------------------------------------------------------------------

#include <cstdio>

#include "../../include/buffgpu.h"
#include "buff_runtime.h"

namespace buffgpu {

namespace {

std::once_flag g_pow5_once;
std::vector<Pow5> g_pow5;

const std::vector<Pow5>& pow5_table() {
  std::call_once(g_pow5_once, [] {
    g_pow5.resize(kPow5Max - kPow5Min + 1);
    csv_pow5_table(g_pow5.data());
  });
  return g_pow5;
}

}  // namespace

int csv_parse_device(Ctx* ctx, const uint8_t* text, uint64_t len, uint8_t delim, uint32_t skip, double* out,
                     uint64_t cap, uint64_t* count) {
  if (!ctx || !count || (len && !text)) return fail(BUFF_E_INVALID, "null argument");
  if (delim == '\r' || delim >= 0x80) return fail(BUFF_E_INVALID, "delimiter 0x%02x: an ASCII byte other than CR", delim);
  *count = 0;
  if (len == 0) return BUFF_OK;
  const uint64_t nb = (len + kCsvBlock - 1) / kCsvBlock;
  if (nb > 0x7FFFFFFFull) return fail(BUFF_E_INVALID, "text of %llu bytes", (unsigned long long)len);
  if (!ctx->csv_tab_ready) {
    const std::vector<Pow5>& tab = pow5_table();
    BUFF_TRY(ctx->scratch(ctx->s_csvtab, tab.size() * sizeof(Pow5)));
    HIP_TRY(hipMemcpyAsync(ctx->s_csvtab.ptr, tab.data(), tab.size() * sizeof(Pow5), hipMemcpyHostToDevice,
                           ctx->stream));
    ctx->csv_tab_ready = true;
  }
  BUFF_TRY(ctx->scratch(ctx->s_csv, csv_scratch_bytes(nb)));
  uint8_t* scr = (uint8_t*)ctx->s_csv.ptr;
  // the items are parsed straight into `out` when it has room for all of them
  // (the parse returns at once when it has not, known only on the device), with
  // a small queue for the items the 19-digit rounding leaves open (more than 19
  // digits close to a rounding boundary: rare; k_csv_slow decides them exactly)
  unsigned long long tot[kCsvWords];
  double* dst = out;
  uint64_t room = out ? cap : 0, slow_cap = 4096;
  CsvSlow* slow = nullptr;
  auto parse = [&]() -> int {
    BUFF_TRY(ctx->scratch(ctx->s_csvslow, slow_cap * sizeof(CsvSlow)));
    slow = (CsvSlow*)ctx->s_csvslow.ptr;
    {
      ProfScope ps(ctx, "k_csv_parse");
      HIP_TRY(launch_csv_parse(text, len, delim, skip, (const Pow5*)ctx->s_csvtab.ptr, scr, nb, dst, room, slow,
                               slow_cap, ctx->stream));
    }
    return d2h_small(ctx, tot, scr + csv_totals_offset(nb), sizeof(tot));
  };
  {
    ProfScope ps(ctx, "k_csv_count");
    HIP_TRY(launch_csv_count(text, len, delim, scr, nb, ctx->stream));
  }
  BUFF_TRY(parse());
  if (tot[1])
    return fail(BUFF_E_UNSUPPORTED, "bytes >= 0x80: the reference drops every line that is not UTF-8");
  const uint64_t items = tot[0];
  if (items == 0) return BUFF_OK;
  const bool direct = items <= room;
  if (!direct) {
    BUFF_TRY(ctx->scratch(ctx->s_csvtmp, items * 8));
    dst = (double*)ctx->s_csvtmp.ptr;
    room = items;
    BUFF_TRY(parse());
  }
  if (tot[4] && items / 64 > slow_cap) {   // more open items than the queue holds
    slow_cap = items / 64;
    BUFF_TRY(parse());
  }
  if (tot[3] && !tot[4]) {
    ProfScope ps(ctx, "k_csv_slow");
    HIP_TRY(launch_csv_slow(text, slow, std::min<uint64_t>(tot[3], slow_cap), scr, nb, dst, ctx->stream));
    BUFF_TRY(d2h_small(ctx, tot, scr + csv_totals_offset(nb), sizeof(tot)));
  }
  if (tot[4])
    return fail(BUFF_E_UNSUPPORTED, "%llu items (the first at byte %llu) have more than %d significant digits or "
                "exceed the exact path's queue", (unsigned long long)tot[4], (unsigned long long)tot[5], 300);
  uint64_t ok = items;
  for (uint32_t k = 0; k < kCsvSlots; ++k) ok -= tot[kCsvTotals + k];
  *count = ok;
  if (ok > cap) return fail(BUFF_E_SMALL_BUFFER, "%llu values, room for %llu", (unsigned long long)ok,
                            (unsigned long long)cap);
  if (ok && !out) return fail(BUFF_E_INVALID, "null output");
  if (ok < items || !direct) {
    const double* src = dst;
    if (direct) {  // the values sit in out at their items' slots: move them through scratch
      BUFF_TRY(ctx->scratch(ctx->s_csvtmp, items * 8));
      HIP_TRY(hipMemcpyAsync(ctx->s_csvtmp.ptr, out, items * 8, hipMemcpyDeviceToDevice, ctx->stream));
      src = (const double*)ctx->s_csvtmp.ptr;
    }
    ProfScope ps(ctx, "k_csv_compact");
    HIP_TRY(launch_csv_compact(scr, nb, src, out, ctx->stream));
  }
  return BUFF_OK;
}

int csv_parse_host(Ctx* ctx, const uint8_t* text, uint64_t len, uint8_t delim, uint32_t skip, double* out,
                   uint64_t cap, uint64_t* count) {
  if (!ctx || !count || (len && !text)) return fail(BUFF_E_INVALID, "null argument");
  *count = 0;
  if (len == 0) return BUFF_OK;
  BUFF_TRY(ctx->scratch(ctx->s_stream, len));
  HIP_TRY(hipMemcpyAsync(ctx->s_stream.ptr, text, len, hipMemcpyHostToDevice, ctx->stream));
  // every parsed item takes at least one byte and a delimiter
  const uint64_t most = len / 2 + 1;
  BUFF_TRY(ctx->scratch(ctx->s_values, most * 8));
  uint64_t n = 0;
  BUFF_TRY(csv_parse_device(ctx, (const uint8_t*)ctx->s_stream.ptr, len, delim, skip, (double*)ctx->s_values.ptr,
                            most, &n));
  *count = n;
  if (n > cap) return fail(BUFF_E_SMALL_BUFFER, "%llu values, room for %llu", (unsigned long long)n,
                           (unsigned long long)cap);
  if (n) {
    if (!out) return fail(BUFF_E_INVALID, "null output");
    HIP_TRY(hipMemcpyAsync(out, ctx->s_values.ptr, n * 8, hipMemcpyDeviceToHost, ctx->stream));
  }
  HIP_TRY(hipStreamSynchronize(ctx->stream));
  return BUFF_OK;
}

}  // namespace buffgpu

using namespace buffgpu;

extern "C" {

int buff_csv_parse_device(buff_ctx* ctx, const uint8_t* text_dev, uint64_t len, uint8_t delim, uint32_t skip_val,
                          double* out_dev, uint64_t cap, uint64_t* count) {
  return csv_parse_device(reinterpret_cast<Ctx*>(ctx), text_dev, len, delim, skip_val, out_dev, cap, count);
}

int buff_csv_parse(buff_ctx* ctx, const uint8_t* text, uint64_t len, uint8_t delim, uint32_t skip_val, double* out,
                   uint64_t cap, uint64_t* count) {
  return csv_parse_host(reinterpret_cast<Ctx*>(ctx), text, len, delim, skip_val, out, cap, count);
}

int buff_construct_file_iterator_skip_newline(const char* file, uint32_t skip_val, uint8_t delim, double* out,
                                              uint64_t cap, uint64_t* count) {
  if (!file || !count) return fail(BUFF_E_INVALID, "null argument");
  FILE* f = std::fopen(file, "rb");
  if (!f) return fail(BUFF_E_INVALID, "cannot open %s", file);  // the reference's Err(())
  std::vector<uint8_t> text;
  uint8_t buf[1 << 16];
  size_t got;
  while ((got = std::fread(buf, 1, sizeof(buf), f)) > 0) text.insert(text.end(), buf, buf + got);
  const bool err = std::ferror(f) != 0;
  std::fclose(f);
  if (err) return fail(BUFF_E_INVALID, "read error on %s", file);
  Ctx* c = nullptr;
  BUFF_TRY(default_ctx(&c));
  return csv_parse_host(c, text.data(), text.size(), delim, skip_val, out, cap, count);
}

}  // extern "C"
