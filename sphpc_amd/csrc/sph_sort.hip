// Stable key/value radix sort, exclusive scan and cell bounds for gfx950.
//
// Replaces the Thrust wrappers of the reference (thrust_c.cu:86-120):
//  - SortByKey: LSD radix sort, digits of 8 or 10 bits.  Each pass is an
//    upsweep (per-tile digit histogram), a scan of each digit's row of it, and a
//    downsweep that ranks keys inside the tile with wavefront ballots (peers with
//    the same digit), stages the tile in LDS in digit order and writes each digit
//    run out contiguously.  Ranks follow input position (wave, round, lane), so
//    the sort is stable.
//  - FindLowerBounds/FindUpperBounds: a key histogram followed by a scan:
//    exclusive it is lower_bound(c) for every cell, inclusive upper_bound(c).
#include <mutex>

#include "sph_internal.h"

namespace sph {

constexpr int RS_THREADS = 256;
constexpr int RS_ITEMS = 16;
constexpr int RS_TILE = RS_THREADS * RS_ITEMS;  // 4096 keys per block
constexpr int RS_WAVES = RS_THREADS / 64;
constexpr int SC_THREADS = 256;
constexpr int SC_ITEMS = 16;
constexpr int SC_TILE = SC_THREADS * SC_ITEMS;
static_assert(SC_TILE == kScanTile, "scratch sized by scan_tiles");

// Every lane of the wave calls it.  Data-parallel moves (shifts within 16 lanes,
// then lane 15 of each row and lane 31 passed on) in place of six LDS round trips.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
  const auto from = [&x](auto ctrl, auto rows) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value,
                                                 decltype(rows)::value, 0xF, false);
  };
  using std::integral_constant;
  const integral_constant<int, 0xF> all;
  x += from(integral_constant<int, 0x111>{}, all);
  x += from(integral_constant<int, 0x112>{}, all);
  x += from(integral_constant<int, 0x114>{}, all);
  x += from(integral_constant<int, 0x118>{}, all);
  x += from(integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{});
  x += from(integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{});
  return x;
}

// Exclusive scan over a 256-thread block; *tot receives the block total.
__device__ __forceinline__ uint32_t block_excl_scan_256(uint32_t x, uint32_t *wtot,
                                                        uint32_t *tot) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t inc = wave_incl_scan(x);
  if (lane == 63) wtot[w] = inc;
  __syncthreads();
  uint32_t pre = 0, all = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t t = wtot[i];
    if (i < w) pre += t;
    all += t;
  }
  __syncthreads();
  *tot = all;
  const uint32_t before = __shfl_up(inc, 1, 64);
  return pre + (lane ? before : 0u);
}

// Lanes of the wave holding the same digit (valid lanes only).
template <int BITS>
__device__ __forceinline__ uint64_t match_digit(uint32_t d, bool valid) {
  uint64_t peers = __ballot(valid);
#pragma unroll
  for (int b = 0; b < BITS; ++b) {
    const bool bit = (d >> b) & 1u;
    const uint64_t bb = __ballot(bit);
    peers &= bit ? bb : ~bb;
  }
  return peers;
}

__device__ __forceinline__ uint64_t lanemask_lt() {
  const int lane = threadIdx.x & 63;
  return lane ? (~0ull >> (64 - lane)) : 0ull;
}

// --------------------------------------------------------------------------
// Scan
// --------------------------------------------------------------------------
// A wave owns 1024 consecutive entries of a tile, a lane four of each 256 of
// them: one 16-byte load and store a quarter, side by side over the lanes.
constexpr int SC_QUARTERS = SC_ITEMS / 4;
__device__ __forceinline__ uint32_t first_item(int q) {
  return blockIdx.x * SC_TILE + (threadIdx.x >> 6) * (64 * SC_ITEMS) + q * 256 +
         (threadIdx.x & 63) * 4;
}

__device__ __forceinline__ void load_items(const uint32_t *in, uint32_t len,
                                           uint4 (&x)[SC_QUARTERS]) {
#pragma unroll
  for (int q = 0; q < SC_QUARTERS; ++q) {
    const uint32_t i = first_item(q);
    if (i + 4 <= len) {
      x[q] = *reinterpret_cast<const uint4 *>(in + i);
    } else {
      x[q].x = i < len ? in[i] : 0u;
      x[q].y = i + 1 < len ? in[i + 1] : 0u;
      x[q].z = i + 2 < len ? in[i + 2] : 0u;
      x[q].w = 0u;
    }
  }
}

__global__ __launch_bounds__(SC_THREADS) void k_scan_tile_sums(const uint32_t *__restrict__ in,
                                                               uint32_t len,
                                                               uint32_t *__restrict__ sums) {
  __shared__ uint32_t wtot[4];
  uint4 x[SC_QUARTERS];
  load_items(in, len, x);
  uint32_t s = 0;
#pragma unroll
  for (int q = 0; q < SC_QUARTERS; ++q) s += (x[q].x + x[q].y) + (x[q].z + x[q].w);
  uint32_t tot;
  block_excl_scan_256(s, wtot, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ __launch_bounds__(SC_THREADS) void k_scan_spine(uint32_t *sums, uint32_t tiles) {
  __shared__ uint32_t wtot[4];
  uint32_t carry = 0;
  for (uint32_t base = 0; base < tiles; base += SC_THREADS) {
    const uint32_t i = base + threadIdx.x;
    const uint32_t x = i < tiles ? sums[i] : 0u;
    uint32_t tot;
    const uint32_t e = block_excl_scan_256(x, wtot, &tot);
    if (i < tiles) sums[i] = carry + e;
    carry += tot;
  }
}

// Where a tile takes the sum of the tiles before it from.
enum ScanFrom {
  SCAN_INPUT,  // the input itself (up to kScanSelfTiles tiles: no other launch)
  SCAN_SUMS,   // the tiles' sums (up to kScanSumTiles tiles)
  SCAN_SPINE   // their exclusive scan
};
// One launch costs 4-5 us of a small substep (kernel and gap), and reading up
// to 7 tiles (28,672 words, all of L2) again costs less; a block reads 2048
// sums in 8 loads per thread, less than the spine's launch.
constexpr uint32_t kScanSelfTiles = 8, kScanLateTiles = 256, kScanSumTiles = 2048;

// in and out may alias with SCAN_SUMS and SCAN_SPINE (in-place scan).
// Bounded by the writes of a large table (5.9M cells, 23 MB, of which particles are
// in a tenth): with 16 consecutive entries a thread, each store left in 64 pieces of
// 16 bytes, 13.4 us; side by side and without reading the empty tiles 6.9.
template <ScanFrom FROM>
__global__ __launch_bounds__(SC_THREADS) void k_scan_apply(const uint32_t *in, uint32_t *out,
                                                           uint32_t len,
                                                           const uint32_t *__restrict__ sums,
                                                           int inclusive, int write_total) {
  __shared__ uint32_t wtot[4];
  uint4 x[SC_QUARTERS] = {};
  // of many tiles, one without a count is not read (a table of cells is mostly
  // empty); of few, its loads go out before its sum is known
  const bool late = FROM == SCAN_SUMS && gridDim.x > kScanLateTiles;
  if (!late) load_items(in, len, x);
  uint32_t before = 0;
  if (FROM == SCAN_SPINE) {
    before = sums[blockIdx.x];
  } else {
    uint32_t own = 0;
    if (FROM == SCAN_SUMS) {
      if (late && sums[blockIdx.x] != 0u) load_items(in, len, x);
      for (uint32_t t = threadIdx.x; t < blockIdx.x; t += SC_THREADS) own += sums[t];
    } else {
      for (uint32_t t = 0; t < blockIdx.x; ++t) {
        const uint4 *v = reinterpret_cast<const uint4 *>(in + t * SC_TILE) + threadIdx.x;
#pragma unroll
        for (int q = 0; q < SC_QUARTERS; ++q) {
          const uint4 a = v[q * SC_THREADS];
          own += (a.x + a.y) + (a.z + a.w);
        }
      }
    }
    block_excl_scan_256(own, wtot, &before);
  }
  // scan within the quarters, the quarters' sums before them, the waves' before those
  uint32_t pre[SC_QUARTERS], run = 0;
#pragma unroll
  for (int q = 0; q < SC_QUARTERS; ++q) {
    const uint32_t own = (x[q].x + x[q].y) + (x[q].z + x[q].w), inc = wave_incl_scan(own);
    pre[q] = run + inc - own;
    run += (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) wtot[w] = run;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (i < w) before += wtot[i];
  const bool aligned = (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
#pragma unroll
  for (int q = 0; q < SC_QUARTERS; ++q) {
    const uint32_t i = first_item(q), e0 = before + pre[q], e1 = e0 + x[q].x, e2 = e1 + x[q].y,
                   e3 = e2 + x[q].z, e4 = e3 + x[q].w;
    const uint4 o = inclusive ? make_uint4(e1, e2, e3, e4) : make_uint4(e0, e1, e2, e3);
    if (i + 4 <= len && aligned) {
      *reinterpret_cast<uint4 *>(out + i) = o;
    } else {
      if (i < len) out[i] = o.x;
      if (i + 1 < len) out[i + 1] = o.y;
      if (i + 2 < len) out[i + 2] = o.z;
      if (i + 3 < len) out[i + 3] = o.w;
    }
    // the thread holding entry len-1 writes the total after it
    if (write_total && i < len && len <= i + 4) out[len] = e4;
  }
}

__global__ void k_fill_u32(uint32_t *p, uint32_t v, uint32_t len) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < len) p[i] = v;
}

int scan(const uint32_t *in, uint32_t *out, uint32_t len, bool inclusive, bool write_total,
         ScanScratch *sc, hipStream_t s, sph_ctx *prof) {
  if (len == 0) {
    if (write_total) {
      k_fill_u32<<<1, 64, 0, s>>>(out, 0u, 1u);
      SPH_HIP(hipGetLastError());
    }
    return SPH_OK;
  }
  if ((uintptr_t)in & 15u) {
    set_error("scan: the input must be 16-byte aligned");
    return SPH_ERR_ARG;
  }
  const uint32_t tiles = (len + SC_TILE - 1) / SC_TILE;
  const bool self = tiles <= kScanSelfTiles && in != out;
  if (!self && sc->tile_cap < tiles) {
    if (sc->tile_sums) SPH_HIP(hipFree(sc->tile_sums));
    sc->tile_sums = nullptr;
    sc->tile_cap = 0;
    SPH_HIP(hipMalloc(&sc->tile_sums, sizeof(uint32_t) * tiles));
    sc->tile_cap = tiles;
  }
  const int incl = inclusive ? 1 : 0, total = write_total ? 1 : 0;
  hipEvent_t ev = nullptr;
  if (prof) prof_begin(prof, K_SCAN, &ev);
  if (self) {
    k_scan_apply<SCAN_INPUT><<<tiles, SC_THREADS, 0, s>>>(in, out, len, nullptr, incl, total);
  } else {
    k_scan_tile_sums<<<tiles, SC_THREADS, 0, s>>>(in, len, sc->tile_sums);
    if (tiles <= kScanSumTiles) {
      k_scan_apply<SCAN_SUMS><<<tiles, SC_THREADS, 0, s>>>(in, out, len, sc->tile_sums, incl,
                                                           total);
    } else {
      k_scan_spine<<<1, SC_THREADS, 0, s>>>(sc->tile_sums, tiles);
      k_scan_apply<SCAN_SPINE><<<tiles, SC_THREADS, 0, s>>>(in, out, len, sc->tile_sums, incl,
                                                            total);
    }
  }
  if (prof) prof_end(prof, K_SCAN, ev);
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

// --------------------------------------------------------------------------
// Radix sort
// --------------------------------------------------------------------------
// hist[digit * tiles + tile]: the tile's count of the digit.
template <int BITS>
__global__ __launch_bounds__(RS_THREADS) void k_radix_upsweep(const uint32_t *__restrict__ keys,
                                                              uint32_t n, int shift,
                                                              uint32_t *__restrict__ hist,
                                                              uint32_t tiles) {
  constexpr int D = 1 << BITS;
  __shared__ uint32_t h[RS_WAVES][D];
  for (int i = threadIdx.x; i < RS_WAVES * D; i += RS_THREADS) (&h[0][0])[i] = 0u;
  __syncthreads();
  const int w = threadIdx.x >> 6;
  const uint64_t lt = lanemask_lt();
  const uint32_t base = blockIdx.x * RS_TILE;
  uint32_t kk[RS_ITEMS];
#pragma unroll
  for (int r = 0; r < RS_ITEMS; ++r) {
    const uint32_t i = base + r * RS_THREADS + threadIdx.x;
    kk[r] = i < n ? keys[i] : 0u;
  }
#pragma unroll
  for (int r = 0; r < RS_ITEMS; ++r) {
    const uint32_t i = base + r * RS_THREADS + threadIdx.x;
    const bool valid = i < n;
    const uint32_t d = (kk[r] >> shift) & (D - 1u);
    const uint64_t peers = match_digit<BITS>(d, valid);
    // one leader per digit per wave adds the digit's count (a non-returning
    // LDS add: no wait between rounds)
    if (valid && (peers & lt) == 0) atomicAdd(&h[w][d], (uint32_t)__popcll(peers));
  }
  __syncthreads();
  for (int d = threadIdx.x; d < D; d += RS_THREADS) {
    uint32_t s = 0;
#pragma unroll
    for (int ww = 0; ww < RS_WAVES; ++ww) s += h[ww][d];
    hist[(size_t)d * tiles + blockIdx.x] = s;
  }
}

// Exclusive scan of each digit's row of the histogram and its total, a block per
// digit.  With the digits' own scan left to the downsweep (a block scan of the
// totals) this is one launch, where a scan of the whole histogram takes three.
__global__ __launch_bounds__(RS_THREADS) void k_radix_rows(uint32_t *__restrict__ hist,
                                                           uint32_t tiles,
                                                           uint32_t *__restrict__ totals) {
  __shared__ uint32_t wtot[4];
  uint32_t *row = hist + (size_t)blockIdx.x * tiles;
  uint32_t carry = 0;
  for (uint32_t t0 = 0; t0 < tiles; t0 += RS_THREADS) {
    const uint32_t t = t0 + threadIdx.x;
    uint32_t tot;
    const uint32_t e = block_excl_scan_256(t < tiles ? row[t] : 0u, wtot, &tot);
    if (t < tiles) row[t] = carry + e;
    carry += tot;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// ROWS: the histogram's rows are scanned and `totals` holds their sums;
// otherwise each block sums the rows itself (few tiles: no launch between).
template <int BITS, bool ROWS>
__global__ __launch_bounds__(RS_THREADS) void k_radix_downsweep(
    const uint32_t *__restrict__ kin, const uint32_t *__restrict__ vin,
    uint32_t *__restrict__ kout, uint32_t *__restrict__ vout, uint32_t n, int shift,
    const uint32_t *__restrict__ hist, const uint32_t *__restrict__ totals, uint32_t tiles) {
  constexpr int D = 1 << BITS, DPT = D / RS_THREADS;  // digits per thread, consecutive
  __shared__ uint32_t wcnt[RS_WAVES][D];
  __shared__ uint32_t dstart[D];
  __shared__ uint32_t goff[D];
  __shared__ uint32_t wtot[4];
  __shared__ uint32_t sk[RS_TILE];
  __shared__ uint32_t sv[RS_TILE];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  for (int i = tid; i < RS_WAVES * D; i += RS_THREADS) (&wcnt[0][0])[i] = 0u;
  __syncthreads();
  const uint64_t lt = lanemask_lt();
  const uint32_t tile0 = blockIdx.x * RS_TILE;
  const uint32_t wbase = tile0 + (uint32_t)w * 64u * RS_ITEMS;
  uint32_t k[RS_ITEMS], v[RS_ITEMS], rk[RS_ITEMS];
#pragma unroll
  for (int r = 0; r < RS_ITEMS; ++r) {
    const uint32_t i = wbase + (uint32_t)r * 64u + (uint32_t)lane;
    const bool valid = i < n;
    k[r] = valid ? kin[i] : 0u;
    v[r] = valid ? (vin ? vin[i] : i) : 0u;
  }
#pragma unroll
  for (int r = 0; r < RS_ITEMS; ++r) {
    const uint32_t i = wbase + (uint32_t)r * 64u + (uint32_t)lane;
    const bool valid = i < n;
    const uint32_t d = (k[r] >> shift) & (D - 1u);
    const uint64_t peers = match_digit<BITS>(d, valid);
    const uint32_t below = (uint32_t)__popcll(peers & lt);
    // the digit's leader (lowest peer) takes the wave's running count and adds
    // the peers; LDS operations of a wave complete in order, so later rounds
    // see this one's add without waiting for its result
    uint32_t old = 0u;
    if (valid && below == 0) old = atomicAdd(&wcnt[w][d], (uint32_t)__popcll(peers));
    const int leader = peers ? (int)__builtin_ctzll(peers) : lane;
    rk[r] = __shfl(old, leader, 64) + below;
  }
  // where the digits of this thread begin in the output, over all tiles and in
  // this one's share
  uint32_t all[DPT], before[DPT], sum = 0u;
#pragma unroll
  for (int q = 0; q < DPT; ++q) {
    const int d = tid * DPT + q;
    const uint32_t *row = hist + (size_t)d * tiles;
    if (ROWS) {
      all[q] = totals[d];
      before[q] = row[blockIdx.x];
    } else {
      all[q] = before[q] = 0u;
      for (uint32_t t = 0; t < tiles; ++t) {
        const uint32_t x = row[t];
        all[q] += x;
        before[q] += t < blockIdx.x ? x : 0u;
      }
    }
    sum += all[q];
  }
  uint32_t tot, run = block_excl_scan_256(sum, wtot, &tot);  // its barriers end the counting
#pragma unroll
  for (int q = 0; q < DPT; ++q) {
    goff[tid * DPT + q] = run + before[q];
    run += all[q];
  }
  // prefix over the waves, then tile-level digit starts
  uint32_t mine[DPT];
  sum = 0u;
#pragma unroll
  for (int q = 0; q < DPT; ++q) {
    uint32_t c = 0u;
#pragma unroll
    for (int ww = 0; ww < RS_WAVES; ++ww) {
      const uint32_t x = wcnt[ww][tid * DPT + q];
      wcnt[ww][tid * DPT + q] = c;
      c += x;
    }
    mine[q] = c;
    sum += c;
  }
  run = block_excl_scan_256(sum, wtot, &tot);
#pragma unroll
  for (int q = 0; q < DPT; ++q) {
    dstart[tid * DPT + q] = run;
    run += mine[q];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RS_ITEMS; ++r) {
    const uint32_t i = wbase + (uint32_t)r * 64u + (uint32_t)lane;
    if (i < n) {
      const uint32_t d = (k[r] >> shift) & (D - 1u);
      const uint32_t lp = dstart[d] + wcnt[w][d] + rk[r];
      sk[lp] = k[r];
      sv[lp] = v[r];
    }
  }
  __syncthreads();
  const uint32_t tile_n = min((uint32_t)RS_TILE, n - tile0);
  for (uint32_t i = tid; i < tile_n; i += RS_THREADS) {
    const uint32_t kk = sk[i];
    const uint32_t d = (kk >> shift) & (D - 1u);
    const uint32_t o = goff[d] + (i - dstart[d]);
    kout[o] = kk;
    vout[o] = sv[i];
  }
}

// Digits of 8 bits, or of 10 where that saves a pass and the launches of a pass
// weigh: a wider digit ranks with more ballots, holds more LDS (57 KB a block
// against 39) and leaves shorter runs to write.  Measured for 20-bit keys, two
// passes of 10 against three of 8, with the copy in and the wait: 1,000 pairs 45 /
// 58 us, 30k 60 / 66, 300k 65 / 76, 1M 76 / 87, 4M 172 / 150.  Three of 10 for
// 30-bit keys give nothing over four of 8 (1M: 107 / 100), nor do 11 bits for 22
// (1M: 95 / 87).
static void radix_digits(uint32_t n, int key_bits, int *bits, int *passes) {
  *bits = 8;
  *passes = key_bits <= 0 ? 1 : (key_bits + 7) / 8;
  const int wide = (key_bits + 9) / 10;
  if (n <= (1u << 21) && wide < *passes && wide <= 2) {
    *bits = 10;
    *passes = wide;
  }
}

// A block sums the rows itself up to so many words per thread.
constexpr uint32_t kRadixSelfWords = 32;

size_t radix_words(uint32_t n, int key_bits) {
  int bits = 8, passes = 1;
  radix_digits(n, key_bits, &bits, &passes);
  const size_t tiles = (n + RS_TILE - 1) / RS_TILE;
  return ((size_t)1 << bits) * (tiles + 1);
}

template <int BITS>
static int radix_passes(int passes, const uint32_t *ck, const uint32_t *cv, uint32_t *k0,
                        uint32_t *v0, uint32_t *k1, uint32_t *v1, uint32_t n, uint32_t *hist,
                        hipStream_t s, const uint32_t **kout, const uint32_t **vout) {
  constexpr uint32_t D = 1u << BITS;
  const uint32_t tiles = (n + RS_TILE - 1) / RS_TILE;
  uint32_t *totals = hist + (size_t)D * tiles;
  const bool self = D / RS_THREADS * tiles <= kRadixSelfWords;
  for (int p = 0; p < passes; ++p) {
    uint32_t *ok = (p & 1) ? k1 : k0;
    uint32_t *ov = (p & 1) ? v1 : v0;
    const int shift = BITS * p;
    k_radix_upsweep<BITS><<<tiles, RS_THREADS, 0, s>>>(ck, n, shift, hist, tiles);
    if (self) {
      k_radix_downsweep<BITS, false><<<tiles, RS_THREADS, 0, s>>>(ck, cv, ok, ov, n, shift, hist,
                                                                  nullptr, tiles);
    } else {
      k_radix_rows<<<D, RS_THREADS, 0, s>>>(hist, tiles, totals);
      k_radix_downsweep<BITS, true><<<tiles, RS_THREADS, 0, s>>>(ck, cv, ok, ov, n, shift, hist,
                                                                 totals, tiles);
    }
    SPH_HIP(hipGetLastError());
    ck = ok;
    cv = ov;
  }
  *kout = ck;
  *vout = cv;
  return SPH_OK;
}

int radix_sort_pairs(const uint32_t *kin, const uint32_t *vin, uint32_t *k0, uint32_t *v0,
                     uint32_t *k1, uint32_t *v1, uint32_t n, int key_bits, uint32_t *hist,
                     hipStream_t s, const uint32_t **kout, const uint32_t **vout) {
  *kout = kin;
  *vout = vin;
  if (n == 0) return SPH_OK;
  int bits = 8, passes = 1;
  radix_digits(n, key_bits, &bits, &passes);
  const auto go = bits == 8 ? radix_passes<8> : radix_passes<10>;
  return go(passes, kin, vin, k0, v0, k1, v1, n, hist, s, kout, vout);
}

// Counts of the keys below `cells`.  A run of equal keys in a wave (sorted keys
// are nothing else) adds with one atomic: lanes of a run serialise on its word,
// and a lower bound of a million sorted pairs took 46 us, now 24.
__global__ void k_count_keys(const uint32_t *__restrict__ keys, uint32_t n,
                             uint32_t *__restrict__ count, uint32_t cells) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const uint32_t k = i < n ? keys[i] : 0xFFFFFFFFu;
  const uint32_t left = __shfl_up(k, 1, 64);
  const bool first = lane == 0 || left != k;
  const uint64_t firsts = __ballot(first);
  const uint64_t after = lane == 63 ? 0ull : firsts >> (lane + 1);
  const int next = after ? lane + 1 + __builtin_ctzll(after) : 64;
  // the lanes of the last wave that lie past n end the last run, or are one
  const uint32_t in = i < n ? min((uint32_t)(next - lane), n - i) : 0u;
  if (first && i < n && k < cells) atomicAdd(&count[k], in);
}

int count_keys(const uint32_t *keys, uint32_t n, uint32_t *count, uint32_t cells,
               hipStream_t s) {
  k_fill_u32<<<blocks_for(cells), kBlock, 0, s>>>(count, 0u, cells);
  if (n) k_count_keys<<<blocks_for(n), kBlock, 0, s>>>(keys, n, count, cells);
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

}  // namespace sph

using namespace sph;

// --------------------------------------------------------------------------
// C ABI: native sort / bounds (replacing thrust_c.cu:86-120)
// --------------------------------------------------------------------------
// Scratch of the native sort / bounds entry points, kept per device between
// calls (grow-only, held until the process ends) so that a caller that sorts
// every substep does not allocate each time.  Calls on one device take turns;
// each ends with a synchronize of the caller's stream.
namespace {
struct AbiScratch {
  std::mutex m;
  uint32_t *a = nullptr, *b = nullptr;  // `words` each
  size_t words = 0;
  uint32_t *hist = nullptr;
  size_t hist_cap = 0;
  ScanScratch sc;
  uint32_t *word = nullptr;   // the keys' OR and the count of finished blocks
  uint32_t *found = nullptr;  // the OR again, in pinned host memory
};
constexpr int kAbiDevices = 64;
AbiScratch g_abi[kAbiDevices];

int abi_scratch(AbiScratch **out) {
  int dev = 0;
  SPH_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kAbiDevices) {
    set_error("device index beyond the native entry points' scratch table");
    return SPH_ERR_ARG;
  }
  *out = &g_abi[dev];
  return SPH_OK;
}

// a and b hold at least `words` words each (contents not kept on growth)
int abi_words(AbiScratch *w, size_t words) {
  if (w->words >= words) return SPH_OK;
  if (w->a) SPH_HIP(hipFree(w->a));
  if (w->b) SPH_HIP(hipFree(w->b));
  w->a = w->b = nullptr;
  w->words = 0;
  hipError_t e = hipMalloc(&w->a, sizeof(uint32_t) * words);
  if (e == hipSuccess) e = hipMalloc(&w->b, sizeof(uint32_t) * words);
  if (e != hipSuccess) return hip_fail(e, "hipMalloc (native entry point scratch)");
  w->words = words;
  return SPH_OK;
}
}  // namespace

// OR of all keys: the highest set bit gives the radix passes a 32-bit sort
// needs.  One device-scope atomic per block (with one per wave, 4096 of them on
// one word took 50 us); the last block to finish puts the result into pinned
// host memory and both words back to zero for the next call.
constexpr uint32_t kOrBlocks = 256;
__global__ __launch_bounds__(kBlock) void k_or_keys(const uint32_t *__restrict__ keys,
                                                    uint32_t n, uint32_t *words,
                                                    uint32_t *found) {
  __shared__ uint32_t part[kBlock / kWave];
  uint32_t v = 0;
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
    v |= keys[i];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v |= __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kBlock / kWave; ++w) v |= part[w];
    atomicOr(&words[0], v);
    __threadfence();
    if (atomicAdd(&words[1], 1u) == gridDim.x - 1u) {
      *found = atomicExch(&words[0], 0u);
      atomicExch(&words[1], 0u);
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_copy_pairs(uint32_t n, const uint32_t *__restrict__ k,
                                                       const uint32_t *__restrict__ v,
                                                       uint32_t *__restrict__ kout,
                                                       uint32_t *__restrict__ vout) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  kout[i] = k[i];
  vout[i] = v[i];
}

// The word pair and the pinned word of k_or_keys, on first use.
static int or_words(AbiScratch *w, hipStream_t s) {
  if (w->word && w->found) return SPH_OK;
  hipError_t e = hipSuccess;
  if (!w->word) {
    e = hipMalloc(&w->word, 2 * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMemsetAsync(w->word, 0, 2 * sizeof(uint32_t), s);
    if (e != hipSuccess) {
      if (w->word) (void)hipFree(w->word);
      w->word = nullptr;
      return hip_fail(e, "hipMalloc (key range)");
    }
  }
  e = hipHostMalloc((void **)&w->found, sizeof(uint32_t), hipHostMallocDefault);
  if (e != hipSuccess) {
    w->found = nullptr;
    return hip_fail(e, "hipHostMalloc (key range)");
  }
  return SPH_OK;
}

static int sort_impl(uint32_t *keys, uint32_t *values, int n, int key_bits, void *stream) {
  if (n < 0 || (n > 0 && (!keys || !values)) || key_bits < 0 || key_bits > 32) {
    set_error("sph_sort_by_key: invalid argument");
    return SPH_ERR_ARG;
  }
  if (n <= 1) return SPH_OK;
  hipStream_t s = (hipStream_t)stream;
  AbiScratch *w = nullptr;
  int rc = abi_scratch(&w);
  if (rc) return rc;
  std::lock_guard<std::mutex> lock(w->m);
  if ((rc = abi_words(w, (size_t)n))) return rc;
  if (key_bits == 0) {  // unknown key range: from the keys' OR
    if ((rc = or_words(w, s))) return rc;
    k_or_keys<<<std::min(blocks_for((uint32_t)n), kOrBlocks), kBlock, 0, s>>>(
        keys, (uint32_t)n, w->word, w->found);
    SPH_HIP(hipGetLastError());
    SPH_HIP(hipStreamSynchronize(s));
    const uint32_t all = *(volatile uint32_t *)w->found;
    key_bits = all ? 32 - __builtin_clz(all) : 1;
  }
  const size_t need = radix_words((uint32_t)n, key_bits);
  if (w->hist_cap < need) {
    if (w->hist) SPH_HIP(hipFree(w->hist));
    w->hist = nullptr;
    w->hist_cap = 0;
    SPH_HIP(hipMalloc(&w->hist, sizeof(uint32_t) * need));
    w->hist_cap = need;
  }
  const uint32_t *kout = nullptr, *vout = nullptr;
  rc = radix_sort_pairs(keys, values, w->a, w->b, keys, values, (uint32_t)n, key_bits, w->hist, s,
                        &kout, &vout);
  if (rc == SPH_OK && kout != keys) {
    k_copy_pairs<<<blocks_for((uint32_t)n), kBlock, 0, s>>>((uint32_t)n, kout, vout, keys, values);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) rc = hip_fail(e, "k_copy_pairs");
  }
  const hipError_t e = hipStreamSynchronize(s);
  if (rc == SPH_OK && e != hipSuccess) rc = hip_fail(e, "hipStreamSynchronize (sort)");
  return rc;
}

extern "C" int sph_sort_by_key_bits(uint32_t *keys, uint32_t *values, int n, int key_bits,
                                    void *stream) {
  if (key_bits < 1) {
    set_error("sph_sort_by_key: invalid argument");
    return SPH_ERR_ARG;
  }
  return sort_impl(keys, values, n, key_bits, stream);
}

// Keys of any range: the passes follow the keys' highest set bit.
extern "C" int sph_sort_by_key(uint32_t *keys, uint32_t *values, int n, void *stream) {
  return sort_impl(keys, values, n, 0, stream);
}

// --------------------------------------------------------------------------
// Sort without allocation: scratch in a file-scope device array
// --------------------------------------------------------------------------
// For callers that cannot allocate device memory (code under stream capture,
// serving loops, harnesses that forbid hipMalloc).  Layout, in words: the two
// ping-pong buffers (kStaticPairs each) and the digit histogram with its totals
// (for the widest digits); each part starts on a 16-byte boundary.
namespace {
constexpr size_t kStaticPairs = size_t(1) << 21;
constexpr size_t kStaticTiles = (kStaticPairs + RS_TILE - 1) / RS_TILE;
constexpr size_t kStaticHist = 1024 * (kStaticTiles + 1);
constexpr size_t kStaticWords = 2 * kStaticPairs + kStaticHist;
static_assert(kStaticPairs % 4 == 0 && kStaticHist % 4 == 0, "16-byte aligned parts");
static_assert(kStaticPairs == SPH_SORT_NOALLOC_MAX_PAIRS, "header limit");
}  // namespace

// Each GPU holds its own copy until the process ends (about 19 MB).
static __device__ __align__(256) uint32_t scratch[kStaticWords];

namespace {
// Device address of `scratch` on each device, looked up once per device with
// that device current (the host-side name is not a device address).
std::mutex g_static_m;
uint32_t *g_static_ptr[kAbiDevices] = {};

int static_scratch(uint32_t **out) {
  int dev = 0;
  SPH_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kAbiDevices) {
    set_error("device index beyond the native entry points' scratch table");
    return SPH_ERR_ARG;
  }
  std::lock_guard<std::mutex> lock(g_static_m);
  if (!g_static_ptr[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress (sort scratch)");
    g_static_ptr[dev] = static_cast<uint32_t *>(p);
  }
  *out = g_static_ptr[dev];
  return SPH_OK;
}
}  // namespace

extern "C" int sph_sort_by_key_bits_noalloc(uint32_t *keys, uint32_t *values, int n,
                                            int key_bits, void *stream) {
  if (n < 0 || (n > 0 && (!keys || !values)) || key_bits < 1 || key_bits > 32) {
    set_error("sph_sort_by_key_bits_noalloc: invalid argument");
    return SPH_ERR_ARG;
  }
  if ((size_t)n > kStaticPairs) {
    set_error("sph_sort_by_key_bits_noalloc: n exceeds SPH_SORT_NOALLOC_MAX_PAIRS (2^21)");
    return SPH_ERR_ARG;
  }
  if (n <= 1) return SPH_OK;
  uint32_t *base = nullptr;
  int rc = static_scratch(&base);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  uint32_t *a = base, *b = base + kStaticPairs, *hist = base + 2 * kStaticPairs;
  const uint32_t *kout = nullptr, *vout = nullptr;
  rc = radix_sort_pairs(keys, values, a, b, keys, values, (uint32_t)n, key_bits, hist, s, &kout,
                        &vout);
  if (rc) return rc;
  if (kout != keys) {  // an odd number of passes ends in the scratch buffers
    k_copy_pairs<<<blocks_for((uint32_t)n), kBlock, 0, s>>>((uint32_t)n, kout, vout, keys, values);
    SPH_HIP(hipGetLastError());
  }
  return SPH_OK;
}

static int bounds_impl(const uint32_t *keys, int n, int cells, uint32_t *out, void *stream,
                       bool upper) {
  if (n < 0 || cells < 0 || (cells > 0 && !out) || (n > 0 && !keys)) {
    set_error("sph_find_bounds: invalid argument");
    return SPH_ERR_ARG;
  }
  if (cells == 0) return SPH_OK;
  hipStream_t s = (hipStream_t)stream;
  AbiScratch *w = nullptr;
  int rc = abi_scratch(&w);
  if (rc) return rc;
  std::lock_guard<std::mutex> lock(w->m);
  if ((rc = abi_words(w, (size_t)cells))) return rc;
  rc = count_keys(keys, (uint32_t)n, w->a, (uint32_t)cells, s);
  if (rc == SPH_OK) rc = scan(w->a, out, (uint32_t)cells, upper, false, &w->sc, s, nullptr);
  const hipError_t e = hipStreamSynchronize(s);
  if (rc == SPH_OK && e != hipSuccess) rc = hip_fail(e, "hipStreamSynchronize (bounds)");
  return rc;
}

extern "C" int sph_find_lower_bounds(const uint32_t *keys, int n, int cells, uint32_t *out,
                                     void *stream) {
  return bounds_impl(keys, n, cells, out, stream, false);
}

extern "C" int sph_find_upper_bounds(const uint32_t *keys, int n, int cells, uint32_t *out,
                                     void *stream) {
  return bounds_impl(keys, n, cells, out, stream, true);
}
