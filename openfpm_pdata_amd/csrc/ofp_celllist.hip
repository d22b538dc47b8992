// ofp_celllist.hip -- CellList_gpu construction, reorder and restore.
//
// Build (per updateCellListGPU): a stable LSD radix sort of the particles by
// cell id, started from the identity order, so inside every cell the particles
// come out in ascending original index (domain ids < ghost ids: domain first).
// That is the canonical order, reached without atomics on cell counters.
//   1. k_rx_hist     pass 0: cell id per particle (the key), and per tile of
//                    4096 particles (1024 in small builds) the histogram of the
//                    pass's digit (<= 8 bits), counted per wave with ballots, one
//                    LDS add per digit run.
//   2. column sums   of the [tile][digit] histogram table give every (tile,
//                    digit) its first output slot: summed in the scatter up to
//                    kRxChunked tiles, in kernels of their own beyond.
//   3. k_rx_scatter  per tile: stable rank of each key inside the tile (ballot
//                    peer masks, per-wave running counts in LDS), staged in LDS in
//                    digit order, then written out as contiguous runs.
//   Passes 1.. repeat 1-3 on the next digit (k_rx_hist reads the keys).
//   Positions to be reordered ride along as a payload when pass 0 counts many
//   descents (input far from cell order); otherwise step 6 gathers them.
//   4. k_cl_runs     per run of equal sorted keys (one occupied cell): its
//                    length and its number of domain particles, from ballots of
//                    run starts and domain flags over 64 consecutive slots.
//   5. scan (u64)    packed (domain << 32 | count) per cell -> cell starts (low
//                    word) and domain-id starts (high word).
//   6. k_cl_emit     per sorted slot: nonsort_to_sort, domain sort ids, reordered
//                    positions and planes, and the quantised cell-relative stream.
//                    From 2^22 particles far from cell order, nonsort_to_sort and
//                    the planes go by ranges of destinations (permute_far), as
//                    restores and reorders then do.
// The particle count may be read from device memory (ensembles whose ghost count
// stays on the device): every kernel is launched for the capacity and returns
// past the count.
#include "ofp_internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <mutex>

struct ofp_cl {
  ofp::HandleLife life;
  int dtype = OFP_F32;
  uint32_t opt = 0;
  ofp::CellGeom<float> gf;
  ofp::CellGeom<double> gd;
  double lo[3], sp[3];
  uint32_t div[3], divc[3];
  uint64_t n_cells = 0;
  uint64_t n_part = 0, gm = 0;
  bool built = false;
  uint32_t box_nn = 1;
  // ensemble mode: per-system grids in device memory (owned by the caller)
  uint32_t n_sys = 0;               // 0: one grid
  const void* sys = nullptr;        // SysGrid<T>[n_sys]
  const uint32_t* sid = nullptr;    // system of each particle, input order
  const uint32_t* rbase = nullptr;  // first global x-row of each system (n_sys + 1)
  uint32_t n_rows = 0;              // x-rows of all grids
  const uint32_t* n_dev = nullptr;  // particle count in device memory (or null)
  // target-item work queue (built on first use after each construct)
  bool items_valid = false;
  size_t items_cap = 0;
  ofp::DevBuf packed, scan64, keys, keys2, s2n, vals2, n2s, dom, quant, scantmp, hist, sid_sorted, payload;
  ofp::DevBuf colpart;  // chunk sums of the histogram table
  // the last construct's particles were many and far from cell order, and there is
  // scratch for permute_far (payload, cursors).  It serves one call after another:
  // restores and reorders may come from several threads and streams
  bool far = false;
  ofp::DevBuf cursors;
  mutable std::mutex far_lock;
  hipEvent_t far_done = nullptr;
  // the order check's result on the host (pinned) and its event
  unsigned long long* desc = nullptr;
  hipEvent_t checked = nullptr;
  ofp::DevBuf items;
  ofp::DevBuf aux;            // pair kernels' per-particle record stream (cell tiles)
  // sparse view (ofp_cl_build_sparse): non-empty cells only
  ofp::DevBuf nz_flag, nz_key, nz_start, nz_nn, nz_inv;
  uint64_t n_nz = 0;
  bool sparse_valid = false;
  uint32_t nz_box_nn = 1;  // stencil half-width of the sparse view's neighbour table
};

namespace ofp {

constexpr int kRxBlock = 256;
constexpr int kRxWaves = kRxBlock / kWave;
// 64-key rounds per wave, and so the keys per tile (256 x rounds): 4096 for long
// runs per digit, 1024 below kRxSmall particles, where tiles of 4096 leave most
// CUs without a block and a wave works through 16 rounds one after another (and
// through four times the code, fetched cold): 17,000 keys, a scatter 26 -> 13 us.
constexpr int kRxLong = 16, kRxShort = 4;
constexpr size_t kRxSmall = size_t(1) << 20;
constexpr int kRxMaxBits = 8;
// Up to kRxDirect tiles a scatter block sums the tiles' histograms itself; up to
// kRxChunked it sums those of its own chunk of tiles and the chunks' sums, which
// the histogram blocks add up with atomics (at most 32 adds per word): two launches
// per pass.  The rows a block sums are loaded kColBatch at a time, one batch after
// another: at 65 tiles 2 batches with chunks, 5 without.  Beyond kRxChunked, the
// column kernels do it (four launches): a block would read over 100 rows of 1 KB
// for its 4096 keys.
constexpr uint32_t kRxDirect = 32;
constexpr uint32_t kRxChunked = 2048;
// Below this many particles the host does not wait for the order check before it
// launches the passes: their kernels return at once if the check found the input in
// cell order.  Whole builds with and without the wait (us): input in order 47 and 53
// at 17,000 particles, 70 and 64 at 2^20, 133 and 134 at 8e6; one exchanged pair 81
// and 62, 186 and 163, 438 and 417.  From here on the empty grids cost more.
constexpr size_t kRxNoSync = size_t(1) << 23;
constexpr int kRxBins = 1 << kRxMaxBits;

__device__ __forceinline__ uint32_t lanes_below(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
}

// Lanes of `act` whose digit equals this lane's (digit < 2^bits).
__device__ __forceinline__ unsigned long long rx_peers(uint32_t d, int bits, unsigned long long act) {
  unsigned long long m = act;
  for (int b = 0; b < bits; ++b) {
    const bool bit = ((d >> b) & 1u) != 0u;
    const unsigned long long v = __ballot(bit);
    m &= bit ? v : ~v;
  }
  return m;
}

__device__ __forceinline__ uint32_t count_of(uint32_t n_host, const uint32_t* n_dev) {
  return n_dev ? *n_dev : n_host;
}


// Grid-uniform: the order check (*check = its descents; null = no check was
// made) found the input in cell order, so the build is done.
__device__ __forceinline__ bool in_order(const unsigned long long* check) { return check && *check == 0ull; }

// Tile histogram of one digit.  Pass 0 (kin == null) evaluates the key, stores
// it to kout, clears the cells' counts (clear[0 .. n_clear), null: not needed),
// adds the digits' counts to the tile's chunk (part != null; cleared before), and,
// where no order check ran before (disorder != null), adds the tile's
// descents (k[e] > k[e+1] inside each 64-key round) to *disorder, which then
// tells how far the input is from cell order.
template <class Key, int kIters>
__global__ __launch_bounds__(kRxBlock) void k_rx_hist(Key key, const uint32_t* __restrict__ kin,
                                                      uint32_t* __restrict__ kout, uint32_t n_host,
                                                      const uint32_t* __restrict__ n_dev, int shift, int bits,
                                                      uint32_t n_tiles, uint32_t* __restrict__ hist,
                                                      unsigned long long* __restrict__ disorder,
                                                      const unsigned long long* __restrict__ check,
                                                      unsigned long long* __restrict__ clear, uint64_t n_clear,
                                                      uint32_t* __restrict__ part, uint32_t ch) {
  if (in_order(check)) return;
  constexpr uint32_t kRxTile = uint32_t(kRxBlock * kIters);
  __shared__ uint32_t h[kRxBins];
  __shared__ uint32_t wdesc[kRxWaves];
  const uint32_t n = count_of(n_host, n_dev);
  const uint32_t t = blockIdx.x;
  if (clear)
    for (uint64_t i = uint64_t(t) * kRxBlock + threadIdx.x; i < n_clear; i += uint64_t(gridDim.x) * kRxBlock)
      clear[i] = 0ull;
  for (int d = threadIdx.x; d < kRxBins; d += kRxBlock) h[d] = 0;
  __syncthreads();
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const uint32_t mask = (1u << bits) - 1u;
  const uint64_t base = uint64_t(t) * kRxTile + uint64_t(w) * (kIters * kWave);
  uint32_t desc = 0;
  // batches of rounds: the batch's loads first, then its stores, then the
  // counting; all 16 rounds at once for stored keys, 4 when the keys are
  // evaluated from the positions (their registers)
  auto rounds = [&](auto batch) {
    constexpr int kB = decltype(batch)::value;
#pragma unroll 1
    for (int b = 0; b < kIters; b += kB) {
      uint32_t kr[kB];
#pragma unroll
      for (int i = 0; i < kB; ++i) {
        const uint64_t e = base + uint64_t(b + i) * kWave + uint64_t(lane);
        kr[i] = 0u;
        if (e < n) kr[i] = kin ? kin[e] : key(uint32_t(e));
      }
      if (!kin) {
#pragma unroll
        for (int i = 0; i < kB; ++i) {
          const uint64_t e = base + uint64_t(b + i) * kWave + uint64_t(lane);
          if (e < n) kout[e] = kr[i];
        }
      }
#pragma unroll
      for (int i = 0; i < kB; ++i) {
        const uint64_t e = base + uint64_t(b + i) * kWave + uint64_t(lane);
        const bool v = e < n;
        const unsigned long long act = __ballot(v);
        if (act == 0ull) continue;  // wave-uniform: a round past n
        const uint32_t k = kr[i];
        if (!kin && disorder) {
          const uint32_t next = __shfl_down(k, 1, kWave);
          const bool nv = lane + 1 < kWave && ((act >> (lane + 1)) & 1ull);
          desc += (v && nv && k > next) ? 1u : 0u;
        }
        const uint32_t d = (k >> shift) & mask;
        const unsigned long long peers = rx_peers(d, bits, act);
        if (v && lanes_below(peers) == 0u) atomicAdd(&h[d], uint32_t(__popcll(peers)));
      }
    }
  };
  if (kin)
    rounds(std::integral_constant<int, kIters>{});
  else
    rounds(std::integral_constant<int, 4>{});
  if (!kin && disorder) {
    desc = wave_sum(desc);
    if (lane == 0) wdesc[w] = desc;
  }
  __syncthreads();
  for (int d = threadIdx.x; d < (1 << bits); d += kRxBlock) {
    const uint32_t v = h[d];
    hist[size_t(t) * kRxBins + d] = v;
    if (part && v) atomicAdd(&part[size_t(t / ch) * kRxBins + d], v);
  }
  if (!kin && disorder && threadIdx.x == 0) {
    uint32_t s = 0;
    for (int ww = 0; ww < kRxWaves; ++ww) s += wdesc[ww];
    if (s) atomicAdd(disorder, static_cast<unsigned long long>(s));
  }
}

// Carry the positions through the radix passes (instead of one gather at the
// end) when at least one key in kDisorderDen is followed by a smaller one: a
// gather from input that far from cell order reads a cache line per coordinate.
constexpr uint64_t kDisorderDen = 8;
__device__ __forceinline__ bool carry_positions(const unsigned long long* disorder, uint32_t n) {
  return disorder && *disorder * kDisorderDen > uint64_t(n);
}

// Offsets of the [tile][digit] table (rows of kRxBins, written and read as
// coalesced rows): offs[t][d] = sum of all counts of digits < d + sum of the
// counts of digit d in tiles < t.  The tiles form at most kColChunks chunks;
// every loop below loads kColBatch rows before it uses them.
constexpr uint32_t kColChunks = 64;
constexpr uint32_t kColBatch = 16;
constexpr int kColGroups = 4;  // of kRxBins threads

// Sum of rows [a, b) of the table's column d.
__device__ __forceinline__ uint32_t col_sum(const uint32_t* __restrict__ tab, uint32_t a, uint32_t b, int d) {
  uint32_t s = 0;
  for (uint32_t t = a; t < b; t += kColBatch) {
    uint32_t v[kColBatch];
#pragma unroll
    for (uint32_t i = 0; i < kColBatch; ++i) v[i] = t + i < b ? tab[size_t(t + i) * kRxBins + d] : 0u;
#pragma unroll
    for (uint32_t i = 0; i < kColBatch; ++i) s += v[i];
  }
  return s;
}

// Exclusive scan of one value per digit over the first kRxBins threads of the
// block (ws: a word per wave of them); every thread of the block calls it.
__device__ __forceinline__ uint32_t digit_excl_scan(uint32_t v, uint32_t* ws) {
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const uint32_t inc = wave_incl_scan(v);
  if (lane == kWave - 1 && w < kRxBins / kWave) ws[w] = inc;
  __syncthreads();
  uint32_t base = inc - v;
  if (w < kRxBins / kWave)
    for (int i = 0; i < w; ++i) base += ws[i];
  __syncthreads();
  return base;
}

// part[c][d] = counts of digit d in the tiles of chunk c
__global__ __launch_bounds__(kRxBins) void k_rx_colsum(const uint32_t* __restrict__ tab, uint32_t n_tiles,
                                                       uint32_t ch, int nb, uint32_t* __restrict__ part,
                                                       const unsigned long long* __restrict__ check) {
  if (in_order(check)) return;
  const uint32_t c = blockIdx.x;
  const int d = threadIdx.x;
  const uint32_t t0 = c * ch;
  const uint32_t t1 = t0 + ch < n_tiles ? t0 + ch : n_tiles;
  part[size_t(c) * kRxBins + d] = d < nb ? col_sum(tab, t0, t1, d) : 0u;
}

// tab[t][d] of chunk c becomes offs[t][d].  Every block sums the chunks' counts
// itself, a quarter of them per group of kRxBins threads (one batch of loads), so
// no launch of one block stands between the sums and their use.
__global__ __launch_bounds__(kColGroups* kRxBins) void k_rx_colapply(uint32_t* __restrict__ tab, uint32_t n_tiles,
                                                                      uint32_t ch, int nb, uint32_t n_chunks,
                                                                      const uint32_t* __restrict__ part,
                                                                      const unsigned long long* __restrict__ check) {
  if (in_order(check)) return;
  __shared__ uint32_t below[kColGroups][kRxBins];  // chunks before c
  __shared__ uint32_t total[kColGroups][kRxBins];
  __shared__ uint32_t run_of[kColGroups][kRxBins];  // tiles of the chunk before the group's
  __shared__ uint32_t ws[kRxBins / kWave];
  const uint32_t c = blockIdx.x;
  const int d = int(threadIdx.x) % kRxBins, g = int(threadIdx.x) / kRxBins;
  const uint32_t per = (n_chunks + kColGroups - 1) / kColGroups;
  const uint32_t a = uint32_t(g) * per, b = a + per < n_chunks ? a + per : n_chunks;
  const uint32_t lo = c < a ? a : (c < b ? c : b);  // [a, lo) lie before c
  const uint32_t s0 = a < b ? col_sum(part, a, lo, d) : 0u;
  below[g][d] = s0;
  total[g][d] = a < b ? s0 + col_sum(part, lo, b, d) : 0u;
  // the chunk's tiles, a quarter per group
  const uint32_t t0 = c * ch;
  const uint32_t t1 = t0 + ch < n_tiles ? t0 + ch : n_tiles;
  const uint32_t pt = (t1 - t0 + kColGroups - 1) / kColGroups;
  const uint32_t ta = t0 + uint32_t(g) * pt < t1 ? t0 + uint32_t(g) * pt : t1;
  const uint32_t tb = ta + pt < t1 ? ta + pt : t1;
  run_of[g][d] = d < nb ? col_sum(tab, ta, tb, d) : 0u;
  __syncthreads();
  uint32_t all = 0, run = 0;
#pragma unroll
  for (int q = 0; q < kColGroups; ++q) {
    all += total[q][d];
    run += below[q][d];
    if (q < g) run += run_of[q][d];
  }
  const uint32_t base = digit_excl_scan(all, ws);  // of group 0's threads
  if (g == 0) below[0][d] = base;
  __syncthreads();
  if (d >= nb) return;
  run += below[0][d];
  for (uint32_t t = ta; t < tb; t += kColBatch) {
    uint32_t v[kColBatch];
#pragma unroll
    for (uint32_t i = 0; i < kColBatch; ++i) v[i] = t + i < tb ? tab[size_t(t + i) * kRxBins + d] : 0u;
#pragma unroll
    for (uint32_t i = 0; i < kColBatch; ++i) {
      if (t + i < tb) tab[size_t(t + i) * kRxBins + d] = run;
      run += v[i];
    }
  }
}

// Stable scatter of one tile by one digit; offs = [tile][digit] offset table, or
// (direct) the tiles' histograms, from which the block sums its row, with the sums
// of the chunks of ch tiles where part is given.
// vin == null stands for the identity (pass 0).  Payload: three planes of T
// (positions) that travel with the keys, pin (stride si) in the input order,
// pout (stride so) in the output order; null = none.  Keys, values and each
// payload plane are read in input order (coalesced), placed in LDS at their
// staged slot, and written out in staged order: runs of one digit each.
template <class T, int kIters>
__global__ __launch_bounds__(kRxBlock) void k_rx_scatter(const uint32_t* __restrict__ kin,
                                                         const uint32_t* __restrict__ vin, uint32_t n_host,
                                                         const uint32_t* __restrict__ n_dev, int shift,
                                                         int bits, uint32_t n_tiles,
                                                         const uint32_t* __restrict__ offs,
                                                         uint32_t* __restrict__ kout,
                                                         uint32_t* __restrict__ vout, const T* __restrict__ pin,
                                                         size_t si, T* __restrict__ pout, size_t so,
                                                         const unsigned long long* __restrict__ disorder,
                                                         const unsigned long long* __restrict__ check,
                                                         int direct, const uint32_t* __restrict__ part,
                                                         uint32_t ch, uint32_t n_chunks) {
  if (in_order(check)) return;
  constexpr uint32_t kRxTile = uint32_t(kRxBlock * kIters);
  __shared__ uint32_t wh[kRxWaves][kRxBins];  // running count per wave, then wave prefix
  __shared__ uint32_t tstart[kRxBins];        // first staged slot of each digit
  __shared__ uint32_t goff[kRxBins];          // first output slot of each digit
  __shared__ uint32_t wsum[kRxWaves + 1];
  __shared__ uint32_t sk[kRxTile];                       // staged keys, then their output slots
  __shared__ uint32_t sv[kRxTile * (sizeof(T) / 4)];     // staged values, then one payload plane
  T* const sp = reinterpret_cast<T*>(sv);
  const uint32_t n = count_of(n_host, n_dev);
  const uint32_t t = xcd_tile(blockIdx.x, gridDim.x);
  const uint64_t tile0 = uint64_t(t) * kRxTile;
  if (tile0 >= n) return;  // block-uniform
  const int nb = 1 << bits;
  const uint32_t mask = uint32_t(nb) - 1u;
  for (int d = threadIdx.x; d < kRxBins; d += kRxBlock) {
#pragma unroll
    for (int w = 0; w < kRxWaves; ++w) wh[w][d] = 0;
    if (!direct) goff[d] = d < nb ? offs[size_t(t) * kRxBins + d] : 0u;
  }
  if (direct) {
    const int d = threadIdx.x;
    static_assert(kRxBlock == kRxBins, "a thread per digit");
    const uint32_t c = t / ch;
    uint32_t before = 0, all = 0;
    if (d < nb) {
      if (part) {
        before = col_sum(part, 0, c, d);
        all = before + col_sum(part, c, n_chunks, d);
        before += col_sum(offs, c * ch, t, d);
      } else {
        before = col_sum(offs, 0, t, d);
        all = before + col_sum(offs, t, n_tiles, d);
      }
    }
    goff[d] = digit_excl_scan(all, wsum) + before;
  }
  __syncthreads();
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const uint64_t base = tile0 + uint64_t(w) * (kIters * kWave);
  uint32_t key[kIters], lr[kIters], val[kIters];
  // all loads of the wave's rounds first
#pragma unroll
  for (int it = 0; it < kIters; ++it) {
    const uint64_t e = base + uint64_t(it) * kWave + uint64_t(lane);
    key[it] = 0u;
    val[it] = uint32_t(e);
    if (e < n) {
      key[it] = kin[e];
      if (vin) val[it] = vin[e];
    }
  }
#pragma unroll
  for (int it = 0; it < kIters; ++it) {
    const uint64_t e = base + uint64_t(it) * kWave + uint64_t(lane);
    const bool v = e < n;
    const unsigned long long act = __ballot(v);
    const uint32_t k = key[it];
    const uint32_t d = (k >> shift) & mask;
    uint32_t r = 0;
    if (act != 0ull) {
      const unsigned long long peers = rx_peers(d, bits, act);
      const uint32_t below = lanes_below(peers);
      const uint32_t prior = v ? wh[w][d] : 0u;
      r = prior + below;
      if (v && below == 0u) wh[w][d] = prior + uint32_t(__popcll(peers));
    }
    lr[it] = r;
  }
  __syncthreads();
  // wave prefixes per digit and the tile's digit totals
  uint32_t tot = 0;
  if (threadIdx.x < kRxBins) {
    const int d = threadIdx.x;
#pragma unroll
    for (int ww = 0; ww < kRxWaves; ++ww) {
      const uint32_t c = wh[ww][d];
      wh[ww][d] = tot;
      tot += c;
    }
  }
  // exclusive scan of the digit totals (one digit per thread)
  const uint32_t inc = wave_incl_scan(tot);
  if (lane == kWave - 1) wsum[w] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t s = 0;
    for (int ww = 0; ww < kRxWaves; ++ww) {
      const uint32_t c = wsum[ww];
      wsum[ww] = s;
      s += c;
    }
  }
  __syncthreads();
  if (threadIdx.x < kRxBins) tstart[threadIdx.x] = wsum[w] + inc - tot;
  __syncthreads();
  // lr[it] becomes the staged slot of element it
#pragma unroll
  for (int it = 0; it < kIters; ++it) {
    const uint64_t e = base + uint64_t(it) * kWave + uint64_t(lane);
    if (e < n) {
      const uint32_t d = (key[it] >> shift) & mask;
      const uint32_t slot = tstart[d] + wh[w][d] + lr[it];
      lr[it] = slot;
      sk[slot] = key[it];
      sv[slot] = val[it];
    }
  }
  __syncthreads();
  const uint32_t len = uint32_t(n - tile0 < kRxTile ? n - tile0 : kRxTile);
  constexpr uint32_t kNone = 0xFFFFFFFFu;
  for (uint32_t s = threadIdx.x; s < len; s += kRxBlock) {
    const uint32_t k = sk[s];
    const uint32_t d = (k >> shift) & mask;
    const uint32_t o = goff[d] + (s - tstart[d]);
    // o < n always holds for a consistent table; the test keeps a bad one in bounds
    if (o < n) {
      kout[o] = k;
      vout[o] = sv[s];
    }
    sk[s] = o < n ? o : kNone;
  }
  if (!pin || !carry_positions(disorder, n)) return;  // grid-uniform
  for (int q = 0; q < 3; ++q) {
    __syncthreads();  // sv / the previous plane has been read
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
      const uint64_t e = base + uint64_t(it) * kWave + uint64_t(lane);
      if (e < n) sp[lr[it]] = pin[size_t(q) * si + e];
    }
    __syncthreads();
    for (uint32_t s = threadIdx.x; s < len; s += kRxBlock) {
      const uint32_t o = sk[s];
      if (o != kNone) pout[size_t(q) * so + o] = sp[s];
    }
  }
}

// Per occupied cell, from the sorted keys (packed[] cleared before): (domain
// particles << 32 | particles).  Each wave covers 64 consecutive sorted slots;
// ballots of "a run of equal keys starts here" and "domain particle" split the
// wave into run segments, whose lengths and domain counts are bit counts.  A
// segment that is a whole run is stored; the pieces of a run that crosses a
// wave boundary are added atomically.  One coalesced read of keys and
// sort_to_nonsort; empty cells keep 0.  A wave takes kRounds rounds of 64
// slots with all loads issued first (the work per slot is a few bit operations,
// so the loads' latency is what there is to hide).

// The runs of one wave's kRounds rounds of 64 consecutive sorted slots from
// w0: kk = keys, kp = the previous slot's key, dmf = domain particle.  The run
// that reaches the end of a round is carried (wave-uniform) into the next
// round: only a run that crosses the wave's first or last slot is added
// atomically, every other run is stored once.
template <int kRounds>
__device__ __forceinline__ void runs_of_wave(const uint32_t (&kk)[kRounds], const uint32_t (&kp)[kRounds],
                                             const bool (&dmf)[kRounds], uint64_t w0, uint32_t n,
                                             uint64_t n_cells, unsigned long long* __restrict__ packed) {
  const int lane = threadIdx.x & (kWave - 1);
  uint32_t ck = 0;              // carried run: key,
  unsigned long long cval = 0;  // (domain << 32 | count) so far,
  bool copen = false;           // open,
  bool cown = false;            // started inside this wave
  auto seg_val = [](unsigned long long D, int a, int e) {
    const unsigned long long upto = e == kWave - 1 ? ~0ull : (1ull << (e + 1)) - 1ull;
    const unsigned long long seg = upto & ~((1ull << a) - 1ull);
    return (static_cast<unsigned long long>(__popcll(D & seg)) << 32) | static_cast<unsigned long long>(e - a + 1);
  };
  auto close = [&]() {
    if (copen && lane == 0 && uint64_t(ck) < n_cells) {
      if (cown)
        packed[ck] = cval;
      else
        atomicAdd(&packed[ck], cval);
    }
    copen = false;
  };
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const uint64_t f = w0 + uint64_t(r) * kWave + uint64_t(lane);
    const bool v = f < n;
    const uint32_t k = kk[r];
    const bool st = v && (f == 0 || kp[r] != k);
    const bool dm = v && dmf[r];
    const unsigned long long S = __ballot(st), D = __ballot(dm), V = __ballot(v);
    if (V == 0ull) break;  // wave-uniform: this and later rounds are past n
    const int last = 63 - __builtin_clzll(V);
    const uint64_t f0 = w0 + uint64_t(r) * kWave;  // slot of lane 0
    const bool ends_at_n = f0 + uint64_t(last) + 1 == n;
    if (S & 1ull) {
      close();  // the carried run ended at the previous round's last slot
    } else {
      // lanes [0, e0] continue the run of the previous slot
      const unsigned long long up = S & ~1ull;
      const int e0 = up ? __builtin_ctzll(up) - 1 : last;
      const unsigned long long v0 = seg_val(D, 0, e0);
      if (copen) {
        cval += v0;
      } else {
        ck = uint32_t(__builtin_amdgcn_readfirstlane(int(k)));
        cval = v0;
        cown = false;
        copen = true;
      }
      if (up || ends_at_n) close();
    }
    // runs starting in this round: stored here when they end in the round, the
    // last one carried otherwise
    const int hi = S ? 63 - __builtin_clzll(S) : -1;
    const bool hi_open = hi >= 0 && !ends_at_n;
    if (st && uint64_t(k) < n_cells && !(hi_open && lane == hi)) {
      const unsigned long long above = lane == kWave - 1 ? 0ull : (S >> (lane + 1)) << (lane + 1);
      const int e = above ? __builtin_ctzll(above) - 1 : last;
      packed[k] = seg_val(D, lane, e);
    }
    if (hi_open) {
      ck = uint32_t(__builtin_amdgcn_readlane(int(k), hi));
      cval = seg_val(D, hi, last);
      cown = true;
      copen = true;
    }
  }
  // a run open at the wave's end may go on in the next wave
  if (copen) {
    cown = false;
    close();
  }
}

// Per occupied cell, from the sorted keys (packed[] cleared before): (domain
// particles << 32 | particles).  Each wave covers 64 consecutive sorted slots
// per round; ballots of "a run of equal keys starts here" and "domain particle"
// split the wave into run segments, whose lengths and domain counts are bit
// counts (runs_of_wave).  One coalesced read of keys and sort_to_nonsort; empty
// cells keep 0.  All loads of the wave's kRounds rounds are issued first
// (the work per slot is a few bit operations, so the loads' latency is what
// there is to hide).
template <int kRounds>
__global__ __launch_bounds__(256) void k_cl_runs(const uint32_t* __restrict__ keys,
                                                 const uint32_t* __restrict__ s2n, uint32_t n_host,
                                                 const uint32_t* __restrict__ n_dev, uint32_t gm,
                                                 uint64_t n_cells, unsigned long long* __restrict__ packed,
                                                 const unsigned long long* __restrict__ check) {
  if (in_order(check)) return;
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t w0 = (uint64_t(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave) * (kRounds * kWave);
  const uint32_t n = count_of(n_host, n_dev);
  uint32_t kk[kRounds], kp[kRounds];
  bool dm[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const uint64_t f = w0 + uint64_t(r) * kWave + uint64_t(lane);
    kk[r] = 0u;
    kp[r] = ~0u;
    dm[r] = false;
    if (f < n) {
      kk[r] = keys[f];
      dm[r] = s2n[f] < gm;
      if (f > 0) kp[r] = keys[f - 1];
    }
  }
  runs_of_wave<kRounds>(kk, kp, dm, w0, n, n_cells, packed);
}

template <class T>
struct EmitArgs {
  const T* pos;
  size_t stride;
  T* pos_sorted;
  size_t sorted_stride;
  int4* quant;
  double qlo[3], qsp[3], qinv[3];  // cell origin, spacing, 2^28 / spacing
  uint32_t divc[3];
  uint32_t gm;
  uint32_t* n2s;
  uint32_t* dom;
  PlaneArgs pa;
  // ensembles: grid of each particle's system
  const SysGrid<T>* sys;
  const uint32_t* sid;
  uint32_t* sid_sorted;
  // the passes carried the positions into pos_sorted when *disorder says so, or they
  // have been placed there
  const unsigned long long* disorder;
  bool placed;
};

template <class T>
__device__ __forceinline__ void cl_emit(const EmitArgs<T>& A, uint32_t o, uint32_t f, uint32_t c,
                                        uint32_t dstart, uint32_t rank, bool pos_done) {
  if (A.n2s) A.n2s[o] = f;  // else by permute_far
  if (o < A.gm) A.dom[dstart + rank] = f;
  uint32_t s = 0;
  if (A.sys) {
    s = A.sid[o];
    A.sid_sorted[f] = s;
  }
  if (A.pos_sorted || A.quant) {
    T x, y, z;
    if (pos_done) {
      x = A.pos_sorted[f];
      y = A.pos_sorted[A.sorted_stride + f];
      z = A.pos_sorted[2 * A.sorted_stride + f];
    } else {
      x = A.pos[o];
      y = A.pos[A.stride + o];
      z = A.pos[2 * A.stride + o];
    }
    if (A.pos_sorted && !pos_done) {
      A.pos_sorted[f] = x;
      A.pos_sorted[A.sorted_stride + f] = y;
      A.pos_sorted[2 * A.sorted_stride + f] = z;
    }
    if (A.quant) {
      const double xs[3] = {double(x), double(y), double(z)};
      if (A.sys) {
        const SysGrid<T>& G = A.sys[s];
        const uint32_t cl = c - G.cbase;
        const uint32_t cc[3] = {cl % G.divc[0], (cl / G.divc[0]) % G.divc[1], cl / (G.divc[0] * G.divc[1])};
        A.quant[f] = quantise(xs, cc, G.qlo, G.qsp, G.qinv);
      } else {
        const uint32_t cc[3] = {c % A.divc[0], (c / A.divc[0]) % A.divc[1], c / (A.divc[0] * A.divc[1])};
        A.quant[f] = quantise(xs, cc, A.qlo, A.qsp, A.qinv);
      }
    }
  }
  copy_planes(A.pa, o, f);
}

template <class T>
__global__ __launch_bounds__(256) void k_cl_emit(EmitArgs<T> A, const uint32_t* __restrict__ keys,
                                                 const uint32_t* __restrict__ s2n, uint32_t n_host,
                                                 const uint32_t* __restrict__ n_dev,
                                                 const unsigned long long* __restrict__ cs,
                                                 const unsigned long long* __restrict__ check) {
  if (in_order(check)) return;
  const uint32_t f = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t n = count_of(n_host, n_dev);
  if (f >= n) return;
  const bool pos_done = A.placed || (A.pos_sorted && carry_positions(A.disorder, n));
  const uint32_t c = keys[f];
  const unsigned long long s0 = cs[c];
  cl_emit(A, s2n[f], f, c, uint32_t(s0 >> 32), f - uint32_t(s0), pos_done);
}

// The build of input already in cell order, speculatively, with the check of
// that order.  Per tile of 256 kIters particles: the cell keys and the descents
// k[f-1] > k[f] (the key before a wave's first slot recomputed from its
// position), added to *disorder.  A tile without descents writes what the
// build gives for its particles when the whole input is in cell order: the
// identity permutations, the positions and planes copied, the domain sort
// ids, the quantised stream, and its cells' (domain << 32 | count) into
// packed (cleared before).  If *disorder ends at zero these are the build's
// results; otherwise the radix passes (from the positions: neither keys nor
// histograms are kept here) and k_cl_emit overwrite every one of them.
template <class T, int kIters>
__global__ __launch_bounds__(kRxBlock) void k_cl_first(CellGeom<T> g, EmitArgs<T> A, uint32_t n,
                                                       uint32_t* __restrict__ s2n,
                                                       unsigned long long* __restrict__ disorder,
                                                       unsigned long long* __restrict__ packed, uint64_t n_cells) {
  constexpr uint32_t kRxTile = uint32_t(kRxBlock * kIters);
  __shared__ uint32_t wdesc[kRxWaves];
  const uint32_t t = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const uint64_t base = uint64_t(t) * kRxTile + uint64_t(w) * (kIters * kWave);
  const T* pos = A.pos;
  const size_t st = A.stride;
  uint32_t kk[kIters], kp[kIters];
  // keys, four rounds' loads at a time; the positions stay in registers for
  // the identity build below (read once from memory)
  T x[kIters], y[kIters], z[kIters];
#pragma unroll
  for (int b = 0; b < kIters; b += 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint64_t e = base + uint64_t(b + i) * kWave + uint64_t(lane);
      x[b + i] = y[b + i] = z[b + i] = T(0);
      if (e < n) {
        x[b + i] = pos[e];
        y[b + i] = pos[st + e];
        z[b + i] = pos[2 * st + e];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint64_t e = base + uint64_t(b + i) * kWave + uint64_t(lane);
      uint32_t cx, cy, cz;
      kk[b + i] = e < n ? cell_of(g, x[b + i], y[b + i], z[b + i], &cx, &cy, &cz) : 0u;
    }
  }
  // the key of the slot before the wave's first one
  uint32_t before = ~0u;
  if (base > 0 && base - 1 < n) {
    uint32_t cx, cy, cz;
    const uint64_t e = base - 1;
    before = cell_of(g, pos[e], pos[st + e], pos[2 * st + e], &cx, &cy, &cz);
  }
  uint32_t desc = 0;
#pragma unroll
  for (int r = 0; r < kIters; ++r) {
    const uint64_t e = base + uint64_t(r) * kWave + uint64_t(lane);
    const uint32_t up = __shfl_up(kk[r], 1, kWave);
    const uint32_t prev_last = r == 0 ? before : uint32_t(__builtin_amdgcn_readlane(int(kk[r - 1]), kWave - 1));
    kp[r] = lane == 0 ? prev_last : up;
    desc += (e < n && e > 0 && kp[r] > kk[r]) ? 1u : 0u;
  }
  desc = wave_sum(desc);
  if (lane == 0) wdesc[w] = desc;
  __syncthreads();
  uint32_t tile_desc = 0;
  for (int ww = 0; ww < kRxWaves; ++ww) tile_desc += wdesc[ww];
  if (threadIdx.x == 0 && tile_desc) atomicAdd(disorder, static_cast<unsigned long long>(tile_desc));
  if (tile_desc != 0) return;  // block-uniform
  // the identity build of this tile
  bool dm[kIters];
#pragma unroll
  for (int r = 0; r < kIters; ++r) {
    const uint64_t e = base + uint64_t(r) * kWave + uint64_t(lane);
    dm[r] = e < A.gm;
    if (e >= n) continue;
    const uint32_t f = uint32_t(e);
    s2n[f] = f;
    A.n2s[f] = f;
    if (f < A.gm) A.dom[f] = f;
    if (A.pos_sorted) {
      A.pos_sorted[f] = x[r];
      A.pos_sorted[A.sorted_stride + f] = y[r];
      A.pos_sorted[2 * A.sorted_stride + f] = z[r];
    }
    if (A.quant) {
      const uint32_t c = kk[r];
      const uint32_t cc[3] = {c % A.divc[0], (c / A.divc[0]) % A.divc[1], c / (A.divc[0] * A.divc[1])};
      const double xs[3] = {double(x[r]), double(y[r]), double(z[r])};
      A.quant[f] = quantise(xs, cc, A.qlo, A.qsp, A.qinv);
    }
    copy_planes(A.pa, f, f);
  }
  runs_of_wave<kIters>(kk, kp, dm, base, n, n_cells, packed);
}

// out[idx[j]] = in[j] for a permutation idx whose neighbours lie far apart, in two
// steps.  A plain scatter over a plane much larger than the L2 (4 MB per XCD) writes
// each value as a piece of a line of its own, 70e9 values/s.  Here the destinations
// are cut into ranges of 32768, each as large as a block's LDS:
//   k_far_stage  brings a tile of 32768 values into the order of their ranges in LDS
//                and appends them, with their places in the range, to the ranges'
//                parts of the scratch planes (2^25 values: runs of 32);
//   k_far_place  brings a range's values into order in LDS and writes them out.
// Each part is exactly as long as its range (idx is a permutation), so nothing is
// counted in advance; the order inside a part does not matter.  Bound by memory:
// each value is read and written twice, its place once.  A second step that
// scattered in the L2 instead (128 ranges, all blocks of a range on one XCD) took
// 200-230 us per 2^27 bytes, the L2's rate of partial stores.  Restore of 2^25
// particles from random order, 5 planes of 24 bytes: 2.40 -> 0.94 ms.
constexpr int kFarBlock = 1024;
constexpr int kFarIters = 32;
constexpr int kFarShift = 15;
constexpr uint32_t kFarTile = uint32_t(kFarBlock * kFarIters);
static_assert(kFarTile == 1u << kFarShift, "a range is a tile");
constexpr int kFarPer = 3;  // ranges a thread counts: the most the LDS holds beside a tile
constexpr uint32_t kFarRanges = kFarPer * kFarBlock;
constexpr size_t kFarFrom = size_t(1) << 22;  // restore of 24 bytes: 128 us at 2^21 (143 direct), 132 (265) here
constexpr size_t kFarTo = size_t(kFarRanges) << kFarShift;
constexpr size_t kFarScratch = 10;      // least scratch, bytes per particle
constexpr size_t kFarScratchFull = 26;  // six 4-byte planes at a time

// Barrier over the block's LDS only: loads and stores of global memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Two 16-bit values a register: 64 registers of a plane's values and a thread's
// slots and runs have to fit into the 128 that 1024 threads leave.
struct Halves {
  uint32_t w[kFarIters / 2] = {};
  __device__ __forceinline__ uint32_t get(int i) const { return i & 1 ? w[i / 2] >> 16 : w[i / 2] & 0xFFFFu; }
  __device__ __forceinline__ void put(int i, uint32_t v) {
    w[i / 2] = i & 1 ? (w[i / 2] & 0xFFFFu) | v << 16 : (w[i / 2] & 0xFFFF0000u) | v;
  }
  // opaque to the compiler, which would keep the 32 unpacked values across planes
  __device__ __forceinline__ void hide() {
#pragma unroll
    for (int i = 0; i < kFarIters / 2; ++i) asm volatile("" : "+v"(w[i]));
  }
};

// The planes of pa one after another through st: slot.get(i) is the place that value
// i of the thread takes in st, to(i, l) the index that place l of st goes to.  Of a
// last tile of len < kFarTile values the loads past the end read its last value,
// which takes the place past the end that no value has.
// 8-byte values pass in halves (32768 of them fill twice the LDS).
template <class To>
__device__ __forceinline__ void far_planes(const PlaneArgs& pa, uint32_t e0, uint32_t len, uint32_t (&st)[kFarTile],
                                           Halves& slot, To&& to) {
  uint32_t tid = threadIdx.x;
  auto each = [&](auto&& f) {
#pragma unroll
    for (int i = 0; i < kFarIters; ++i) f(i, uint32_t(i) * kFarBlock + tid);
  };
  const uint32_t last = len - 1;
  auto at = [&](uint32_t l) { return l < last ? l : last; };
  for (int k = 0; k < pa.n; ++k) {
    const uint64_t src = pa.src[k], dst = pa.dst[k];
    slot.hide();
    asm volatile("" : "+v"(tid));
    uint32_t v[kFarIters];
    if (pa.esz[k] == 4) {
      const uint32_t* in = reinterpret_cast<const uint32_t*>(src) + e0;
      each([&](int i, uint32_t l) { v[i] = src ? in[at(l)] : e0 + l; });
      lds_barrier();  // st has been read
      each([&](int i, uint32_t) { st[slot.get(i)] = v[i]; });
      lds_barrier();
      each([&](int i, uint32_t l) {
        if (l < len) reinterpret_cast<uint32_t*>(dst)[to(i, l)] = st[l];
      });
    } else {
      const uint2* in = reinterpret_cast<const uint2*>(src) + e0;
      uint32_t hi[kFarIters];
      each([&](int i, uint32_t l) {
        const uint2 w = in[at(l)];
        v[i] = w.x;
        hi[i] = w.y;
      });
      lds_barrier();
      each([&](int i, uint32_t) { st[slot.get(i)] = v[i]; });
      lds_barrier();
      each([&](int i, uint32_t l) { v[i] = st[l]; });
      lds_barrier();
      slot.hide();
      each([&](int i, uint32_t) { st[slot.get(i)] = hi[i]; });
      lds_barrier();
      asm volatile("" : "+v"(tid));
      each([&](int i, uint32_t l) {
        if (l < len) reinterpret_cast<uint2*>(dst)[to(i, l)] = uint2{v[i], st[l]};
      });
    }
  }
}

// pa: planes to stage (src 0: the values are the indexes j); dst: scratch planes.
__global__ __launch_bounds__(kFarBlock) void k_far_stage(const uint32_t* __restrict__ idx, uint32_t n,
                                                         uint32_t* __restrict__ cursor, PlaneArgs pa,
                                                         uint16_t* __restrict__ place) {
  __shared__ uint32_t st[kFarTile];
  __shared__ uint32_t cnt[kFarRanges];   // counts, then the first slots of the runs
  __shared__ uint32_t goff[kFarRanges];  // where slot 0 of the tile would go, by run
  __shared__ uint32_t wsum[kFarBlock / kWave];
  const uint32_t tid = threadIdx.x;
  const uint32_t tile0 = blockIdx.x << kFarShift;
  const uint32_t len = n - tile0 < kFarTile ? n - tile0 : kFarTile;
#pragma unroll
  for (int q = 0; q < kFarPer; ++q) cnt[tid + q * kFarBlock] = 0;
  uint32_t d[kFarIters];
  Halves slot;
#pragma unroll
  for (int i = 0; i < kFarIters; ++i) {
    const uint32_t l = uint32_t(i) * kFarBlock + tid;
    d[i] = idx[tile0 + (l < len ? l : len - 1)];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kFarIters; ++i)
    slot.put(i, uint32_t(i) * kFarBlock + tid < len ? atomicAdd(&cnt[d[i] >> kFarShift], 1u) : 0u);
  __syncthreads();
  // first slots of the tile's runs, in the tile and in the ranges' parts: consecutive
  // ranges a thread
  uint32_t c[kFarPer], g[kFarPer], own = 0;
#pragma unroll
  for (int q = 0; q < kFarPer; ++q) {
    const uint32_t r = kFarPer * tid + q;
    c[q] = cnt[r];
    own += c[q];
    g[q] = (r << kFarShift) + (c[q] ? atomicAdd(&cursor[r], c[q]) : 0u);
  }
  const uint32_t inc = wave_incl_scan(own);
  if ((tid & (kWave - 1)) == kWave - 1) wsum[tid / kWave] = inc;
  __syncthreads();
  uint32_t first = inc - own;
  for (uint32_t w = 0; w < tid / kWave; ++w) first += wsum[w];
#pragma unroll
  for (int q = 0; q < kFarPer; ++q) {
    cnt[kFarPer * tid + q] = first;
    goff[kFarPer * tid + q] = g[q] - first;
    first += c[q];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kFarIters; ++i) {
    const uint32_t l = uint32_t(i) * kFarBlock + tid;
    const uint32_t t = l < len ? slot.get(i) + cnt[d[i] >> kFarShift] : l;
    slot.put(i, t);
    st[t] = d[i];
  }
  __syncthreads();
  Halves run;
#pragma unroll
  for (int i = 0; i < kFarIters; ++i) {
    const uint32_t l = uint32_t(i) * kFarBlock + tid;
    const uint32_t v = st[l];
    run.put(i, v >> kFarShift);
    if (l < len) place[goff[v >> kFarShift] + l] = uint16_t(v & (kFarTile - 1));
  }
  auto to = [&](int i, uint32_t l) {
    if (i == 0) run.hide();
    return goff[run.get(i)] + l;
  };
  far_planes(pa, tile0, len, st, slot, to);
}

// pa: scratch planes (src) of values staged by range, brought into order to dst.
__global__ __launch_bounds__(kFarBlock) void k_far_place(const uint16_t* __restrict__ place, uint32_t n,
                                                         PlaneArgs pa) {
  __shared__ uint32_t st[kFarTile];
  const uint32_t e0 = blockIdx.x << kFarShift;
  const uint32_t len = n - e0 < kFarTile ? n - e0 : kFarTile;
  Halves d;
#pragma unroll
  for (int i = 0; i < kFarIters; ++i) {
    const uint32_t l = uint32_t(i) * kFarBlock + threadIdx.x;
    const uint32_t p = place[e0 + (l < len ? l : len - 1)];
    d.put(i, l < len ? p : l);
  }
  auto to = [&](int, uint32_t l) { return e0 + l; };
  far_planes(pa, e0, len, st, d, to);
}

// out[idx[j]] = in[j], j < n, for every plane (pa.src 0: in[j] = j), through
// `scratch` (bytes >= kFarScratch (n + 8)); cursors: kFarRanges words.
static int permute_far(const uint32_t* idx, uint32_t n, const PlaneArgs& pa, void* scratch, size_t bytes,
                       uint32_t* cursors, hipStream_t s) {
  const unsigned tiles = unsigned((uint64_t(n) + kFarTile - 1) >> kFarShift);
  const size_t step = (size_t(n) + 7) & ~size_t(7);  // values per scratch plane
  for (int k = 0; k < pa.n;) {
    PlaneArgs in{}, out{};
    size_t used = step * 2;
    for (; k < pa.n && (in.n == 0 || used + step * pa.esz[k] <= bytes); ++k) {
      const int m = in.n;
      in.src[m] = pa.src[k];
      in.dst[m] = out.src[m] = reinterpret_cast<uint64_t>(static_cast<char*>(scratch) + used);
      out.dst[m] = pa.dst[k];
      in.esz[m] = out.esz[m] = pa.esz[k];
      in.n = out.n = m + 1;
      used += step * pa.esz[k];
    }
    OFP_TRY(fill_u32(cursors, 0, kFarRanges, s));
    k_far_stage<<<tiles, kFarBlock, 0, s>>>(idx, n, cursors, in, static_cast<uint16_t*>(scratch));
    OFP_LAUNCHED();
    k_far_place<<<tiles, kFarBlock, 0, s>>>(static_cast<const uint16_t*>(scratch), n, out);
    OFP_LAUNCHED();
  }
  return OFP_OK;
}

// out[j] = in[s2n[j]] (gather into sorted order)
__global__ __launch_bounds__(256) void k_cl_reorder(uint32_t n, const uint32_t* __restrict__ s2n,
                                                    PlaneArgs pa) {
  uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  copy_planes(pa, s2n[j], j);
}

// out[s2n[j]] = in[j] (scatter back to the original order)
__global__ __launch_bounds__(256) void k_cl_restore(uint32_t n, const uint32_t* __restrict__ s2n,
                                                    PlaneArgs pa) {
  uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  copy_planes(pa, j, s2n[j]);
}

// permute_far with the list's scratch (which is there).
static int go_far(ofp_cl* h, const uint32_t* idx, uint32_t n, const PlaneArgs& pa, hipStream_t s) {
  if (pa.n == 0) return OFP_OK;
  std::lock_guard<std::mutex> lock(h->far_lock);
  if (h->far_done)
    OFP_HIP(hipStreamWaitEvent(s, h->far_done, 0));
  else
    OFP_HIP(hipEventCreateWithFlags(&h->far_done, hipEventDisableTiming));
  OFP_TRY(permute_far(idx, n, pa, h->payload.p, h->payload.cap, h->cursors.as<uint32_t>(), s));
  OFP_HIP(hipEventRecord(h->far_done, s));
  return OFP_OK;
}

// A reorder or restore (out[idx[j]] = in[j]) by ranges, where the list's particles
// are many and far from cell order; *done: it is.  A captured call takes the direct
// kernel: the graph may be replayed beside other calls that use the scratch.
static int permute_route(const ofp_cl* h, const uint32_t* idx, const PlaneArgs& pa, hipStream_t s, bool* done) {
  *done = false;
  if (!h->far) return OFP_OK;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  OFP_HIP(hipStreamIsCapturing(s, &cap));
  if (cap != hipStreamCaptureStatusNone) return OFP_OK;
  OFP_TRY(go_far(const_cast<ofp_cl*>(h), idx, uint32_t(h->n_part), pa, s));  // its scratch only
  *done = true;
  return OFP_OK;
}

// p[0 .. n) = 0 unless the order check found the input in cell order.
__global__ __launch_bounds__(256) void k_clear_unless(unsigned long long* __restrict__ p, uint64_t n,
                                                      const unsigned long long* __restrict__ check) {
  if (in_order(check)) return;
  for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += uint64_t(gridDim.x) * 256) p[i] = 0ull;
}

// Digit widths of the radix passes for keys < n_cells: as few passes of at most
// 8 bits as cover the key, widths as even as possible.
static int radix_plan(uint64_t n_cells, int* widths) {
  int bits = 1;
  while (bits < 32 && (uint64_t(1) << bits) < n_cells) ++bits;
  const int passes = (bits + kRxMaxBits - 1) / kRxMaxBits;
  for (int p = 0; p < passes; ++p) widths[p] = bits / passes + (p < bits % passes ? 1 : 0);
  return passes;
}

// n_cap: particles the buffers hold (the count itself is n_host or *n_dev).
// g1 (one grid, count on the host): k_cl_first first checks the input's order
// while writing the build of ordered input; for input already in cell order the
// build ends with the scan of the cell counts it wrote, otherwise the radix build
// follows (see kRxNoSync for how the two are told apart).
// Ensembles (g1 null) keep every step on the device (their rebuilds are
// captured in graphs).
template <class T, int kIters, class Key>
static int cl_build_t(ofp_cl* h, const Key& key, const EmitArgs<T>& A0, size_t n_cap, uint32_t n_host,
                      const uint32_t* n_dev, size_t gm, hipStream_t s, const CellGeom<T>* g1) {
  constexpr uint32_t kRxTile = uint32_t(kRxBlock * kIters);
  const uint64_t C = h->n_cells;
  const uint32_t n_tiles = uint32_t((n_cap + kRxTile - 1) / kRxTile);
  const size_t hist_n = size_t(kRxBins) * (n_tiles ? n_tiles : 1);
  const bool first = g1 != nullptr && n_dev == nullptr;
  if (first && n_tiles > 0) {  // a build of a count on the host is none for a graph: the count and the buffers are this call's
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    OFP_HIP(hipStreamIsCapturing(s, &cap));
    if (cap != hipStreamCaptureStatusNone) OFP_HIP(hipErrorStreamCaptureUnsupported);
  }
  int widths[4];
  const int passes = radix_plan(C, widths);
  // behind the cells' counts, and cleared with them: the descents counted, the items'
  // queue heads and their count (captured pair passes name these: their place must not
  // depend on the particles, nor the buffer grow with them), the chunks' sums
  const int direct = n_tiles <= kRxChunked ? 1 : 0;
  const bool chunked = direct && n_tiles > kRxDirect;
  // the [tile][digit] table in at most kColChunks chunks of ch tiles
  const uint32_t ch = std::max((n_tiles + kColChunks - 1) / kColChunks, kColBatch);
  const uint32_t n_chunks = (n_tiles + ch - 1) / ch;
  const uint64_t sums_at = C + 1 + kQueueWords / 2 + 1;
  const uint64_t n_clear = sums_at + (chunked ? uint64_t(passes) * n_chunks * (kRxBins / 2) : 0);
  OFP_TRY(h->packed.ensure((sums_at + uint64_t(passes) * kColChunks * (kRxBins / 2)) * 8));
  OFP_TRY(h->scan64.ensure((C + 1) * 8));
  OFP_TRY(h->scantmp.ensure(scan_tmp_bytes(C)));
  if (!direct) OFP_TRY(h->colpart.ensure(size_t(kColChunks) * kRxBins * 4));
  OFP_TRY(h->keys.ensure((n_cap + 1) * 4));
  OFP_TRY(h->keys2.ensure((n_cap + 1) * 4));
  OFP_TRY(h->s2n.ensure((n_cap + 1) * 4));
  OFP_TRY(h->vals2.ensure((n_cap + 1) * 4));
  OFP_TRY(h->n2s.ensure((n_cap + 1) * 4));
  OFP_TRY(h->dom.ensure((gm + 1) * 4));
  OFP_TRY(h->hist.ensure((hist_n + 1) * 4));
  const bool want_quant = (h->opt & OFP_CL_QUANT) != 0;
  if (want_quant) OFP_TRY(h->quant.ensure((n_cap + 1) * 16));
  if (h->n_sys) OFP_TRY(h->sid_sorted.ensure((n_cap + 1) * 4));

  // With sorted positions requested they may travel with the keys as a payload
  // (the passes before the last alternate between two payload buffers, the last
  // one writes the sorted positions); the kernels carry them only when the
  // descents say the input is far from cell order (carry_positions), else
  // k_cl_emit gathers them.  Few particles' positions stay in the caches and are
  // gathered in any order (300,000 random ones: build 91 -> 82 us, 2^20: 205 -> 192);
  // many are placed by permute_far (build of 2^25: 2.37 -> 1.92 ms).
  const bool payload = A0.pos_sorted != nullptr && n_cap > kRxSmall &&
                       !(first && n_cap >= kFarFrom && n_cap <= kFarTo);
  if (payload && passes > 1) OFP_TRY(h->payload.ensure(2 * 3 * n_cap * sizeof(T)));
  T* pbuf[2] = {h->payload.as<T>(), h->payload.as<T>() + 3 * n_cap};
  // ping-pong buffers chosen so that the last pass lands in keys / s2n
  uint32_t* kbuf[2] = {h->keys.as<uint32_t>(), h->keys2.as<uint32_t>()};
  uint32_t* vbuf[2] = {h->s2n.as<uint32_t>(), h->vals2.as<uint32_t>()};
  uint32_t* hist = h->hist.as<uint32_t>();
  auto* packed = h->packed.as<unsigned long long>();
  auto* disorder = packed + C;
  auto* cs = h->scan64.as<unsigned long long>();
  auto emit_args = [&]() {
    EmitArgs<T> A = A0;
    A.quant = want_quant ? h->quant.as<int4>() : nullptr;
    A.gm = uint32_t(gm);
    A.n2s = h->n2s.as<uint32_t>();
    A.dom = h->dom.as<uint32_t>();
    A.sid_sorted = h->n_sys ? h->sid_sorted.as<uint32_t>() : nullptr;
    A.disorder = payload ? disorder : nullptr;
    return A;
  };
  auto scan_and_finish = [&]() -> int {
    OFP_TRY(scan_excl_u64(reinterpret_cast<const uint64_t*>(packed), reinterpret_cast<uint64_t*>(cs), C,
                          h->scantmp.p, s));
    h->n_part = n_dev ? n_cap : n_host;
    h->gm = gm;
    h->n_dev = n_dev;
    h->built = true;
    h->sparse_valid = false;
    h->items_valid = false;
    return OFP_OK;
  };
  h->far = false;
  OFP_TRY(fill_u64(reinterpret_cast<uint64_t*>(packed), 0, n_clear, s));
  if (n_tiles == 0) return scan_and_finish();
  const unsigned long long* check = nullptr;  // the kernels below return if *check == 0
  if (first) {
    k_cl_first<T, kIters><<<n_tiles, kRxBlock, 0, s>>>(*g1, emit_args(), n_host, vbuf[0], disorder, packed, C);
    OFP_LAUNCHED();
    if (n_cap >= kFarFrom) {
      // the descents to the host, for the emission's route: read there while the passes run
      if (!h->desc) OFP_HIP(hipHostMalloc(reinterpret_cast<void**>(&h->desc), sizeof(*h->desc)));
      if (!h->checked) OFP_HIP(hipEventCreateWithFlags(&h->checked, hipEventDisableTiming));
      OFP_HIP(hipMemcpyAsync(h->desc, disorder, sizeof(*h->desc), hipMemcpyDeviceToHost, s));
      OFP_HIP(hipEventRecord(h->checked, s));
    }
    static_assert(kFarFrom <= kRxNoSync, "a build that waits has the descents");
    if (n_cap < kRxNoSync) {
      check = disorder;
    } else {
      OFP_HIP(hipEventSynchronize(h->checked));
      if (*h->desc == 0) return scan_and_finish();  // every tile wrote its identity build
    }
  }
  uint32_t* kin = kbuf[passes % 2];  // pass-0 keys
  const uint32_t* vin = nullptr;
  const T* pin = payload ? A0.pos : nullptr;
  size_t si = A0.stride;
  int shift = 0;
  // pass 0 clears the counts that the order check's tiles wrote; many more cells
  // than particles are left to a launch of their own
  const bool clear_in_hist = first && C <= 16 * n_cap;
  if (first && !clear_in_hist) {
    k_clear_unless<<<2048, 256, 0, s>>>(packed, C, check);
    OFP_LAUNCHED();
  }
  for (int p = 0; p < passes; ++p) {
    const int bits = widths[p];
    uint32_t* kout = kbuf[(passes - 1 - p) % 2];
    uint32_t* vout = vbuf[(passes - 1 - p) % 2];
    T* pout = nullptr;
    size_t so = 0;
    if (payload) {
      const bool last = p == passes - 1;
      pout = last ? A0.pos_sorted : pbuf[p % 2];
      so = last ? A0.sorted_stride : n_cap;
    }
    uint32_t* part = chunked ? reinterpret_cast<uint32_t*>(packed + sums_at) + size_t(p) * n_chunks * kRxBins
                             : h->colpart.as<uint32_t>();
    k_rx_hist<Key, kIters><<<n_tiles, kRxBlock, 0, s>>>(
        key, p ? kin : nullptr, p ? nullptr : kin, n_host, n_dev, shift, bits, n_tiles, hist,
        p || first ? nullptr : disorder, check, p == 0 && clear_in_hist ? packed : nullptr, C,
        chunked ? part : nullptr, ch);
    OFP_LAUNCHED();
    if (!direct) {
      k_rx_colsum<<<n_chunks, kRxBins, 0, s>>>(hist, n_tiles, ch, 1 << bits, part, check);
      OFP_LAUNCHED();
      k_rx_colapply<<<n_chunks, kColGroups * kRxBins, 0, s>>>(hist, n_tiles, ch, 1 << bits, n_chunks, part, check);
      OFP_LAUNCHED();
    }
    k_rx_scatter<T, kIters><<<n_tiles, kRxBlock, 0, s>>>(kin, vin, n_host, n_dev, shift, bits, n_tiles, hist, kout,
                                                         vout, pin, si, pout, so, disorder, check, direct,
                                                         chunked ? part : nullptr, ch, n_chunks);
    OFP_LAUNCHED();
    kin = kout;
    vin = vout;
    pin = pout;
    si = so;
    shift += bits;
  }
  k_cl_runs<kIters><<<grid_for(n_cap, 256 * kIters), 256, 0, s>>>(h->keys.as<uint32_t>(), h->s2n.as<uint32_t>(),
                                                                  n_host, n_dev, uint32_t(gm), C, packed, check);
  OFP_LAUNCHED();
  OFP_TRY(scan_and_finish());
  EmitArgs<T> A = emit_args();
  if (first && n_cap >= kFarFrom && n_cap <= kFarTo) {
    OFP_HIP(hipEventSynchronize(h->checked));
    if (*h->desc * kDisorderDen > n_cap) {
      // scratch for five or six floats at a time, or for what there is memory
      h->far = h->cursors.ensure(kFarRanges * 4) == OFP_OK &&
               (h->payload.ensure(kFarScratchFull * (n_cap + 8)) == OFP_OK ||
                h->payload.ensure(kFarScratch * (n_cap + 8)) == OFP_OK);
      clear_error();  // without it, if there is none
    }
  }
  if (h->far) {
    PlaneArgs index{};  // n2s[s2n[f]] = f
    index.n = 1;
    index.esz[0] = 4;
    index.dst[0] = reinterpret_cast<uint64_t>(h->n2s.p);
    OFP_TRY(go_far(h, h->s2n.as<uint32_t>(), n_host, index, s));
    PlaneArgs planes = A0.pa;
    if (A0.pos_sorted) {
      PlaneArgs pos{};
      for (int k = 0; k < 3; ++k) {
        pos.src[k] = reinterpret_cast<uint64_t>(A0.pos + size_t(k) * A0.stride);
        pos.dst[k] = reinterpret_cast<uint64_t>(A0.pos_sorted + size_t(k) * A0.sorted_stride);
        pos.esz[k] = uint32_t(sizeof(T));
      }
      pos.n = 3;
      for (int k = 0; k < planes.n && pos.n < kMaxPlanes; ++k, ++pos.n) {
        pos.src[pos.n] = planes.src[k];
        pos.dst[pos.n] = planes.dst[k];
        pos.esz[pos.n] = planes.esz[k];
      }
      OFP_TRY(go_far(h, h->n2s.as<uint32_t>(), n_host, pos, s));
      const int done = pos.n - 3;
      planes.n -= done;
      for (int k = 0; k < planes.n; ++k) {
        planes.src[k] = planes.src[k + done];
        planes.dst[k] = planes.dst[k + done];
        planes.esz[k] = planes.esz[k + done];
      }
      A.placed = true;
    }
    OFP_TRY(go_far(h, h->n2s.as<uint32_t>(), n_host, planes, s));
    A.n2s = nullptr;
    A.pa.n = 0;
  }
  k_cl_emit<T><<<grid_for(n_cap, 256), 256, 0, s>>>(A, h->keys.as<uint32_t>(), h->s2n.as<uint32_t>(), n_host, n_dev,
                                                     cs, check);
  OFP_LAUNCHED();
  return OFP_OK;
}

template <class T, class Key>
static int cl_build(ofp_cl* h, const Key& key, const EmitArgs<T>& A0, size_t n_cap, uint32_t n_host,
                    const uint32_t* n_dev, size_t gm, hipStream_t s, const CellGeom<T>* g1 = nullptr) {
  if (n_cap < kRxSmall) return cl_build_t<T, kRxShort>(h, key, A0, n_cap, n_host, n_dev, gm, s, g1);
  return cl_build_t<T, kRxLong>(h, key, A0, n_cap, n_host, n_dev, gm, s, g1);
}

template <class T>
static int cl_construct(ofp_cl* h, const CellGeom<T>& g, const void* pos_v, size_t stride,
                        size_t n_tot, size_t gm, void* pos_sorted_v, size_t sorted_stride,
                        const PlaneArgs& pa, hipStream_t s) {
  const T* pos = static_cast<const T*>(pos_v);
  EmitArgs<T> A;
  std::memset(&A, 0, sizeof(A));
  A.pos = pos;
  A.stride = stride;
  A.pos_sorted = static_cast<T*>(pos_sorted_v);
  A.sorted_stride = sorted_stride;
  for (int k = 0; k < 3; ++k) {
    A.qlo[k] = double(g.lo[k]);
    A.qsp[k] = double(g.sp[k]);
    A.qinv[k] = double(kQuantOne) / double(g.sp[k]);
    A.divc[k] = g.divc[k];
  }
  A.pa = pa;
  KeyOne<T> key{g, pos, stride};
  return cl_build<T>(h, key, A, n_tot, uint32_t(n_tot), nullptr, gm, s, &g);
}

template <class T>
static int cl_construct_many_t(ofp_cl* h, const void* pos_v, size_t stride, size_t n_cap, const uint32_t* n_dev,
                             size_t gm, void* pos_sorted_v, size_t sorted_stride, hipStream_t s) {
  const T* pos = static_cast<const T*>(pos_v);
  EmitArgs<T> A;
  std::memset(&A, 0, sizeof(A));
  A.pos = pos;
  A.stride = stride;
  A.pos_sorted = static_cast<T*>(pos_sorted_v);
  A.sorted_stride = sorted_stride;
  A.sys = static_cast<const SysGrid<T>*>(h->sys);
  A.sid = h->sid;
  KeyMany<T> key{A.sys, h->sid, pos, stride};
  return cl_build<T>(h, key, A, n_cap, uint32_t(n_cap), n_dev, gm, s);
}

// Target items of the Verlet build and the cell tiles.  A row of cells is cut into
// blocks of kItemBlock cells, and a block's domain particles (consecutive domain
// rows) into items of up to kItemTargets that span at most kItemMaxCells cells,
// those of its first to its last particle.  Every domain particle is in exactly
// one item.  In an ensemble the rows of all grids are numbered consecutively and the item
// carries its system in ncx >> 8.
// One wave per row, a lane per block; kItemRows rows take their place in the
// queue with one atomic.  A thread per row that grouped whole cells one after
// another and drew a place per item spent 335 us on 13,700 rows of 117 cells and
// 1.2e5 items (clustered, 4.2e6 particles), this 42 us; whole cells left an item
// short of 64 targets by half a cell on average, blocks by half an item in 16 cells.
constexpr uint32_t kItemTargets = 64;
constexpr int kItemRows = 16;
constexpr uint32_t kItemBlock = 16;

__global__ __launch_bounds__(kItemRows* kWave) void k_cl_items(const unsigned long long* __restrict__ cs,
                                                               uint32_t divc0_one, uint32_t nrows, uint32_t n_sys,
                                                               const uint32_t* __restrict__ rbase,
                                                               const uint32_t* __restrict__ sysdesc,
                                                               uint32_t sys_words, TargetItem* __restrict__ items,
                                                               uint32_t* __restrict__ nitems) {
  __shared__ uint32_t cnt[kItemRows];
  __shared__ uint32_t place;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t r = blockIdx.x * uint32_t(kItemRows) + w;
  uint32_t base = 0, divc0 = 0, tag = 0;  // a row past the last: no cells
  if (r < nrows) {
    base = r * divc0_one;
    divc0 = divc0_one;
    if (n_sys) {
      // system of row r: last s with rbase[s] <= r
      uint32_t lo = 0, hi = n_sys;
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (rbase[mid] <= r)
          lo = mid;
        else
          hi = mid;
      }
      const uint32_t* G = sysdesc + size_t(lo) * sys_words;  // divc[3], cbase at word offset 0..3
      divc0 = G[0];
      base = G[3] + (r - rbase[lo]) * divc0;
      tag = lo << 8;
    }
  }
  // the lane's block of cells [c, c + kItemBlock): first domain row of each, and
  // the block's items one after another
  uint32_t d[kItemBlock + 1];
  auto load = [&](uint32_t c) {
#pragma unroll
    for (uint32_t i = 0; i <= kItemBlock; ++i) {
      const uint32_t ci = c + i < divc0 ? c + i : divc0;
      d[i] = c < divc0 ? uint32_t(cs[base + ci] >> 32) : 0u;
    }
  };
  auto items_of = [&](auto&& emit) -> uint32_t {
    uint32_t n = 0;
    for (uint32_t row = d[0]; row < d[kItemBlock]; ++n) {
      // the cell of a row: the first whose end lies past it
      uint32_t ca = 0, cb = 0, end = 0;
#pragma unroll
      for (uint32_t q = 1; q < kItemBlock; ++q) ca += d[q] <= row ? 1u : 0u;
#pragma unroll
      for (uint32_t q = 1; q <= kItemBlock; ++q) end = q <= ca + kItemMaxCells ? d[q] : end;
      const uint32_t m = min(kItemTargets, end - row);
#pragma unroll
      for (uint32_t q = 1; q < kItemBlock; ++q) cb += d[q] <= row + m - 1 ? 1u : 0u;
      emit(n, row, m, ca, cb);
      row += m;
    }
    return n;
  };
  constexpr uint32_t kSpan = kWave * kItemBlock;  // cells per round
  uint32_t k = 0;  // the row's items
  for (uint32_t c0 = 0; c0 < divc0; c0 += kSpan) {
    load(c0 + lane * kItemBlock);
    k += wave_sum(items_of([](uint32_t, uint32_t, uint32_t, uint32_t, uint32_t) {}));
  }
  if (lane == 0) cnt[w] = k;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t all = 0;
    for (int i = 0; i < kItemRows; ++i) {
      const uint32_t c = cnt[i];
      cnt[i] = all;
      all += c;
    }
    place = all ? atomicAdd(nitems, all) : 0u;
  }
  __syncthreads();
  uint32_t at = place + cnt[w];
  for (uint32_t c0 = 0; c0 < divc0; c0 += kSpan) {
    const uint32_t c = c0 + lane * kItemBlock;
    load(c);
    const uint32_t n = items_of([](uint32_t, uint32_t, uint32_t, uint32_t, uint32_t) {});
    const uint32_t inc = wave_incl_scan(n);
    items_of([&](uint32_t i, uint32_t row, uint32_t m, uint32_t ca, uint32_t cb) {
      items[at + inc - n + i] = TargetItem{row, m, base + c + ca, (cb - ca + 1u) | tag};
    });
    at += __builtin_amdgcn_readlane(inc, kWave - 1);
  }
}

// Sparse view: flag[c] = 1 for a non-empty cell (cell_start is the packed
// scan: low 32 bits = first sorted index).
__global__ void k_nz_flag(const uint64_t* __restrict__ cs, uint64_t n_cells, uint32_t* __restrict__ flag) {
  const uint64_t c = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (c < n_cells) flag[c] = uint32_t(cs[c + 1]) > uint32_t(cs[c]) ? 1u : 0u;
}

// pos = exclusive scan of the flags: the non-empty cell c is entry pos[c];
// inv[c] = that entry or -1.  The entry after the last holds the particle total.
__global__ void k_nz_scatter(const uint64_t* __restrict__ cs, uint64_t n_cells, const uint32_t* __restrict__ pos,
                             uint32_t* __restrict__ key, uint32_t* __restrict__ start, int32_t* __restrict__ inv) {
  const uint64_t c = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (c > n_cells) return;
  if (c == n_cells) {
    start[pos[n_cells]] = uint32_t(cs[n_cells]);
    return;
  }
  const bool nz = uint32_t(cs[c + 1]) > uint32_t(cs[c]);
  inv[c] = nz ? int32_t(pos[c]) : -1;
  if (nz) {
    key[pos[c]] = uint32_t(c);
    start[pos[c]] = uint32_t(cs[c]);
  }
}

// The (2B + 1)^3 neighbour cells of each non-empty cell, B = the list's box_nn
// (offsets dz, dy, dx in -B..B, x fastest), as entries of the sparse view, -1
// where empty or off the grid.  One thread per (cell, offset).
__global__ void k_nz_nn(const uint32_t* __restrict__ key, uint64_t n_nz, uint32_t d0, uint32_t d1, uint32_t d2,
                        int B, const int32_t* __restrict__ inv, int32_t* __restrict__ nn) {
  const int W = 2 * B + 1, K = W * W * W;
  const uint64_t t = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n_nz * uint64_t(K)) return;
  const uint64_t m = t / uint64_t(K);
  const int k = int(t - m * uint64_t(K));
  const int dx = k % W - B, dy = (k / W) % W - B, dz = k / (W * W) - B;
  const uint32_t c = key[m];
  const int x = int(c % d0) + dx, y = int((c / d0) % d1) + dy, z = int(c / (uint64_t(d0) * d1)) + dz;
  const bool in = x >= 0 && y >= 0 && z >= 0 && x < int(d0) && y < int(d1) && z < int(d2);
  nn[t] = in ? inv[uint64_t(x) + uint64_t(d0) * (uint64_t(y) + uint64_t(d1) * uint64_t(z))] : -1;
}

}  // namespace ofp

using namespace ofp;

// ------------------------------------------------------- ensemble internals
int ofp::cl_create_many(ofp_cl** out, int dtype, uint32_t n_sys, const void* sys_dev, const uint32_t* rbase_dev,
                        uint32_t n_rows, uint64_t n_cells, uint32_t opt) {
  OFP_CHECK(out && sys_dev && rbase_dev && n_sys > 0, OFP_E_ARG, "cl_create_many: null argument");
  OFP_CHECK(n_cells < (1ull << 31), OFP_E_LIMIT, "too many cells (%llu)", (unsigned long long)n_cells);
  ofp_cl* h = new ofp_cl();
  h->dtype = dtype;
  h->opt = opt;
  h->n_cells = n_cells;
  h->n_sys = n_sys;
  h->sys = sys_dev;
  h->rbase = rbase_dev;
  h->n_rows = n_rows;
  *out = h;
  return OFP_OK;
}

int ofp::cl_construct_many(ofp_cl* h, const void* pos, size_t stride, const uint32_t* sid, size_t n_cap,
                           const uint32_t* n_dev, size_t gm, void* pos_sorted, size_t sorted_stride,
                           hipStream_t s) {
  OFP_CHECK(h && h->n_sys, OFP_E_ARG, "cl_construct_many: not an ensemble cell list");
  OFP_CHECK(n_cap < 0xFFFFFFF0ull, OFP_E_LIMIT, "particle capacity must fit 32 bits");
  h->sid = sid;
  if (h->dtype == OFP_F32)
    return ofp::cl_construct_many_t<float>(h, pos, stride, n_cap, n_dev, gm, pos_sorted, sorted_stride, s);
  return ofp::cl_construct_many_t<double>(h, pos, stride, n_cap, n_dev, gm, pos_sorted, sorted_stride, s);
}

int ofp::cl_far(const ofp_cl* hc, size_t n, bool* far, hipStream_t s) {
  *far = false;
  ofp_cl* h = const_cast<ofp_cl*>(hc);  // its scratch only
  if (!h->built || n < kFarFrom || n > kFarTo || h->payload.cap < kFarScratch * (n + 8)) return OFP_OK;
  if (h->cursors.ensure(kFarRanges * 4) != OFP_OK) {
    clear_error();
    return OFP_OK;
  }
  unsigned long long desc = 0;
  OFP_HIP(hipMemcpyAsync(&desc, h->packed.as<unsigned long long>() + h->n_cells, sizeof(desc), hipMemcpyDeviceToHost,
                         s));
  OFP_HIP(hipStreamSynchronize(s));
  *far = desc * kDisorderDen > n;
  return OFP_OK;
}

int ofp::cl_permute(const ofp_cl* hc, const uint32_t* idx, size_t n, const PlaneArgs& pa, bool* done,
                    hipStream_t s) {
  *done = false;
  ofp_cl* h = const_cast<ofp_cl*>(hc);  // its scratch only
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  OFP_HIP(hipStreamIsCapturing(s, &cap));
  if (cap != hipStreamCaptureStatusNone || n > kFarTo || h->payload.cap < kFarScratch * (n + 8) || !h->cursors.p)
    return OFP_OK;
  OFP_TRY(go_far(h, idx, uint32_t(n), pa, s));
  *done = true;
  return OFP_OK;
}

int ofp::cl_sid_sorted(const ofp_cl* h, const uint32_t** sid_sorted) {
  OFP_CHECK(h && h->built && h->n_sys, OFP_E_STATE, "ensemble cell list not constructed");
  *sid_sorted = h->sid_sorted.as<uint32_t>();
  return OFP_OK;
}

extern "C" {

int ofp_cl_create(ofp_cl** out, int dtype, const void* box_lo, const void* box_hi,
                  const uint32_t* div, uint32_t opt) {
  OFP_CHECK(out && box_lo && box_hi && div, OFP_E_ARG, "ofp_cl_create: null argument");
  OFP_CHECK(dtype == OFP_F32 || dtype == OFP_F64, OFP_E_ARG, "bad dtype %d", dtype);
  uint64_t C = 1;
  for (int k = 0; k < 3; ++k) {
    OFP_CHECK(div[k] >= 1, OFP_E_ARG, "div[%d] must be >= 1", k);
    C *= uint64_t(div[k]) + 2;
  }
  OFP_CHECK(C < (1ull << 31), OFP_E_LIMIT, "too many cells (%llu)", (unsigned long long)C);
  if (opt & OFP_CL_QUANT)
    OFP_CHECK(div[0] + 2 <= 2048 && div[1] + 2 <= 2048 && div[2] + 2 <= 1024, OFP_E_LIMIT,
              "OFP_CL_QUANT packs cell coordinates in 11/11/10 bits");
  ofp_cl* h = new ofp_cl();
  h->dtype = dtype;
  h->opt = opt;
  h->n_cells = C;
  for (int k = 0; k < 3; ++k) {
    h->div[k] = div[k];
    h->divc[k] = div[k] + 2;
  }
  h->n_rows = h->divc[1] * h->divc[2];
  if (dtype == OFP_F32) {
    const float* lo = (const float*)box_lo;
    const float* hi = (const float*)box_hi;
    for (int k = 0; k < 3; ++k) {
      h->gf.lo[k] = lo[k];
      h->gf.sp[k] = (hi[k] - lo[k]) / float(div[k]);
      h->gf.divc[k] = h->divc[k];
      h->lo[k] = h->gf.lo[k];
      h->sp[k] = h->gf.sp[k];
    }
  } else {
    const double* lo = (const double*)box_lo;
    const double* hi = (const double*)box_hi;
    for (int k = 0; k < 3; ++k) {
      h->gd.lo[k] = lo[k];
      h->gd.sp[k] = (hi[k] - lo[k]) / double(div[k]);
      h->gd.divc[k] = h->divc[k];
      h->lo[k] = h->gd.lo[k];
      h->sp[k] = h->gd.sp[k];
    }
  }
  *out = h;
  return OFP_OK;
}

int ofp_cl_destroy(ofp_cl* h) {
  if (!h) return OFP_OK;
  DevBuf* bufs[] = {&h->packed, &h->scan64, &h->keys,    &h->keys2, &h->s2n,        &h->vals2, &h->n2s,
                    &h->dom,    &h->quant,  &h->scantmp, &h->hist,  &h->sid_sorted, &h->items,
                    &h->payload, &h->colpart, &h->cursors, &h->nz_flag, &h->nz_key, &h->nz_start, &h->nz_nn,
                    &h->nz_inv, &h->aux};
  for (DevBuf* b : bufs) b->release();
  if (h->far_done) (void)hipEventDestroy(h->far_done);
  if (h->checked) (void)hipEventDestroy(h->checked);
  if (h->desc) (void)hipHostFree(h->desc);
  delete h;
  return OFP_OK;
}

int ofp_cl_construct(ofp_cl* h, const void* pos, size_t stride, size_t n_tot, size_t gm,
                     void* pos_sorted, size_t sorted_stride, const ofp_plane* planes_in,
                     const ofp_plane* planes_out, int n_planes, void* stream) {
  OFP_CHECK(h, OFP_E_ARG, "ofp_cl_construct: null handle");
  OFP_CHECK(!h->n_sys, OFP_E_STATE, "ofp_cl_construct: ensemble cell lists are built by their ensemble");
  OFP_CHECK(n_tot == 0 || pos, OFP_E_ARG, "ofp_cl_construct: null positions");
  OFP_CHECK(gm <= n_tot, OFP_E_ARG, "ghost_marker %zu > n_tot %zu", gm, n_tot);
  OFP_CHECK(stride >= n_tot, OFP_E_ARG, "stride %zu < n_tot %zu", stride, n_tot);
  OFP_CHECK(!pos_sorted || sorted_stride >= n_tot, OFP_E_ARG, "sorted_stride < n_tot");
  OFP_CHECK(n_tot < 0xFFFFFFF0ull, OFP_E_LIMIT, "n_tot must fit 32 bits");
  OFP_CHECK(n_planes == 0 || planes_out, OFP_E_ARG, "reordered planes need outputs");
  PlaneArgs pa;
  OFP_TRY(make_plane_args(planes_in, planes_out, n_planes, &pa));
  if (h->dtype == OFP_F32)
    return cl_construct(h, h->gf, pos, stride, n_tot, gm, pos_sorted, sorted_stride, pa,
                        as_stream(stream));
  return cl_construct(h, h->gd, pos, stride, n_tot, gm, pos_sorted, sorted_stride, pa,
                      as_stream(stream));
}

int ofp_cl_set_box_nn(ofp_cl* h, uint32_t box_nn) {
  OFP_CHECK(h, OFP_E_ARG, "ofp_cl_set_box_nn: null handle");
  OFP_CHECK(box_nn >= 1 && box_nn <= uint32_t(kMaxBoxNN), OFP_E_LIMIT,
            "box_nn must be in [1, %d] (got %u)", kMaxBoxNN, box_nn);
  h->box_nn = box_nn;
  return OFP_OK;
}

int ofp_cl_dev_(const ofp_cl* h, ClDev* d, ofp_cl_view* v) {
  OFP_TRY(ofp_cl_get_view(h, v));
  d->cs = h->scan64.as<unsigned long long>();
  d->dom = h->dom.as<uint32_t>();
  d->quant = (h->opt & OFP_CL_QUANT) ? h->quant.as<int4>() : nullptr;
  for (int k = 0; k < 3; ++k) d->divc[k] = h->divc[k];
  d->n_dom = uint32_t(h->gm);
  d->box_nn = h->box_nn;
  d->n_cells = h->n_cells;
  return OFP_OK;
}

int ofp_cl_items_(const ofp_cl* hc, const TargetItem** items, const uint32_t** n_items,
                  uint32_t** counter, size_t* cap, hipStream_t s) {
  ofp_cl* h = const_cast<ofp_cl*>(hc);
  OFP_CHECK(h && h->built, OFP_E_STATE, "cell list not constructed");
  // the consumers' queue heads (kQueueWords), then the item count: see cl_build_t
  uint32_t* heads = reinterpret_cast<uint32_t*>(h->packed.as<unsigned long long>() + h->n_cells + 1);
  if (!h->items_valid) {
    size_t need = size_t(h->gm) + 1;
    OFP_TRY(h->items.ensure(need * sizeof(TargetItem)));
    // cleared by the build, once: a captured call, which may be replayed, clears itself
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    OFP_HIP(hipStreamIsCapturing(s, &cap));
    if (cap != hipStreamCaptureStatusNone) OFP_TRY(fill_u32(heads, 0, kQueueWords + 1, s));
    const uint32_t words = h->dtype == OFP_F32 ? uint32_t(sizeof(SysGrid<float>) / 4)
                                               : uint32_t(sizeof(SysGrid<double>) / 4);
    const uint32_t off = h->dtype == OFP_F32 ? uint32_t(offsetof(SysGrid<float>, divc) / 4)
                                             : uint32_t(offsetof(SysGrid<double>, divc) / 4);
    const uint32_t* desc = h->n_sys ? static_cast<const uint32_t*>(h->sys) + off : nullptr;
    k_cl_items<<<grid_for(h->n_rows, kItemRows), kItemRows * kWave, 0, s>>>(
        h->scan64.as<unsigned long long>(), h->divc[0], h->n_rows, h->n_sys, h->rbase, desc, words,
        h->items.as<TargetItem>(), heads + kQueueWords);
    OFP_LAUNCHED();
    h->items_cap = need;
    h->items_valid = true;
  }
  *items = h->items.as<TargetItem>();
  *n_items = heads + kQueueWords;
  *counter = heads;
  *cap = h->items_cap;
  return OFP_OK;
}

int ofp_cl_aux_(const ofp_cl* h, size_t bytes, void** p) {
  OFP_CHECK(h && p, OFP_E_ARG, "ofp_cl_aux_: null argument");
  ofp_cl* m = const_cast<ofp_cl*>(h);
  OFP_TRY(m->aux.ensure(bytes));
  *p = m->aux.p;
  return OFP_OK;
}

int ofp_cl_get_view(const ofp_cl* h, ofp_cl_view* v) {
  OFP_CHECK(h && v, OFP_E_ARG, "ofp_cl_get_view: null argument");
  OFP_CHECK(h->built, OFP_E_STATE, "cell list not constructed");
  std::memset(v, 0, sizeof(*v));
  v->cell_start = h->scan64.as<uint64_t>();
  v->sort_to_nonsort = h->s2n.as<uint32_t>();
  v->nonsort_to_sort = h->n2s.as<uint32_t>();
  v->dom_sort_ids = h->dom.as<uint32_t>();
  v->quant = (h->opt & OFP_CL_QUANT) ? h->quant.as<int32_t>() : nullptr;
  for (int k = 0; k < 3; ++k) {
    v->lo[k] = h->lo[k];
    v->spacing[k] = h->sp[k];
    v->div[k] = h->div[k];
    v->divc[k] = h->divc[k];
  }
  v->n_cells = h->n_cells;
  v->n_part = h->n_part;
  v->ghost_marker = h->gm;
  v->dtype = h->dtype;
  return OFP_OK;
}

int ofp_cl_build_sparse(ofp_cl* h, void* stream) {
  OFP_CHECK(h && h->built, OFP_E_STATE, "ofp_cl_build_sparse: cell list not constructed");
  OFP_CHECK(h->n_sys == 0, OFP_E_ARG, "ofp_cl_build_sparse: ensemble cell lists are not supported");
  OFP_CHECK(h->n_cells < (uint64_t(1) << 31), OFP_E_LIMIT, "ofp_cl_build_sparse: more than 2^31 cells");
  hipStream_t s = as_stream(stream);
  const uint64_t C = h->n_cells;
  OFP_TRY(h->nz_flag.ensure((C + 1) * sizeof(uint32_t)));
  OFP_TRY(h->nz_inv.ensure((C + 1) * sizeof(int32_t)));
  OFP_TRY(h->nz_key.ensure((C + 1) * sizeof(uint32_t)));
  OFP_TRY(h->nz_start.ensure((C + 1) * sizeof(uint32_t)));
  OFP_TRY(h->scantmp.ensure(scan_tmp_bytes(C)));
  DevBuf& pos = h->nz_nn;  // holds the scanned flags first, the neighbour table after
  OFP_TRY(pos.ensure((C + 1) * sizeof(uint32_t)));
  const uint64_t* cs = h->scan64.as<uint64_t>();
  k_nz_flag<<<grid_for(C, 256), 256, 0, s>>>(cs, C, h->nz_flag.as<uint32_t>());
  OFP_LAUNCHED();
  OFP_TRY(scan_excl_u32(h->nz_flag.as<uint32_t>(), pos.as<uint32_t>(), C, h->scantmp.p, s));
  k_nz_scatter<<<grid_for(C + 1, 256), 256, 0, s>>>(cs, C, pos.as<uint32_t>(), h->nz_key.as<uint32_t>(),
                                                     h->nz_start.as<uint32_t>(), h->nz_inv.as<int32_t>());
  OFP_LAUNCHED();
  uint32_t m = 0;
  OFP_HIP(hipMemcpyAsync(&m, pos.as<uint32_t>() + C, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
  OFP_HIP(hipStreamSynchronize(s));
  const uint32_t W = 2 * h->box_nn + 1, K = W * W * W;
  OFP_TRY(h->nz_nn.ensure((size_t(m) * K + 1) * sizeof(int32_t)));
  if (m > 0) {
    k_nz_nn<<<grid_for(size_t(m) * K, 256), 256, 0, s>>>(h->nz_key.as<uint32_t>(), m, h->divc[0], h->divc[1],
                                                         h->divc[2], int(h->box_nn), h->nz_inv.as<int32_t>(),
                                                         h->nz_nn.as<int32_t>());
    OFP_LAUNCHED();
  }
  h->n_nz = m;
  h->nz_box_nn = h->box_nn;
  h->sparse_valid = true;
  return OFP_OK;
}

int ofp_cl_get_sparse_view(const ofp_cl* h, ofp_cl_sparse_view* v) {
  OFP_CHECK(h && v, OFP_E_ARG, "ofp_cl_get_sparse_view: null argument");
  OFP_CHECK(h->built && h->sparse_valid, OFP_E_STATE, "ofp_cl_get_sparse_view: no sparse view of this build");
  v->cell_key = h->nz_key.as<uint32_t>();
  v->cell_start = h->nz_start.as<uint32_t>();
  v->cell_nn = h->nz_nn.as<int32_t>();
  v->n_cells = h->n_nz;
  v->box_nn = h->nz_box_nn;
  v->nn_per_cell = (2 * h->nz_box_nn + 1) * (2 * h->nz_box_nn + 1) * (2 * h->nz_box_nn + 1);
  return OFP_OK;
}

int ofp_cl_restore(const ofp_cl* h, const ofp_plane* sorted_in, const ofp_plane* orig_out,
                   int n_planes, void* stream) {
  OFP_CHECK(h && h->built, OFP_E_STATE, "ofp_cl_restore: cell list not constructed");
  OFP_CHECK(!h->n_dev, OFP_E_STATE, "ofp_cl_restore: particle count is on the device");
  OFP_CHECK(n_planes == 0 || orig_out, OFP_E_ARG, "ofp_cl_restore: null outputs");
  PlaneArgs pa;
  OFP_TRY(make_plane_args(sorted_in, orig_out, n_planes, &pa));  // every plane checked before any is written
  if (h->n_part == 0 || n_planes == 0) return OFP_OK;
  hipStream_t s = as_stream(stream);
  bool done = false;
  OFP_TRY(permute_route(h, h->s2n.as<uint32_t>(), pa, s, &done));
  if (done) return OFP_OK;
  // planes scattered together while their destinations fit the Infinity Cache
  // (256 MB), where the scattered values of a line meet: 2^25 particles from random
  // order, 24 bytes each, 2.4 ms plane by plane, 3.2 ms with the three coordinates
  // together, 5.6 ms all at once; 8,192 particles 13 us in four launches, 4 us in one
  constexpr size_t kTogether = size_t(160) << 20;
  for (int k = 0; k < n_planes;) {
    size_t bytes = 0;
    int m = 0;
    do bytes += h->n_part * sorted_in[k + m++].elem_bytes;
    while (k + m < n_planes && bytes + h->n_part * sorted_in[k + m].elem_bytes <= kTogether);
    OFP_TRY(make_plane_args(sorted_in + k, orig_out + k, m, &pa));
    k_cl_restore<<<grid_for(h->n_part, 256), 256, 0, s>>>(uint32_t(h->n_part), h->s2n.as<uint32_t>(), pa);
    OFP_LAUNCHED();
    k += m;
  }
  return OFP_OK;
}

int ofp_cl_reorder(const ofp_cl* h, const ofp_plane* orig_in, const ofp_plane* sorted_out,
                   int n_planes, void* stream) {
  OFP_CHECK(h && h->built, OFP_E_STATE, "ofp_cl_reorder: cell list not constructed");
  OFP_CHECK(!h->n_dev, OFP_E_STATE, "ofp_cl_reorder: particle count is on the device");
  OFP_CHECK(n_planes == 0 || sorted_out, OFP_E_ARG, "ofp_cl_reorder: null outputs");
  PlaneArgs pa;
  OFP_TRY(make_plane_args(orig_in, sorted_out, n_planes, &pa));
  if (h->n_part == 0 || n_planes == 0) return OFP_OK;
  hipStream_t s = as_stream(stream);
  bool done = false;
  OFP_TRY(permute_route(h, h->n2s.as<uint32_t>(), pa, s, &done));
  if (done) return OFP_OK;
  k_cl_reorder<<<grid_for(h->n_part, 256), 256, 0, s>>>(uint32_t(h->n_part), h->s2n.as<uint32_t>(), pa);
  OFP_LAUNCHED();
  return OFP_OK;
}

}  // extern "C"
