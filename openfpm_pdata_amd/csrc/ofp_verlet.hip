// ofp_verlet.hip -- getVerlet on the GPU: non-symmetric Verlet lists (self
// included) from a built cell list, in two passes over target items pulled
// from a device-side work queue.
//
// A target item is up to 64 domain particles (one per lane) whose cells lie on
// one x-row of the grid; its candidates are the (2B+1)^2 x-runs of the stencil
// (B = box_nn), each a contiguous range of sorted indices, cut into blocks of 32
// candidates.  The blocks of an item are numbered through its runs; a target's
// hits in a block are one 32-bit word, a target's words are consecutive, the
// targets one after another.
//  * count: the squared distances of 64 targets and the 64 candidates of two
//    blocks come from the matrix cores (FP32, K = 4: 2 x 2 tiles of 32 x 32), the
//    sign bits of d^2 - r^2 are the targets' words.  Blocks in which some square
//    is too near r^2 for FP32 products to decide are tested again with the
//    reference's rounding (distance2 unfused, in the position dtype), so the
//    words are those of the exact test.
//  * fill: an item's words, in order, are its rows, in order, so the wave takes 64
//    words at a time, one per lane, finds each lane's place by a prefix sum of
//    the bit counts, and expands the bits into LDS, from where whole 1 KB stores
//    go to the list.
// Entries of a row come out in ascending sorted index, which is the reference
// traversal order (cells in ascending linear id, ascending index inside a cell).
// Persistent waves: each wave takes the next unit (an item, or a part of one
// where there are too few items for the chip) from its queue and leaves when that
// is empty, so every wave reaches its exit.
// A mask buffer too small for the items is flagged (mstate[1]); the fill then
// writes nothing and the host grows the buffer and counts again.
#include "ofp_internal.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>

struct ofp_vl {
  ofp::HandleLife life;
  ofp::DevBuf cnt, off, nbr, scantmp, masks, place, xyz;
  ofp::DevBuf rmask;  // thread-per-row build: the rows' hit masks, count pass to fill
  ofp::DevBuf aux;  // pair kernels' per-particle gather stream over the rows
  ofp::DevBuf rec;  // the density pass's 12-byte records
  std::mutex rec_lock;  // its allocation: passes over one list may come from several threads
  size_t mask_cap = 0;  // pairs of mask words (8 bytes) the buffer holds (0: not sized yet)
  bool rows_path = false;  // the last build ran the thread-per-row kernels
  uint64_t n_rows = 0, n_entries = 0;
  uint64_t n_state = 0;  // rows of the last build: mstate lies behind its offsets
  bool built = false;
  bool symmetric = false;  // built by ofp_vl_build_sym (each interaction once)
  const ofp_cl* cl = nullptr;
};

namespace ofp {

constexpr int kVlBlock = 256;
constexpr int kVlWaves = kVlBlock / kWave;
constexpr uint32_t kBlk = 32;  // candidates per block (bits of a mask word)

// The coordinates of 8 consecutive particles, x y z interleaved (read with
// scalar loads; the element alignment is all a scalar load needs).
template <class T>
struct alignas(sizeof(T)) Run8 {
  T v[24];
};
template <class T>
struct Run1 {
  T v[3];
};
// A load of read-only data at a wave-uniform address, as scalar loads (the
// constant address space tells the compiler that no store of the kernel changes
// it).
template <class S>
__device__ __forceinline__ S scalar_load(const void* p) {
  using W = const uint32_t __attribute__((address_space(4)));
  static_assert(sizeof(S) % 4 == 0, "whole dwords");
  W* q = (W*)(reinterpret_cast<uintptr_t>(p));
  uint32_t w[sizeof(S) / 4];
#pragma unroll
  for (size_t i = 0; i < sizeof(S) / 4; ++i) w[i] = q[i];
  S s;
  __builtin_memcpy(&s, w, sizeof(S));
  return s;
}

// Sorted positions (three planes of stride `stride`) to one interleaved xyz
// stream: the count pass reads the candidates of a run as one contiguous range,
// whatever the planes' stride (planes a large power of two apart would share
// cache sets).
// Also clears the build's counts (cnt) and control words (ctl).
template <class T>
__global__ void k_vl_pack(const T* __restrict__ pos, size_t stride, uint32_t n, T* __restrict__ xyz,
                          uint32_t* __restrict__ cnt, uint32_t n_cnt, uint32_t* __restrict__ ctl, uint32_t n_ctl) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_cnt) cnt[i] = 0u;
  if (i < n_ctl) ctl[i] = 0u;
  if (i >= n) return;
  xyz[3 * size_t(i)] = pos[i];
  xyz[3 * size_t(i) + 1] = pos[stride + i];
  xyz[3 * size_t(i) + 2] = pos[2 * stride + i];
}

// An item's runs in the lanes: lane r < (2B+1)^2 holds run r (traversal order),
// its bounds and the number of its first block; blocks = the item's total.
struct ItemRuns {
  uint32_t ja, jb, first, blocks;
};
template <class T>
__device__ __forceinline__ ItemRuns item_runs(const ClDev& c, const ItemGeom<T>& G, int lane) {
  const uint2 run = lane_run(c, G, lane);
  ItemRuns R{run.x, run.y, 0, 0};
  const uint32_t nb = (R.jb - R.ja + kBlk - 1) / kBlk;
  const uint32_t inc = wave_incl_scan(nb);
  R.first = inc - nb;
  R.blocks = __builtin_amdgcn_readlane(inc, kWave - 1);
  return R;
}

// Orders a wave's LDS accesses for the compiler (the LDS itself serves a wave's
// accesses in order).
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The first candidates and lengths of blocks [w0, w0 + N) of the item into the
// wave's LDS table (entries past the item's blocks are not written).
template <uint32_t N>
__device__ __forceinline__ void block_table(const ItemRuns& R, uint32_t w0, uint2* tab) {
  lds_order();
  uint32_t q = R.first > w0 ? R.first : w0;
  uint32_t j = R.ja + (q - R.first) * kBlk;
  for (; j < R.jb && q < w0 + N; ++q, j += kBlk) tab[q - w0] = make_uint2(j, R.jb - j < kBlk ? R.jb - j : kBlk);
  lds_order();
}

// Part `part` of P of `total` (monotonic in part, 0 and total at the ends).
__device__ __forceinline__ uint32_t part_begin(uint32_t total, uint32_t part, uint32_t P) {
  return P == 1 ? (part ? total : 0u) : uint32_t(uint64_t(total) * part / P);
}

// An item's words in the mask buffer: the first (in pairs of words) and the words
// per target, a multiple of four (16-byte stores).
struct ItemPlace {
  unsigned long long first;
  uint32_t words;
  uint32_t pad;
};

// The places of all items and their total (mstate[0], cleared before), a thread
// per item and one atomic per block of threads.
template <class T>
__global__ __launch_bounds__(kVlBlock) void k_vl_place(ClDev c, const SysGrid<T>* __restrict__ sys,
                                                       const TargetItem* __restrict__ items,
                                                       const uint32_t* __restrict__ n_items_p,
                                                       unsigned long long* __restrict__ mstate,
                                                       ItemPlace* __restrict__ place) {
  __shared__ unsigned long long ws[kVlWaves + 1];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const uint32_t n_items = *n_items_p;
  for (uint32_t i0 = blockIdx.x * kVlBlock; i0 < n_items; i0 += gridDim.x * kVlBlock) {
    const uint32_t it = i0 + threadIdx.x;
    uint32_t words = 0, n = 0;
    if (it < n_items) {
      const TargetItem ti = items[it];
      const ItemGeom<T> G = item_geom(c, ti, T(0), sys, static_cast<const T*>(nullptr));
      const int B = int(c.box_nn);
      const int xa = G.cx0 - B > 0 ? G.cx0 - B : 0;
      const int xe = G.cx0 + G.ncx - 1 + B;
      const int xb = xe < int(G.d0) - 1 ? xe : int(G.d0) - 1;
      for (int dz = -B; dz <= B; ++dz) {
        const int zz = G.cz + dz;
        if (zz < 0 || zz >= int(G.d2)) continue;
        // a plane's rows at once, those outside the grid as an empty run of the
        // item's own (small builds wait for nothing but these loads)
        uint32_t ja[2 * kMaxBoxNN + 1], jb[2 * kMaxBoxNN + 1];
#pragma unroll
        for (int k = 0; k < 2 * kMaxBoxNN + 1; ++k) {
          const int yy = G.cy - B + k;
          const bool in = k <= 2 * B && yy >= 0 && yy < int(G.d1);
          const uint32_t rowc = G.cbase + G.d0 * (uint32_t(in ? yy : G.cy) + G.d1 * uint32_t(zz));
          ja[k] = uint32_t(c.cs[rowc + uint32_t(xa)]);
          jb[k] = uint32_t(c.cs[rowc + (in ? uint32_t(xb) + 1u : uint32_t(xa))]);
        }
#pragma unroll
        for (int k = 0; k < 2 * kMaxBoxNN + 1; ++k) words += (jb[k] - ja[k] + kBlk - 1) / kBlk;
      }
      words = (words + 3u) & ~3u;
      n = ti.n;
    }
    const unsigned long long need = static_cast<unsigned long long>(words / 2u) * n;
    const unsigned long long inc = wave_incl_scan(need);
    if (lane == kWave - 1) ws[w] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned long long all = 0;
      for (int k = 0; k < kVlWaves; ++k) {
        const unsigned long long x = ws[k];
        ws[k] = all;
        all += x;
      }
      ws[kVlWaves] = all ? atomicAdd(&mstate[0], all) : 0ull;
    }
    __syncthreads();
    if (it < n_items) place[it] = ItemPlace{ws[kVlWaves] + ws[w] + inc - need, words, 0u};
    __syncthreads();
  }
}

// Count pass.  Lane t builds the words of target t, two blocks at a time.  A unit
// is a part (of P) of an item's words; with P > 1 the parts' hits are added to cnt
// (cleared before).  mstate[0]: pairs of words of all items, mstate[1]: overflow
// flag (then no words are stored).
//
// With coordinates relative to one of the item's targets, a tile of the matrix
// product of (x, y, z, |c|^2) and (-2x, -2y, -2z, 1), on top of |t|^2 - r^2, is
// d^2 - r^2 for 32 candidates (rows) and 32 targets (columns): 128 matrix-core
// cycles per 1024 pairs, and the vector ALU is left one instruction per 64 pairs
// for the sign bit and half a one for the smallest |d^2 - r^2|, where the
// distance test in the vector ALU took ten.  Rows are assigned to candidates so
// that a lane's 16 results of a tile are 16 consecutive candidates, highest
// first.
// Undecided squares: with S = (R_c + R_t)^2 + r^2, R the farthest candidate and
// target from the origin, relative coordinates, norms and products in FP32
// (unit roundoff u) differ from the exact square by less than 24 u S, and the
// reference's own roundings by less than 6 u d^2; |d^2 - r^2| < 32 u S = 2^-19 S
// is tested exactly.  R comes from the cell geometry; blocks or an item with a
// particle beyond it (outside its cell, or not a number) are tested exactly too, and
// so are items whose squares FP32 cannot hold: FP64 coordinates are scaled by
// matrix_unit first, FP32 ones are not, for the reference's own squares of them leave
// the range where those of the products do.
// 4.2e6 clustered particles (cells of r/2, 150 words a target): 6.4 -> 3.8 ms; 3e5:
// 0.46 -> 0.27 ms; 4e5 in FP64 0.85 -> 0.36 ms.
template <class T>
__global__ __launch_bounds__(kVlBlock, 4) void k_vl_count(ClDev c, const T* __restrict__ xyz, T r2_one, T spx,
                                                       T spy, T spz, const SysGrid<T>* __restrict__ sys,
                                                       const T* __restrict__ r2_sys,
                                                       const TargetItem* __restrict__ items,
                                                       const uint32_t* __restrict__ n_items_p, uint32_t P,
                                                       uint32_t* __restrict__ counter, uint32_t* __restrict__ cnt,
                                                       unsigned long long* __restrict__ mstate,
                                                       const ItemPlace* __restrict__ place,
                                                       unsigned long long* __restrict__ masks,
                                                       unsigned long long mask_cap) {
  __shared__ uint2 tabs[kVlWaves][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  uint2* const tab = tabs[threadIdx.x / kWave];
  const uint32_t n_units = *n_items_p * P;
  const bool keep = mstate[0] <= mask_cap;  // grid-uniform
  if (!keep && blockIdx.x == 0 && threadIdx.x == 0) atomicOr(&mstate[1], 1ull);
  const uint32_t mine = matrix_candidate(uint32_t(lane));
  for (;;) {
    const uint32_t un = next_unit(counter);
    if (un >= n_units) break;
    const uint32_t it = P == 1 ? un : un / P, part = P == 1 ? 0u : un % P;
    const TargetItem ti = items[it];
    const ItemGeom<T> G = item_geom(c, ti, r2_one, sys, r2_sys);
    const T r2 = G.r2;
    if (sys) {
      const uint32_t sy = ti.ncx >> 8;
      spx = sys[sy].sp[0];
      spy = sys[sy].sp[1];
      spz = sys[sy].sp[2];
    }
    const bool valid = uint32_t(lane) < ti.n;
    const uint32_t row = ti.row0 + (valid ? uint32_t(lane) : 0u);
    const uint32_t p = c.dom[row];
    const ItemPlace at = place[it];
    const ItemRuns R = item_runs(c, G, lane);
    const T xp = xyz[3 * size_t(p)], yp = xyz[3 * size_t(p) + 1], zp = xyz[3 * size_t(p) + 2];
    // targets relative to the middle one, and the bounds of the FP32 squares
    const uint32_t mid = ti.n / 2;
    const T ox = lane_value(xp, mid), oy = lane_value(yp, mid), oz = lane_value(zp, mid);
    const T unit = std::is_same_v<T, double> ? T(matrix_unit(spx, spy, spz)) : T(1);
    auto rel = [&](T a, T o) {
      if constexpr (std::is_same_v<T, double>) return float((a - o) * unit);
      return float(a - o);
    };
    const float ux = float(spx * unit), uy = float(spy * unit), uz = float(spz * unit);
    const float B1 = float(c.box_nn + 1u), nx = float(G.ncx), bx = nx + float(c.box_nn);
    const float rt2 = nx * nx * ux * ux + uy * uy + uz * uz;
    const float rc2 = bx * bx * ux * ux + B1 * B1 * (uy * uy + uz * uz);
    MatrixTest mt;
    const bool fast = mt.template targets<false>(rel(xp, ox), rel(yp, oy), rel(zp, oz), rt2, rc2,
                                                 float(r2 * unit * unit), ti.n > 32u);
    // Exact hit bits of candidates j0 .. j0 + m - 1 (1 <= m <= 32, uniform), bit k
    // for candidate j0 + k; the coordinates come in through scalar loads.  Lanes
    // past the item's targets compute bits that are never stored.
    auto hit_word = [&](uint32_t j0, uint32_t m) -> uint32_t {
      uint32_t w = 0;  // candidate j0 + k at bit (k' - 1 - k) after k' shifts
      uint32_t k = 0;
      for (; k + 8 <= m; k += 8) {
        const Run8<T> Q = scalar_load<Run8<T>>(xyz + 3 * size_t(j0 + k));
#pragma unroll
        for (int i = 0; i < 8; ++i)
          w = shift_in(w, dist2_unfused<T>(Q.v[3 * i] - xp, Q.v[3 * i + 1] - yp, Q.v[3 * i + 2] - zp) < r2);
      }
      for (; k < m; ++k) {
        const Run1<T> q = scalar_load<Run1<T>>(xyz + 3 * size_t(j0 + k));
        w = shift_in(w, dist2_unfused<T>(q.v[0] - xp, q.v[1] - yp, q.v[2] - zp) < r2);
      }
      return __builtin_bitreverse32(w << (32u - m));
    };
    uint32_t n = 0;
    // the unit's words [wa, wb), whole quads; blocks past the item's last are empty
    const uint32_t wa = 4u * part_begin(at.words / 4u, part, P), wb = 4u * part_begin(at.words / 4u, part + 1, P);
    uint2 tv = make_uint2(0u, 0u);  // block (w & ~63) + lane: first candidate, length
    T cx, cy, cz;                   // this lane's candidate of the next two blocks
    struct Two {
      uint32_t ja, ma, jb, mb;
    };
    auto fetch = [&](uint32_t w) {
      if ((w & 63u) == 0u || w == wa) {
        block_table<kWave>(R, w & ~63u, tab);
        tv = (w & ~63u) + uint32_t(lane) < R.blocks ? tab[lane] : make_uint2(0u, 0u);
      }
      Two b;
      b.ja = __builtin_amdgcn_readlane(tv.x, w & 63u);
      b.ma = __builtin_amdgcn_readlane(tv.y, w & 63u);
      b.jb = __builtin_amdgcn_readlane(tv.x, (w & 63u) + 1u);
      b.mb = __builtin_amdgcn_readlane(tv.y, (w & 63u) + 1u);
      const uint32_t j = lane < 32 ? b.ja : b.jb, m = lane < 32 ? b.ma : b.mb;
      const T* s = xyz + 3 * size_t(j + (mine < m ? mine : (m ? m - 1u : 0u)));
      cx = s[0];
      cy = s[1];
      cz = s[2];
      return b;
    };
    Two cur{0, 0, 0, 0};
    if (wa < wb) cur = fetch(wa);
    uint32_t* const out = reinterpret_cast<uint32_t*>(masks + at.first) + size_t(lane) * at.words;
    uint32_t q0 = 0, q1 = 0;  // the quad's first two words
    for (uint32_t w = wa; w < wb; w += 2) {
      const Two b = cur;
      const float x0 = rel(cx, ox), y0 = rel(cy, oy), z0 = rel(cz, oz);
      if (w + 2 < wb) cur = fetch(w + 2);
      uint32_t lo = 0, hi = 0;
      if (b.ma) {
        if (!fast || !mt.template words<true>(x0, y0, z0, b.mb != 0u, &lo, &hi)) {  // a few per hundred
          lo = hit_word(b.ja, b.ma);
          hi = b.mb ? hit_word(b.jb, b.mb) : 0u;
        } else {
          lo &= 0xFFFFFFFFu >> (32u - b.ma);
          hi &= b.mb ? 0xFFFFFFFFu >> (32u - b.mb) : 0u;
        }
      }
      n += uint32_t(__builtin_popcount(lo)) + uint32_t(__builtin_popcount(hi));
      if ((w & 2u) == 0u) {
        q0 = lo;
        q1 = hi;
      } else if (keep && valid) {
        *reinterpret_cast<uint4*>(out + (w - 2u)) = make_uint4(q0, q1, lo, hi);
      }
    }
    if (valid) {
      if (P == 1)
        cnt[row] = n;
      else if (n)
        atomicAdd(&cnt[row], n);
    }
  }
}

// Fill pass from the words.  A unit is the words of TQ consecutive targets of an
// item, the wave's stream; its entries are consecutive in the list.  Words with a
// hit are queued in LDS with their blocks' first candidates (in the clustered
// workload half of all words are empty), and 64 queued words are expanded at a time:
// a prefix sum of the bit counts gives each lane its place in the staged row, and
// each lane writes out its own word's bits.  Staged entries go to the list 16
// bytes per lane.
// Storing each word's hits straight to the list, a chunk of 64 candidates in the
// lanes and a target's mask as exec mask, was bound by the 20 cycles a store
// takes of the CU's address unit, for 8 entries on average.
// e_total / e_cap: the list's entry count (device) and the capacity of nbr; a list
// that does not fit, or whose masks did not, is not written.
// 4.2e6 clustered particles (4.4e9 entries, 17.7 GB): 8.4 -> 6.4 ms (2.8 TB/s
// written; instructions of the expansion, 45 % of the kernel's lanes on, and LDS
// conflicts, 56 % of its LDS cycles); 3e5: 0.58 -> 0.35 ms; 4e5 in FP64 0.83 -> 0.55 ms.
// LDS: 24 KB a block, six blocks per CU (32 KB and five: 6.8 ms).
constexpr uint32_t kStage = 1024;  // entries staged per wave
constexpr uint32_t kTab = 192;     // blocks tabulated per item (more: searched in its runs)
template <class T>
__global__ __launch_bounds__(kVlBlock) void k_vl_fill(ClDev c, const SysGrid<T>* __restrict__ sys,
                                                      const TargetItem* __restrict__ items,
                                                      const uint32_t* __restrict__ n_items_p, uint32_t TQ,
                                                      uint32_t* __restrict__ counter,
                                                      const unsigned long long* __restrict__ off,
                                                      const unsigned long long* __restrict__ e_total,
                                                      unsigned long long e_cap,
                                                      const unsigned long long* __restrict__ mstate,
                                                      const ItemPlace* __restrict__ place,
                                                      const unsigned long long* __restrict__ masks,
                                                      uint32_t* __restrict__ nbr) {
  static_assert(kStage >= 32 * kWave / 2, "half a wave of full words fits the empty row");
  __shared__ uint4 stages[kVlWaves][kStage / 4];
  __shared__ uint2 queues[kVlWaves][2 * kWave];
  __shared__ uint32_t tabs[kVlWaves][kTab];
  const int lane = threadIdx.x & (kWave - 1);
  uint32_t* const tab = tabs[threadIdx.x / kWave];
  uint2* const queue = queues[threadIdx.x / kWave];
  uint4* const st4 = stages[threadIdx.x / kWave];
  uint32_t* const st = reinterpret_cast<uint32_t*>(st4);
  const uint32_t Q = kWave / TQ;  // units per item
  const uint32_t n_units = *n_items_p * Q;
  if (*e_total > e_cap || mstate[1] != 0ull) return;
  for (;;) {
    const uint32_t un = next_unit(counter);
    if (un >= n_units) break;
    const uint32_t it = un / Q;
    const TargetItem ti = items[it];
    const uint32_t ta = (un % Q) * TQ, tb = ta + TQ < ti.n ? ta + TQ : ti.n;
    if (ta >= ti.n) continue;
    const ItemPlace at = place[it];
    const uint32_t W = at.words;
    if (W == 0) continue;
    const unsigned long long e0 = off[ti.row0 + ta];
    const uint32_t* __restrict__ words = reinterpret_cast<const uint32_t*>(masks + at.first) + size_t(ta) * W;
    const uint32_t total = (tb - ta) * W;
    const ItemGeom<T> G = item_geom(c, ti, T(0), sys, static_cast<const T*>(nullptr));
    const ItemRuns R = item_runs(c, G, lane);
    lds_order();
    const bool small = W <= kTab;
    if (small) {  // tab[block] = its first candidate
      for (uint32_t q = R.first, j = R.ja; j < R.jb; ++q, j += kBlk) tab[q] = j;
    } else {  // tab[run] = its first block, tab[64 + run] = its first candidate
      tab[lane] = R.first;
      tab[kWave + lane] = R.ja;
    }
    lds_order();
    auto block_first = [&](uint32_t w) -> uint32_t {
      if (small) return tab[w];
      uint32_t lo = 0;  // the last run that starts at or before w (empty runs start where the next one does)
#pragma unroll
      for (uint32_t d = kWave / 2; d > 0; d >>= 1) lo += tab[lo + d] <= w ? d : 0u;
      return tab[kWave + lo] + (w - tab[lo]) * kBlk;
    };
    uint32_t* out = nbr + e0;
    uint32_t staged = 0, queued = 0;
    auto flush = [&]() {
      lds_order();
      for (uint32_t k = uint32_t(lane); k < (staged >> 2); k += kWave) {
        const uint4 v = st4[k];
        __builtin_memcpy(out + 4 * k, &v, sizeof(v));
      }
      const uint32_t k = (staged & ~3u) + uint32_t(lane);
      if (k < staged) out[k] = st[k];
      out += staged;
      staged = 0;
      lds_order();
    };
    // the first m <= 64 queued words
    auto expand = [&](uint32_t m) {
      lds_order();
      uint2 v = make_uint2(0u, 0u);
      if (uint32_t(lane) < m) v = queue[lane];
      const uint32_t pc = uint32_t(__builtin_popcount(v.x));
      const uint32_t inc = wave_incl_scan(pc);
      const uint32_t all = __builtin_amdgcn_readlane(inc, kWave - 1);
      auto write = [&](uint32_t bits, uint32_t place_) {
        uint32_t* p = st + place_;
        while (bits) {
          *p++ = v.y + uint32_t(__builtin_ctz(bits));
          bits &= bits - 1u;
        }
      };
      if (staged + all > kStage) flush();
      if (all <= kStage) {
        write(v.x, staged + inc - pc);
        staged += all;
      } else {  // more hits than the row holds: half a wave at a time
        const uint32_t first = __builtin_amdgcn_readlane(inc, kWave / 2 - 1);
        write(lane < kWave / 2 ? v.x : 0u, inc - pc);
        staged = first;
        flush();
        write(lane < kWave / 2 ? 0u : v.x, inc - pc - first);
        staged = all - first;
      }
    };
    uint32_t w = uint32_t(lane) % W;  // this lane's word of its target
    const uint32_t step = kWave % W;
    uint32_t next = uint32_t(lane) < total ? words[lane] : 0u;
    for (uint32_t f = 0; f < total; f += kWave) {
      const uint32_t bits = next;
      const uint32_t fn = f + kWave + uint32_t(lane);
      next = fn < total ? words[fn] : 0u;
      const unsigned long long nz = __ballot(bits != 0u);
      if (bits) {
        const uint32_t lo = __builtin_amdgcn_mbcnt_lo(uint32_t(nz), 0u);
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(uint32_t(nz >> 32), lo);
        const uint32_t k = queued + below;
        queue[k] = make_uint2(bits, block_first(w));
      }
      queued += uint32_t(__popcll(nz));
      w += step;
      w = w >= W ? w - W : w;
      if (queued >= uint32_t(kWave)) {
        expand(kWave);
        queued -= kWave;
        if (uint32_t(lane) < queued) queue[lane] = queue[kWave + lane];
      }
    }
    if (queued) expand(queued);
    if (staged) flush();
  }
}

// Thread-per-row build for dilute lists (few candidates per target: the item
// kernels' 64 lanes would mostly idle).  Thread k takes row k (domain particle
// dom[k]), finds its cell with the build's key formula, and walks the
// (2B+1)^2 x-runs of its own stencil in traversal order.
//  * count (kFill = false): every candidate is tested with the same rounding
//    as the item kernels (distance2 unfused, in the position dtype); each test
//    appends one bit to the row's hit mask (candidate c of the row is bit
//    31 - c % 32 of word c / 32), staged in LDS and stored for the row's first
//    kRowWords words (word w of the wave's rows at one 256-byte line), and the
//    hits are counted.
//  * fill (kFill = true): the row's entries come from its mask words (the
//    tests of candidates past kRowWords words are repeated), in ascending
//    sorted index as the item kernels write them, gathered in LDS up to
//    kSeg of them per wave and written out with coalesced stores; past
//    kSeg they go straight to the list.
// Ensembles: the row's system from sid_sorted.
constexpr int kRowAhead = 4;  // candidates in flight per thread
constexpr uint32_t kRowWords = 16;  // mask words kept per row (32 candidates each)
// Entries per wave staged in LDS by the fill; the others go to the list one by one, a
// line each.  The larger where the mean wave (the host knows the list's entries, or
// its capacity) does not fit the smaller: 10 KB a wave are 16 waves per CU, with the
// next run's bounds loaded ahead.  1e6 rows of 46 entries: fill 256 -> 167 us (3072:
// 208, 5120: 253); the 857,000 rows of 64 boxes 247 -> 197 us.
constexpr uint32_t kRowSegFew = 1024, kRowSegMany = 2560;
constexpr int kRowWaves = 256 / kWave;

// kB: the stencil half-width B (c.box_nn) as a constant, so the row's
// (2B+1)^2 run bounds are all loaded before its first candidate is read.
// masks: kRowWords x 64 words per wave of rows.
// kSeg: kRowSegFew or kRowSegMany.
template <class T, bool kFill, int kB, uint32_t kSeg>
__global__ __launch_bounds__(256) void k_vl_rows(ClDev c, CellGeom<T> g1, const T* __restrict__ xyz, T r2_one,
                                                 const SysGrid<T>* __restrict__ sys, const T* __restrict__ r2_sys,
                                                 const uint32_t* __restrict__ sid_sorted, uint32_t* __restrict__ cnt,
                                                 uint32_t* __restrict__ masks,
                                                 const unsigned long long* __restrict__ off,
                                                 const unsigned long long* __restrict__ e_total,
                                                 unsigned long long e_cap, uint32_t* __restrict__ nbr) {
  __shared__ uint32_t lds[kRowWaves][kFill ? kSeg : kRowWords * kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t k0 = k - uint32_t(lane);  // the wave's first row
  if (k0 >= c.n_dom) return;               // wave-uniform
  if constexpr (kFill) {
    if (*e_total > e_cap) return;  // the list does not fit: nothing is written (grid-uniform)
  }
  const bool valid = k < c.n_dom;
  uint32_t* const wl = lds[threadIdx.x / kWave];
  uint32_t* const wmask = masks + size_t(k0 / uint32_t(kWave)) * (kRowWords * kWave);
  T xp = T(0), yp = T(0), zp = T(0), r2 = r2_one;
  CellGeom<T> g = g1;
  uint32_t cbase = 0;
  int cxi = 0, cyi = 0, czi = 0;
  if (valid) {
    const uint32_t p = c.dom[k];
    xp = xyz[3 * size_t(p)];
    yp = xyz[3 * size_t(p) + 1];
    zp = xyz[3 * size_t(p) + 2];
    if (sys) {
      const uint32_t s = sid_sorted[p];
      g = sys[s].geom();
      cbase = sys[s].cbase;
      if (r2_sys) r2 = r2_sys[s];
    }
    uint32_t cx, cy, cz;
    (void)cell_of(g, xp, yp, zp, &cx, &cy, &cz);
    cxi = int(cx);
    cyi = int(cy);
    czi = int(cz);
  }
  const int d0 = int(g.divc[0]), d1 = int(g.divc[1]), d2 = int(g.divc[2]);
  const int xa = cxi - kB > 0 ? cxi - kB : 0;
  const int xb = cxi + kB < d0 - 1 ? cxi + kB : d0 - 1;
  // the stencil's x-runs [a, b) of sorted indices in traversal order (dz, then
  // dy); runs off the grid (and every run of an invalid lane) are empty
  auto run_bounds = [&](int r, uint32_t* a, uint32_t* b) {
    const int zz = czi + r / (2 * kB + 1) - kB, yy = cyi + r % (2 * kB + 1) - kB;
    const bool in = valid && zz >= 0 && zz < d2 && yy >= 0 && yy < d1;
    const uint32_t rowc = cbase + uint32_t(d0) * (uint32_t(in ? yy : 0) + uint32_t(d1) * uint32_t(in ? zz : 0));
    *a = in ? uint32_t(c.cs[rowc + uint32_t(xa)]) : 0u;
    *b = in ? uint32_t(c.cs[rowc + uint32_t(xb) + 1]) : 0u;
  };
  constexpr int kRuns = (2 * kB + 1) * (2 * kB + 1);
  constexpr bool kKeep = kB == 1;  // the 9 runs' bounds loaded up front, kept in registers
  uint32_t run_a[kKeep ? kRuns : 1], run_b[kKeep ? kRuns : 1];
  if constexpr (kKeep) {
#pragma unroll
    for (int r = 0; r < kRuns; ++r) run_bounds(r, &run_a[r], &run_b[r]);
  }
  auto for_runs = [&](auto&& fn) {
    if constexpr (kKeep) {
#pragma unroll
      for (int r = 0; r < kRuns; ++r) fn(run_a[r], run_b[r]);
    } else {
      uint32_t a, b;
      run_bounds(0, &a, &b);
      for (int r = 0; r < kRuns; ++r) {
        uint32_t na = 0, nb = 0;  // the next run's, loaded ahead
        if (r + 1 < kRuns) run_bounds(r + 1, &na, &nb);
        fn(a, b);
        a = na;
        b = nb;
      }
    }
  };
  if constexpr (!kFill) {
    // the candidates in groups of kRowAhead from each run's start, all of a
    // group's coordinates loaded before any is tested (up to kRowAhead - 1
    // candidates past the run's end are read, from the next run or the
    // coordinate stream's padding; their tests are dropped).  A group appends its m tests to the
    // pending bits (acc, the newest lowest; fill of them not yet stored), and
    // every 32 of them go to the next mask word.
    uint32_t n = 0, nwd = 0, fill = 0;  // hits, mask words completed, bits pending
    unsigned long long acc = 0;
    for_runs([&](uint32_t ja, uint32_t jb) {
      for (uint32_t j0 = ja; j0 < jb; j0 += kRowAhead) {
        const T* __restrict__ q = xyz + 3 * size_t(j0);
        T c[kRowAhead][3];
#pragma unroll
        for (int u = 0; u < kRowAhead; ++u) {
          c[u][0] = q[3 * u];
          c[u][1] = q[3 * u + 1];
          c[u][2] = q[3 * u + 2];
        }
        const uint32_t m = jb - j0 < uint32_t(kRowAhead) ? jb - j0 : uint32_t(kRowAhead);
        uint32_t h = 0;  // the group's tests, its first candidate highest
#pragma unroll
        for (int u = 0; u < kRowAhead; ++u) {
          const bool hit = dist2_unfused<T>(c[u][0] - xp, c[u][1] - yp, c[u][2] - zp) < r2;
          h |= (hit && uint32_t(u) < m ? 1u : 0u) << (kRowAhead - 1 - u);
        }
        h >>= uint32_t(kRowAhead) - m;
        n += uint32_t(__popc(h));
        acc = (acc << m) | h;
        fill += m;
        if (fill >= 32u) {
          fill -= 32u;
          if (nwd < kRowWords) wl[nwd * kWave + uint32_t(lane)] = uint32_t(acc >> fill);
          ++nwd;
        }
      }
    });
    // the last, partial word, its first candidate at bit 31
    if (fill != 0u && nwd < kRowWords) wl[nwd * kWave + uint32_t(lane)] = uint32_t(acc << (32u - fill));
    const uint32_t cand = nwd * 32u + fill;
    if (valid) cnt[k] = n;
    // the mask words out, word w of the wave's rows on one line (a lane past
    // its own words stores what is there; nothing reads it)
    uint32_t nw = (cand + 31u) >> 5;
    nw = nw < kRowWords ? nw : kRowWords;
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
      const uint32_t o = __shfl_xor(nw, d, kWave);
      nw = o > nw ? o : nw;
    }
    __builtin_amdgcn_wave_barrier();
    for (uint32_t w = 0; w < nw; ++w) wmask[w * kWave + uint32_t(lane)] = wl[w * kWave + uint32_t(lane)];
  } else {
    const unsigned long long base = off[k0];
    const unsigned long long lo = valid ? off[k] - base : 0;
    uint32_t i = 0;  // entries of the row written
    auto emit = [&](uint32_t j) {
      const unsigned long long at = lo + i;
      if (at < kSeg)
        wl[at] = j;
      else
        nbr[base + at] = j;
      ++i;
    };
    uint32_t cb = 0;              // candidate index of the run's first candidate
    uint32_t cw = ~0u, cbits = 0;  // the mask word last read
    for_runs([&](uint32_t ja, uint32_t jb) {
      const uint32_t end = cb + (jb - ja);
      const uint32_t lim = end < 32u * kRowWords ? end : 32u * kRowWords;
      uint32_t cc = cb;
      while (cc < lim) {
        const uint32_t w = cc >> 5, sh = cc & 31u;
        const uint32_t wend = (w + 1u) * 32u < lim ? (w + 1u) * 32u : lim;
        const uint32_t m = wend - cc;  // the run's candidates in word w (1-32)
        if (w != cw) {
          cw = w;
          cbits = wmask[w * kWave + uint32_t(lane)];
        }
        uint32_t bm = cbits << sh;
        if (m < 32u) bm &= ~(0xFFFFFFFFu >> m);
        while (bm) {
          const uint32_t lead = uint32_t(__builtin_clz(bm));
          bm ^= 0x80000000u >> lead;
          emit(ja + (cc - cb) + lead);
        }
        cc = wend;
      }
      for (uint32_t j = ja + (cc - cb); j < jb; ++j)
        if (dist2_unfused<T>(xyz[3 * size_t(j)] - xp, xyz[3 * size_t(j) + 1] - yp, xyz[3 * size_t(j) + 2] - zp) < r2)
          emit(j);
      cb = end;
    });
    // the wave's staged entries, written out by all its lanes (the wave's LDS
    // writes all precede these reads in its program order)
    __builtin_amdgcn_wave_barrier();
    const uint32_t k1 = k0 + uint32_t(kWave) < c.n_dom ? k0 + uint32_t(kWave) : c.n_dom;
    const unsigned long long len = off[k1] - base;
    const uint32_t ms = len < kSeg ? uint32_t(len) : kSeg;
    for (uint32_t e = uint32_t(lane); e < ms; e += kWave) nbr[base + e] = wl[e];
  }
}

static unsigned persistent_grid() {
  static unsigned g = 0;
  if (!g) {
    int dev = 0, ncu = 256;
    if (hipGetDevice(&dev) == hipSuccess) {
      hipDeviceProp_t prop;
      if (hipGetDeviceProperties(&prop, dev) == hipSuccess) ncu = prop.multiProcessorCount;
    }
    g = unsigned(ncu) * 8;  // 8 workgroups of 4 waves per CU
  }
  return g;
}

// How the item kernels split their work: count units of 1/parts of an item's
// words, fill units of `targets` of its targets.  Whole items (one prologue, no
// atomic adds to the counts) where n targets, at about 32 per item, give the waves
// of the grid several units each; below that an item's serial walk would leave
// most of the chip idle.
struct VlSplit {
  uint32_t parts, targets;
};
static VlSplit vl_split(size_t n) {
  VlSplit s{1u, 64u};
  while (s.parts < 8u && n * s.parts < size_t(1) << 18) s.parts *= 2u;
  while (s.targets > 4u && n * (64u / s.targets) < size_t(1) << 20) s.targets /= 2u;
  return s;
}

// One build.  sys/r2_sys: ensemble tables (null: one grid, radius r2_one).
// sync: the counts are read back (entries, mask total), nbr and the mask
// buffer grow to fit (the count pass is repeated if the masks did not fit), and
// e_cap_io becomes max(e_cap_io, E x headroom); without sync nothing is read
// back and the capacities stay (a list that would not fit is flagged).
// rows_mode: 1 = the item kernels (targets in the lanes), 2 = thread per row,
// 0 = by the mean candidates per target, n_part (2B+1)^3 / n_cells: thread per row
// below kRowsBelow, the item kernels from there on (their 64 x 64 tiles need
// candidates to fill).  Rebuilds of 2^20 uniform particles, items against rows, ms:
// at 48 candidates 0.58 / 0.42, 110 1.17 / 0.63, 180 0.61 / 0.55, 222 0.90 / 0.91,
// 359 0.72 / 0.86 (110 and 222 on cells of r/2, the others on cells of r).  Fewer than
// kRowsFrom rows leave most of the chip without a wave, which the item kernels'
// parts fill: 3,000 particles at 124 candidates 0.249 / 0.277, 10,000 at 132 0.219 /
// 0.224, 30,000 at 144 0.286 / 0.258; below kRowsBelowFew candidates rows win there too.
constexpr double kRowsBelow = 200.0, kRowsBelowFew = 64.0;
constexpr size_t kRowsFrom = 16384;
template <class T>
static int vl_build_t(ofp_vl* h, const ofp_cl* cl, const void* pos_v, size_t stride, T r2_one, const void* sys_v,
                      const void* r2_sys_v, bool sync, size_t* e_cap_io, double headroom, unsigned grid,
                      uint64_t* e_count, hipStream_t s, int rows_mode = 0) {
  ClDev c;
  ofp_cl_view v;
  OFP_TRY(ofp_cl_dev_(cl, &c, &v));
  const T* pos = static_cast<const T*>(pos_v);
  const SysGrid<T>* sys = static_cast<const SysGrid<T>*>(sys_v);
  const T* r2_sys = static_cast<const T*>(r2_sys_v);
  const size_t n = c.n_dom;
  OFP_TRY(h->cnt.ensure((n + 1) * 4));
  // behind the n + 1 offsets: mstate[2] (read back with the last offset) and the
  // queue heads of the count and fill passes
  constexpr uint32_t kCtl = 4u + 2u * kQueueWords;
  OFP_TRY(h->off.ensure((n + 1) * 8 + kCtl * 4));
  h->n_state = n;
  auto* mstate = h->off.as<unsigned long long>() + n + 1;
  auto* heads = reinterpret_cast<uint32_t*>(mstate + 2);
  OFP_TRY(h->scantmp.ensure(scan_tmp_bytes(n)));
  OFP_TRY(h->xyz.ensure((v.n_part + kRowAhead) * 3 * sizeof(T)));  // the row count reads whole groups
  const double stencil = std::pow(2.0 * double(c.box_nn) + 1.0, 3.0);
  const double below = n < kRowsFrom ? kRowsBelowFew : kRowsBelow;
  const bool rows = rows_mode == 2 || (rows_mode == 0 && double(v.n_part) * stencil < below * double(v.n_cells));
  if (rows) {
    // no masks: mstate stays 0, nothing to overflow
    k_vl_pack<T><<<grid_for(std::max<size_t>(v.n_part, 4), 256), 256, 0, s>>>(
        pos, stride, uint32_t(v.n_part), h->xyz.as<T>(), nullptr, 0u, reinterpret_cast<uint32_t*>(mstate), 4u);
    OFP_LAUNCHED();
    CellGeom<T> g1;
    for (int k = 0; k < 3; ++k) {
      g1.lo[k] = T(v.lo[k]);
      g1.sp[k] = T(v.spacing[k]);
      g1.divc[k] = v.divc[k];
    }
    const uint32_t* sid = nullptr;
    if (sys) OFP_TRY(cl_sid_sorted(cl, &sid));
    const unsigned g = grid_for(n, 256);
    const size_t n_waves = (n + kWave - 1) / kWave;
    OFP_TRY(h->rmask.ensure(n_waves * kRowWords * kWave * 4 + 4));
    auto launch = [&](auto fill, auto kb, auto seg, size_t e_cap) {
      k_vl_rows<T, decltype(fill)::value, decltype(kb)::value, decltype(seg)::value><<<g, 256, 0, s>>>(
          c, g1, h->xyz.as<T>(), r2_one, sys, r2_sys, sid, h->cnt.as<uint32_t>(), h->rmask.as<uint32_t>(),
          h->off.as<unsigned long long>(), h->off.as<unsigned long long>() + n, (unsigned long long)e_cap,
          h->nbr.as<uint32_t>());
    };
    auto pass = [&](auto fill, auto seg, size_t e_cap) {
      if (c.box_nn == 1)
        launch(fill, std::integral_constant<int, 1>{}, seg, e_cap);
      else if (c.box_nn == 2)
        launch(fill, std::integral_constant<int, 2>{}, seg, e_cap);
      else
        launch(fill, std::integral_constant<int, 3>{}, seg, e_cap);
    };
    using Few = std::integral_constant<uint32_t, kRowSegFew>;
    using Many = std::integral_constant<uint32_t, kRowSegMany>;
    if (n > 0) {
      pass(std::false_type{}, Few{}, 0);
      OFP_LAUNCHED();
    }
    OFP_TRY(scan_excl_u32_to_u64(h->cnt.as<uint32_t>(), h->off.as<uint64_t>(), n, h->scantmp.p, s));
    uint64_t E = 0;
    if (sync) {
      OFP_HIP(hipMemcpyAsync(&E, h->off.as<uint64_t>() + n, 8, hipMemcpyDeviceToHost, s));
      OFP_HIP(hipStreamSynchronize(s));
      const size_t want = size_t(double(E) * (headroom > 1.0 ? headroom : 1.0)) + 1024;
      if (want > *e_cap_io) *e_cap_io = want;
      if (e_count) *e_count = E;
    }
    const size_t e_cap = *e_cap_io;
    OFP_TRY(h->nbr.ensure((e_cap + 4) * 4));  // + 3: the one-lane row kernels read whole groups of four entries
    if (n > 0) {
      const double entries = sync ? double(E) : double(e_cap) / std::max(1.0, headroom);
      if (entries * kWave <= double(kRowSegFew) * double(n))
        pass(std::true_type{}, Few{}, e_cap);
      else
        pass(std::true_type{}, Many{}, e_cap);
      OFP_LAUNCHED();
    }
    h->n_rows = n;
    h->n_entries = sync ? E : 0;
    h->built = true;
    h->symmetric = false;
    h->cl = cl;
    h->rows_path = true;
    return OFP_OK;
  }
  h->rows_path = false;
  const TargetItem* items;
  const uint32_t* n_items;
  uint32_t* counter;  // the cell tiles' queue heads; a list's passes have their own
  size_t cap;
  OFP_TRY(ofp_cl_items_(cl, &items, &n_items, &counter, &cap, s));
  grid = queue_grid(grid ? grid : persistent_grid(), kVlWaves);
  const VlSplit sp = vl_split(n);
  const bool add = sp.parts > 1;  // the parts add their hits to the counts
  k_vl_pack<T><<<grid_for(std::max<size_t>(v.n_part, kCtl), 256), 256, 0, s>>>(
      pos, stride, uint32_t(v.n_part), h->xyz.as<T>(), h->cnt.as<uint32_t>(), add ? uint32_t(n) : 0u,
      reinterpret_cast<uint32_t*>(mstate), kCtl);
  OFP_LAUNCHED();
  OFP_TRY(h->place.ensure((n + 1) * sizeof(ItemPlace)));
  if (n > 0) {
    k_vl_place<T><<<n < size_t(1) << 18 ? grid_for(n, kVlBlock) : 1024u, kVlBlock, 0, s>>>(
        c, sys, items, n_items, mstate, h->place.as<ItemPlace>());
    OFP_LAUNCHED();
  }
  if (h->mask_cap == 0) {
    // a handle's first build: the words its items need (sync), or an estimate that
    // a sizing build corrects
    h->mask_cap = size_t(stencil) * n + 4096;
    if (sync && n > 0) {
      unsigned long long need = 0;
      OFP_HIP(hipMemcpyAsync(&need, mstate, 8, hipMemcpyDeviceToHost, s));
      OFP_HIP(hipStreamSynchronize(s));
      h->mask_cap = size_t(double(need) * (headroom > 1.0 ? headroom : 1.0)) + 4096;
    }
  }
  OFP_TRY(h->masks.ensure(h->mask_cap * 8));
  auto count = [&](bool again) -> int {
    if (n == 0) return OFP_OK;
    if (again) {
      OFP_TRY(fill_u64(reinterpret_cast<uint64_t*>(mstate) + 1, 0, 1, s));
      OFP_TRY(fill_u32(heads, 0, kQueueWords, s));
      if (add) OFP_TRY(fill_u32(h->cnt.as<uint32_t>(), 0, n, s));
    }
    k_vl_count<T><<<grid, kVlBlock, 0, s>>>(c, h->xyz.as<T>(), r2_one, T(v.spacing[0]), T(v.spacing[1]),
                                            T(v.spacing[2]), sys, r2_sys, items, n_items, sp.parts, heads,
                                            h->cnt.as<uint32_t>(), mstate, h->place.as<ItemPlace>(),
                                            h->masks.as<unsigned long long>(), (unsigned long long)h->mask_cap);
    OFP_LAUNCHED();
    return OFP_OK;
  };
  OFP_TRY(count(false));
  OFP_TRY(scan_excl_u32_to_u64(h->cnt.as<uint32_t>(), h->off.as<uint64_t>(), n, h->scantmp.p, s));
  uint64_t E = 0;
  if (sync) {
    unsigned long long back[3] = {0, 0, 0};  // the last offset, mstate
    OFP_HIP(hipMemcpyAsync(back, h->off.as<uint64_t>() + n, sizeof(back), hipMemcpyDeviceToHost, s));
    OFP_HIP(hipStreamSynchronize(s));
    E = back[0];
    if (back[2] != 0) {  // masks did not fit: grow to the exact total (+ headroom) and count again
      h->mask_cap = size_t(double(back[1]) * (headroom > 1.0 ? headroom : 1.0)) + 4096;
      OFP_TRY(h->masks.ensure(h->mask_cap * 8));
      OFP_TRY(count(true));
    }
    const size_t want = size_t(double(E) * (headroom > 1.0 ? headroom : 1.0)) + 1024;
    if (want > *e_cap_io) *e_cap_io = want;
    if (e_count) *e_count = E;
  }
  const size_t e_cap = *e_cap_io;
  OFP_TRY(h->nbr.ensure((e_cap + 4) * 4));  // + 3: the one-lane row kernels read whole groups of four entries
  if (n > 0) {
    k_vl_fill<T><<<grid, kVlBlock, 0, s>>>(c, sys, items, n_items, sp.targets, heads + kQueueWords,
                                           h->off.as<unsigned long long>(), h->off.as<unsigned long long>() + n,
                                           (unsigned long long)e_cap, mstate, h->place.as<ItemPlace>(),
                                           h->masks.as<unsigned long long>(), h->nbr.as<uint32_t>());
    OFP_LAUNCHED();
  }
  h->n_rows = n;
  h->n_entries = sync ? E : 0;  // otherwise on the device: off[n_rows]
  h->built = true;
  h->symmetric = false;
  h->cl = cl;
  return OFP_OK;
}

template <class T>
static int vl_build(ofp_vl* h, const ofp_cl* cl, const void* pos, size_t stride, double r_cut, hipStream_t s) {
  ClDev c;
  ofp_cl_view v;
  OFP_TRY(ofp_cl_dev_(cl, &c, &v));
  for (int k = 0; k < 3; ++k)
    OFP_CHECK(v.spacing[k] * c.box_nn >= r_cut * (1.0 - 1e-6), OFP_E_ARG,
              "stencil %u x spacing %g is smaller than the Verlet radius %g", c.box_nn, v.spacing[k], r_cut);
  const T rc = T(r_cut);
  size_t e_cap = 0;
  return vl_build_t<T>(h, cl, pos, stride, rc * rc, nullptr, nullptr, true, &e_cap, 1.0, 0, nullptr, s);
}

// Symmetric list from a full one: row r keeps the entries whose particle comes
// after the row's own in one total order, so every unordered interaction is kept
// once.  Domain neighbour j: kept iff j > i (sorted indices).  Ghost neighbour
// (ghost k of source particle q, shift id sid): kept iff sorted(q) > i, or
// q is the row's own particle and sid > 13 (shift ids s and -s are id and
// 26 - id, 13 the zero shift, so one image of each pair is kept).  One wave
// per row; kFill = false counts, true writes the kept entries in row order.
template <bool kFill>
__global__ __launch_bounds__(256) void k_vl_sym(const uint64_t* __restrict__ off, const uint32_t* __restrict__ nbr,
                                                uint64_t n_rows, const uint32_t* __restrict__ dom,
                                                const uint32_t* __restrict__ s2n, const uint32_t* __restrict__ n2s,
                                                uint32_t gm, const uint32_t* __restrict__ opid,
                                                const uint32_t* __restrict__ osid, uint32_t* __restrict__ cnt,
                                                const uint64_t* __restrict__ off_sym,
                                                uint32_t* __restrict__ nbr_sym) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t r = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) / kWave;
  if (r >= n_rows) return;  // wave-uniform
  const uint32_t i = dom[r];
  const uint64_t e1 = off[r + 1];
  uint64_t out = kFill ? off_sym[r] : 0;
  uint32_t kept = 0;
  for (uint64_t e0 = off[r]; e0 < e1; e0 += kWave) {
    const uint64_t e = e0 + uint64_t(lane);
    bool keep = false;
    uint32_t j = 0;
    if (e < e1) {
      j = nbr[e];
      const uint32_t o = s2n[j];
      if (o < gm) {
        keep = j > i;
      } else {
        const uint32_t k = o - gm;
        const uint32_t q = n2s[opid[k]];
        keep = q > i || (q == i && osid[k] > 13u);
      }
    }
    const unsigned long long m = __ballot(keep);
    if (kFill && keep)
      nbr_sym[out + __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u))] = j;
    out += uint64_t(__popcll(m));
    kept += uint32_t(__popcll(m));
  }
  if (!kFill && lane == 0) cnt[r] = kept;
}

}  // namespace ofp

using namespace ofp;

int ofp::vl_build_many(ofp_vl* h, const ofp_cl* cl, int dtype, const void* pos_sorted, size_t stride,
                       const void* sys_dev, const void* r2_sys_dev, size_t* e_cap, double headroom, int sizing,
                       unsigned grid, uint64_t* e_count, hipStream_t s, int rows_mode) {
  OFP_CHECK(h && cl && sys_dev && r2_sys_dev && e_cap, OFP_E_ARG, "vl_build_many: null argument");
  if (dtype == OFP_F32)
    return vl_build_t<float>(h, cl, pos_sorted, stride, 0.f, sys_dev, r2_sys_dev, sizing != 0, e_cap, headroom,
                             grid, e_count, s, rows_mode);
  return vl_build_t<double>(h, cl, pos_sorted, stride, 0.0, sys_dev, r2_sys_dev, sizing != 0, e_cap, headroom, grid,
                            e_count, s, rows_mode);
}

int ofp::vl_offsets(const ofp_vl* h, const unsigned long long** off) {
  OFP_CHECK(h && h->built, OFP_E_STATE, "Verlet list not built");
  *off = h->off.as<unsigned long long>();
  return OFP_OK;
}

int ofp::vl_mask_state(const ofp_vl* h, const unsigned long long** mstate) {
  OFP_CHECK(h && h->built, OFP_E_STATE, "Verlet list not built");
  *mstate = h->off.as<unsigned long long>() + h->n_state + 1;
  return OFP_OK;
}

int ofp::vl_set_mask_cap(ofp_vl* h, size_t mask_cap, size_t* old_cap) {
  OFP_CHECK(h && mask_cap > 0, OFP_E_ARG, "vl_set_mask_cap: null handle or zero capacity");
  if (old_cap) *old_cap = h->mask_cap;
  h->masks.release();
  h->mask_cap = mask_cap;
  return h->masks.ensure(mask_cap * 8);
}

extern "C" {

// accessor for the pair kernels (same library)
int ofp_vl_dev_(const ofp_vl* h, const ofp_cl* cl, int symmetric, const unsigned long long** off,
                const uint32_t** nbr) {
  OFP_CHECK(h && h->built, OFP_E_STATE, "Verlet list not built");
  OFP_CHECK(h->cl == cl, OFP_E_STATE, "Verlet list not built from this cell list");
  OFP_CHECK(h->symmetric == (symmetric != 0), OFP_E_ARG,
            symmetric ? "a symmetric pass needs a list from ofp_vl_build_sym"
                      : "a symmetric list holds each interaction once: use the symmetric pair passes");
  *off = h->off.as<unsigned long long>();
  *nbr = h->nbr.as<uint32_t>();
  return OFP_OK;
}

// A device buffer of at least `bytes` owned by the list, for a pair kernel's
// per-particle stream over the rows' entries (rebuilt by each pass that uses it).
int ofp_vl_aux_(const ofp_vl* h, size_t bytes, void** p) {
  OFP_CHECK(h && p, OFP_E_ARG, "ofp_vl_aux_: null argument");
  ofp_vl* m = const_cast<ofp_vl*>(h);
  OFP_TRY(m->aux.ensure(bytes));
  *p = m->aux.p;
  return OFP_OK;
}

// A buffer of the list for the density pass's records, apart from ofp_vl_aux_ so that
// a density and a force pass may run side by side (density passes write the same
// records).  Null where it would have to grow and cannot: in a captured call, or for
// want of memory.
int ofp_vl_rec_(const ofp_vl* h, size_t bytes, void** p, hipStream_t s) {
  OFP_CHECK(h && p, OFP_E_ARG, "ofp_vl_rec_: null argument");
  ofp_vl* m = const_cast<ofp_vl*>(h);
  *p = nullptr;
  std::lock_guard<std::mutex> lock(m->rec_lock);
  if (m->rec.cap < bytes) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    OFP_HIP(hipStreamIsCapturing(s, &cap));
    if (cap != hipStreamCaptureStatusNone) return OFP_OK;
    if (m->rec.ensure(bytes) != OFP_OK) {
      clear_error();
      return OFP_OK;
    }
  }
  *p = m->rec.p;
  return OFP_OK;
}

// Test hook (not in the public header): whether the last build ran the
// thread-per-row kernels (else the item kernels).
int ofp_vl_test_rows_(const ofp_vl* h, int* rows) {
  OFP_CHECK(h && h->built && rows, OFP_E_STATE, "ofp_vl_test_rows_: list not built");
  *rows = h->rows_path ? 1 : 0;
  return OFP_OK;
}

int ofp_vl_create(ofp_vl** h) {
  OFP_CHECK(h, OFP_E_ARG, "ofp_vl_create: null handle pointer");
  *h = new ofp_vl();
  return OFP_OK;
}

int ofp_vl_destroy(ofp_vl* h) {
  if (!h) return OFP_OK;
  DevBuf* bufs[] = {&h->cnt, &h->off, &h->nbr, &h->scantmp, &h->masks, &h->place,
                    &h->xyz, &h->aux, &h->rec, &h->rmask};
  for (DevBuf* b : bufs) b->release();
  delete h;
  return OFP_OK;
}

int ofp_vl_build(ofp_vl* h, const ofp_cl* cl, const void* pos_sorted, size_t stride, double r_cut,
                 void* stream) {
  OFP_CHECK(h && cl, OFP_E_ARG, "ofp_vl_build: null handle");
  OFP_CHECK(r_cut > 0, OFP_E_ARG, "r_cut must be positive");
  ofp_cl_view v;
  OFP_TRY(ofp_cl_get_view(cl, &v));
  OFP_CHECK(v.n_part == 0 || pos_sorted, OFP_E_ARG, "null sorted positions");
  OFP_CHECK(stride >= v.n_part, OFP_E_ARG, "stride < n_part");
  if (v.dtype == OFP_F32) return vl_build<float>(h, cl, pos_sorted, stride, r_cut, as_stream(stream));
  return vl_build<double>(h, cl, pos_sorted, stride, r_cut, as_stream(stream));
}

int ofp_vl_build_sym(ofp_vl* h, const ofp_vl* full, const ofp_ghost* g, void* stream) {
  OFP_CHECK(h && full && g && h != full, OFP_E_ARG, "ofp_vl_build_sym: null or aliased handle");
  OFP_CHECK(full->built && full->cl, OFP_E_STATE, "ofp_vl_build_sym: full list not built");
  ofp_cl_view v;
  OFP_TRY(ofp_cl_get_view(full->cl, &v));
  const uint32_t *pid = nullptr, *sid = nullptr;
  size_t n_ghost = 0;
  OFP_TRY(ofp_ghost_opart(g, &pid, &sid, &n_ghost));
  OFP_CHECK(v.n_part == v.ghost_marker + n_ghost, OFP_E_STATE,
            "ofp_vl_build_sym: the cell list holds %llu particles, the ghost list %zu after %llu",
            (unsigned long long)v.n_part, n_ghost, (unsigned long long)v.ghost_marker);
  OFP_CHECK(full->n_rows == v.ghost_marker, OFP_E_STATE, "ofp_vl_build_sym: rows %llu != domain particles %llu",
            (unsigned long long)full->n_rows, (unsigned long long)v.ghost_marker);
  hipStream_t s = as_stream(stream);
  const size_t n = full->n_rows;
  OFP_TRY(h->cnt.ensure((n + 1) * sizeof(uint32_t)));
  OFP_TRY(h->off.ensure((n + 1) * sizeof(uint64_t)));
  OFP_TRY(h->scantmp.ensure(scan_tmp_bytes(n)));
  const unsigned grid = grid_for(n * kWave, 256);
  if (n > 0) {
    k_vl_sym<false><<<grid, 256, 0, s>>>(full->off.as<uint64_t>(), full->nbr.as<uint32_t>(), n, v.dom_sort_ids,
                                          v.sort_to_nonsort, v.nonsort_to_sort, uint32_t(v.ghost_marker), pid, sid,
                                          h->cnt.as<uint32_t>(), nullptr, nullptr);
    OFP_LAUNCHED();
  }
  OFP_TRY(scan_excl_u32_to_u64(h->cnt.as<uint32_t>(), h->off.as<uint64_t>(), n, h->scantmp.p, s));
  uint64_t E = 0;
  OFP_HIP(hipMemcpyAsync(&E, h->off.as<uint64_t>() + n, 8, hipMemcpyDeviceToHost, s));
  OFP_HIP(hipStreamSynchronize(s));
  OFP_TRY(h->nbr.ensure((E + 1) * sizeof(uint32_t)));
  if (n > 0) {
    k_vl_sym<true><<<grid, 256, 0, s>>>(full->off.as<uint64_t>(), full->nbr.as<uint32_t>(), n, v.dom_sort_ids,
                                         v.sort_to_nonsort, v.nonsort_to_sort, uint32_t(v.ghost_marker), pid, sid,
                                         nullptr, h->off.as<uint64_t>(), h->nbr.as<uint32_t>());
    OFP_LAUNCHED();
  }
  h->n_rows = n;
  h->n_entries = E;
  h->cl = full->cl;
  h->built = true;
  h->symmetric = true;
  return OFP_OK;
}

int ofp_vl_get_view(const ofp_vl* h, ofp_vl_view* v) {
  OFP_CHECK(h && v, OFP_E_ARG, "ofp_vl_get_view: null argument");
  OFP_CHECK(h->built, OFP_E_STATE, "Verlet list not built");
  v->offsets = h->off.as<uint64_t>();
  v->nbr = h->nbr.as<uint32_t>();
  v->n_rows = h->n_rows;
  v->n_entries = h->n_entries;
  return OFP_OK;
}

}  // extern "C"
