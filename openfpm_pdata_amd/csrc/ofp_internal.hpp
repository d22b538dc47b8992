// ofp_internal.hpp -- shared helpers of libofp_nn.so (gfx950 only).
//
// Error reporting, grow-only device buffers, the plane-copy argument block, the
// cell-key formula shared by every kernel, and the wave/block scan primitives.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <limits>
#include <string>

#include "ofp_nn.h"

namespace ofp {

// ------------------------------------------------------------------ errors
int set_error(int code, const char* fmt, ...);
void clear_error();

#define OFP_HIP(call)                                                                    \
  do {                                                                                   \
    hipError_t e_ = (call);                                                              \
    if (e_ != hipSuccess)                                                                \
      return ::ofp::set_error(OFP_E_HIP, "%s:%d %s -> %s", __FILE__, __LINE__, #call,    \
                              hipGetErrorString(e_));                                    \
  } while (0)

#define OFP_CHECK(cond, code, ...)                                                       \
  do {                                                                                   \
    if (!(cond)) return ::ofp::set_error((code), __VA_ARGS__);                           \
  } while (0)

#define OFP_TRY(expr)                                                                    \
  do {                                                                                   \
    int r_ = (expr);                                                                     \
    if (r_ != OFP_OK) return r_;                                                         \
  } while (0)

// Last launch error (a bad launch configuration is reported here).
#define OFP_LAUNCHED() OFP_HIP(hipGetLastError())

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// ------------------------------------------------------- device buffers
// Process-wide count of device-buffer (re)allocations and releases.  A captured
// hipGraph holds buffer addresses and capacities as kernel arguments, so it is
// valid only while this count is unchanged since its capture.
uint64_t realloc_epoch();
void bump_realloc_epoch();

// Device blocks.  A released block is kept for the next allocation of about its
// size on the same device, by any handle: a program that makes its lists anew
// each time its particles moved (getVerletGPU) otherwise spends most of the call
// in hipMalloc and hipFree (LJ over a new list of 1e6 particles: 9.3 -> 1.26 ms a call,
// up to 41 ms before where calls follow each other without a wait).
//  * A block is handed out again only after the device has finished everything
//    submitted before the block's release (one wait covers all earlier releases;
//    hipFree waits the same way), so its former users may have run on any stream and
//    been called from any thread.
//  * Kept blocks are bounded (1/128 of the device's memory; the oldest go first),
//    given back when an allocation fails or the program asks (ofp_trim), and all
//    given back when the library's last handle is destroyed.
int block_alloc(void** p, size_t bytes, size_t* cap, int* dev);
void block_free(void* p, size_t cap, int dev);

// One library handle (a member of every handle type): counts the live ones.
struct HandleLife {
  HandleLife();
  ~HandleLife();
  HandleLife(const HandleLife&) = delete;
  HandleLife& operator=(const HandleLife&) = delete;
};

// Grow-only device allocation owned by a handle.
struct DevBuf {
  void* p = nullptr;
  size_t cap = 0;
  int dev = 0;
  int ensure(size_t bytes) {
    if (bytes <= cap && p) return OFP_OK;
    release();
    bump_realloc_epoch();
    return block_alloc(&p, bytes < 256 ? 256 : bytes, &cap, &dev);
  }
  void release() {
    if (p) {
      bump_realloc_epoch();
      block_free(p, cap, dev);
    }
    p = nullptr;
    cap = 0;
  }
  template <class U>
  U* as() const {
    return reinterpret_cast<U*>(p);
  }
};

// --------------------------------------------------------- plane copies
constexpr int kMaxPlanes = 24;

// Up to kMaxPlanes (src, dst) plane pairs, passed to kernels by value.
struct PlaneArgs {
  uint64_t src[kMaxPlanes];
  uint64_t dst[kMaxPlanes];
  uint32_t esz[kMaxPlanes];
  int n;
};

int make_plane_args(const ofp_plane* in, const ofp_plane* out, int n, PlaneArgs* a);

__device__ __forceinline__ void copy_planes(const PlaneArgs& a, size_t from, size_t to) {
  for (int k = 0; k < a.n; ++k) {
    if (a.esz[k] == 8) {
      reinterpret_cast<uint64_t*>(a.dst[k])[to] = reinterpret_cast<const uint64_t*>(a.src[k])[from];
    } else {
      reinterpret_cast<uint32_t*>(a.dst[k])[to] = reinterpret_cast<const uint32_t*>(a.src[k])[from];
    }
  }
}

// ------------------------------------------------------------ cell key
// Cell grid of CellList_gpu: one padding layer, key_d = floor((x_d - lo_d) /
// spacing_d) + 1 in the position dtype, linearised x-fastest over divc = div + 2.
// Coordinates outside the padded grid are clamped to it.
template <class T>
struct CellGeom {
  T lo[3];
  T sp[3];
  uint32_t divc[3];
};

template <class T>
__host__ __device__ __forceinline__ uint32_t cell_coord(T x, T lo, T sp, uint32_t divc) {
#pragma clang fp contract(off)
  T f = floor((x - lo) / sp);
  if (!(f == f)) return 0u;  // NaN -> padding cell
  if (f < T(-1)) return 0u;
  if (f > T(divc) - T(2)) return divc - 1u;
  return uint32_t(int(f) + 1);
}

template <class T>
__host__ __device__ __forceinline__ uint32_t cell_of(const CellGeom<T>& g, T x, T y, T z,
                                                     uint32_t* cx, uint32_t* cy,
                                                     uint32_t* cz) {
  *cx = cell_coord(x, g.lo[0], g.sp[0], g.divc[0]);
  *cy = cell_coord(y, g.lo[1], g.sp[1], g.divc[1]);
  *cz = cell_coord(z, g.lo[2], g.sp[2], g.divc[2]);
  return *cx + g.divc[0] * (*cy + g.divc[1] * *cz);
}

// One system of an ensemble: its cell grid (same formula as CellGeom) placed at
// global cell ids [cbase, cbase + divc0 divc1 divc2), and the FP64 copies the
// quantised stream is computed from.
template <class T>
struct SysGrid {
  T lo[3];
  T sp[3];
  uint32_t divc[3];
  uint32_t cbase;
  double qlo[3], qsp[3], qinv[3];
  __host__ __device__ CellGeom<T> geom() const {
    CellGeom<T> g;
    for (int k = 0; k < 3; ++k) {
      g.lo[k] = lo[k];
      g.sp[k] = sp[k];
      g.divc[k] = divc[k];
    }
    return g;
  }
};

// Cell key of particle i: one grid, or the grid of the particle's system.
template <class T>
struct KeyOne {
  CellGeom<T> g;
  const T* pos;
  size_t stride;
  __device__ __forceinline__ uint32_t operator()(uint32_t i) const {
    uint32_t cx, cy, cz;
    return cell_of(g, pos[i], pos[stride + i], pos[2 * stride + i], &cx, &cy, &cz);
  }
};

template <class T>
struct KeyMany {
  const SysGrid<T>* sys;
  const uint32_t* sid;  // system of every particle (domain and ghost)
  const T* pos;
  size_t stride;
  __device__ __forceinline__ uint32_t operator()(uint32_t i) const {
    const SysGrid<T>& G = sys[sid[i]];
    uint32_t cx, cy, cz;
    return G.cbase + cell_of(G.geom(), pos[i], pos[stride + i], pos[2 * stride + i], &cx, &cy, &cz);
  }
};

// ------------------------------------------------------------ ghost boxes
// Local ghost boxes of one single-domain periodic system (sorted by shift id)
// and its 27 shift vectors.
constexpr int kMaxBoxes = 26;

// in_lo / in_hi: a region that no box reaches (filt != 0), so a particle
// inside it has no ghost and skips the box tests.  Every box is a slab of the
// boxes' bounding box in some dimension d: it starts at the lower face (then
// in_lo[d] >= its upper bound) or ends at the upper face (then in_hi[d] <= its
// lower bound); a particle with in_lo <= x < in_hi in every dimension is thus
// outside every box.  A box that is a slab in no dimension turns the filter off.
template <class T>
struct GhostBoxes {
  T lo[kMaxBoxes][3];
  T hi[kMaxBoxes][3];
  T shift[27][3];
  uint32_t sv[kMaxBoxes];
  int nb;
  int filt;
  T in_lo[3], in_hi[3];
};

// Box::isInsideNP: half-open on every side.  All six compares, no branches
// between them: a box's bounds are scalar loads, and the loops over the boxes can
// have several boxes' loads in flight.
template <class T>
__device__ __forceinline__ bool inside_np(const GhostBoxes<T>& B, int b, T x, T y, T z) {
  return (x >= B.lo[b][0]) & (x < B.hi[b][0]) & (y >= B.lo[b][1]) & (y < B.hi[b][1]) & (z >= B.lo[b][2]) &
         (z < B.hi[b][2]);
}

// True when (x, y, z) lies in the region no box reaches (no ghost).
template <class T>
__device__ __forceinline__ bool no_box(const GhostBoxes<T>& B, T x, T y, T z) {
  return B.filt && x >= B.in_lo[0] && x < B.in_hi[0] && y >= B.in_lo[1] && y < B.in_hi[1] && z >= B.in_lo[2] &&
         z < B.in_hi[2];
}

template <class T>
inline void fill_boxes(GhostBoxes<T>& B, int nb, const void* blo, const void* bhi, const uint32_t* sv,
                       const void* shifts27) {
  B = GhostBoxes<T>{};
  const T* lo = static_cast<const T*>(blo);
  const T* hi = static_cast<const T*>(bhi);
  const T* sh = static_cast<const T*>(shifts27);
  B.nb = nb;
  for (int b = 0; b < nb; ++b) {
    for (int k = 0; k < 3; ++k) {
      B.lo[b][k] = lo[3 * b + k];
      B.hi[b][k] = hi[3 * b + k];
    }
    B.sv[b] = sv[b];
  }
  for (int s = 0; s < 27; ++s)
    for (int k = 0; k < 3; ++k) B.shift[s][k] = sh[3 * s + k];
  // the region no box reaches
  T dlo[3], dhi[3];
  for (int k = 0; k < 3; ++k) {
    dlo[k] = std::numeric_limits<T>::max();
    dhi[k] = std::numeric_limits<T>::lowest();
    B.in_lo[k] = std::numeric_limits<T>::lowest();
    B.in_hi[k] = std::numeric_limits<T>::max();
  }
  for (int b = 0; b < nb; ++b)
    for (int k = 0; k < 3; ++k) {
      dlo[k] = B.lo[b][k] < dlo[k] ? B.lo[b][k] : dlo[k];
      dhi[k] = B.hi[b][k] > dhi[k] ? B.hi[b][k] : dhi[k];
    }
  B.filt = nb > 0 ? 1 : 0;
  for (int b = 0; b < nb; ++b) {
    bool slab = false;
    for (int k = 0; k < 3; ++k) {
      const bool at_lo = B.lo[b][k] <= dlo[k], at_hi = B.hi[b][k] >= dhi[k];
      if (at_lo && at_hi) continue;  // spans the dimension
      if (at_lo) {
        B.in_lo[k] = B.hi[b][k] > B.in_lo[k] ? B.hi[b][k] : B.in_lo[k];
        slab = true;
      } else if (at_hi) {
        B.in_hi[k] = B.lo[b][k] < B.in_hi[k] ? B.lo[b][k] : B.in_hi[k];
        slab = true;
      }
    }
    if (!slab) B.filt = 0;
  }
}

// distance2 as the reference's Point::distance2: ((dx^2 + dy^2) + dz^2), unfused,
// in the position dtype -- the Verlet test must round exactly like the oracle.
template <class T>
__device__ __forceinline__ T dist2_unfused(T dx, T dy, T dz) {
#pragma clang fp contract(off)
  T r = dx * dx;
  r = r + dy * dy;
  r = r + dz * dz;
  return r;
}

// Cell-relative quantised coordinates of the FP32 pair kernels: per dim,
// u = rint((x - cell_low) / q) with q = spacing / 2^28, stored as
// g = u + c 2^28 (mod 2^32), c the cell coordinate.  The separation of two
// particles whose cells are at most kMaxBoxNN apart is the exact integer
//   d_int = u_q - u_p + (c_q - c_p) 2^28 = int32(g_q - g_p),
// |d_int| < (kMaxBoxNN + 1) 2^28 <= 2^30, so the wrapped subtraction is exact.
constexpr int kQuantBits = 28;
constexpr int kMaxBoxNN = 3;
constexpr int32_t kQuantOne = int32_t(1) << kQuantBits;
// cell coordinates packed in the 4th int: cx | cy << 11 | cz << 22.
__host__ __device__ __forceinline__ int32_t pack_cell(uint32_t cx, uint32_t cy, uint32_t cz) {
  return int32_t(cx | (cy << 11) | (cz << 22));
}

// g = u + c 2^28 (mod 2^32) with u = rint((x - cell_low) / q), u clamped to
// +-2^29 (a particle may drift past its cell between rebuilds).  qlo, qsp:
// cell-list box low corner and spacing, qinv = 2^28 / spacing, cc = cell coords.
__device__ __forceinline__ uint32_t quantise_one(double x, uint32_t cc, double qlo, double qsp, double qinv) {
  const double org = qlo + double(int(cc) - 1) * qsp;
  double u = rint((x - org) * qinv);
  u = u < -536870912.0 ? -536870912.0 : (u > 536870912.0 ? 536870912.0 : u);
  return uint32_t(int(u)) + (cc << kQuantBits);
}
__device__ __forceinline__ int4 quantise(const double xs[3], const uint32_t cc[3], const double qlo[3],
                                         const double qsp[3], const double qinv[3]) {
  uint32_t q[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) q[k] = quantise_one(xs[k], cc[k], qlo[k], qsp[k], qinv[k]);
  return make_int4(int(q[0]), int(q[1]), int(q[2]), pack_cell(cc[0], cc[1], cc[2]));
}

// ------------------------------------------------------------- launch
constexpr int kWave = 64;

inline unsigned grid_for(size_t n, unsigned block) {
  size_t g = (n + block - 1) / block;
  return unsigned(g == 0 ? 1 : g);
}

// ------------------------------------------------------------- scans
// Exclusive scans with the total appended at out[n]: out has n + 1 entries.
// tmp must hold scan_tmp_bytes(n) bytes.  No host synchronisation.
size_t scan_tmp_bytes(size_t n);
int scan_excl_u32(const uint32_t* in, uint32_t* out, size_t n, void* tmp, hipStream_t s);
int scan_excl_u64(const uint64_t* in, uint64_t* out, size_t n, void* tmp, hipStream_t s);
// 32-bit counts widened to 64-bit prefix sums (Verlet offsets can exceed 2^32).
int scan_excl_u32_to_u64(const uint32_t* in, uint64_t* out, size_t n, void* tmp,
                         hipStream_t s);

// Fill helper (graph-safe replacement for hipMemsetAsync).
int fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s);
int fill_u64(uint64_t* p, uint64_t v, size_t n, hipStream_t s);

// Wave-level inclusive scan (64 lanes).
template <class V>
__device__ __forceinline__ V wave_incl_scan(V x) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    V y = __shfl_up(x, d, kWave);
    if (lane >= d) x += y;
  }
  return x;
}

template <class V>
__device__ __forceinline__ V wave_sum(V x) {
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) x += __shfl_xor(x, d, kWave);
  return x;
}

// w * 2 + hit, per lane: the compare's lane mask enters v_addc as its carry-in,
// so appending a hit bit costs one VALU op after the compare.  (s_nop 1: the wait
// states between a write of an SGPR by the vector ALU and a read of it there, which
// the compiler does not add before inline asm.)
__device__ __forceinline__ uint32_t shift_in(uint32_t w, bool hit) {
  const unsigned long long m = __ballot(hit);
  uint32_t r;
  asm("s_nop 1\n\tv_addc_co_u32 %0, vcc, %1, %1, %2" : "=v"(r) : "v"(w), "s"(m) : "vcc");
  return r;
}

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own L2):
// block b runs on XCD b % 8.  This maps the blocks of XCD x onto one contiguous
// range of tiles, so the tiles that run side by side on one XCD are neighbours
// and their writes to adjacent output runs meet in the same L2.
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t xcd_tile(uint32_t b, uint32_t n_blocks) {
  const uint32_t x = b % kXcds, i = b / kXcds;
  const uint32_t per = n_blocks / kXcds, rem = n_blocks % kXcds;
  return x * per + (x < rem ? x : rem) + i;
}

// ---------------------------------------------------------- work queues
// The units of a persistent launch (numbered from 0) lie in kQueues interleaved
// queues, unit u in queue u % kQueues, each with a head of its own cache line;
// a wave draws from the queue of its number until that is empty.  One head for
// all served one draw per ~6 ns, 0.7 ms for 1.2e5 items, longer than the smaller
// passes take (65,536 FP64 particles over cells: 193 -> 99 us).  Interleaving gives every queue units from all over
// the grid, and waves w and w + kQueues, which share one, run on the same XCD.
constexpr uint32_t kQueues = 64;
constexpr uint32_t kQueueStride = 32;  // u32 words between heads
constexpr uint32_t kQueueWords = kQueues * kQueueStride;
// A queue that no wave draws from keeps its units: blocks of such a launch, no fewer
// than bring a wave to every queue (few CUs, as in a partition of the card).
inline unsigned queue_grid(unsigned blocks, unsigned waves_per_block) {
  const unsigned least = (kQueues + waves_per_block - 1) / waves_per_block;
  return blocks < least ? least : blocks;
}
__device__ __forceinline__ uint32_t next_unit(uint32_t* __restrict__ heads) {
  const uint32_t q =
      __builtin_amdgcn_readfirstlane((blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave) % kQueues);
  uint32_t k = 0;
  if ((threadIdx.x & (kWave - 1)) == 0) k = atomicAdd(&heads[q * kQueueStride], 1u);
  return __builtin_amdgcn_readfirstlane(k) * kQueues + q;
}

// ------------------------------------------- distances on the matrix cores
typedef float v16f __attribute__((ext_vector_type(16)));
// Lane halves: {a_lo, b_lo} and {a_hi, b_hi}.
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void swap_halves(float& a, float& b) {
  uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
  swap_halves(x, y);
  a = __uint_as_float(x);
  b = __uint_as_float(y);
}
template <class T>
__device__ __forceinline__ T lane_value(T v, uint32_t lane);
template <>
__device__ __forceinline__ float lane_value<float>(float v, uint32_t lane) {
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}
template <>
__device__ __forceinline__ double lane_value<double>(double v, uint32_t lane) {
  const unsigned long long u = static_cast<unsigned long long>(__double_as_longlong(v));
  const uint32_t lo = __builtin_amdgcn_readlane(uint32_t(u), lane);
  const uint32_t hi = __builtin_amdgcn_readlane(uint32_t(u >> 32), lane);
  return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}


// min(m, |a|, |b|): one instruction, which the compiler has to write itself.  Inline
// asm would hide from it that a and b come out of the matrix cores, and the wait
// states that such a read needs would be missing.
__device__ __forceinline__ float min3_abs(float m, float a, float b) {
  return __builtin_fminf(__builtin_fminf(m, __builtin_fabsf(a)), __builtin_fabsf(b));
}

// Row of this lane in a 32 x 32 product: row 8 q + 4 h + m of a 32-block is candidate
// 16 h + 15 - (4 q + m), so a lane's results i = 4 q + m (rows 8 (i / 4) +
// 4 (lane / 32) + i % 4) are candidates 15 - i of its half.
__device__ __forceinline__ uint32_t matrix_candidate(uint32_t lane) {
  const uint32_t r = lane & 31u;
  return 16u * ((r >> 2) & 1u) + 15u - (4u * (r >> 3) + (r & 3u));
}

// The power of two that brings the largest of a grid's spacings to [1, 2): FP64
// coordinates relative to an origin are multiplied by it before their conversion to
// FP32, so that their squares stay in FP32's range whatever the unit of length
// (squares of 1e-21 or 1e19 do not).  1 for spacings so small or large that FP64
// squares leave FP64's range too (MatrixTest then declines).
__device__ __forceinline__ double matrix_unit(double spx, double spy, double spz) {
  const double m = __builtin_fmax(spx, __builtin_fmax(spy, spz));
  const int e = int((static_cast<unsigned long long>(__double_as_longlong(m)) >> 52) & 0x7FFull) - 1023;
  if (e < -500 || e > 500) return 1.0;
  return __longlong_as_double(static_cast<long long>(1023 - e) << 52);
}

// Candidates that may lie within a cut-off of a wave's targets (target = lane), from
// tiles of the matrix product of (x, y, z, |c|^2) and (-2x, -2y, -2z, 1) on top of
// |t|^2 - r^2 (coordinates relative to a common origin): the sign of 32 x 32 squares
// less r^2.  eps, the bound of the FP32 error: 2^-19 S with S = (R_c + R_t)^2 + r^2, R
// the farthest candidate's and target's distance from the origin.
struct MatrixTest {
  v16f C0, C1;
  float b00, b01, b10, b11, lim_c, eps;
  bool two;  // more than 32 targets
  // (x, y, z): the lane's target; rt2, rc2: squares of the farthest target's and
  // candidate's distance from the origin by the cell geometry; r2: the cut-off's
  // square.  kWide: every pair within the cut-off gets its bit, and a few beyond
  // (r2 + eps).  False if a target lies beyond its bound or is not a number, or if the
  // squares are not FP32's: from 2^-100 to 2^100, eps is normal and no smaller than
  // what the flush of denormals could cost, and no product overflows.
  template <bool kWide>
  __device__ __forceinline__ bool targets(float x, float y, float z, float rt2, float rc2, float r2,
                                          bool more_than_32) {
    eps = (2.05f * (rt2 + rc2) + r2) * 0x1p-19f;  // (a + b)^2 <= 2 a^2 + 2 b^2
    const float tn = __builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z));
    float k0 = tn - (kWide ? r2 + eps : r2), k1 = k0;
    b00 = -2.f * x, b01 = -2.f * y;  // columns of the target halves: k = 0, 1
    swap_halves(b00, b01);
    b10 = -2.f * z, b11 = 1.f;  // k = 2, 3
    swap_halves(b10, b11);
    swap_halves(k0, k1);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      C0[i] = k0;
      C1[i] = k1;
    }
    lim_c = rc2 * 1.01f;
    two = more_than_32;
    return eps >= 0x1p-100f && eps <= 0x1p100f && __ballot(!(tn <= rt2 * 1.01f)) == 0ull;
  }
  // kNear: the smallest |square less r^2| in dm too.
  template <bool kNear>
  __device__ __forceinline__ void tile(float a0, float a1, float b0, float b1, const v16f& K, uint32_t& w,
                                       float& dm) const {
    v16f D = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, K, 0, 0, 0);
    D = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, D, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) w = __builtin_amdgcn_alignbit(w, __float_as_uint(D[i]), 31);
    if constexpr (kNear) {
#pragma unroll
      for (int i = 0; i < 16; i += 2) dm = min3_abs(dm, D[i], D[i + 1]);
    }
  }
  // (x, y, z): candidate matrix_candidate(lane) of the first block in the lower
  // lanes, of the second (if any) in the upper.  Words of the two blocks for target
  // = lane.  False (words void) if a candidate lies beyond the bound or is not a
  // number, or (kNear) some square is too near r^2 for FP32 products to decide.
  template <bool kNear>
  __device__ __forceinline__ bool words(float x, float y, float z, bool second, uint32_t* lo, uint32_t* hi) const {
    const float cn = __builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z));
    if (__ballot(!(cn <= lim_c)) != 0ull) return false;
    float dm = __builtin_inff();
    float a00 = x, a01 = y, a10 = z, a11 = cn;
    swap_halves(a00, a01);  // a00: x, y of the first block; a01: of the second
    swap_halves(a10, a11);
    uint32_t w0 = 0, w1 = 0;
    if (second) {
      tile<kNear>(a01, a11, b00, b10, C0, w0, dm);
      if (two) tile<kNear>(a01, a11, b01, b11, C1, w1, dm);
    }
    tile<kNear>(a00, a10, b00, b10, C0, w0, dm);
    if (two) tile<kNear>(a00, a10, b01, b11, C1, w1, dm);
    // w_k: targets 32 k + lane % 32; of each block candidates 16 h + (0-15), h =
    // lane / 32, the second block's in the high half.  To lane = target: w0 the
    // h = 0 bits, w1 the h = 1 bits
    swap_halves(w0, w1);
    *lo = __builtin_amdgcn_perm(w1, w0, 0x05040100u);
    *hi = __builtin_amdgcn_perm(w1, w0, 0x07060302u);
    if constexpr (kNear) return !__any(dm < eps);
    return true;
  }
};

// ------------------------------------------------------ cell-list view
// What the walkers need of a built cell list, passed to kernels by value.
struct ClDev {
  const unsigned long long* cs;  // packed starts: low = sorted index, high = domain position
  const uint32_t* dom;           // domain sort ids
  const int4* quant;             // cell-relative stream (or null)
  uint32_t divc[3];
  uint32_t n_dom;
  uint32_t box_nn;  // stencil half-width in cells
  uint64_t n_cells;
};

// Target items of the Verlet build: up to 64 consecutive domain rows whose
// cells lie on one x-row of the grid (cells [cx0, cx0 + ncx) at (cy, cz)).
// An item spans at most kItemMaxCells cells (the FP32C cell-tile kernels rely
// on it for their separations).
constexpr uint32_t kItemMaxCells = 8;
struct TargetItem {
  uint32_t row0;
  uint32_t n;
  uint32_t cell0;  // linear id of the first cell
  uint32_t ncx;
};

// Grid, stencil origin and radius of one target item: the cell list's own grid,
// or (ensembles) the grid of the item's system, whose cells start at cbase.
template <class T>
struct ItemGeom {
  uint32_t d0, d1, d2, cbase;
  int cx0, cy, cz, ncx;
  T r2;
};

template <class T>
__device__ __forceinline__ ItemGeom<T> item_geom(const ClDev& c, const TargetItem& ti, T r2,
                                                 const SysGrid<T>* sys, const T* r2_sys) {
  ItemGeom<T> g;
  g.ncx = int(ti.ncx & 0xFFu);
  g.r2 = r2;
  if (sys) {
    const uint32_t s = ti.ncx >> 8;
    g.d0 = sys[s].divc[0];
    g.d1 = sys[s].divc[1];
    g.d2 = sys[s].divc[2];
    g.cbase = sys[s].cbase;
    if (r2_sys) g.r2 = r2_sys[s];
  } else {
    g.d0 = c.divc[0];
    g.d1 = c.divc[1];
    g.d2 = c.divc[2];
    g.cbase = 0;
  }
  const uint32_t cl = ti.cell0 - g.cbase;
  g.cx0 = int(cl % g.d0);
  g.cy = int((cl / g.d0) % g.d1);
  g.cz = int(cl / (g.d0 * g.d1));
  return g;
}

// Run r of the item (traversal order) in lane r < (2B+1)^2: [x, y), empty outside the
// grid and in the other lanes.
template <class T>
__device__ __forceinline__ uint2 lane_run(const ClDev& c, const ItemGeom<T>& G, int lane) {
  const int B = int(c.box_nn), W = 2 * B + 1;
  const int xa = G.cx0 - B > 0 ? G.cx0 - B : 0;
  const int xe = G.cx0 + G.ncx - 1 + B;
  const int xb = xe < int(G.d0) - 1 ? xe : int(G.d0) - 1;
  const int zz = G.cz + lane / W - B, yy = G.cy + lane % W - B;
  if (lane >= W * W || zz < 0 || zz >= int(G.d2) || yy < 0 || yy >= int(G.d1)) return make_uint2(0u, 0u);
  const uint32_t rowc = G.cbase + G.d0 * (uint32_t(yy) + G.d1 * uint32_t(zz));
  return make_uint2(uint32_t(c.cs[rowc + uint32_t(xa)]), uint32_t(c.cs[rowc + uint32_t(xb) + 1]));
}
static_assert((2 * kMaxBoxNN + 1) * (2 * kMaxBoxNN + 1) <= kWave, "one lane per run");

// Ensemble cell lists: one sort over the grids of all systems (global cell ids).
// sys_dev = SysGrid<T>[n_sys], rbase_dev = first global x-row of each system
// (n_sys + 1 entries); both stay owned by the caller.
int cl_create_many(ofp_cl** out, int dtype, uint32_t n_sys, const void* sys_dev, const uint32_t* rbase_dev,
                   uint32_t n_rows, uint64_t n_cells, uint32_t opt);
// sid = system of every particle; the particle count is *n_dev (<= n_cap).
int cl_construct_many(ofp_cl* h, const void* pos, size_t stride, const uint32_t* sid, size_t n_cap,
                      const uint32_t* n_dev, size_t gm, void* pos_sorted, size_t sorted_stride, hipStream_t s);
int cl_sid_sorted(const ofp_cl* h, const uint32_t** sid_sorted);
// Whether the last build found its n particles many and far from cell order, and the
// list holds all scratch for cl_permute (read from the device: synchronous).
int cl_far(const ofp_cl* h, size_t n, bool* far, hipStream_t s);
// out[idx[j]] = in[j] (pa.src 0: in[j] = j), idx a permutation of n, by ranges of
// destinations in the list's scratch; *done = false: not done (captured, no scratch).
int cl_permute(const ofp_cl* h, const uint32_t* idx, size_t n, const PlaneArgs& pa, bool* done, hipStream_t s);
// Ensemble Verlet build (no host synchronisation); the entry count stays on the
// device at offsets[n_rows] and the list is written only if it fits e_cap.
// r2_sys = squared Verlet radius per system in the position dtype.
// sizing != 0: the count is read back (synchronous), *e_cap grows to at least
// count x headroom and nbr with it.  grid = persistent workgroups (0: default).
// rows_mode: 0 = chosen by the mean candidates per target, 1 = the item
// kernels, 2 = thread per row.
int vl_build_many(ofp_vl* h, const ofp_cl* cl, int dtype, const void* pos_sorted, size_t stride,
                  const void* sys_dev, const void* r2_sys_dev, size_t* e_cap, double headroom, int sizing,
                  unsigned grid, uint64_t* e_count, hipStream_t s, int rows_mode);
int vl_offsets(const ofp_vl* h, const unsigned long long** off);
// [0] masks used by the last count pass, [1] != 0 if they did not fit
int vl_mask_state(const ofp_vl* h, const unsigned long long** mstate);
// Replace the mask buffer by one of exactly mask_cap masks (the next build
// that needs more flags the overflow); *old_cap (may be null) = the previous one.
int vl_set_mask_cap(ofp_vl* h, size_t mask_cap, size_t* old_cap);
// Ensemble LJ over the Verlet rows: per-system constant tables (built once by
// lj_tables_many for fixed output arrays), `lanes` lanes per row (8, 16, 32);
// with_u = 0 writes the forces only (energy and n_neigh are left as they are).
// all_cubic (may be null) tells whether every system's cells are cubic; pass it
// to pair_lj_many as `cubic`.
int lj_tables_many(int precision, uint32_t n_sys, const ofp_lj_params* prm, const double* spacing, void* fx,
                   void* fy, void* fz, void* energy, uint32_t* n_neigh, const void* pos_sorted, size_t pstride,
                   int pos_f64, DevBuf* tab, DevBuf* qtab, int* all_cubic);
// Per-system dynamics constants of an ensemble.
template <class T>
struct SysDyn {
  T lo[3], hi[3], L[3];  // periodic box
  T lim2;                // (skin r_cut / 2)^2, rebuild threshold on the squared displacement
  T inv_m;
};

// Velocity Verlet between two force evaluations, for particle i (storage
// order) with force a: the second half kick v += dt/(2m) a of the step that
// ends, the next step's first half kick and its drift x += dt v, and the
// displacement check against the position at the last build (flags[0] |= 1
// when the squared displacement exceeds lim2).
// The arithmetic on values: v, x updated in place; returns whether the
// displacement exceeds the threshold.
// One component; returns the square of its displacement since the build.
template <class T>
__device__ __forceinline__ T kick_kick_drift_one(T& v, T& x, T xb, const SysDyn<T>& D, T dt, T a) {
#pragma clang fp contract(off)
  const T h = (T(0.5) * dt) * D.inv_m;
  const T v1 = v + h * a;  // end of this step
  v = v1 + h * a;          // first half kick of the next
  x = x + dt * v;
  const T r = x - xb;
  return r * r;
}
template <class T>
__device__ __forceinline__ bool kick_kick_drift_v(T (&v)[3], T (&x)[3], const T (&xb)[3], const SysDyn<T>& D, T dt,
                                                  const T (&a)[3]) {
#pragma clang fp contract(off)
  T dd = 0;
#pragma unroll
  for (int d = 0; d < 3; ++d) dd = dd + kick_kick_drift_one<T>(v[d], x[d], xb[d], D, dt, a[d]);
  return dd > D.lim2;
}
// xo: the new position.
template <class T>
__device__ inline void kick_kick_drift(uint32_t i, size_t cap, T* __restrict__ pos, T* __restrict__ vel,
                                       const T* __restrict__ xb, const SysDyn<T>& D, T dt, const T (&a)[3],
                                       uint32_t* __restrict__ flags, T (&xo)[3]) {
  T v[3], b[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    v[d] = vel[d * cap + i];
    xo[d] = pos[d * cap + i];
    b[d] = xb[d * cap + i];
  }
  const bool far = kick_kick_drift_v<T>(v, xo, b, D, dt, a);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    vel[d * cap + i] = v[d];
    pos[d * cap + i] = xo[d];
  }
  if (far) atomicOr(&flags[0], 1u);
}

// The pair kernels that end a step of an ensemble run apply kick_kick_drift to
// the particle of each row as soon as its force is summed (the force is not
// stored).  s2n maps a row's sorted slot p to its storage index; per_sys = 0:
// one system, constants dyn[0] / sys[0], else those of the row's system.  The
// position of before is the sorted one that the pass has read anyway.  The
// new position also goes to slot p of the next step's sorted positions (snext)
// and, for FP32C, of its quantised records (qnext, against the cell of the
// last build, w of the row's current record): the pair pass of the next step
// reads those, while this one reads the current ones, which no lane changes.
// Rows of kSplitLanes lanes and more: lane d takes component d (lanes past 2
// repeat it for the loads), so that a wave's kick is 2 loads and 4 stores in
// place of 6 and 10 of an eighth of the lanes each.
struct NoKick {
  static constexpr bool kOn = false;
  struct Pre {};
  __device__ __forceinline__ uint32_t index(uint32_t) const { return 0u; }
  template <int kLanes>
  __device__ __forceinline__ Pre prefetch(uint32_t, unsigned) const {
    return Pre{};
  }
};
template <class T>
struct StepKick {
  static constexpr bool kOn = true;
  static constexpr int kSplitLanes = 4;
  using Tv = T;
  const uint32_t* s2n;
  T* pos;
  T* vel;
  const T* xb;
  size_t cap;
  const SysDyn<T>* dyn;
  int per_sys;
  T dt;
  uint32_t* flags;
  T* snext;
  int4* qnext;  // null: no quantised records (FP64 pass)
  const SysGrid<T>* sys;
  // the particle's storage index and state (component 0: the lane's own, of a
  // split row), loaded ahead of the kick (the kernels issue these loads before
  // their last gathers, so they wait once)
  struct Pre {
    uint32_t i;
    T v[3], xb[3];
  };
  __device__ __forceinline__ uint32_t index(uint32_t p) const { return s2n[p]; }
  template <int kLanes>
  __device__ __forceinline__ Pre prefetch(uint32_t i, unsigned lane) const {
    Pre q;
    q.i = i;
    if constexpr (kLanes >= kSplitLanes) {
      const size_t at = (lane < 2u ? lane : 2u) * cap + i;
      q.v[0] = vel[at];
      q.xb[0] = xb[at];
    } else {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        q.v[d] = vel[d * cap + i];
        q.xb[d] = xb[d * cap + i];
      }
    }
    return q;
  }
  // One lane for all components.  xp: the current position.
  __device__ __forceinline__ void apply(const Pre& q, uint32_t p, uint32_t sy, int w, const T (&a)[3],
                                        const T (&xp)[3]) const {
    const uint32_t s = per_sys ? sy : 0u;
    T v[3] = {q.v[0], q.v[1], q.v[2]};
    T x[3] = {xp[0], xp[1], xp[2]};
    const bool far = kick_kick_drift_v<T>(v, x, q.xb, dyn[s], dt, a);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      vel[d * cap + q.i] = v[d];
      pos[d * cap + q.i] = x[d];
      snext[d * cap + p] = x[d];
    }
    if (far) atomicOr(&flags[0], 1u);
    if (qnext) {
      const uint32_t cc[3] = {uint32_t(w) & 2047u, (uint32_t(w) >> 11) & 2047u, (uint32_t(w) >> 22) & 1023u};
      const double xs[3] = {double(x[0]), double(x[1]), double(x[2])};
      const SysGrid<T>& G = sys[s];
      qnext[p] = quantise(xs, cc, G.qlo, G.qsp, G.qinv);
    }
  }
  // Lane d of a row for component d, called by every lane of the row; the
  // arithmetic of apply.
  template <int kLanes>
  __device__ __forceinline__ void apply_split(const Pre& q, uint32_t p, uint32_t sy, int w, const T (&a)[3],
                                              const T (&xp)[3], unsigned lane) const {
    const uint32_t s = per_sys ? sy : 0u;
    auto own = [&](auto a0, auto a1, auto a2) { return lane == 0 ? a0 : (lane == 1 ? a1 : a2); };
    T v = q.v[0], x = own(xp[0], xp[1], xp[2]);
    const T rr = kick_kick_drift_one<T>(v, x, q.xb[0], dyn[s], dt, own(a[0], a[1], a[2]));
    T dd = T(0);
#pragma unroll
    for (int d = 0; d < 3; ++d) dd = dd + __shfl(rr, d, kLanes);
    const bool far = dd > dyn[s].lim2;
    if (lane < 3u) {
      vel[lane * cap + q.i] = v;
      pos[lane * cap + q.i] = x;
      snext[lane * cap + p] = x;
    }
    if (far && lane == 0u) atomicOr(&flags[0], 1u);
    if (qnext && lane < 4u) {
      const SysGrid<T>& G = sys[s];
      const uint32_t cc = own(uint32_t(w) & 2047u, (uint32_t(w) >> 11) & 2047u, (uint32_t(w) >> 22) & 1023u);
      const uint32_t g = quantise_one(double(x), cc, own(G.qlo[0], G.qlo[1], G.qlo[2]),
                                      own(G.qsp[0], G.qsp[1], G.qsp[2]), own(G.qinv[0], G.qinv[1], G.qinv[2]));
      // (lane 3: the cell, as it was)
      reinterpret_cast<uint32_t*>(qnext + p)[lane] = lane == 3u ? uint32_t(w) : g;
    }
  }
};

// vl == null: the cell-tile pass over the cell list's item queue (the cells of
// the last build, whose stencil covers r_cut + skin), sysgrid = SysGrid<T>[n_sys]
// of the position dtype.  one_system: every row's constants are the tables' first
// entry.  kick (Verlet rows only, with_u = 0): a StepKick<T>
// of the position dtype, applied to every row in place of storing its force.
// Over Verlet rows, pos_sorted (sorted positions, plane stride `stride`) and
// quant (FP32C records; null: the cell list's own) are what the pass reads.
int pair_lj_many(const ofp_cl* cl, const ofp_vl* vl, int dtype, const void* pos_sorted, size_t stride,
                 int precision, const void* tab, const void* qtab, int lanes, size_t e_cap, int with_u, int cubic,
                 bool one_system, hipStream_t s, const void* sysgrid = nullptr, const void* kick = nullptr,
                 const void* quant = nullptr);

}  // namespace ofp

// Internal cell-list accessor shared by the pair and Verlet sources.
extern "C" int ofp_cl_dev_(const ofp_cl* cl, ofp::ClDev* d, ofp_cl_view* v);
// A device buffer of at least `bytes` owned by the cell list, for the pair
// kernels' per-particle records (its contents belong to the last caller).
extern "C" int ofp_cl_aux_(const ofp_cl* cl, size_t bytes, void** p);
// Work queue of target items of a built cell list (built on first use).
extern "C" int ofp_cl_items_(const ofp_cl* cl, const ofp::TargetItem** items,
                             const uint32_t** n_items, uint32_t** counter, size_t* cap,
                             hipStream_t s);
