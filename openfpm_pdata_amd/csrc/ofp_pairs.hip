// ofp_pairs.hip -- pair-interaction loops (LJ, SPH density, SPH pressure force)
// in plain FP64 and in FP32 on quantised cell-relative coordinates with FP64
// per-particle sums (FP32C), plus the Tait EOS and the FP64 reductions.
//
// Two walkers:
//  * Verlet-driven (vl != NULL): 16 lanes per row, 4 rows per wave; the lanes of
//    a row read 16 consecutive entries (coalesced index stream), gather the
//    neighbours, and the partial sums are combined across the 16 lanes at the
//    end.
//  * cell tiles (vl == NULL): persistent waves over the cell list's target
//    items (up to 64 domain particles of one x-row run of cells, one per lane);
//    the item's (2B+1)^2 stencil x-runs are staged through LDS and every lane
//    tests and evaluates its own target against them.
//
// FP32C arithmetic: x_q - x_p per dim is the exact int32 u_q - u_p + (c_q -
// c_p) 2^28 (quantum q_k = spacing_k / 2^28, see the cell-list build); all
// lengths are in units of q_0, so no rounded scale factor touches a distance.
// Every pair gets the exact square (integer products summed in FP64, split once
// into an FP32 hi/lo pair); the cut-off test compares its hi part.  Physical
// constants in q_0 units that enter a power are carried as (hi, lo) FP32 pairs.
// Each pair's FP32 factor times its FP64 separation (an exact product) is summed
// in FP64 (on this GPU an FP64 add or FMA issues at the rate of an FP32 one, so
// this costs less than a compensated FP32 sum), and the remaining scale factors
// are applied once per particle in FP64.
#include "ofp_internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

extern "C" int ofp_vl_dev_(const ofp_vl* h, const ofp_cl* cl, int symmetric, const unsigned long long** off,
                           const uint32_t** nbr);
extern "C" int ofp_vl_aux_(const ofp_vl* h, size_t bytes, void** p);
extern "C" int ofp_vl_rec_(const ofp_vl* h, size_t bytes, void** p, hipStream_t s);

namespace ofp {

constexpr int kRowLanes = 16;
constexpr int kUnroll = 4;  // Verlet entries in flight per lane

// ----------------------------------------------------------------- walkers
// exact x_q - x_p in quanta from the wrapped per-particle coordinates
__device__ __forceinline__ int wrap_diff(int gq, int gp) { return int(uint32_t(gq) - uint32_t(gp)); }

// ------------------------------------------------------------ cubic spline
// With t = 1 - r/(2h) and u = 1 - r/h, both clamped to [0, 1], the spline without
// its normalisation is W = 2 t^3 - u^3 and dW/dq = 3 (u^2 - t^2): no branch on
// q < 1 or q < 2, and a pair past the cut-off (t = u = 0) adds an exact zero, so
// a pass needs no cut-off decision (both go to zero with the distance to 2h, as
// (1 - r/2h)^3 and (1 - r/2h)^2; a pair that one rounding puts on either side
// adds less than any rounding of the sums).  The particle itself has
// t = u = 1: W = 1.  A force needs dW/dq / r: (u^2 - t^2) / r taken as it stands
// cancels for close pairs (relative error 2e-16 / q); as (u + t) (u - t) / r, where
// (u - t) / r is -1/(2h) below r = h and -t / r from there on, the larger of the two,
// it does not.
// max(min(1 + a b, 1), 0) in one instruction: the FMA's clamp modifier (a NaN
// gives 0 in the clamp mode kernels run in).
__device__ __forceinline__ double sat1(double a, double b) {
  double r;
  asm("v_fma_f64 %0, %1, %2, 1.0 clamp" : "=v"(r) : "v"(a), "s"(b));
  return r;
}
struct Spline {
  double n2, n1;  // -1/(2h), -1/h in the unit of the pass
  __device__ __forceinline__ double t(double r) const { return sat1(r, n2); }
  __device__ __forceinline__ double u(double r) const { return sat1(r, n1); }
  // dW/dq / (3 r), inv = 1 / r
  __device__ __forceinline__ double slope(double r, double inv) const {
    const double t_ = t(r);
    return (u(r) + t_) * __builtin_fmax(n2, -t_ * inv);
  }
};
// sqrt(x) and 1/sqrt(x) of an FP64 pass (x > 0): Goldschmidt's iteration from the
// hardware estimate (2^-23), then one correction of each by its residual, which
// leaves 2^-90 before the last rounding: the IEEE root in each of 2e7 samples, its
// reciprocal as near to the true one as the IEEE quotient (1.49 units in the last place).
__device__ __forceinline__ double sqrt_full(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
__device__ __forceinline__ double sqrt_full(double x, double* inv) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  const double y1 = h + h;
  *inv = __builtin_fma(y1, __builtin_fma(-g, y1, 1.0), y1);
  return g;
}

// -------------------------------------------------- FP64 plain physics
// kU: also the per-particle energy and neighbour count (en / nn); the forms
// share one layout, so one constant table serves both.
template <bool kU>
struct LJ64T {
  static constexpr bool kSmooth = false;
  double rc2, sig2, eps24, eps4;
  double* fx;
  double* fy;
  double* fz;
  double* en;
  uint32_t* nn;
  struct St {
    double fx = 0, fy = 0, fz = 0, u = 0;
    uint32_t n = 0;
  };
  __device__ void start(St&, uint32_t) const {}
  __device__ __forceinline__ double aux(uint32_t) const { return 0.0; }
  __device__ __forceinline__ void pair(St& s, double, double rx, double ry, double rz, double d2) const {
    if constexpr (kU) ++s.n;
    if (d2 == 0.0) return;
    double inv = 1.0 / d2;
    double s2 = sig2 * inv;
    double s6 = s2 * s2 * s2;
    double s12 = s6 * s6;
    double f = eps24 * (2.0 * s12 - s6) * inv;
    s.fx += f * rx;
    s.fy += f * ry;
    s.fz += f * rz;
    if constexpr (kU) s.u += eps4 * (s12 - s6);
  }
  __device__ __forceinline__ void reduce(St& s, int w) const {
    for (int d = w / 2; d > 0; d >>= 1) {
      s.fx += __shfl_xor(s.fx, d, w);
      s.fy += __shfl_xor(s.fy, d, w);
      s.fz += __shfl_xor(s.fz, d, w);
      if constexpr (kU) {
        s.u += __shfl_xor(s.u, d, w);
        s.n += __shfl_xor(s.n, d, w);
      }
    }
  }
  // the force finish stores, in the position dtype (what a kick reads back)
  template <class T>
  __device__ __forceinline__ void force_as(const St& s, T (&a)[3]) const {
    a[0] = T(s.fx);
    a[1] = T(s.fy);
    a[2] = T(s.fz);
  }
  __device__ __forceinline__ void finish(const St& s, uint32_t p) const {
    if (fx) {
      fx[p] = s.fx;
      fy[p] = s.fy;
      fz[p] = s.fz;
    }
    if constexpr (kU) {
      if (en) en[p] = s.u;
      if (nn) nn[p] = s.n;
    }
  }
};
using LJ64 = LJ64T<true>;

// SPH physics (both forms): kSmooth, pairs that vanish at the cut-off; pair()
// takes every pair of the candidates, the particle itself included.
struct Dens64 {
  static constexpr bool kSmooth = true;
  static constexpr bool kAux = false;
  double rc2;   // the cell walk's own test
  Spline sp;
  double sk_m;  // m / (pi h^3)
  double* rho;
  struct St {
    double t3 = 0, u3 = 0;
  };
  __device__ void start(St&, uint32_t) const {}
  __device__ __forceinline__ double aux(uint32_t) const { return 0.0; }
  __device__ __forceinline__ void pair(St& s, double, double, double, double, double d2) const {
    const double r = sqrt_full(d2);
    const double t = sp.t(r), u = sp.u(r);
    s.t3 = __builtin_fma(t * t, t, s.t3);
    s.u3 = __builtin_fma(u * u, u, s.u3);
  }
  __device__ __forceinline__ void reduce(St& s, int w) const {
    for (int d = w / 2; d > 0; d >>= 1) {
      s.t3 += __shfl_xor(s.t3, d, w);
      s.u3 += __shfl_xor(s.u3, d, w);
    }
  }
  // self: W(0) of the particle itself where its candidates did not hold it
  __device__ __forceinline__ void finish(const St& s, uint32_t p, double self) const {
    rho[p] = sk_m * (__builtin_fma(2.0, s.t3, -s.u3) + self);
  }
};

struct Force64 {
  static constexpr bool kSmooth = true;
  static constexpr bool kAux = true;
  double rc2;
  Spline sp;
  double sd_m;          // 3 m / (pi h^4)
  const double* pterm;  // P / rho^2 per sorted particle
  double* fx;
  double* fy;
  double* fz;
  struct St {
    double fx = 0, fy = 0, fz = 0, pi = 0;
  };
  __device__ __forceinline__ void start(St& s, uint32_t p) const { s.pi = pterm[p]; }
  __device__ __forceinline__ double aux(uint32_t j) const { return pterm[j]; }
  __device__ __forceinline__ void pair(St& s, double pj, double rx, double ry, double rz, double d2) const {
    double inv;
    const double r = sqrt_full(d2, &inv);
    const double c = (s.pi + pj) * sp.slope(r, inv);
    s.fx = __builtin_fma(c, rx, s.fx);
    s.fy = __builtin_fma(c, ry, s.fy);
    s.fz = __builtin_fma(c, rz, s.fz);
  }
  __device__ __forceinline__ void reduce(St& s, int w) const {
    for (int d = w / 2; d > 0; d >>= 1) {
      s.fx += __shfl_xor(s.fx, d, w);
      s.fy += __shfl_xor(s.fy, d, w);
      s.fz += __shfl_xor(s.fz, d, w);
    }
  }
  __device__ __forceinline__ void finish(const St& s, uint32_t p, double) const {
    fx[p] = -sd_m * s.fx;
    fy[p] = -sd_m * s.fy;
    fz[p] = -sd_m * s.fz;
  }
};

// ------------------------------------------------- FP32C physics (q_0 units)
// FP32 storage (16-byte quantised records, FP32 P/rho^2 and forces); the pair
// is evaluated in FP64 from the FP64 separation.  On this GPU, with packed FP32
// off, an FP64 add, multiply or FMA issues at the rate of an FP32 one, and the
// FP64 reciprocal / reciprocal square root estimates at half the rate of the
// FP32 ones, so one FP64 Newton step on the estimate replaces the (hi, lo) FP32
// pairs an FP32 evaluation needed to stay near 1e-6: the pair costs about the
// same time (the kernels are bound by their gathers), and the error left is
// that of the FP32 inputs (P/rho^2, the quantum), near 1e-7 or below.
//
// One pair in q_0 units: x_p - x_q and its square in FP64 (integer components;
// for non-cubic cells times the FP64 axis ratio), and the square rounded to
// FP32 (d2), on which the cut-off test decides.
struct QPair {
  double rx, ry, rz, r2;
  float d2;
};

// 1/x and 1/sqrt(x) (x > 0) from the hardware estimates (about 2^-23 relative)
// and one Newton step each (about 2^-46).
__device__ __forceinline__ double rcp_refined(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = __builtin_fma(-x, y, 1.0);
  return __builtin_fma(y, e, y);
}
__device__ __forceinline__ double rsqrt_refined(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-x * y, y, 1.0);  // 1 - x y^2
  return __builtin_fma(0.5 * y, e, y);
}
// sqrt(x) on the same terms
__device__ __forceinline__ double sqrt_refined(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double s = x * y;
  return __builtin_fma(0.5 * s, __builtin_fma(-s, y, 1.0), s);
}

// Butterfly sum over groups of w lanes (every lane of a group ends with the
// same value: FP addition is commutative).
__device__ __forceinline__ void lane_sum(double& a, int w) {
  for (int d = w / 2; d > 0; d >>= 1) a += __shfl_xor(a, d, w);
}

// Cut-off decisions identical to the FP64 form.  The quantised square differs
// from the exact one by at most 2 sqrt(3) q_m r + 3 q_m^2 (q_m = the largest
// quantum, in q_0 units) and is then rounded to FP32, so a pair whose FP32
// square lies in [lo2, hi2) around the cut-off is decided again as the FP64
// kernels decide it: x_p - x_q per component in FP64 from the stored (sorted)
// positions, the squares summed unfused, compared with the FP64 form's r_c^2.
// Outside the band both forms agree.  A few pairs per million fall in the band,
// so the divergent path costs nothing measurable.
struct ExactCut {
  const void* pos;  // sorted positions, 3 planes pstride apart
  size_t pstride;
  int pos_f64;
  float lo2, hi2;  // band of the FP32 square (q_0 units)
  double rc2;      // r_c^2 in position units, the FP64 form's constant
  __device__ __forceinline__ bool in_band(float d2) const { return d2 >= lo2 && d2 < hi2; }
  __device__ bool hit(uint32_t p, uint32_t j) const {
    double dx, dy, dz;
    if (pos_f64) {
      const double* P = static_cast<const double*>(pos);
      dx = P[p] - P[j];
      dy = P[pstride + p] - P[pstride + j];
      dz = P[2 * pstride + p] - P[2 * pstride + j];
    } else {
      const float* P = static_cast<const float*>(pos);
      dx = double(P[p]) - double(P[j]);
      dy = double(P[pstride + p]) - double(P[pstride + j]);
      dz = double(P[2 * pstride + p]) - double(P[2 * pstride + j]);
    }
    return dist2_unfused<double>(dx, dy, dz) < rc2;
  }
  // the same decision from the two stored positions (dtype T), loaded by the caller
  template <class T>
  __device__ __forceinline__ bool hit_from(const T (&a)[3], const T (&b)[3]) const {
    const double dx = double(a[0]) - double(b[0]);
    const double dy = double(a[1]) - double(b[1]);
    const double dz = double(a[2]) - double(b[2]);
    return dist2_unfused<double>(dx, dy, dz) < rc2;
  }
};

// kU as for LJ64T.
template <bool kU>
struct LJ32T {
  static constexpr bool kSmooth = false;
  static constexpr bool kAuxInQuant = false;
  float rc2;      // (r_c / q0)^2
  double sig2;    // (sigma / q0)^2
  double fscale;  // 24 eps / q0
  double uscale;  // 4 eps
  float* fx;
  float* fy;
  float* fz;
  float* en;
  uint32_t* nn;
  ExactCut xc;
  // Close pairs (r < sigma, where the repulsion is steep and strong): the
  // quantised separation (error < 1 quantum) is replaced by the FP64
  // difference of the stored positions, since the r^-13 repulsion multiplies
  // its relative error by 13 and a pair force there exceeds 24 eps / sigma.
  double inv_q0;  // 1 / q0
  float close2;   // (sigma / q0)^2
  struct St {
    double fx = 0, fy = 0, fz = 0, u = 0;
    uint32_t n = 0;
  };
  // The refined separation from the two stored positions, loaded by the
  // caller (same arithmetic as refine), so that a group of pairs can issue all
  // its loads before the first use.
  template <class T>
  __device__ __forceinline__ void refine_from(QPair& r, const T (&a)[3], const T (&b)[3]) const {
    const double dx = (double(a[0]) - double(b[0])) * inv_q0;
    const double dy = (double(a[1]) - double(b[1])) * inv_q0;
    const double dz = (double(a[2]) - double(b[2])) * inv_q0;
    r.rx = dx;
    r.ry = dy;
    r.rz = dz;
    r.r2 = __builtin_fma(dx, dx, __builtin_fma(dy, dy, dz * dz));
  }
  __device__ void refine(QPair& r, uint32_t p, uint32_t j) const {
    double dx, dy, dz;
    if (xc.pos_f64) {
      const double* P = static_cast<const double*>(xc.pos);
      dx = P[p] - P[j];
      dy = P[xc.pstride + p] - P[xc.pstride + j];
      dz = P[2 * xc.pstride + p] - P[2 * xc.pstride + j];
    } else {
      const float* P = static_cast<const float*>(xc.pos);
      dx = double(P[p]) - double(P[j]);
      dy = double(P[xc.pstride + p]) - double(P[xc.pstride + j]);
      dz = double(P[2 * xc.pstride + p]) - double(P[2 * xc.pstride + j]);
    }
    dx *= inv_q0;
    dy *= inv_q0;
    dz *= inv_q0;
    r.rx = dx;
    r.ry = dy;
    r.rz = dz;
    r.r2 = __builtin_fma(dx, dx, __builtin_fma(dy, dy, dz * dz));
  }
  __device__ void start(St&, uint32_t) const {}
  __device__ __forceinline__ float aux(uint32_t) const { return 0.f; }
  // (sigma/r)^6 and ^12 and the force factor (2 (sigma/r)^12 - (sigma/r)^6) / r^2
  // from 1/r^2 in FP64.
  __device__ __forceinline__ void eval(double r2, double* f, double* u) const {
    const double inv = rcp_refined(r2);
    const double s2 = sig2 * inv;
    const double s6 = s2 * s2 * s2;
    const double s12 = s6 * s6;
    *f = __builtin_fma(2.0, s12, -s6) * inv;
    *u = s12 - s6;
  }
  __device__ __forceinline__ void pair(St& s, float, const QPair& r) const {
    if constexpr (kU) ++s.n;
    if (r.r2 == 0.0) return;
    double f, u;
    eval(r.r2, &f, &u);
    s.fx = __builtin_fma(f, r.rx, s.fx);
    s.fy = __builtin_fma(f, r.ry, s.fy);
    s.fz = __builtin_fma(f, r.rz, s.fz);
    if constexpr (kU) s.u += u;
  }
  __device__ __forceinline__ void pair_masked(St& s, float, const QPair& r, bool hit) const {
    if constexpr (kU) s.n += hit ? 1u : 0u;
    const bool live = hit && r.r2 != 0.0;
    // a miss is evaluated at r = sigma (every power finite) and weighted by 0
    // (a product rather than a select keeps the evaluation branch-free)
    double f, u;
    eval(live ? r.r2 : sig2, &f, &u);
    const double m = live ? 1.0 : 0.0;
    f *= m;
    s.fx = __builtin_fma(f, r.rx, s.fx);
    s.fy = __builtin_fma(f, r.ry, s.fy);
    s.fz = __builtin_fma(f, r.rz, s.fz);
    if constexpr (kU) s.u = __builtin_fma(u, m, s.u);
  }
  __device__ __forceinline__ void reduce(St& s, int w) const {
    lane_sum(s.fx, w);
    lane_sum(s.fy, w);
    lane_sum(s.fz, w);
    if constexpr (kU) {
      lane_sum(s.u, w);
      for (int d = w / 2; d > 0; d >>= 1) s.n += __shfl_xor(s.n, d, w);
    }
  }
  template <class T>
  __device__ __forceinline__ void force_as(const St& s, T (&a)[3]) const {
    a[0] = T(float(fscale * s.fx));
    a[1] = T(float(fscale * s.fy));
    a[2] = T(float(fscale * s.fz));
  }
  __device__ __forceinline__ void finish(const St& s, uint32_t p) const {
    if (fx) {
      fx[p] = float(fscale * s.fx);
      fy[p] = float(fscale * s.fy);
      fz[p] = float(fscale * s.fz);
    }
    if constexpr (kU) {
      if (en) en[p] = float(uscale * s.u);
      if (nn) nn[p] = s.n;
    }
  }
};
using LJ32 = LJ32T<true>;

// pair(): the separation x_q - x_p and its square (> 0) in q_0 units.
struct Dens32 {
  static constexpr bool kSmooth = true;
  static constexpr bool kAuxInQuant = false;
  float rc2;    // (2h / q0)^2, the cell walk's pre-test
  Spline sp;
  double sk_m;  // m / (pi h^3)
  double* rho;  // output in FP64
  struct St {
    double t3 = 0, u3 = 0;
  };
  __device__ void start(St&, uint32_t) const {}
  __device__ __forceinline__ float aux(uint32_t) const { return 0.f; }
  __device__ __forceinline__ void pair(St& s, float, double, double, double, double r2) const {
    const double r = sqrt_refined(r2);
    const double t = sp.t(r), u = sp.u(r);
    s.t3 = __builtin_fma(t * t, t, s.t3);
    s.u3 = __builtin_fma(u * u, u, s.u3);
  }
  __device__ __forceinline__ void reduce(St& s, int w) const {
    lane_sum(s.t3, w);
    lane_sum(s.u3, w);
  }
  __device__ __forceinline__ void finish(const St& s, uint32_t p, double self) const {
    rho[p] = sk_m * (__builtin_fma(2.0, s.t3, -s.u3) + self);
  }
};

struct Force32 {
  static constexpr bool kSmooth = true;
  // the passes gather (q_x, q_y, q_z, pterm) as one 16-byte record per pair
  static constexpr bool kAuxInQuant = true;
  float rc2;
  double cut2;  // (2h / q0)^2
  Spline sp;
  double fscale;       // 3 m / (pi h^4): of the separation x_q - x_p
  const float* pterm;  // P / rho^2
  float* fx;
  float* fy;
  float* fz;
  struct St {
    double fx = 0, fy = 0, fz = 0;
    double pi = 0;
  };
  __device__ __forceinline__ void start(St& s, uint32_t p) const { s.pi = pterm[p]; }
  __device__ __forceinline__ float aux(uint32_t j) const { return pterm[j]; }
  // (P_p/rho_p^2 + P_q/rho_q^2) dW/dq / (3 r); coincident particles have no
  // separation to multiply it with
  __device__ __forceinline__ void pair(St& s, float pj, double dx, double dy, double dz, double r2) const {
    const double inv = rsqrt_refined(r2);
    const double r = r2 * inv;
    const double c = (s.pi + double(pj)) * sp.slope(r, inv);
    s.fx = __builtin_fma(c, dx, s.fx);
    s.fy = __builtin_fma(c, dy, s.fy);
    s.fz = __builtin_fma(c, dz, s.fz);
  }
  __device__ __forceinline__ void reduce(St& s, int w) const {
    lane_sum(s.fx, w);
    lane_sum(s.fy, w);
    lane_sum(s.fz, w);
  }
  __device__ __forceinline__ void finish(const St& s, uint32_t p, double) const {
    fx[p] = float(fscale * s.fx);
    fy[p] = float(fscale * s.fy);
    fz[p] = float(fscale * s.fz);
  }
};

// x_p - x_q in q_0 units; exact squared distance for hits.
struct QGeom {
  float ry, rz;       // q_y / q_0, q_z / q_0 (1 for cubic cells)
  double ryd, rzd;
};

// A pair gets x_p - x_q in FP64 (integer components; for non-cubic cells times
// the FP64 axis ratio, rounded once) and its square in FP64 (products summed
// with FMAs; the (sigma/r)^12 chain needs the exact square); the cut-off test compares
// the square rounded to FP32, and a square in the ExactCut band is decided on the
// stored positions as the FP64 form decides.
// The cell walk first drops candidates whose FP32 square exceeds the cut-off by
// more than any rounding and the band (pre_cut), then decides like the Verlet
// rows.
// kCubic: cubic cells (q_y = q_z = q_0), no component scaling.
// The quantised separation of a hit closer than close2 is replaced by the exact one
// from the stored positions.
constexpr float kPreCut = 1.0f + 1.0f / 65536.0f;

template <bool kCubic>
__device__ __forceinline__ QPair quant_geom(const QGeom& qg, int ix, int iy, int iz, float* d2f) {
  QPair p;
  const double dx = double(ix);
  const double dy = kCubic ? double(iy) : double(iy) * qg.ryd;
  const double dz = kCubic ? double(iz) : double(iz) * qg.rzd;
  const double r2 = __builtin_fma(dx, dx, __builtin_fma(dy, dy, dz * dz));
  p.rx = -dx;
  p.ry = -dy;
  p.rz = -dz;
  p.r2 = r2;
  p.d2 = float(r2);
  *d2f = p.d2;
  return p;
}
// kSmooth physics: x_q - x_p and its square in FP64 from the integer separation.
// The square of coincident particles is kTiny instead of 0 (every other one is
// an integer, or for non-cubic cells at least the squared axis ratio, to which
// adding kTiny changes nothing), so 1/r stays finite.
constexpr double kTiny = 1e-30;
// careful (wave-uniform): the pairs may come with values that are infinite or no
// number, so the particle itself and pairs beyond the cut-off, which the candidate
// masks let through, are left out rather than multiplied by zero.  (Deciding every
// pair: 16 us of the 400 of a force pass of 1.09e6 particles on a lattice, this 4.)
template <class Ph, bool kCubic>
__device__ __forceinline__ void smooth_pair(const Ph& ph, typename Ph::St& st, const QGeom& qg, float aux, int ix,
                                            int iy, int iz, bool careful) {
  const double dx = double(ix);
  const double dy = kCubic ? double(iy) : double(iy) * qg.ryd;
  const double dz = kCubic ? double(iz) : double(iz) * qg.rzd;
  const double r2 = __builtin_fma(dx, dx, __builtin_fma(dy, dy, __builtin_fma(dz, dz, kTiny)));
  if constexpr (Ph::kAuxInQuant) {
    if (careful && ((ix | iy | iz) == 0 || r2 >= ph.cut2)) return;
  }
  ph.pair(st, aux, dx, dy, dz, r2);
}

template <class Ph>
__device__ __forceinline__ void refine_close(const Ph& ph, QPair& p, bool hit, uint32_t ip, uint32_t jq) {
  if (hit && p.d2 < ph.close2) ph.refine(p, ip, jq);  // rare, divergent
}

template <class Ph, bool kCubic>
__device__ __forceinline__ void quant_pair(const Ph& ph, typename Ph::St& st, const QGeom& qg, float aux,
                                           int ix, int iy, int iz, uint32_t ip, uint32_t jq) {
  const float fx = float(ix);
  const float fy = kCubic ? float(iy) : float(iy) * qg.ry;
  const float fz = kCubic ? float(iz) : float(iz) * qg.rz;
  const float pre = __builtin_fmaf(fx, fx, __builtin_fmaf(fy, fy, fz * fz));
  if (pre < ph.rc2 * kPreCut) {
    float d2;
    QPair p = quant_geom<kCubic>(qg, ix, iy, iz, &d2);
    bool hit = d2 < ph.rc2;
    if (ph.xc.in_band(d2)) hit = ph.xc.hit(ip, jq);  // rare, divergent
    if (hit) {
      refine_close(ph, p, true, ip, jq);
      ph.pair(st, aux, p);
    }
  }
}

// Branch-free variant for Verlet rows (most entries are hits): the pair is
// evaluated for every entry with a safe distance and its contributions are
// multiplied by the hit mask.  j == p enters with hit = false.
template <class Ph, bool kCubic>
__device__ __forceinline__ void quant_pair_masked(const Ph& ph, typename Ph::St& st, const QGeom& qg, float aux,
                                                  int ix, int iy, int iz, bool not_self, uint32_t ip,
                                                  uint32_t jq) {
  float d2;
  QPair p = quant_geom<kCubic>(qg, ix, iy, iz, &d2);
  bool hit = not_self && d2 < ph.rc2;
  if (not_self && ph.xc.in_band(d2)) hit = ph.xc.hit(ip, jq);  // rare, divergent
  refine_close(ph, p, hit, ip, jq);
  ph.pair_masked(st, aux, p, hit);
}

// Four Verlet entries of one row, for physics with close-pair refinement, in
// three passes: the decisions of all four from their quantised separations
// (hit, in the ExactCut band, possibly close); the stored positions (sref,
// dtype T, the positions the records were made from) of the entries that need
// them gathered together, so a group waits for
// memory once rather than once per such pair; then each entry decided and
// evaluated in turn, its separation recomputed from the records (only the
// decisions and the gathered positions stay live across the passes, which
// keeps down the register count, and with it the waves per SIMD that hide the
// gathers).  Same results as four quant_pair_masked calls.  pp: the row
// particle's stored position.
template <class T, class Ph, bool kCubic>
__device__ __forceinline__ void quant_group_masked(const Ph& ph, typename Ph::St& st, const QGeom& qg,
                                                   const float (&aux)[4], const int4 (&Q)[4], const int4& P,
                                                   const uint32_t (&j)[4], const bool (&not_self)[4],
                                                   const T (&pp)[3], const T* __restrict__ sref, size_t sstride) {
  bool hit[4], band[4], need[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    float d2;
    const QPair r =
        quant_geom<kCubic>(qg, wrap_diff(Q[u].x, P.x), wrap_diff(Q[u].y, P.y), wrap_diff(Q[u].z, P.z), &d2);
    hit[u] = not_self[u] && d2 < ph.rc2;
    band[u] = not_self[u] && ph.xc.in_band(d2);
    // close pairs are refined; a band pair's final decision may still be a hit
    need[u] = band[u] || (hit[u] && r.d2 < ph.close2);
  }
  T xq[4][3];
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (need[u]) {
      xq[u][0] = sref[j[u]];
      xq[u][1] = sref[sstride + j[u]];
      xq[u][2] = sref[2 * sstride + j[u]];
    }
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (band[u]) hit[u] = ph.xc.hit_from(pp, xq[u]);  // rare
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    int ix = wrap_diff(Q[u].x, P.x), iy = wrap_diff(Q[u].y, P.y), iz = wrap_diff(Q[u].z, P.z);
    // fresh values for the compiler: the separation is recomputed here rather
    // than kept from the first pass
    asm volatile("" : "+v"(ix), "+v"(iy), "+v"(iz));
    float d2;
    QPair r = quant_geom<kCubic>(qg, ix, iy, iz, &d2);
    if (hit[u] && r.d2 < ph.close2) ph.refine_from(r, pp, xq[u]);
    ph.pair_masked(st, aux[u], r, hit[u]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// One lane per row: close pairs are not refined inside the loop (where one
// lane's close pair costs every lane of the wave a second memory round trip
// per group) but set aside, up to kDefer of them, and evaluated after the
// row's last group, their stored positions gathered together.  A row with more
// close pairs refines the others in place.  The row's sum takes its terms in
// another order than quant_group_masked's; the pairs and their separations
// are the same.
constexpr int kDefer = 4;
struct Deferred {
  uint32_t j[kDefer];
  float a[kDefer];
  int n = 0;
  // j[0] is the newest (a shift register: no dynamic indexing of registers)
  __device__ __forceinline__ void push(uint32_t jj, float aa) {
#pragma unroll
    for (int k = kDefer - 1; k > 0; --k) {
      j[k] = j[k - 1];
      a[k] = a[k - 1];
    }
    j[0] = jj;
    a[0] = aa;
    ++n;
  }
};

template <class T, class Ph, bool kCubic>
__device__ __forceinline__ void quant_group_defer(const Ph& ph, typename Ph::St& st, const QGeom& qg,
                                                  const float (&aux)[4], const int4 (&Q)[4], const int4& P,
                                                  const uint32_t (&j)[4], const bool (&not_self)[4],
                                                  const T (&pp)[3], const T* __restrict__ sref, size_t sstride,
                                                  Deferred& df) {
  bool hit[4], need[4], close[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    float d2;
    const QPair r =
        quant_geom<kCubic>(qg, wrap_diff(Q[u].x, P.x), wrap_diff(Q[u].y, P.y), wrap_diff(Q[u].z, P.z), &d2);
    hit[u] = not_self[u] && d2 < ph.rc2;
    const bool band = not_self[u] && ph.xc.in_band(d2);
    close[u] = hit[u] && !band && r.d2 < ph.close2;
    if (close[u] && df.n < kDefer) {
      df.push(j[u], aux[u]);
      hit[u] = false;
      close[u] = false;
    }
    need[u] = band || close[u];  // rare: the band, or a row past kDefer close pairs
  }
  T xq[4][3];
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (need[u]) {
      xq[u][0] = sref[j[u]];
      xq[u][1] = sref[sstride + j[u]];
      xq[u][2] = sref[2 * sstride + j[u]];
      if (!close[u]) hit[u] = ph.xc.hit_from(pp, xq[u]);  // the band decision
    }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    int ix = wrap_diff(Q[u].x, P.x), iy = wrap_diff(Q[u].y, P.y), iz = wrap_diff(Q[u].z, P.z);
    asm volatile("" : "+v"(ix), "+v"(iy), "+v"(iz));  // recomputed, not kept from the first pass
    float d2;
    QPair r = quant_geom<kCubic>(qg, ix, iy, iz, &d2);
    if (close[u]) ph.refine_from(r, pp, xq[u]);
    ph.pair_masked(st, aux[u], r, hit[u]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The set-aside close pairs of a row: positions gathered together, then each
// evaluated from the refined separation.
template <class T, class Ph>
__device__ __forceinline__ void flush_deferred(const Ph& ph, typename Ph::St& st, const T (&pp)[3],
                                               const T* __restrict__ sref, size_t sstride, const Deferred& df) {
  if (df.n == 0) return;
  T xq[kDefer][3];
#pragma unroll
  for (int k = 0; k < kDefer; ++k)
    if (k < df.n) {
      xq[k][0] = sref[df.j[k]];
      xq[k][1] = sref[sstride + df.j[k]];
      xq[k][2] = sref[2 * sstride + df.j[k]];
    }
#pragma unroll
  for (int k = 0; k < kDefer; ++k)
    if (k < df.n) {
      QPair r;
      ph.refine_from(r, pp, xq[k]);
      ph.pair(st, df.a[k], r);
    }
}

// ---------------------------------------------------------- FP64 kernels
template <class T, class Ph>
__global__ __launch_bounds__(256) void k_pairs_f64(ClDev c, const T* __restrict__ pos,
                                                   size_t stride, const unsigned long long* __restrict__ voff,
                                                   const uint32_t* __restrict__ vnbr, Ph ph) {
  const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t k = tid / kRowLanes;
  const bool valid = k < c.n_dom;
  const uint32_t p = c.dom[valid ? k : 0];
  const T tx = pos[p], ty = pos[stride + p], tz = pos[2 * stride + p];
  const double xp = tx, yp = ty, zp = tz;
  typename Ph::St st;
  ph.start(st, p);
  // x_p - x_q; unfused square, as the oracle, so the neighbour decision is
  // bit-identical
  auto body = [&](uint32_t j, T qx, T qy, T qz, double a) {
    if (j == p) return;
    double rx = xp - double(qx);
    double ry = yp - double(qy);
    double rz = zp - double(qz);
    double d2 = dist2_unfused<double>(rx, ry, rz);
    if (d2 < ph.rc2) ph.pair(st, a, rx, ry, rz, d2);
  };
  const unsigned lane = threadIdx.x & (kRowLanes - 1);
  if (valid) {
    const unsigned long long e1 = voff[k + 1];
    for (unsigned long long e = voff[k] + lane; e < e1; e += kUnroll * kRowLanes) {
      uint32_t j[kUnroll];
      T qx[kUnroll], qy[kUnroll], qz[kUnroll];
      double a[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const unsigned long long ee = e + u * kRowLanes;
        j[u] = ee < e1 ? vnbr[ee] : p;
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        qx[u] = pos[j[u]];
        qy[u] = pos[stride + j[u]];
        qz[u] = pos[2 * stride + j[u]];
        a[u] = ph.aux(j[u]);
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) body(j[u], qx[u], qy[u], qz[u], a[u]);
    }
  }
  ph.reduce(st, kRowLanes);
  if (valid && lane == 0) ph.finish(st, p);
}

// --------------------------------------------------------- FP32C kernels
template <class Ph, bool kCubic>
__global__ __launch_bounds__(256) void k_pairs_f32c(ClDev c, QGeom qg, const unsigned long long* __restrict__ voff,
                                                    const uint32_t* __restrict__ vnbr, Ph ph) {
  const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t k = tid / kRowLanes;
  const bool valid = k < c.n_dom;
  const uint32_t p = c.dom[valid ? k : 0];
  const int4 P = c.quant[p];
  typename Ph::St st;
  ph.start(st, p);
  const unsigned lane = threadIdx.x & (kRowLanes - 1);
  if (valid) {
    const unsigned long long e1 = voff[k + 1];
    // the row's entries of the next step are loaded before the current step's
    // gathers are used, so the row stream's latency hides behind the pairs.
    // The loads are unconditional, so the compiler can count them in its
    // waits: past the row end a lane reads the row's last entry (entry 0 when
    // the list's first row is empty; the buffer holds at least one entry) and
    // its pair is masked off.
    const unsigned long long elast = e1 > 0 ? e1 - 1 : 0;
    uint32_t jn[kUnroll];
    bool okn[kUnroll];
    auto load_j = [&](unsigned long long e) {
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const unsigned long long ee = e + u * kRowLanes;
        okn[u] = ee < e1;
        jn[u] = vnbr[okn[u] ? ee : elast];
      }
    };
    load_j(voff[k] + lane);
    for (unsigned long long e = voff[k] + lane; e < e1; e += kUnroll * kRowLanes) {
      uint32_t j[kUnroll];
      bool ok[kUnroll];
      int4 Q[kUnroll];
      float a[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        j[u] = jn[u];
        ok[u] = okn[u] && jn[u] != p;
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        Q[u] = c.quant[j[u]];
        a[u] = ph.aux(j[u]);
      }
      load_j(e + kUnroll * kRowLanes);
      // one entry's evaluation at a time (its FP64 temporaries are what sets
      // the kernel's register count, and with it the waves per SIMD that
      // hide the gathers' latency)
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        quant_pair_masked<Ph, kCubic>(ph, st, qg, a[u], wrap_diff(Q[u].x, P.x), wrap_diff(Q[u].y, P.y),
                                      wrap_diff(Q[u].z, P.z), ok[u], p, j[u]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  ph.reduce(st, kRowLanes);
  if (valid && lane == 0) ph.finish(st, p);
}

// ------------------------------------------- smooth physics, Verlet rows
// SPH passes over Verlet rows, 16 lanes per row.  A row holds the particle itself
// (unless its position was not a number at the build: then the row is empty, which
// counts as W(0)), and its skin's entries vanish by themselves.  In FP32C, whose
// separations are integers, whole steps of 64 entries so run without a decision, a
// mask or a branch; only the row's last, partial step masks its lanes past the end
// (their square becomes kFar).  In FP64 a pair is decided: a value of the skin, or a
// position since the build, may be infinite or no number, which zero does not undo.
// The rows' entries of the next step are loaded before the current step's
// gathers are used.
// A pass was bound by VALU issue (62 and 45 instructions per entry in the force
// and density passes); without the decisions and with the clamped spline it is
// 33 and 26, and the texture path is what it waits for (data unit busy 97 %, address
// unit 93 %, VALU 62-69 %).  4.4e9 entries (clustered, 4.2e6 particles): density
// 8.8 -> 7.1 ms, force 9.9 -> 8.1 ms.
constexpr double kFar = 1e200;

// A pair of plain FP64 positions: taken within the cut-off (which a square that is no
// number is not), coincident particles by the densities alone, as r = 1e-154.
template <class Ph>
__device__ __forceinline__ bool plain_pair(const Ph& ph, typename Ph::St& st, double aux, double rx, double ry,
                                           double rz, double r2) {
  if (!(r2 < ph.rc2)) return false;
  if (Ph::kAux && r2 == 0.0) return false;
  ph.pair(st, aux, rx, ry, rz, __builtin_fmax(r2, __DBL_MIN__));
  return true;
}

// FP32C: 12-byte (q_x, q_y, q_z) or 16-byte (q, pterm) records; kWide: the
// quantised stream itself, where there is no room for 12-byte records.
template <class Ph, bool kCubic, bool kWide = false>
struct QuantRows {
  using St = typename Ph::St;
  using Rec = std::conditional_t<Ph::kAuxInQuant || kWide, int4, int3>;
  const Rec* rec;
  QGeom qg;
  Ph ph;
  __device__ __forceinline__ Rec target(uint32_t p) const { return rec[p]; }
  __device__ __forceinline__ Rec gather(uint32_t j) const { return rec[j]; }
  // whether a row's own entry was taken
  __device__ __forceinline__ bool holds_itself(const Rec&) const { return true; }
  template <bool kMask>
  __device__ __forceinline__ void eval(St& st, const Rec& P, const Rec& Q, bool ok) const {
    const double dx = double(wrap_diff(Q.x, P.x));
    double dy = double(wrap_diff(Q.y, P.y)), dz = double(wrap_diff(Q.z, P.z));
    if constexpr (!kCubic) {
      dy *= qg.ryd;
      dz *= qg.rzd;
    }
    double r2 = __builtin_fma(dx, dx, __builtin_fma(dy, dy, __builtin_fma(dz, dz, kTiny)));
    if constexpr (kMask) r2 = ok ? r2 : kFar;
    float a = 0.f;
    if constexpr (Ph::kAuxInQuant) a = __int_as_float(Q.w);
    ph.pair(st, a, dx, dy, dz, r2);
  }
};

// Plain FP64: the stored positions (three planes) and the physics' own value.
template <class T, class Ph>
struct PlainRows {
  using St = typename Ph::St;
  struct Rec {
    T x, y, z;
    double a;
  };
  const T* pos;
  size_t stride;
  Ph ph;
  __device__ __forceinline__ Rec target(uint32_t p) const { return gather(p); }
  __device__ __forceinline__ Rec gather(uint32_t j) const {
    Rec r{pos[j], pos[stride + j], pos[2 * stride + j], 0.0};
    if constexpr (Ph::kAux) r.a = ph.aux(j);
    return r;
  }
  // not if the particle's position is infinite or not a number (inf - inf)
  __device__ __forceinline__ bool holds_itself(const Rec& P) const {
    const double rx = double(P.x) - double(P.x), ry = double(P.y) - double(P.y), rz = double(P.z) - double(P.z);
    return rx + ry + rz == 0.0;
  }
  template <bool kMask>
  __device__ __forceinline__ void eval(St& st, const Rec& P, const Rec& Q, bool ok) const {
    const double rx = double(P.x) - double(Q.x), ry = double(P.y) - double(Q.y), rz = double(P.z) - double(Q.z);
    const double r2 = __builtin_fma(rx, rx, __builtin_fma(ry, ry, rz * rz));
    if (kMask && !ok) return;
    plain_pair(ph, st, Q.a, rx, ry, rz, r2);
  }
};

template <class W>
__global__ __launch_bounds__(256) void k_rows_smooth(ClDev c, const unsigned long long* __restrict__ voff,
                                                     const uint32_t* __restrict__ vnbr, W w) {
  constexpr uint32_t kStep = uint32_t(kUnroll * kRowLanes);
  const uint32_t k = (blockIdx.x * blockDim.x + threadIdx.x) / kRowLanes;
  const bool valid = k < c.n_dom;
  const uint32_t p = c.dom[valid ? k : 0];
  const typename W::Rec P = w.target(p);
  typename W::St st;
  w.ph.start(st, p);
  const uint32_t lane = threadIdx.x & (kRowLanes - 1);
  uint32_t len = 0;
  if (valid) {
    const unsigned long long e0 = voff[k];
    len = uint32_t(voff[k + 1] - e0);
    if (len > 0) {
      const uint32_t* __restrict__ row = vnbr + e0;
      const uint32_t last = len - 1;
      uint32_t jn[kUnroll];
      // past the row's end a lane reads the row's last entry
      auto load_j = [&](uint32_t b) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const uint32_t i = b + uint32_t(u * kRowLanes) + lane;
          jn[u] = row[i < last ? i : last];
        }
      };
      load_j(0);
      const uint32_t full = len & ~(kStep - 1);
      typename W::Rec Q[kUnroll];
      for (uint32_t b = 0; b < full; b += kStep) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) Q[u] = w.gather(jn[u]);
        load_j(b + kStep);
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          w.template eval<false>(st, P, Q[u], true);
          __builtin_amdgcn_sched_barrier(0);  // one entry's temporaries at a time (registers)
        }
      }
      if (full < len) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) Q[u] = w.gather(jn[u]);
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const uint32_t i = full + uint32_t(u * kRowLanes);
          if (i < len) w.template eval<true>(st, P, Q[u], i + lane < len);
        }
      }
    }
  }
  w.ph.reduce(st, kRowLanes);
  if (valid && lane == 0) w.ph.finish(st, p, len == 0 || !w.holds_itself(P) ? 1.0 : 0.0);
}

// ---------------------------------------------- LDS-staged cell tiles
// The pair pass over a cell list without a Verlet list.  Persistent waves take
// target items from the cell list's item queue: up to 64 domain particles of
// consecutive cells on one x-row of the grid, one per lane.  The item's
// candidates are the (2B+1)^2 x-runs of its stencil, each a contiguous range
// of sorted indices; they pass through the wave's LDS region tile_chunk() at a
// time (coalesced loads).  Check: the matrix cores give every target a bit per
// staged candidate that may lie within the cut-off (MatrixTest; tested one by one
// in the vector ALU where coordinates lie beyond its bounds).
// Evaluate: each lane walks its own set bits in ascending order and evaluates
// those pairs from the staged records, deciding the cut-off where the physics does
// not vanish there by itself.  A target's pairs are summed in one
// lane in ascending sorted index, so the results do not depend on the order in
// which the items are taken.  Candidates that lie in the union of the item's
// stencils but outside a target's own stencil are more than B cells away in x
// from it, so they are misses for it.
// Bound by the evaluation's instructions (31 an entry of the density pass) and its
// idle lanes (38 % busy with rounds of 128 candidates, whose runs' hits depend on a
// target's place in its cell; larger rounds even that out).  Tests in the vector
// ALU, eleven instructions per candidate and wave, took half of the passes.
// 1,092,727 particles on a lattice (FP32C, density and force): 632 and 682 -> 372
// and 400 us (128 candidates a round 445 and 453); 65,536 of a
// gas, FP64 LJ: 112 -> 55 us.
//
// FP32C separations: the union spans at most kItemMaxCells - 1 + B cells in x
// from any of the item's targets, so a candidate is either within 2^31 quanta
// (the wrapped subtraction is exact) or its wrapped separation is still more
// than B cells (one cell of slack for positions that have drifted since the
// cells were built): no far candidate's pair is within the cut-off.  The masks'
// coordinates are relative to the middle of the item's cells, from which no
// candidate within a target's cut-off is 2^31 quanta away (static_assert below).
// Candidates staged per round: a lane's hits of a run of cells vary with its place
// in y and z, those of several runs less, and a round takes as long as its busiest
// lane.  Four blocks of four waves fit a CU's registers, 40 KB of LDS each.
template <class R>
constexpr int tile_chunk() {
  return sizeof(R) <= 16 ? 384 : 256;
}
constexpr int kTileBlock = 256;  // four independent waves
constexpr int kTileWaves = kTileBlock / kWave;
static_assert(int(kItemMaxCells) / 2 + 1 + kMaxBoxNN <= 8, "wrapped FP32C coordinates of the masks");
static_assert(16 - (int(kItemMaxCells) - 1 + kMaxBoxNN) - 2 > kMaxBoxNN, "wrapped FP32C separations");

// Hit bits of staged candidates k0 .. k0 + cnt - 1 (cnt <= 32, uniform) for
// this lane's target, candidate k0 + k at bit k; `test(Q)` is the lane's check.
template <class R, class F>
__device__ __forceinline__ uint32_t staged_hits(const R* buf, uint32_t k0, uint32_t cnt, F&& test) {
  if (cnt == 0) return 0u;
  uint32_t w = 0, k = 0;
  for (; k + 8 <= cnt; k += 8) {
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) w = shift_in(w, test(buf[k0 + k + i]));
  }
  for (; k < cnt; ++k) w = shift_in(w, test(buf[k0 + k]));
  return __builtin_bitreverse32(w << (32u - cnt));
}

// Calls fn(k) for the set bits k of the lane's `words` 64-bit words (mk[q][lane]),
// lowest first, one bit per lane per round, until no lane has bits left (an empty
// word costs its lane a round).
template <class F>
__device__ __forceinline__ void for_each_hit(const unsigned long long (*mk)[kWave], uint32_t words, int lane, F&& fn) {
  unsigned long long w = mk[0][lane];
  uint32_t q = 0;
  for (;;) {
    if (w == 0ull && q + 1 < words) w = mk[++q][lane];
    if (__ballot(w != 0ull || q + 1 < words) == 0ull) return;
    if (w != 0ull) {
      const uint32_t k = q * 64u + uint32_t(__builtin_ctzll(w));
      w &= w - 1ull;
      fn(k);
    }
  }
}

// The item's candidates through the wave's buffer, kChunk at a time across the
// ends of the runs: put(slot, j) stages sorted index j, eval(m) takes the m staged.
// Lane r holds run r.  The wave's LDS operations execute in issue order; the
// barriers keep the compiler from moving the reads of one round across the writes
// of the next.
template <int kChunk, class T, class P, class E>
__device__ __forceinline__ void for_each_chunk(const ClDev& c, const ItemGeom<T>& G, int lane, P&& put, E&& eval) {
  const uint2 R = lane_run(c, G, lane);
  const uint32_t runs = (2u * c.box_nn + 1u) * (2u * c.box_nn + 1u);
  uint32_t r = 0, done = 0;  // the run in hand, and how much of it has been staged
  for (;;) {
    uint32_t m = 0;
    __builtin_amdgcn_wave_barrier();
    while (m < uint32_t(kChunk) && r < runs) {
      const uint32_t ja = __builtin_amdgcn_readlane(R.x, r) + done, left = __builtin_amdgcn_readlane(R.y, r) - ja;
      const uint32_t n = left < uint32_t(kChunk) - m ? left : uint32_t(kChunk) - m;
      for (uint32_t k = uint32_t(lane); k < n; k += kWave) put(m + k, ja + k);
      m += n;
      done = n < left ? done + n : 0u;
      r += n < left ? 0u : 1u;
    }
    __builtin_amdgcn_wave_barrier();
    if (m == 0) return;
    eval(m);
  }
}

// Hit words of m staged candidates to mk: from the matrix cores, two blocks of 32 at
// a time (rel: the coordinates of a staged candidate relative to the origin), or by
// the exact test where they decline.
template <class R, class Rel, class Test>
__device__ __forceinline__ void chunk_hits(const MatrixTest& mt, bool fast, const R* buf, uint32_t m, int lane,
                                           bool valid, unsigned long long (*mk)[kWave], Rel&& rel, Test&& test) {
  const uint32_t mine = matrix_candidate(uint32_t(lane)) + (lane < 32 ? 0u : 32u);
  for (uint32_t k0 = 0; k0 < m; k0 += 64u) {
    const uint32_t n = m - k0 < 64u ? m - k0 : 64u;
    float x, y, z;
    rel(buf[k0 + (mine < n ? mine : n - 1u)], &x, &y, &z);
    uint32_t lo = 0, hi = 0;
    if (fast && mt.words<false>(x, y, z, n > 32u, &lo, &hi)) {
      lo &= n < 32u ? 0xFFFFFFFFu >> (32u - n) : 0xFFFFFFFFu;
      hi &= n > 32u ? 0xFFFFFFFFu >> (64u - n) : 0u;
    } else {
      lo = staged_hits(buf, k0, n < 32u ? n : 32u, test);
      hi = n > 32u ? staged_hits(buf, k0 + 32u, n - 32u, test) : 0u;
    }
    mk[k0 / 64u][lane] = valid ? static_cast<unsigned long long>(hi) << 32 | lo : 0ull;
  }
}

// FP32C.  rec: per sorted particle the quantised record; with Ph::kAuxInQuant
// its fourth word is the physics' per-particle value (P / rho^2), otherwise
// the fourth word is not read.  kMany: ensembles, the physics and geometry of
// an item come from the tables of its system (ncx >> 8).
template <class T, class Ph, bool kCubic, bool kMany>
__global__ __launch_bounds__(kTileBlock, 4) void k_tile_f32c(ClDev c, QGeom qg1, Ph ph1, const Ph* __restrict__ tab,
                                                          const QGeom* __restrict__ qtab,
                                                          const SysGrid<T>* __restrict__ sys,
                                                          const int4* __restrict__ rec,
                                                          const TargetItem* __restrict__ items,
                                                          const uint32_t* __restrict__ n_items_p,
                                                          uint32_t* __restrict__ counter) {
  constexpr int kChunk = tile_chunk<int4>();
  __shared__ int4 lds[kTileWaves][kChunk];
  __shared__ unsigned long long ldsm[kTileWaves][kChunk / 64][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  int4* buf = lds[threadIdx.x / kWave];
  unsigned long long(*mk)[kWave] = ldsm[threadIdx.x / kWave];
  const uint32_t n_items = *n_items_p;
  for (;;) {
    const uint32_t it = next_unit(counter);
    if (it >= n_items) break;
    const TargetItem ti = items[it];
    const uint32_t sy = ti.ncx >> 8;
    const Ph ph = kMany ? tab[sy] : ph1;
    const QGeom qg = kMany ? qtab[sy] : qg1;
    const ItemGeom<T> G = item_geom(c, ti, T(0), kMany ? sys : nullptr, static_cast<const T*>(nullptr));
    const bool valid = uint32_t(lane) < ti.n;
    const uint32_t p = c.dom[ti.row0 + (valid ? uint32_t(lane) : 0u)];
    const int4 P = c.quant[p];
    const float pre2 = ph.rc2 * kPreCut;
    typename Ph::St st;
    ph.start(st, p);
    auto sep = [&](const int4& Q, int ox, int oy, int oz, float* x, float* y, float* z) {
      *x = float(wrap_diff(Q.x, ox));
      *y = kCubic ? float(wrap_diff(Q.y, oy)) : float(wrap_diff(Q.y, oy)) * qg.ry;
      *z = kCubic ? float(wrap_diff(Q.z, oz)) : float(wrap_diff(Q.z, oz)) * qg.rz;
    };
    auto test = [&](const int4& Q) {
      float fx, fy, fz;
      sep(Q, P.x, P.y, P.z, &fx, &fy, &fz);
      return __builtin_fmaf(fx, fx, __builtin_fmaf(fy, fy, fz * fz)) < pre2;
    };
    // the origin: the middle of the item's cells, at most ncx / 2 + 1 cells (drift
    // included) from a target in x and B more from a candidate within its cut-off
    const int ox = int(uint32_t(2 * G.cx0 + G.ncx) << (kQuantBits - 1));
    const int oy = int(uint32_t(2 * G.cy + 1) << (kQuantBits - 1));
    const int oz = int(uint32_t(2 * G.cz + 1) << (kQuantBits - 1));
    constexpr float cell = float(kQuantOne);
    const float ry2 = kCubic ? 1.f : qg.ry * qg.ry, rz2 = kCubic ? 1.f : qg.rz * qg.rz;
    const float nx = 0.5f * float(G.ncx) + 1.f, bx = nx + float(c.box_nn), by = 1.5f + float(c.box_nn);
    const float rt2 = cell * cell * (nx * nx + 2.25f * (ry2 + rz2));
    const float rc2 = cell * cell * (bx * bx + by * by * (ry2 + rz2));
    float tx, ty, tz;
    sep(P, ox, oy, oz, &tx, &ty, &tz);
    MatrixTest mt;
    const bool fast = mt.targets<true>(tx, ty, tz, rt2, rc2, pre2, ti.n > 32u);
    bool seen = false;
    bool odd = false;  // a value that is infinite or no number
    if constexpr (Ph::kAuxInQuant) odd = !__builtin_isfinite(ph.aux(p));
    for_each_chunk<kChunk>(
        c, G, lane,
        [&](uint32_t k, uint32_t j) {
          int4 Q = rec[j];
          if constexpr (!Ph::kAuxInQuant) Q.w = int(j);
          if constexpr (Ph::kAuxInQuant) odd |= !__builtin_isfinite(__int_as_float(Q.w));
          buf[k] = Q;
        },
        [&](uint32_t m) {
          chunk_hits(mt, fast, buf, m, lane, valid, mk,
                     [&](const int4& Q, float* x, float* y, float* z) { sep(Q, ox, oy, oz, x, y, z); }, test);
          const bool careful = Ph::kAuxInQuant && __ballot(odd) != 0ull;
          for_each_hit(mk, (m + 63u) / 64u, lane, [&](uint32_t k) {
            seen = true;
            const int4 Q = buf[k];
            const int ix = wrap_diff(Q.x, P.x), iy = wrap_diff(Q.y, P.y), iz = wrap_diff(Q.z, P.z);
            if constexpr (Ph::kSmooth) {  // (the particle itself too)
              float a = 0.f;
              if constexpr (Ph::kAuxInQuant) a = __int_as_float(Q.w);
              smooth_pair<Ph, kCubic>(ph, st, qg, a, ix, iy, iz, careful);
            } else {
              const uint32_t j = uint32_t(Q.w);
              if (j != p) quant_pair<Ph, kCubic>(ph, st, qg, ph.aux(j), ix, iy, iz, p, j);
            }
          });
        });
    if constexpr (Ph::kSmooth) {
      if (valid) ph.finish(st, p, seen ? 0.0 : 1.0);
    } else {
      if (valid) ph.finish(st, p);
    }
  }
}

// Plain FP64 form: positions (three planes) staged per round; the check is the
// pair's own cut-off decision (FP64 separation of the stored positions, squares
// summed unfused), so a set bit is a pair to evaluate.
template <class T>
struct Pos3 {
  T x, y, z;
};

template <class T, class Ph, bool kMany>
__global__ __launch_bounds__(kTileBlock, 4) void k_tile_f64(ClDev c, const T* __restrict__ pos, size_t stride,
                                                         double spx, double spy, double spz, Ph ph1,
                                                         const Ph* __restrict__ tab,
                                                         const SysGrid<T>* __restrict__ sys,
                                                         const TargetItem* __restrict__ items,
                                                         const uint32_t* __restrict__ n_items_p,
                                                         uint32_t* __restrict__ counter) {
  constexpr int kChunk = tile_chunk<Pos3<T>>();
  __shared__ Pos3<T> lds[kTileWaves][kChunk];
  __shared__ uint32_t ldsj[kTileWaves][kChunk];
  __shared__ unsigned long long ldsm[kTileWaves][kChunk / 64][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  Pos3<T>* buf = lds[threadIdx.x / kWave];
  uint32_t* bufj = ldsj[threadIdx.x / kWave];
  unsigned long long(*mk)[kWave] = ldsm[threadIdx.x / kWave];
  const uint32_t n_items = *n_items_p;
  for (;;) {
    const uint32_t it = next_unit(counter);
    if (it >= n_items) break;
    const TargetItem ti = items[it];
    const Ph ph = kMany ? tab[ti.ncx >> 8] : ph1;
    const ItemGeom<T> G = item_geom(c, ti, T(0), kMany ? sys : nullptr, static_cast<const T*>(nullptr));
    const bool valid = uint32_t(lane) < ti.n;
    const uint32_t p = c.dom[ti.row0 + (valid ? uint32_t(lane) : 0u)];
    const double xp = pos[p], yp = pos[stride + p], zp = pos[2 * stride + p];
    typename Ph::St st;
    ph.start(st, p);
    auto test = [&](const Pos3<T>& Q) {
      return dist2_unfused<double>(xp - double(Q.x), yp - double(Q.y), zp - double(Q.z)) < ph.rc2;
    };
    if (kMany) {
      const SysGrid<T>& S = sys[ti.ncx >> 8];
      spx = double(S.sp[0]);
      spy = double(S.sp[1]);
      spz = double(S.sp[2]);
    }
    // relative to the middle target; the bounds as in the Verlet build's count pass
    const uint32_t mid = ti.n / 2;
    const double ox = lane_value(xp, mid), oy = lane_value(yp, mid), oz = lane_value(zp, mid);
    const double unit = matrix_unit(spx, spy, spz);
    const float ux = float(spx * unit), uy = float(spy * unit), uz = float(spz * unit);
    const float B1 = float(c.box_nn + 1u), nx = float(G.ncx), bx = nx + float(c.box_nn);
    const float rt2 = nx * nx * ux * ux + uy * uy + uz * uz;
    const float rc2 = bx * bx * ux * ux + B1 * B1 * (uy * uy + uz * uz);
    MatrixTest mt;
    const bool fast = mt.targets<true>(float((xp - ox) * unit), float((yp - oy) * unit), float((zp - oz) * unit), rt2,
                                       rc2, float(ph.rc2 * unit * unit), ti.n > 32u);
    bool seen = false;
    for_each_chunk<kChunk>(
        c, G, lane,
        [&](uint32_t k, uint32_t j) {
          buf[k] = Pos3<T>{pos[j], pos[stride + j], pos[2 * stride + j]};
          bufj[k] = j;
        },
        [&](uint32_t m) {
          chunk_hits(
              mt, fast, buf, m, lane, valid, mk,
              [&](const Pos3<T>& Q, float* x, float* y, float* z) {
                *x = float((double(Q.x) - ox) * unit);
                *y = float((double(Q.y) - oy) * unit);
                *z = float((double(Q.z) - oz) * unit);
              },
              test);
          for_each_hit(mk, (m + 63u) / 64u, lane, [&](uint32_t k) {
            const Pos3<T> Q = buf[k];
            const uint32_t j = bufj[k];
            const double rx = xp - double(Q.x), ry = yp - double(Q.y), rz = zp - double(Q.z);
            const double d2 = dist2_unfused<double>(rx, ry, rz);
            if constexpr (Ph::kSmooth) {
              seen |= plain_pair(ph, st, ph.aux(j), rx, ry, rz, d2);  // (the particle itself too)
            } else {
              if (d2 < ph.rc2 && j != p) ph.pair(st, ph.aux(j), rx, ry, rz, d2);
            }
          });
        });
    if constexpr (Ph::kSmooth) {
      if (valid) ph.finish(st, p, seen ? 0.0 : 1.0);
    } else {
      if (valid) ph.finish(st, p);
    }
  }
}

// ------------------------------------------------------ ensemble kernels
// One lane per Verlet row: the row's entries [e0, e1) are read in groups of
// four from the row's first entry, so a row of L entries takes ceil(L / 4) groups.
// A wave's rows are consecutive in the list: their entries, where kRowEntries hold
// them, are staged in LDS (RowEntries), 16 bytes per lane of contiguous lines, and
// the lanes read their groups there; else a lane loads a group from the list, 16
// bytes (4-byte aligned; gfx950 takes dword-aligned multi-dword loads).  The list
// buffer holds at least three entries past the list's capacity, so the last group
// read stays inside it.  Slots of the last group past the row's end (the next row's
// entries, or unwritten ones past the list's end) read as p, the row's own
// particle, which the pair evaluation skips.  body(j, next) gets the group and a
// callable that reads the next group; body calls it once its gathers are issued, so
// that it is there after the evaluation.
// The passes are bound by the texture path, which returns a wave's scattered 16-byte
// groups in 64 clocks, against 48 for each of their four gathers.  Step pass of 2^23
// particles, 19 entries a row: FP32C 538 -> 520 us; FP64 40 steps 29.8 -> 24.3 ms.
// 6 KB a wave; 8 KB leave four blocks per CU (FP32C 590 us).
constexpr uint32_t kRowEntries = 1532;
struct RowEntries {
  // (an LDS pointer by type: through a generic one the compiler makes one flat load
  // of the two branches in row_groups)
  typedef const uint32_t __attribute__((address_space(3))) Word;
  Word* lds;
  bool staged;  // wave-uniform
  unsigned long long first;
  // Called by the whole wave with its first row (kw).
  __device__ __forceinline__ RowEntries(uint32_t* buf, const unsigned long long* __restrict__ voff,
                                        const uint32_t* __restrict__ vnbr, unsigned long long e_lim, uint32_t kw,
                                        uint32_t n_rows)
      : lds((Word*)(buf)), staged(false), first(0) {
    if (kw >= n_rows) return;
    first = voff[kw];
    const unsigned long long end = voff[kw + kWave < n_rows ? kw + kWave : n_rows];
    const unsigned long long lim = end < e_lim ? end : e_lim;
    const unsigned long long n = first < lim ? lim - first : 0;
    if (n > kRowEntries) return;
    for (uint32_t i = (threadIdx.x & (kWave - 1)) * 4u; i < uint32_t(n); i += 4u * kWave) {
      uint4 q;
      __builtin_memcpy(&q, vnbr + first + i, sizeof(q));
      *reinterpret_cast<uint4*>(buf + i) = q;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    staged = true;
  }
};
template <class F>
__device__ __forceinline__ void row_groups(const RowEntries& row, const uint32_t* __restrict__ vnbr,
                                           unsigned long long e0, unsigned long long e1, uint32_t p, F&& body) {
  // (an empty row reads nothing: a list cut at its capacity ends before e0)
  if (!(e0 < e1)) return;
  auto walk = [&](auto&& load) {
    uint4 Jn = load(e0);
    for (unsigned long long b = e0; b < e1; b += 4) {
      const uint32_t raw[4] = {Jn.x, Jn.y, Jn.z, Jn.w};
      uint32_t j[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) j[u] = b + u < e1 ? raw[u] : p;
      body(j, [&] { Jn = load(b + 4 < e1 ? b + 4 : b); });
    }
  };
  walk([&](unsigned long long e) {
    uint4 q;
    if (row.staged) {
      const RowEntries::Word* s = row.lds + uint32_t(e - row.first);
      q = make_uint4(s[0], s[1], s[2], s[3]);
    } else {
      __builtin_memcpy(&q, vnbr + e, sizeof(q));
    }
    return q;
  });
}

// The systems of a wave's rows one at a time, so that a system's constants are
// wave-uniform (scalar registers, not a copy per lane): a wave's rows are
// consecutive in cell order and the systems' cells are numbered one system
// after another, so a wave nearly always holds one system (two where one
// system's rows end).  f(sy) runs on the lanes whose rows belong to system sy;
// the lanes of a row share its system, so a row is never split.
template <class F>
__device__ __forceinline__ void by_system(bool valid, uint32_t sy_lane, F&& f) {
  unsigned long long todo = __ballot(valid);
  while (todo) {
    uint32_t sy = __builtin_amdgcn_readlane(sy_lane, int(__builtin_ctzll(todo)));
    // both sides of the test opaque to the compiler, the lane's copy made
    // last: inside the branch it would otherwise use the equal per-lane value
    // for sy (and load the system's constants per lane)
    asm volatile("" : "+s"(sy));
    uint32_t sy_mine = sy_lane;
    asm volatile("" : "+v"(sy_mine));
    const bool mine = valid && sy_mine == sy;
    todo &= ~__ballot(mine);
    if (mine) f(sy);
  }
}

// The end of a row: its force stored (NoKick), or applied to the row's particle
// by the step's kick (StepKick).
// Called by every lane of the row.  x: the row's position.
template <int kLanes, class Ph, class K, class T>
__device__ __forceinline__ void finish_row(const Ph& ph, const typename Ph::St& st, uint32_t p, uint32_t sy, int w,
                                           const K& kick, const typename K::Pre& pre, const T (&x)[3],
                                           unsigned lane) {
  if constexpr (K::kOn) {
    typename K::Tv a[3];
    ph.force_as(st, a);
    // opaque copies: the kick's addresses and the cell terms of its records
    // are computed here, not hoisted above the row's loop where they would
    // hold registers throughout
    uint32_t pk = p;
    int wk = w;
    unsigned lk = lane;
    asm volatile("" : "+v"(pk), "+v"(wk), "+v"(lk));
    if constexpr (kLanes >= K::kSplitLanes)
      kick.template apply_split<kLanes>(pre, pk, sy, wk, a, x, lk);
    else if (lane == 0)
      kick.apply(pre, pk, sy, wk, a, x);
  } else {
    if (lane == 0) ph.finish(st, p);
  }
}

// Verlet rows of an ensemble: the constants of row k are the table entry of its
// system (sid_sorted of the row's particle; null: one system); kLanes lanes per row.  K: NoKick
// (forces stored) or StepKick<T> (the row's particle kicked and drifted).
template <class T, class Ph, int kLanes, bool kCubic, class K>
__global__ __launch_bounds__(256) void k_pairs_many_f32c(ClDev c, const Ph* __restrict__ tab,
                                                         const QGeom* __restrict__ qtab,
                                                         const uint32_t* __restrict__ sid_sorted,
                                                         const unsigned long long* __restrict__ voff,
                                                         const uint32_t* __restrict__ vnbr,
                                                         unsigned long long e_lim, const T* __restrict__ sref,
                                                         size_t sstride, K kick) {
  const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t k = tid / kLanes;
  const bool valid = k < c.n_dom;
  const uint32_t p = c.dom[valid ? k : 0];
  const int4 P = c.quant[p];
  const uint32_t ik = kick.index(p);
  const unsigned lane = threadIdx.x & (kLanes - 1);
  __shared__ __align__(16) uint32_t entries[kLanes == 1 ? 256 / kWave : 1][kLanes == 1 ? kRowEntries + 4 : 1];
  RowEntries staged(entries[kLanes == 1 ? threadIdx.x / kWave : 0], voff, vnbr, e_lim,
                    __builtin_amdgcn_readfirstlane(kLanes == 1 ? k : ~0u), c.n_dom);
  by_system(valid, sid_sorted ? sid_sorted[p] : 0u, [&](uint32_t sy) {
  const Ph ph = tab[sy];
  const QGeom qg = qtab[sy];
  // the stored position, for close pairs
  const T pp[3] = {sref[p], sref[sstride + p], sref[2 * sstride + p]};
  typename Ph::St st;
  ph.start(st, p);
  typename K::Pre pre;
  // the kick's loads after the row's loop (an opaque index, so they are not
  // hoisted above it, where their registers would be held throughout)
  auto prefetch = [&] {
    uint32_t i = ik;
    unsigned l = lane;
    asm volatile("" : "+v"(i), "+v"(l));
    pre = kick.template prefetch<kLanes>(i, l);
  };
  if (kLanes == 1) {
    // e_lim: entries the list holds (a list that overflowed its capacity was not
    // written; its rows are cut at the capacity and the caller rebuilds)
    const unsigned long long e0 = voff[k];
    const unsigned long long e1 = voff[k + 1] < e_lim ? voff[k + 1] : e_lim;
    Deferred df;
    row_groups(staged, vnbr, e0, e1, p, [&](const uint32_t (&j)[4], auto&& next) {
      int4 Q[4];
      float a[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        // slots outside the row (j = p) gather nothing: each gathered record
        // costs the wave a cache-line lookup
        Q[u] = P;
        a[u] = 0.f;
        if (j[u] != p) {
          Q[u] = c.quant[j[u]];
          a[u] = ph.aux(j[u]);
        }
      }
      next();
      const bool ns[4] = {j[0] != p, j[1] != p, j[2] != p, j[3] != p};
      quant_group_defer<T, Ph, kCubic>(ph, st, qg, a, Q, P, j, ns, pp, sref, sstride, df);
    });
    prefetch();
    flush_deferred<T, Ph>(ph, st, pp, sref, sstride, df);
  } else {
    const unsigned long long e1 = voff[k + 1] < e_lim ? voff[k + 1] : e_lim;
    // next step's entries in flight during the current step, unconditional
    // loads (as in k_pairs_f32c): a lane past the row end reads the row's last
    // entry (entry 0 if the first row is empty) and its pair is masked off
    const unsigned long long elast = e1 > 0 ? e1 - 1 : 0;
    uint32_t jn[kUnroll];
    bool okn[kUnroll];
    auto load_j = [&](unsigned long long e) {
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const unsigned long long ee = e + u * kLanes;
        okn[u] = ee < e1;
        jn[u] = vnbr[okn[u] ? ee : elast];
      }
    };
    load_j(voff[k] + lane);
    for (unsigned long long e = voff[k] + lane; e < e1; e += kUnroll * kLanes) {
      uint32_t j[kUnroll];
      bool ok[kUnroll];
      int4 Q[kUnroll];
      float a[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        j[u] = jn[u];
        ok[u] = okn[u] && jn[u] != p;
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        Q[u] = c.quant[j[u]];
        a[u] = ph.aux(j[u]);
      }
      load_j(e + kUnroll * kLanes);
      static_assert(kUnroll == 4, "groups of four entries");
      quant_group_masked<T, Ph, kCubic>(ph, st, qg, a, Q, P, j, ok, pp, sref, sstride);
    }
    prefetch();
  }
  ph.reduce(st, kLanes);
  finish_row<kLanes>(ph, st, p, sy, P.w, kick, pre, pp, lane);
  });
}

template <class T, class Ph, int kLanes, class K>
__global__ __launch_bounds__(256) void k_pairs_many_f64(ClDev c, const Ph* __restrict__ tab,
                                                        const uint32_t* __restrict__ sid_sorted,
                                                        const T* __restrict__ pos, size_t stride,
                                                        const unsigned long long* __restrict__ voff,
                                                        const uint32_t* __restrict__ vnbr,
                                                        unsigned long long e_lim, K kick) {
  const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t k = tid / kLanes;
  const bool valid = k < c.n_dom;
  const uint32_t p = c.dom[valid ? k : 0];
  const double xp = pos[p], yp = pos[stride + p], zp = pos[2 * stride + p];
  const uint32_t ik = kick.index(p);
  const unsigned lane = threadIdx.x & (kLanes - 1);
  __shared__ __align__(16) uint32_t entries[kLanes == 1 ? 256 / kWave : 1][kLanes == 1 ? kRowEntries + 4 : 1];
  RowEntries staged(entries[kLanes == 1 ? threadIdx.x / kWave : 0], voff, vnbr, e_lim,
                    __builtin_amdgcn_readfirstlane(kLanes == 1 ? k : ~0u), c.n_dom);
  by_system(valid, sid_sorted ? sid_sorted[p] : 0u, [&](uint32_t sy) {
  const Ph ph = tab[sy];
  typename Ph::St st;
  ph.start(st, p);
  auto eval = [&](uint32_t j, T qx, T qy, T qz) {
    const double rx = xp - double(qx);
    const double ry = yp - double(qy);
    const double rz = zp - double(qz);
    const double d2 = dist2_unfused<double>(rx, ry, rz);
    if (d2 < ph.rc2) ph.pair(st, 0.0, rx, ry, rz, d2);
  };
  if (kLanes == 1) {
    const unsigned long long e1 = voff[k + 1] < e_lim ? voff[k + 1] : e_lim;
    row_groups(staged, vnbr, voff[k], e1, p, [&](const uint32_t (&j)[4], auto&& next) {
      T qx[4], qy[4], qz[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        qx[u] = pos[j[u]];
        qy[u] = pos[stride + j[u]];
        qz[u] = pos[2 * stride + j[u]];
      }
      next();
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (j[u] != p) eval(j[u], qx[u], qy[u], qz[u]);
    });
  } else {
    const unsigned long long e1 = voff[k + 1] < e_lim ? voff[k + 1] : e_lim;
    for (unsigned long long e = voff[k] + lane; e < e1; e += kUnroll * kLanes) {
      uint32_t j[kUnroll];
      T qx[kUnroll], qy[kUnroll], qz[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const unsigned long long ee = e + u * kLanes;
        j[u] = ee < e1 ? vnbr[ee] : p;
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        qx[u] = pos[j[u]];
        qy[u] = pos[stride + j[u]];
        qz[u] = pos[2 * stride + j[u]];
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
        if (j[u] != p) eval(j[u], qx[u], qy[u], qz[u]);
    }
  }
  uint32_t i = ik;  // opaque: the kick's loads stay after the loop
  asm volatile("" : "+v"(i));
  const typename K::Pre pre = kick.template prefetch<kLanes>(i, lane);
  ph.reduce(st, kLanes);
  const T xr[3] = {T(xp), T(yp), T(zp)};  // stored in T
  finish_row<kLanes>(ph, st, p, sy, 0, kick, pre, xr, lane);
  });
}

// ---------------------------------------------------------------- EOS
template <class PT>
__global__ __launch_bounds__(256) void k_tait(const double* __restrict__ rho, size_t n, double inv_rho0,
                                              double B, double* __restrict__ prs, PT* __restrict__ pterm) {
  size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double rr = rho[i];
  double r = rr * inv_rho0;
  double r2 = r * r, r4 = r2 * r2;
  double P = B * (r4 * r2 * r - 1.0);
  if (prs) prs[i] = P;
  pterm[i] = PT(P / (rr * rr));
}

// ------------------------------------------------------------- reductions
constexpr int kRedBlock = 256;
constexpr unsigned kRedGrid = 1024;

__device__ __forceinline__ double red_op(int op, double a, double b) {
  return op == OFP_RED_SUM ? a + b : (op == OFP_RED_MAX ? fmax(a, b) : fmin(a, b));
}

template <class T>
__global__ __launch_bounds__(kRedBlock) void k_reduce_partial(const T* __restrict__ x, const T* __restrict__ comp,
                                                              size_t n, int op, double ident,
                                                              double* __restrict__ partial) {
  __shared__ double lds[kRedBlock / kWave];
  double acc = ident;
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
    double v = double(x[i]);
    if (comp) v += double(comp[i]);
    acc = red_op(op, acc, v);
  }
  for (int d = kWave / 2; d > 0; d >>= 1) acc = red_op(op, acc, __shfl_xor(acc, d, kWave));
  if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = lds[0];
    for (int w = 1; w < kRedBlock / kWave; ++w) r = red_op(op, r, lds[w]);
    partial[blockIdx.x] = r;
  }
}

// Combines the nb partials and writes the result to *out (for ofp_reduce the
// slot after the partials, for ofp_reduce_noalloc the caller's device word).
__global__ __launch_bounds__(kRedBlock) void k_reduce_final(const double* partial, unsigned nb, int op, double ident,
                                                            double* __restrict__ out) {
  __shared__ double lds[kRedBlock / kWave];
  double acc = ident;
  for (unsigned i = threadIdx.x; i < nb; i += blockDim.x) acc = red_op(op, acc, partial[i]);
  for (int d = kWave / 2; d > 0; d >>= 1) acc = red_op(op, acc, __shfl_xor(acc, d, kWave));
  if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = lds[0];
    for (int w = 1; w < kRedBlock / kWave; ++w) r = red_op(op, r, lds[w]);
    *out = r;
  }
}

// Partials of ofp_reduce_noalloc: one file-scope array per GPU, the most the
// partial kernel's grid can write (kRedGrid) plus one.  In host code the name
// stands for the host-side shadow, never for the device copy: kernels and
// copies get the device address that reduce_scratch() looks up.
constexpr size_t kRedScratch = size_t(kRedGrid) + 1;
static __device__ __align__(256) double scratch[kRedScratch];

// ------------------------------------------------------------- launchers
struct PairCtx {
  const ofp_cl* cl = nullptr;
  ClDev c;
  ofp_cl_view v;
  const unsigned long long* voff = nullptr;
  const uint32_t* vnbr = nullptr;
};

static int pair_ctx(const ofp_cl* cl, const ofp_vl* vl, int precision, double cutoff, PairCtx* x) {
  OFP_CHECK(cl, OFP_E_ARG, "null cell list");
  x->cl = cl;
  OFP_TRY(ofp_cl_dev_(cl, &x->c, &x->v));
  OFP_CHECK(precision == OFP_PREC_F64 || precision == OFP_PREC_F32C, OFP_E_ARG, "bad precision %d", precision);
  if (precision == OFP_PREC_F32C)
    OFP_CHECK(x->c.quant != nullptr, OFP_E_STATE, "FP32C pair kernels need a cell list built with OFP_CL_QUANT");
  if (vl) {
    OFP_TRY(ofp_vl_dev_(vl, cl, 0, &x->voff, &x->vnbr));
  } else {
    for (int k = 0; k < 3; ++k)
      OFP_CHECK(cutoff <= x->v.spacing[k] * x->c.box_nn * (1 + 1e-6), OFP_E_ARG,
                "cut-off %g larger than the stencil (%u x %g)", cutoff, x->c.box_nn, x->v.spacing[k]);
  }
  return OFP_OK;
}

// Persistent cell-tile launches: 8 workgroups of 4 waves per CU.
static unsigned tile_grid() {
  static unsigned g = 0;
  if (!g) {
    int dev = 0, ncu = 256;
    if (ofp_device_info(&dev, &ncu, nullptr, 0) != OFP_OK || ncu <= 0) ncu = 256;
    g = queue_grid(unsigned(ncu) * 8u, kTileWaves);
  }
  return g;
}

struct TileQueue {
  const TargetItem* items = nullptr;
  const uint32_t* n_items = nullptr;
  uint32_t* counter = nullptr;
};

// The cell list's item queue with its consumer head cleared (by a kernel, so a
// caller may capture the launch in a graph).
static int tile_queue(const PairCtx& x, TileQueue* q, hipStream_t s) {
  size_t cap = 0;
  OFP_TRY(ofp_cl_items_(x.cl, &q->items, &q->n_items, &q->counter, &cap, s));
  return fill_u32(q->counter, 0, kQueueWords, s);
}

// Verlet-row launches: kRowLanes lanes per domain row.
static unsigned pair_grid(const PairCtx& x) { return grid_for(size_t(x.c.n_dom) * kRowLanes, 256); }

// With a Verlet list: its rows; without: the cell tiles of the cell list.
template <class Ph>
static int launch_f64(const PairCtx& x, const void* pos, size_t stride, const Ph& ph, hipStream_t s) {
  if (x.c.n_dom == 0) return OFP_OK;
  OFP_CHECK(pos, OFP_E_ARG, "null sorted positions");
  OFP_CHECK(stride >= x.v.n_part, OFP_E_ARG, "stride < n_part");
  auto go = [&](auto tag) -> int {
    using T = decltype(tag);
    const T* P = static_cast<const T*>(pos);
    if (x.voff) {
      if constexpr (Ph::kSmooth)
        k_rows_smooth<<<pair_grid(x), 256, 0, s>>>(x.c, x.voff, x.vnbr, PlainRows<T, Ph>{P, stride, ph});
      else
        k_pairs_f64<T, Ph><<<pair_grid(x), 256, 0, s>>>(x.c, P, stride, x.voff, x.vnbr, ph);
    } else {
      TileQueue q;
      OFP_TRY(tile_queue(x, &q, s));
      k_tile_f64<T, Ph, false><<<tile_grid(), kTileBlock, 0, s>>>(
          x.c, P, stride, x.v.spacing[0], x.v.spacing[1], x.v.spacing[2], ph, nullptr, nullptr, q.items, q.n_items,
          q.counter);
    }
    OFP_LAUNCHED();
    return OFP_OK;
  };
  return x.v.dtype == OFP_F32 ? go(float(0)) : go(double(0));
}

static QGeom qgeom(const PairCtx& x) {
  QGeom q;
  q.ryd = x.v.spacing[1] / x.v.spacing[0];
  q.rzd = x.v.spacing[2] / x.v.spacing[0];
  q.ry = float(q.ryd);
  q.rz = float(q.rzd);
  return q;
}

static double q0_of(const PairCtx& x) { return x.v.spacing[0] / double(kQuantOne); }

// unit: the length unit of the pass in position units (q_0, or 1)
static Spline spline(double h, double unit) { return Spline{-0.5 * unit / h, -unit / h}; }

// The records the FP32C passes gather, made from the quantised stream: (q_x, q_y,
// q_z, aux), or without a value per particle the 12 bytes (q_x, q_y, q_z).  The
// rows' gathers are bound by the cache segments their lanes touch, and 12-byte
// records touch a quarter fewer: density over 4.4e9 entries 8.2 -> 7.2 ms, for
// 0.04 ms here.
__global__ void k_quant_rec(const int4* __restrict__ quant, uint32_t n, int3* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int4 q = quant[i];
  out[i] = make_int3(q.x, q.y, q.z);
}
__global__ void k_quant_rec_aux(const int4* __restrict__ quant, const float* __restrict__ aux, uint32_t n,
                                int4* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int4 q = quant[i];
  out[i] = make_int4(q.x, q.y, q.z, __float_as_int(aux[i]));
}

// rec: kSmooth physics over Verlet rows, int3 (null: the quantised stream) or
// (Ph::kAuxInQuant) int4 records;
// over cell tiles the int4 records (null: the quantised stream).
template <class Ph>
static int launch_f32c(const PairCtx& x, const Ph& ph, hipStream_t s, const void* rec = nullptr) {
  if (x.c.n_dom == 0) return OFP_OK;
  const unsigned grid = pair_grid(x);
  const QGeom qg = qgeom(x);
  const bool cubic = qg.ryd == 1.0 && qg.rzd == 1.0;
  if (x.voff) {
    if constexpr (Ph::kSmooth) {
      using R = typename QuantRows<Ph, true>::Rec;
      const R* r = static_cast<const R*>(rec);
      if constexpr (!Ph::kAuxInQuant) {
        if (!r) {
          if (cubic)
            k_rows_smooth<<<grid, 256, 0, s>>>(x.c, x.voff, x.vnbr, QuantRows<Ph, true, true>{x.c.quant, qg, ph});
          else
            k_rows_smooth<<<grid, 256, 0, s>>>(x.c, x.voff, x.vnbr, QuantRows<Ph, false, true>{x.c.quant, qg, ph});
          OFP_LAUNCHED();
          return OFP_OK;
        }
      }
      if (cubic)
        k_rows_smooth<<<grid, 256, 0, s>>>(x.c, x.voff, x.vnbr, QuantRows<Ph, true>{r, qg, ph});
      else
        k_rows_smooth<<<grid, 256, 0, s>>>(x.c, x.voff, x.vnbr, QuantRows<Ph, false>{r, qg, ph});
    } else {
      if (cubic)
        k_pairs_f32c<Ph, true><<<grid, 256, 0, s>>>(x.c, qg, x.voff, x.vnbr, ph);
      else
        k_pairs_f32c<Ph, false><<<grid, 256, 0, s>>>(x.c, qg, x.voff, x.vnbr, ph);
    }
  } else {
    TileQueue q;
    OFP_TRY(tile_queue(x, &q, s));
    const int4* r = rec ? static_cast<const int4*>(rec) : x.c.quant;
    if (cubic)
      k_tile_f32c<float, Ph, true, false><<<tile_grid(), kTileBlock, 0, s>>>(
          x.c, qg, ph, nullptr, nullptr, nullptr, r, q.items, q.n_items, q.counter);
    else
      k_tile_f32c<float, Ph, false, false><<<tile_grid(), kTileBlock, 0, s>>>(
          x.c, qg, ph, nullptr, nullptr, nullptr, r, q.items, q.n_items, q.counter);
  }
  OFP_LAUNCHED();
  return OFP_OK;
}

// pos: sorted positions of the pass (pstride apart, FP64 if pos_f64) for the
// close-pair refinement, or null.
// The forms of one physics with and without energy share their layout.
static_assert(sizeof(LJ64T<true>) == sizeof(LJ64T<false>) && sizeof(LJ32T<true>) == sizeof(LJ32T<false>));
template <class To, class From>
static To same_layout(const From& f) {
  static_assert(sizeof(To) == sizeof(From) && std::is_trivially_copyable_v<To>);
  To t;
  std::memcpy(&t, &f, sizeof(To));
  return t;
}

// The band of ExactCut for a cut-off r_cut (position units) compared with the
// FP32 square rc2f (q_0 units); qm = the largest quantum in q_0 units (1 for
// cubic cells).  Relative half-width: the quantisation bound at r = r_c with a
// 25 % margin, plus 2^-22 for the FP32 roundings of the square and of rc2f.
static int exact_cut(const void* pos, size_t pstride, int pos_f64, double r_cut, double rc2_pos, double q0,
                     double qm, float rc2f, ExactCut* xc) {
  OFP_CHECK(pos, OFP_E_ARG, "FP32C pair passes need the sorted positions (cut-off ties are decided on them)");
  const double R = r_cut / q0;
  const double rel = 1.25 * (2.0 * std::sqrt(3.0) * qm / R + 3.0 * qm * qm / (R * R)) + std::ldexp(1.0, -22);
  OFP_CHECK(rel < std::ldexp(1.0, -18), OFP_E_LIMIT, "cells too large for the cut-off %g (quantum band %g)", r_cut,
            rel);
  xc->pos = pos;
  xc->pstride = pstride;
  xc->pos_f64 = pos_f64;
  xc->lo2 = std::nextafter(float(double(rc2f) * (1.0 - rel)), 0.0f);
  xc->hi2 = std::nextafter(float(double(rc2f) * (1.0 + rel)), INFINITY);
  xc->rc2 = rc2_pos;
  return OFP_OK;
}

static double quantum_ratio(double ryd, double rzd) { return std::max(1.0, std::max(ryd, rzd)); }

static int lj32_of(const ofp_lj_params& prm, double q0, double qm, const void* pos, size_t pstride, int pos_f64,
                   LJ32* out) {
  LJ32 ph;
  std::memset(&ph, 0, sizeof(ph));
  const double s = prm.sigma / q0;
  ph.rc2 = float((prm.r_cut / q0) * (prm.r_cut / q0));
  ph.sig2 = s * s;
  ph.fscale = 24.0 * prm.eps / q0;
  ph.uscale = 4.0 * prm.eps;
  OFP_TRY(exact_cut(pos, pstride, pos_f64, prm.r_cut, prm.r_cut * prm.r_cut, q0, qm, ph.rc2, &ph.xc));
  ph.inv_q0 = 1.0 / q0;
  ph.close2 = float(s * s);
  *out = ph;
  return OFP_OK;
}

// Device address of this GPU's `scratch` array, looked up once per device
// (with that device current) by hipGetSymbolAddress and kept.  Each GPU holds
// its own copy of the array at its own address.
constexpr int kMaxDevices = 64;
static int reduce_scratch(double** out) {
  static std::mutex mu;
  static double* addr[kMaxDevices] = {};
  int dev = 0;
  OFP_HIP(hipGetDevice(&dev));
  OFP_CHECK(dev >= 0 && dev < kMaxDevices, OFP_E_ARG, "device %d beyond the %d this library serves", dev,
            kMaxDevices);
  std::lock_guard<std::mutex> lk(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_error(OFP_E_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
    addr[dev] = static_cast<double*>(p);
  }
  *out = addr[dev];
  return OFP_OK;
}

}  // namespace ofp

using namespace ofp;

// Per-system constant tables of the ensemble LJ pass (device memory).
// spacing = 3 cell spacings per system; outputs are shared by all systems.
int ofp::lj_tables_many(int precision, uint32_t n_sys, const ofp_lj_params* prm, const double* spacing, void* fx,
                        void* fy, void* fz, void* energy, uint32_t* n_neigh, const void* pos_sorted,
                        size_t pstride, int pos_f64, DevBuf* tab, DevBuf* qtab, int* all_cubic) {
  OFP_CHECK(precision == OFP_PREC_F64 || precision == OFP_PREC_F32C, OFP_E_ARG, "bad precision %d", precision);
  if (all_cubic) {
    *all_cubic = 1;
    for (uint32_t s = 0; s < n_sys; ++s)
      if (spacing[3 * s + 1] != spacing[3 * s] || spacing[3 * s + 2] != spacing[3 * s]) *all_cubic = 0;
  }
  if (precision == OFP_PREC_F64) {
    std::vector<LJ64> t(n_sys);
    for (uint32_t s = 0; s < n_sys; ++s)
      t[s] = LJ64{prm[s].r_cut * prm[s].r_cut, prm[s].sigma * prm[s].sigma, 24.0 * prm[s].eps, 4.0 * prm[s].eps,
                  (double*)fx, (double*)fy, (double*)fz, (double*)energy, n_neigh};
    OFP_TRY(tab->ensure(t.size() * sizeof(LJ64)));
    OFP_HIP(hipMemcpy(tab->p, t.data(), t.size() * sizeof(LJ64), hipMemcpyHostToDevice));
    return OFP_OK;
  }
  std::vector<LJ32> t(n_sys);
  std::vector<QGeom> q(n_sys);
  for (uint32_t s = 0; s < n_sys; ++s) {
    const double q0 = spacing[3 * s] / double(kQuantOne);
    const double qm = quantum_ratio(spacing[3 * s + 1] / spacing[3 * s], spacing[3 * s + 2] / spacing[3 * s]);
    OFP_TRY(lj32_of(prm[s], q0, qm, pos_sorted, pstride, pos_f64, &t[s]));
    t[s].fx = (float*)fx;
    t[s].fy = (float*)fy;
    t[s].fz = (float*)fz;
    t[s].en = (float*)energy;
    t[s].nn = n_neigh;
    q[s].ryd = spacing[3 * s + 1] / spacing[3 * s];
    q[s].rzd = spacing[3 * s + 2] / spacing[3 * s];
    q[s].ry = float(q[s].ryd);
    q[s].rz = float(q[s].rzd);
  }
  OFP_TRY(tab->ensure(t.size() * sizeof(LJ32)));
  OFP_TRY(qtab->ensure(q.size() * sizeof(QGeom)));
  OFP_HIP(hipMemcpy(tab->p, t.data(), t.size() * sizeof(LJ32), hipMemcpyHostToDevice));
  OFP_HIP(hipMemcpy(qtab->p, q.data(), q.size() * sizeof(QGeom), hipMemcpyHostToDevice));
  return OFP_OK;
}

// Lanes per row as a compile-time constant: f(std::integral_constant<int, L>).
template <class F>
static void with_lanes(int lanes, F&& f) {
  switch (lanes) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 16: f(std::integral_constant<int, 16>{}); break;
    case 32: f(std::integral_constant<int, 32>{}); break;
    default: break;
  }
}

// A kick applies to positions of its own dtype only.
template <class K, class T>
constexpr bool kick_fits() {
  if constexpr (K::kOn)
    return std::is_same<typename K::Tv, T>::value;
  else
    return true;
}

// The table memory holds LJ32 / LJ64 (kU = true); the forces-only forms read
// the same bytes (same layout).
template <bool kU, class K>
static void launch_lj_many(const PairCtx& x, int dtype, int precision, const void* pos_sorted, size_t stride,
                           const void* tab, const void* qtab, const uint32_t* sid, int lanes, unsigned long long el,
                           bool cubic, const K& kick, hipStream_t s) {
  const unsigned grid = grid_for(size_t(x.c.n_dom) * unsigned(lanes), 256);
  const auto* vo = x.voff;
  const auto* vn = x.vnbr;
  with_lanes(lanes, [&](auto L) {
    constexpr int kL = decltype(L)::value;
    if (precision == OFP_PREC_F32C) {
      using Ph = LJ32T<kU>;
      const Ph* t = static_cast<const Ph*>(tab);
      const QGeom* q = static_cast<const QGeom*>(qtab);
      auto go = [&](auto T0) {
        using T = decltype(T0);
        const T* sr = static_cast<const T*>(pos_sorted);
        if constexpr (kick_fits<K, T>()) {
          if (cubic)
            k_pairs_many_f32c<T, Ph, kL, true, K><<<grid, 256, 0, s>>>(x.c, t, q, sid, vo, vn, el, sr, stride, kick);
          else
            k_pairs_many_f32c<T, Ph, kL, false, K><<<grid, 256, 0, s>>>(x.c, t, q, sid, vo, vn, el, sr, stride,
                                                                        kick);
        }
      };
      if (dtype == OFP_F32)
        go(float(0));
      else
        go(double(0));
    } else {
      using Ph = LJ64T<kU>;
      const Ph* t = static_cast<const Ph*>(tab);
      if (dtype == OFP_F32) {
        if constexpr (kick_fits<K, float>())
          k_pairs_many_f64<float, Ph, kL, K><<<grid, 256, 0, s>>>(x.c, t, sid, static_cast<const float*>(pos_sorted),
                                                                  stride, vo, vn, el, kick);
      } else {
        if constexpr (kick_fits<K, double>())
          k_pairs_many_f64<double, Ph, kL, K><<<grid, 256, 0, s>>>(
              x.c, t, sid, static_cast<const double*>(pos_sorted), stride, vo, vn, el, kick);
      }
    }
  });
}

// Ensemble LJ over the cell tiles of the last build's cells (no Verlet list):
// one persistent launch over the (system, cell tile) item queue.
template <bool kU, class T>
static int launch_lj_tiles(const PairCtx& x, int precision, const void* pos_sorted, size_t stride, const void* tab,
                           const void* qtab, const void* sysgrid, bool cubic, hipStream_t s) {
  TileQueue q;
  OFP_TRY(tile_queue(x, &q, s));
  const SysGrid<T>* sys = static_cast<const SysGrid<T>*>(sysgrid);
  if (precision == OFP_PREC_F32C) {
    using Ph = LJ32T<kU>;
    const Ph* t = static_cast<const Ph*>(tab);
    const QGeom* qt = static_cast<const QGeom*>(qtab);
    if (cubic)
      k_tile_f32c<T, Ph, true, true><<<tile_grid(), kTileBlock, 0, s>>>(x.c, QGeom{}, Ph{}, t, qt, sys, x.c.quant,
                                                                         q.items, q.n_items, q.counter);
    else
      k_tile_f32c<T, Ph, false, true><<<tile_grid(), kTileBlock, 0, s>>>(x.c, QGeom{}, Ph{}, t, qt, sys, x.c.quant,
                                                                          q.items, q.n_items, q.counter);
  } else {
    using Ph = LJ64T<kU>;
    k_tile_f64<T, Ph, true><<<tile_grid(), kTileBlock, 0, s>>>(x.c, static_cast<const T*>(pos_sorted), stride, 0.0,
                                                               0.0, 0.0, Ph{},
                                                               static_cast<const Ph*>(tab), sys, q.items, q.n_items,
                                                               q.counter);
  }
  OFP_LAUNCHED();
  return OFP_OK;
}

int ofp::pair_lj_many(const ofp_cl* cl, const ofp_vl* vl, int dtype, const void* pos_sorted, size_t stride,
                      int precision, const void* tab, const void* qtab, int lanes, size_t e_cap, int with_u,
                      int cubic, bool one_system, hipStream_t s, const void* sysgrid, const void* kick,
                      const void* quant) {
  PairCtx x;
  OFP_TRY(pair_ctx(cl, vl, precision, 0.0, &x));
  if (quant) x.c.quant = static_cast<const int4*>(quant);
  const uint32_t* sid = nullptr;
  OFP_TRY(cl_sid_sorted(cl, &sid));
  if (one_system) sid = nullptr;
  if (x.c.n_dom == 0) return OFP_OK;
  if (!vl) {
    OFP_CHECK(sysgrid, OFP_E_ARG, "ensemble cell-tile pass needs the systems' grids");
    OFP_CHECK(!kick, OFP_E_ARG, "the cell-tile pass stores its forces (no fused kick)");
    if (dtype == OFP_F32)
      return with_u ? launch_lj_tiles<true, float>(x, precision, pos_sorted, stride, tab, qtab, sysgrid, cubic, s)
                    : launch_lj_tiles<false, float>(x, precision, pos_sorted, stride, tab, qtab, sysgrid, cubic, s);
    return with_u ? launch_lj_tiles<true, double>(x, precision, pos_sorted, stride, tab, qtab, sysgrid, cubic, s)
                  : launch_lj_tiles<false, double>(x, precision, pos_sorted, stride, tab, qtab, sysgrid, cubic, s);
  }
  OFP_CHECK(lanes == 1 || lanes == 2 || lanes == 4 || lanes == 8 || lanes == 16 || lanes == 32, OFP_E_ARG,
            "lanes per row must be 1, 2, 4, 8, 16 or 32 (got %d)", lanes);
  if (kick) {
    OFP_CHECK(!with_u, OFP_E_ARG, "a fused kick writes no energies");
    if (dtype == OFP_F32)
      launch_lj_many<false>(x, dtype, precision, pos_sorted, stride, tab, qtab, sid, lanes, e_cap, cubic != 0,
                            *static_cast<const StepKick<float>*>(kick), s);
    else
      launch_lj_many<false>(x, dtype, precision, pos_sorted, stride, tab, qtab, sid, lanes, e_cap, cubic != 0,
                            *static_cast<const StepKick<double>*>(kick), s);
  } else if (with_u) {
    launch_lj_many<true>(x, dtype, precision, pos_sorted, stride, tab, qtab, sid, lanes, e_cap, cubic != 0, NoKick{},
                         s);
  } else {
    launch_lj_many<false>(x, dtype, precision, pos_sorted, stride, tab, qtab, sid, lanes, e_cap, cubic != 0, NoKick{},
                          s);
  }
  OFP_LAUNCHED();
  return OFP_OK;
}

// LJ over a symmetric list (each interaction once): one wave per row, lanes over
// the row's entries; the pair force goes to the row's particle (+f, summed over
// the wave) and to the neighbour (-f) by FP64 atomic adds, and both neighbour
// counts are incremented.  fx/fy/fz/nn hold every particle, ghosts included
// (sorted index), and start at zero.
template <class T>
__global__ __launch_bounds__(256) void k_lj_sym(const T* __restrict__ pos, size_t stride,
                                                const unsigned long long* __restrict__ off,
                                                const uint32_t* __restrict__ nbr, uint64_t n_rows,
                                                const uint32_t* __restrict__ dom, double rc2, double sig2,
                                                double eps24, double* __restrict__ fx, double* __restrict__ fy,
                                                double* __restrict__ fz, uint32_t* __restrict__ nn) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t r = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) / kWave;
  if (r >= n_rows) return;  // wave-uniform
  const uint32_t i = dom[r];
  const double xi = double(pos[i]), yi = double(pos[stride + i]), zi = double(pos[2 * stride + i]);
  double sx = 0.0, sy = 0.0, sz = 0.0;
  uint32_t cnt = 0;
  const uint64_t e1 = off[r + 1];
  for (uint64_t e = off[r] + uint64_t(lane); e < e1; e += kWave) {
    const uint32_t j = nbr[e];
    const double rx = xi - double(pos[j]), ry = yi - double(pos[stride + j]), rz = zi - double(pos[2 * stride + j]);
    const double d2 = rx * rx + ry * ry + rz * rz;
    if (d2 < rc2) {
      ++cnt;
      if (nn) atomicAdd(nn + j, 1u);
      if (d2 > 0.0) {
        const double inv = 1.0 / d2;
        const double s2 = sig2 * inv;
        const double s6 = s2 * s2 * s2;
        const double f = eps24 * (2.0 * s6 * s6 - s6) * inv;
        sx += f * rx;
        sy += f * ry;
        sz += f * rz;
        unsafeAtomicAdd(fx + j, -f * rx);
        unsafeAtomicAdd(fy + j, -f * ry);
        unsafeAtomicAdd(fz + j, -f * rz);
      }
    }
  }
  for (int d = kWave / 2; d > 0; d >>= 1) {
    sx += __shfl_xor(sx, d);
    sy += __shfl_xor(sy, d);
    sz += __shfl_xor(sz, d);
    cnt += __shfl_xor(cnt, d);
  }
  if (lane == 0) {
    unsafeAtomicAdd(fx + i, sx);
    unsafeAtomicAdd(fy + i, sy);
    unsafeAtomicAdd(fz + i, sz);
    if (nn) atomicAdd(nn + i, cnt);
  }
}

__global__ void k_zero_f64(double* __restrict__ p, size_t n) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0;
}

extern "C" {

int ofp_pair_lj_sym(const ofp_cl* cl, const ofp_vl* vl, const void* pos, size_t stride, const ofp_lj_params* prm,
                    double* fx, double* fy, double* fz, uint32_t* n_neigh, void* stream) {
  OFP_CHECK(cl && vl && pos && prm && fx && fy && fz, OFP_E_ARG, "ofp_pair_lj_sym: null argument");
  ClDev c;
  ofp_cl_view v;
  OFP_TRY(ofp_cl_dev_(cl, &c, &v));
  const unsigned long long* off = nullptr;
  const uint32_t* nbr = nullptr;
  OFP_TRY(ofp_vl_dev_(vl, cl, 1, &off, &nbr));
  OFP_CHECK(stride >= v.n_part, OFP_E_ARG, "stride < particles");
  hipStream_t s = as_stream(stream);
  const size_t n = v.n_part;
  if (n == 0) return OFP_OK;
  double* outs[3] = {fx, fy, fz};
  for (double* o : outs) {
    k_zero_f64<<<grid_for(n, 256), 256, 0, s>>>(o, n);
    OFP_LAUNCHED();
  }
  if (n_neigh) OFP_TRY(fill_u32(n_neigh, 0u, n, s));
  const uint64_t rows = v.ghost_marker;
  if (rows == 0) return OFP_OK;
  const unsigned grid = grid_for(rows * kWave, 256);
  const double rc2 = prm->r_cut * prm->r_cut, sig2 = prm->sigma * prm->sigma, eps24 = 24.0 * prm->eps;
  if (v.dtype == OFP_F32)
    k_lj_sym<float><<<grid, 256, 0, s>>>(static_cast<const float*>(pos), stride, off, nbr, rows, v.dom_sort_ids,
                                         rc2, sig2, eps24, fx, fy, fz, n_neigh);
  else
    k_lj_sym<double><<<grid, 256, 0, s>>>(static_cast<const double*>(pos), stride, off, nbr, rows, v.dom_sort_ids,
                                          rc2, sig2, eps24, fx, fy, fz, n_neigh);
  OFP_LAUNCHED();
  return OFP_OK;
}

int ofp_pair_lj(const ofp_cl* cl, const ofp_vl* vl, const void* pos, size_t stride, int precision,
                const ofp_lj_params* prm, void* fx, void* fy, void* fz, void* energy, uint32_t* n_neigh,
                void* stream) {
  OFP_CHECK(prm, OFP_E_ARG, "ofp_pair_lj: null parameters");
  OFP_CHECK((fx && fy && fz) || (!fx && !fy && !fz), OFP_E_ARG, "force planes: all or none");
  PairCtx x;
  OFP_TRY(pair_ctx(cl, vl, precision, prm->r_cut, &x));
  hipStream_t s = as_stream(stream);
  const bool with_u = energy || n_neigh;  // otherwise the forces-only kernels
  if (precision == OFP_PREC_F64) {
    LJ64 ph{prm->r_cut * prm->r_cut, prm->sigma * prm->sigma, 24.0 * prm->eps, 4.0 * prm->eps,
            (double*)fx, (double*)fy, (double*)fz, (double*)energy, n_neigh};
    return with_u ? launch_f64(x, pos, stride, ph, s)
                  : launch_f64(x, pos, stride, same_layout<LJ64T<false>>(ph), s);
  }
  const double q0 = q0_of(x);
  const QGeom qg = qgeom(x);
  LJ32 ph;
  OFP_TRY(lj32_of(*prm, q0, quantum_ratio(qg.ryd, qg.rzd), pos, stride, x.v.dtype == OFP_F64 ? 1 : 0, &ph));
  ph.fx = (float*)fx;
  ph.fy = (float*)fy;
  ph.fz = (float*)fz;
  ph.en = (float*)energy;
  ph.nn = n_neigh;
  return with_u ? launch_f32c(x, ph, s) : launch_f32c(x, same_layout<LJ32T<false>>(ph), s);
}

int ofp_sph_density(const ofp_cl* cl, const ofp_vl* vl, const void* pos, size_t stride, int precision,
                    const ofp_sph_params* prm, void* rho, void* stream) {
  OFP_CHECK(prm && rho, OFP_E_ARG, "ofp_sph_density: null argument");
  PairCtx x;
  const double h = prm->h;
  OFP_TRY(pair_ctx(cl, vl, precision, 2 * h, &x));
  hipStream_t s = as_stream(stream);
  const double sk_m = prm->mass / (M_PI * h * h * h);
  if (precision == OFP_PREC_F64) {
    Dens64 ph{4 * h * h, spline(h, 1.0), sk_m, (double*)rho};
    return launch_f64(x, pos, stride, ph, s);
  }
  const double q0 = q0_of(x);
  const QGeom qg = qgeom(x);
  Dens32 ph;
  ph.rc2 = float((2 * h / q0) * (2 * h / q0));
  ExactCut xc;  // its limits on the cut-off hold for every FP32C pass
  OFP_TRY(exact_cut(pos, stride, x.v.dtype == OFP_F64 ? 1 : 0, 2 * h, 4 * h * h, q0, quantum_ratio(qg.ryd, qg.rzd),
                    ph.rc2, &xc));
  ph.sp = spline(h, q0);
  ph.sk_m = sk_m;
  ph.rho = (double*)rho;
  void* rec = nullptr;
  if (x.voff && x.c.n_dom > 0) {
    OFP_TRY(ofp_vl_rec_(vl, (x.v.n_part + 1) * sizeof(int3), &rec, s));
    if (rec) {
      k_quant_rec<<<grid_for(x.v.n_part, 256), 256, 0, s>>>(x.c.quant, uint32_t(x.v.n_part),
                                                            static_cast<int3*>(rec));
      OFP_LAUNCHED();
    }
  }
  return launch_f32c(x, ph, s, rec);
}

int ofp_sph_eos(int precision, const void* rho, size_t n, const ofp_sph_params* prm, void* prs, void* pterm,
                void* stream) {
  OFP_CHECK(prm && (n == 0 || (rho && pterm)), OFP_E_ARG, "ofp_sph_eos: null argument");
  if (n == 0) return OFP_OK;
  hipStream_t s = as_stream(stream);
  const double B = prm->c0 * prm->c0 * prm->rho0 / 7.0;
  if (precision == OFP_PREC_F64)
    k_tait<double><<<grid_for(n, 256), 256, 0, s>>>((const double*)rho, n, 1.0 / prm->rho0, B, (double*)prs,
                                                    (double*)pterm);
  else if (precision == OFP_PREC_F32C)
    k_tait<float><<<grid_for(n, 256), 256, 0, s>>>((const double*)rho, n, 1.0 / prm->rho0, B, (double*)prs,
                                                   (float*)pterm);
  else
    return set_error(OFP_E_ARG, "bad precision %d", precision);
  OFP_LAUNCHED();
  return OFP_OK;
}

int ofp_sph_force(const ofp_cl* cl, const ofp_vl* vl, const void* pos, size_t stride, int precision,
                  const ofp_sph_params* prm, const void* pterm, void* fx, void* fy, void* fz, void* stream) {
  OFP_CHECK(prm && pterm && fx && fy && fz, OFP_E_ARG, "ofp_sph_force: null argument");
  PairCtx x;
  const double h = prm->h;
  OFP_TRY(pair_ctx(cl, vl, precision, 2 * h, &x));
  hipStream_t s = as_stream(stream);
  const double sd_m = prm->mass / (M_PI * h * h * h * h);
  if (precision == OFP_PREC_F64) {
    Force64 ph{4 * h * h, spline(h, 1.0), 3.0 * sd_m, (const double*)pterm, (double*)fx, (double*)fy, (double*)fz};
    return launch_f64(x, pos, stride, ph, s);
  }
  const double q0 = q0_of(x);
  const QGeom qg = qgeom(x);
  Force32 ph;
  ph.rc2 = float((2 * h / q0) * (2 * h / q0));
  ExactCut xc;
  OFP_TRY(exact_cut(pos, stride, x.v.dtype == OFP_F64 ? 1 : 0, 2 * h, 4 * h * h, q0, quantum_ratio(qg.ryd, qg.rzd),
                    ph.rc2, &xc));
  ph.sp = spline(h, q0);
  ph.cut2 = (2 * h / q0) * (2 * h / q0);
  ph.fscale = 3.0 * sd_m;
  ph.pterm = (const float*)pterm;
  ph.fx = (float*)fx;
  ph.fy = (float*)fy;
  ph.fz = (float*)fz;
  void* rec = nullptr;
  if (x.c.n_dom > 0) {
    if (x.voff)
      OFP_TRY(ofp_vl_aux_(vl, (x.v.n_part + 1) * sizeof(int4), &rec));
    else
      OFP_TRY(ofp_cl_aux_(cl, (x.v.n_part + 1) * sizeof(int4), &rec));
    k_quant_rec_aux<<<grid_for(x.v.n_part, 256), 256, 0, s>>>(x.c.quant, (const float*)pterm, uint32_t(x.v.n_part),
                                                              static_cast<int4*>(rec));
    OFP_LAUNCHED();
  }
  return launch_f32c(x, ph, s, rec);
}

int ofp_reduce(int dtype, const void* x, const void* comp, size_t n, int op, double* result, void* stream) {
  OFP_CHECK(result, OFP_E_ARG, "ofp_reduce: null result");
  OFP_CHECK(n == 0 || x, OFP_E_ARG, "ofp_reduce: null input");
  OFP_CHECK(op == OFP_RED_SUM || op == OFP_RED_MAX || op == OFP_RED_MIN, OFP_E_ARG, "bad op %d", op);
  const double ident = op == OFP_RED_SUM ? 0.0 : (op == OFP_RED_MAX ? -INFINITY : INFINITY);
  if (n == 0) {
    *result = ident;
    return OFP_OK;
  }
  hipStream_t s = as_stream(stream);
  unsigned grid = grid_for(n, kRedBlock);
  if (grid > kRedGrid) grid = kRedGrid;
  double* partial = nullptr;
  OFP_HIP(hipMallocAsync(reinterpret_cast<void**>(&partial), (grid + 1) * sizeof(double), s));
  if (dtype == OFP_F32)
    k_reduce_partial<float><<<grid, kRedBlock, 0, s>>>((const float*)x, (const float*)comp, n, op, ident, partial);
  else if (dtype == OFP_F64)
    k_reduce_partial<double><<<grid, kRedBlock, 0, s>>>((const double*)x, (const double*)comp, n, op, ident,
                                                        partial);
  else {
    (void)hipFreeAsync(partial, s);
    return set_error(OFP_E_ARG, "bad dtype %d", dtype);
  }
  OFP_LAUNCHED();
  k_reduce_final<<<1, kRedBlock, 0, s>>>(partial, grid, op, ident, partial + grid);
  OFP_LAUNCHED();
  double r = 0;
  OFP_HIP(hipMemcpyAsync(&r, partial + grid, sizeof(double), hipMemcpyDeviceToHost, s));
  OFP_HIP(hipFreeAsync(partial, s));
  OFP_HIP(hipStreamSynchronize(s));
  *result = r;
  return OFP_OK;
}

int ofp_reduce_noalloc(int dtype, const void* x, const void* comp, size_t n, int op, double* result_dev,
                       void* stream) {
  OFP_CHECK(result_dev, OFP_E_ARG, "ofp_reduce_noalloc: null result");
  OFP_CHECK(n == 0 || x, OFP_E_ARG, "ofp_reduce_noalloc: null input");
  OFP_CHECK(op == OFP_RED_SUM || op == OFP_RED_MAX || op == OFP_RED_MIN, OFP_E_ARG, "bad op %d", op);
  OFP_CHECK(dtype == OFP_F32 || dtype == OFP_F64, OFP_E_ARG, "bad dtype %d", dtype);
  OFP_CHECK(n <= OFP_REDUCE_NOALLOC_MAX_N, OFP_E_ARG,
            "ofp_reduce_noalloc: %zu elements exceed the maximum of %llu", n,
            static_cast<unsigned long long>(OFP_REDUCE_NOALLOC_MAX_N));
  double* part = nullptr;
  OFP_TRY(reduce_scratch(&part));
  hipStream_t s = as_stream(stream);
  const double ident = op == OFP_RED_SUM ? 0.0 : (op == OFP_RED_MAX ? -INFINITY : INFINITY);
  // the same grid as ofp_reduce (so the same partials and the same result)
  unsigned grid = n ? grid_for(n, kRedBlock) : 0;
  if (grid > kRedGrid) grid = kRedGrid;
  OFP_CHECK(size_t(grid) + 1 <= kRedScratch, OFP_E_ARG, "ofp_reduce_noalloc: %u partials exceed the scratch", grid);
  if (grid > 0) {
    if (dtype == OFP_F32)
      k_reduce_partial<float><<<grid, kRedBlock, 0, s>>>((const float*)x, (const float*)comp, n, op, ident, part);
    else
      k_reduce_partial<double><<<grid, kRedBlock, 0, s>>>((const double*)x, (const double*)comp, n, op, ident,
                                                          part);
    OFP_LAUNCHED();
  }
  // n == 0: no partials, the final kernel writes the identity
  k_reduce_final<<<1, kRedBlock, 0, s>>>(part, grid, op, ident, result_dev);
  OFP_LAUNCHED();
  return OFP_OK;
}

}  // extern "C"
