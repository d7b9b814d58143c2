// HIP kernels of the MI355X HemeLB timestep (gfx950).
//
// One thread updates one fluid site.  The state holds post-collision
// distributions f*(t) structure-of-arrays (f[d*np + x]); a step pulls the
// values streaming into every slot of a site (the reference pushes them,
// Code/lb/streamers/BulkStreamer.h:31-39), resolves wall and iolet links in
// registers with the reference's link priority (iolet first, then wall,
// StreamerTypeFactory.h:65-78), applies the BFL PostStep correction
// (BouzidiFirdaousLallemand.h:68-91) locally, collides (LBGK.h:140-174 or
// MRT.h:56-105) and writes f*(t+1) to its own slots.  Binary64 arithmetic is
// evaluated in the reference's SSE3 order without contraction, so the plain
// method reproduces the reference bit for bit (up to the sign of zero).
//
// The bandwidth-bound path uses no MFMA.  By default consecutive workgroups
// (dispatched round-robin over the XCDs) cover consecutive x planes of the
// Morton-ordered domain; an XCD-contiguous remap is one of the launch shapes
// the tuner measures.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "lbm_internal.h"

namespace hlb {
namespace {

// ---------------------------------------------------------------------------
// Lattice constants (Code/lb/lattices/D3Q15.h:15-56, D3Q19.h:14-49)
// ---------------------------------------------------------------------------
template <int Q> struct Lat;
template <> struct Lat<15> {
  static constexpr int c[15][3] = {
      {0, 0, 0},   {1, 0, 0},   {-1, 0, 0}, {0, 1, 0},  {0, -1, 0},
      {0, 0, 1},   {0, 0, -1},  {1, 1, 1},  {-1, -1, -1}, {1, 1, -1},
      {-1, -1, 1}, {1, -1, 1},  {-1, 1, -1}, {1, -1, -1}, {-1, 1, 1}};
  static constexpr double w[15] = {
      2.0 / 9.0,  1.0 / 9.0,  1.0 / 9.0,  1.0 / 9.0,  1.0 / 9.0,
      1.0 / 9.0,  1.0 / 9.0,  1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0,
      1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0};
  static constexpr int nmom = 11;
  // DHumieresD3Q15MRTBasis::REDUCED_MOMENT_BASIS (DHumieresD3Q15MRTBasis.h:41-53)
  static constexpr int M[11][15] = {
      {-2, -1, -1, -1, -1, -1, -1, 1, 1, 1, 1, 1, 1, 1, 1},
      {16, -4, -4, -4, -4, -4, -4, 1, 1, 1, 1, 1, 1, 1, 1},
      {0, -4, 4, 0, 0, 0, 0, 1, -1, 1, -1, 1, -1, 1, -1},
      {0, 0, 0, -4, 4, 0, 0, 1, -1, 1, -1, -1, 1, -1, 1},
      {0, 0, 0, 0, 0, -4, 4, 1, -1, -1, 1, 1, -1, -1, 1},
      {0, 2, 2, -1, -1, -1, -1, 0, 0, 0, 0, 0, 0, 0, 0},
      {0, 0, 0, 1, 1, -1, -1, 0, 0, 0, 0, 0, 0, 0, 0},
      {0, 0, 0, 0, 0, 0, 0, 1, 1, 1, 1, -1, -1, -1, -1},
      {0, 0, 0, 0, 0, 0, 0, 1, 1, -1, -1, -1, -1, 1, 1},
      {0, 0, 0, 0, 0, 0, 0, 1, 1, -1, -1, 1, 1, -1, -1},
      {0, 0, 0, 0, 0, 0, 0, 1, -1, -1, 1, -1, 1, 1, -1}};
};
template <> struct Lat<19> {
  static constexpr int c[19][3] = {
      {0, 0, 0},  {1, 0, 0},   {-1, 0, 0}, {0, 1, 0},  {0, -1, 0},
      {0, 0, 1},  {0, 0, -1},  {1, 1, 0},  {-1, -1, 0}, {1, -1, 0},
      {-1, 1, 0}, {1, 0, 1},   {-1, 0, -1}, {1, 0, -1}, {-1, 0, 1},
      {0, 1, 1},  {0, -1, -1}, {0, 1, -1}, {0, -1, 1}};
  static constexpr double w[19] = {
      1.0 / 3.0,  1.0 / 18.0, 1.0 / 18.0, 1.0 / 18.0, 1.0 / 18.0,
      1.0 / 18.0, 1.0 / 18.0, 1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0,
      1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0,
      1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0};
  static constexpr int nmom = 15;
  // DHumieresD3Q19MRTBasis::REDUCED_MOMENT_BASIS (DHumieresD3Q19MRTBasis.h:38-53)
  static constexpr int M[15][19] = {
      {-30, -11, -11, -11, -11, -11, -11, 8, 8, 8, 8, 8, 8, 8, 8, 8, 8, 8, 8},
      {12, -4, -4, -4, -4, -4, -4, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1},
      {0, -4, 4, 0, 0, 0, 0, 1, -1, 1, -1, 1, -1, 1, -1, 0, 0, 0, 0},
      {0, 0, 0, -4, 4, 0, 0, 1, -1, -1, 1, 0, 0, 0, 0, 1, -1, 1, -1},
      {0, 0, 0, 0, 0, -4, 4, 0, 0, 0, 0, 1, -1, -1, 1, 1, -1, -1, 1},
      {0, 2, 2, -1, -1, -1, -1, 1, 1, 1, 1, 1, 1, 1, 1, -2, -2, -2, -2},
      {0, -4, -4, 2, 2, 2, 2, 1, 1, 1, 1, 1, 1, 1, 1, -2, -2, -2, -2},
      {0, 0, 0, 1, 1, -1, -1, 1, 1, 1, 1, -1, -1, -1, -1, 0, 0, 0, 0},
      {0, 0, 0, -2, -2, 2, 2, 1, 1, 1, 1, -1, -1, -1, -1, 0, 0, 0, 0},
      {0, 0, 0, 0, 0, 0, 0, 1, 1, -1, -1, 0, 0, 0, 0, 0, 0, 0, 0},
      {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 1, -1, -1},
      {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 1, -1, -1, 0, 0, 0, 0},
      {0, 0, 0, 0, 0, 0, 0, 1, -1, 1, -1, -1, 1, -1, 1, 0, 0, 0, 0},
      {0, 0, 0, 0, 0, 0, 0, -1, 1, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1},
      {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, -1, -1, 1, -1, 1, 1, -1}};
};

// Inverse directions: both lattices pair d with d+1 for odd d
// (detail::compute_inverses, Lattice.h:49-69).
__host__ __device__ constexpr int inv_dir(int d) {
  return d == 0 ? 0 : ((d & 1) ? d + 1 : d - 1);
}

// Link masks hold direction d in bit d-1, so a pair (d, d+1) sits in bits
// (d-1, d): bit d-1 of pair_swap(x) is bit inv_dir(d)-1 of x.
__host__ __device__ constexpr uint32_t pair_swap(uint32_t x) {
  return ((x & 0x55555555u) << 1) | ((x >> 1) & 0x55555555u);
}

constexpr double kCs2 = 1.0 / 3.0;  // constants.h:41

template <int I, int N, typename F>
__device__ __forceinline__ void sfor(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    sfor<I + 1, N>(f);
  }
}

// acc + C*v for a lattice component C in {-1,0,1}; the zero term is dropped
// (it can only change the sign of an exact zero).
template <int C, typename T>
__device__ __forceinline__ T addc(T acc, T v) {
  if constexpr (C == 0) return acc;
  else if constexpr (C > 0) return acc + v;
  else return acc - v;
}

// (C0*a + C1*b) + C2*c as the reference evaluates the projection of the
// momentum on a lattice vector (Lattice.h:276-285).
template <int C0, int C1, int C2, typename T>
__device__ __forceinline__ T dotc(T a, T b, T c) {
  constexpr bool h0 = C0 != 0, h1 = C1 != 0, h2 = C2 != 0;
  const T s0 = C0 > 0 ? a : -a;
  const T s1 = C1 > 0 ? b : -b;
  const T s2 = C2 > 0 ? c : -c;
  if constexpr (h0 && h1 && h2) return (s0 + s1) + s2;
  else if constexpr (h0 && h1) return s0 + s1;
  else if constexpr (h0 && h2) return s0 + s2;
  else if constexpr (h1 && h2) return s1 + s2;
  else if constexpr (h0) return s0;
  else if constexpr (h1) return s1;
  else if constexpr (h2) return s2;
  else return T(0);
}

// a*b + c.  Binary32 (the reduced-precision forms, which follow no reference
// rounding) fuses it into one FMA; binary64 keeps the reference's separately
// rounded product and sum.
__device__ __forceinline__ float mad(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}
__device__ __forceinline__ double mad(double a, double b, double c) { return a * b + c; }

// 1/x in binary32: the hardware reciprocal (1 ulp).  (Binary64 formulas
// divide.)
__device__ __forceinline__ float recip(float x) { return __builtin_amdgcn_rcpf(x); }

// ---------------------------------------------------------------------------
// Storage: binary64 holds f; binary32/binary16 hold f - w_i*rho0.
// ---------------------------------------------------------------------------
template <typename S> struct Store;
template <> struct Store<double> {
  using T = double;
  static __device__ __forceinline__ double ld(const double* p) { return *p; }
  static __device__ __forceinline__ void st(double* p, double v) { *p = v; }
};
template <> struct Store<float> {
  using T = float;
  static __device__ __forceinline__ float ld(const float* p) { return *p; }
  static __device__ __forceinline__ void st(float* p, float v) { *p = v; }
};
template <> struct Store<_Float16> {
  using T = float;
  static __device__ __forceinline__ float ld(const _Float16* p) { return (float)*p; }
  static __device__ __forceinline__ void st(_Float16* p, float v) { *p = (_Float16)v; }
};

template <typename S> constexpr bool kShifted = !std::is_same<S, double>::value;

// ---------------------------------------------------------------------------
// Moments and equilibrium
// ---------------------------------------------------------------------------
// Lattice::CalculateDensityAndMomentum, SSE3 order (Lattice.h:119-178):
// lane 0 from 0 over even directions, lane 1 from the last (odd Q) direction
// over odd directions; result lane0 + lane1.  For shifted storage the same
// sums give rho - rho0 and the momentum.
template <int Q, typename T>
__device__ __forceinline__ void moments(const T (&f)[Q], T& rho, T& mx, T& my,
                                        T& mz) {
  static_assert(Q & 1, "odd lattices only");
  using L = Lat<Q>;
  T r0 = T(0), r1 = f[Q - 1];
  T x0 = T(0), y0 = T(0), z0 = T(0);
  T x1 = addc<L::c[Q - 1][0]>(T(0), f[Q - 1]);
  T y1 = addc<L::c[Q - 1][1]>(T(0), f[Q - 1]);
  T z1 = addc<L::c[Q - 1][2]>(T(0), f[Q - 1]);
  sfor<0, (Q - 1) / 2>([&](auto p) {
    constexpr int d = 2 * decltype(p)::value;
    r0 = r0 + f[d];
    r1 = r1 + f[d + 1];
    x0 = addc<L::c[d][0]>(x0, f[d]);
    x1 = addc<L::c[d + 1][0]>(x1, f[d + 1]);
    y0 = addc<L::c[d][1]>(y0, f[d]);
    y1 = addc<L::c[d + 1][1]>(y1, f[d + 1]);
    z0 = addc<L::c[d][2]>(z0, f[d]);
    z1 = addc<L::c[d + 1][2]>(z1, f[d + 1]);
  });
  rho = r0 + r1;
  mx = x0 + x1;
  my = y0 + y1;
  mz = z0 + z1;
}

// Common factors of Lattice::CalculateFeq, SSE3 variant (Lattice.h:236-270).
template <typename T>
struct FeqCoef {
  T t1, nine, mx, my, mz;
  __device__ __forceinline__ FeqCoef(T rho, T mx_, T my_, T mz_)
      : mx(mx_), my(my_), mz(mz_) {
    const T three_halves = T(3. / 2.) * ((mx * mx + my * my) + mz * mz);
    t1 = rho - three_halves / rho;
    const T rho_1 = T(1.) / rho;
    nine = T(9. / 2.);
    nine *= rho_1;
  }
  // f_eq[i] = w_i * ((t1 + nine*(e*e)) + 3*e)  (Lattice.h:271-320)
  template <int Q, int I>
  __device__ __forceinline__ T eq() const {
    using L = Lat<Q>;
    const T e = dotc<L::c[I][0], L::c[I][1], L::c[I][2]>(mx, my, mz);
    return T(L::w[I]) * ((t1 + nine * (e * e)) + T(3.) * e);
  }
};

// Shifted equilibrium feq_i - w_i*rho0 for reduced-precision storage, with
// drho = rho - rho0 carried separately (no cancellation against rho0).
template <typename T>
struct FeqShifted {
  T drho, q, nine, mx, my, mz;
  __device__ __forceinline__ FeqShifted(T drho_, T rho, T mx_, T my_, T mz_)
      : drho(drho_), mx(mx_), my(my_), mz(mz_) {
    const T inv = recip(rho);
    q = mad(T(-1.5) * mad(mz, mz, mad(my, my, mx * mx)), inv, drho);
    nine = T(4.5) * inv;
  }
  template <int Q, int I>
  __device__ __forceinline__ T eq() const {
    using L = Lat<Q>;
    const T e = dotc<L::c[I][0], L::c[I][1], L::c[I][2]>(mx, my, mz);
    return T(L::w[I]) * mad(T(3.), e, mad(nine, e * e, q));
  }
};

// ---------------------------------------------------------------------------
// Collision
// ---------------------------------------------------------------------------
template <int Q, typename T>
struct Hydro {
  T rho, mx, my, mz;  // rho is the full density (rho0 added back if shifted)
};

// d'Humieres relaxation rates (DHumieresD3Q15MRTBasis.cc:10-26,
// DHumieresD3Q19MRTBasis.cc:11-36); 0 marks the moments relaxed with 1/tau.
__host__ __device__ constexpr double mrt_rate(int Q, int k) {
  constexpr double r15[11] = {1.6, 1.2, 1.6, 1.6, 1.6, 0, 0, 0, 0, 0, 1.2};
  constexpr double r19[15] = {1.19, 1.4, 1.2, 1.2, 1.2, 0, 1.4, 0,
                              1.4,  0,   0,   0,   1.98, 1.98, 1.98};
  return Q == 15 ? r15[k] : r19[k];
}
// BASIS_TIMES_BASIS_TRANSPOSED (basis_helpers.h:14-26), exact in binary64.
template <int Q>
__host__ __device__ constexpr double mrt_diag(int k) {
  double acc = 0.0;
  for (int i = 0; i < Q; ++i) acc = acc + (double)Lat<Q>::M[k][i] * (double)Lat<Q>::M[k][i];
  return acc;
}

// Parity of MRT moment k under inversion of the directions, which come in
// opposite pairs (d, d+1), d odd: 1 when row k of the basis takes the same
// value on both directions of every pair, -1 when opposite values (and 0 on
// the rest direction), 0 when neither.
template <int Q>
__host__ __device__ constexpr int mrt_parity(int k) {
  bool even = true, odd = Lat<Q>::M[k][0] == 0;
  for (int d = 1; d < Q; d += 2) {
    if (Lat<Q>::M[k][d] != Lat<Q>::M[k][d + 1]) even = false;
    if (Lat<Q>::M[k][d] != -Lat<Q>::M[k][d + 1]) odd = false;
  }
  return even ? 1 : (odd ? -1 : 0);
}
template <int Q>
__host__ __device__ constexpr bool mrt_rows_have_parity() {
  for (int k = 0; k < Lat<Q>::nmom; ++k)
    if (mrt_parity<Q>(k) == 0) return false;
  return true;
}

// Sums over the binary32-rounded weights (exact, in binary64): sum_i w_i and
// sum_i w_i c_ix^2 (the same for y and z on both lattices).
template <int Q>
__host__ __device__ constexpr double rounded_weight_sum() {
  double s = 0.0;
  for (int i = 0; i < Q; ++i) s += (double)(float)Lat<Q>::w[i];
  return s;
}
template <int Q>
__host__ __device__ constexpr double rounded_weight_c2() {
  double s = 0.0;
  for (int i = 0; i < Q; ++i) s += (double)(float)Lat<Q>::w[i] * Lat<Q>::c[i][0] * Lat<Q>::c[i][0];
  return s;
}
// sum_i fl(3 w_i) c_ix^2 with the binary32 coefficients of the linear
// equilibrium term
template <int Q>
__host__ __device__ constexpr double rounded_3w_c2() {
  double s = 0.0;
  for (int i = 0; i < Q; ++i)
    s += (double)(float)(3.0 * Lat<Q>::w[i]) * Lat<Q>::c[i][0] * Lat<Q>::c[i][0];
  return s;
}
template <int Q>
__host__ __device__ constexpr bool pairs_opposite() {
  for (int i = 1; i < Q; i += 2)
    for (int k = 0; k < 3; ++k)
      if (Lat<Q>::c[i + 1][k] != -Lat<Q>::c[i][k]) return false;
  return true;
}

// LBGK of the shifted storage forms in binary32 (these follow no reference
// rounding).  Directions come in opposite pairs (d, d+1), so the moments are
// sums of pair sums and differences, and a pair's equilibria are A +- B with
// A = w (q + 9/2 e^2 / rho) and B = 3 w e, e = c_d . m.
// Conservation: with binary32 coefficients, sum_i w_i = W, sum_i w_i c_i c_i
// = G I and sum_i fl(3 w_i) c_i c_i = K I differ from 1, 1/3 and 1 by 1e-8 to
// 3e-8, so the equilibrium's mass and momentum are W q + (9/2) G m^2/rho and
// K m instead of drho and m.  Relaxing towards it would act as a body force
// of ~1e-8 m per step (a 2e-5 to 3e-5 velocity bias on the vessel tree).
// Two corrections of f_neq before the relaxation, both applied to f_neq,
// whose magnitude keeps them above the rounding of binary32:
// * EXACT (binary32 storage): the mass and momentum of the computed f_neq
//   are removed, n_d -= w_d (s0 + 3 c_d . s) with s0, s its sums; this also
//   removes the rounding noise of each collision (velocity 1e-7 from
//   binary64 on the tree after 10000 steps);
// * otherwise (binary16 storage, whose own rounding is 1e-3): only the
//   systematic amounts above, the mass one on the rest direction and the
//   momentum one split over the axis pairs (1e-6 in binary32 arithmetic),
//   at a fraction of the projection's instructions.
template <int Q, typename T, bool EXACT>
__device__ __forceinline__ Hydro<Q, T> collide_lbgk_shifted(T (&f)[Q], const StepArgs& a) {
  using L = Lat<Q>;
  static_assert(pairs_opposite<Q>(), "directions d and d+1 must be opposite");
  constexpr double W = rounded_weight_sum<Q>(), G = rounded_weight_c2<Q>();
  constexpr double K = rounded_3w_c2<Q>();
  T r = f[0], mx = T(0), my = T(0), mz = T(0);
  sfor<0, (Q - 1) / 2>([&](auto p) {
    constexpr int i = 2 * decltype(p)::value + 1;
    const T dd = f[i] - f[i + 1];
    r = r + (f[i] + f[i + 1]);
    mx = addc<L::c[i][0]>(mx, dd);
    my = addc<L::c[i][1]>(my, dd);
    mz = addc<L::c[i][2]>(mz, dd);
  });
  Hydro<Q, T> h;
  h.rho = T(a.rho0) + r;
  h.mx = mx;
  h.my = my;
  h.mz = mz;
  const T inv = recip(h.rho);
  const T m2 = mad(mz, mz, mad(my, my, mx * mx));
  const T q = mad(T(-1.5) * m2, inv, r);
  const T nine = T(4.5) * inv;
  const T om = T(a.omega_f);
  T n[Q];  // f_neq
  n[0] = f[0] - T(L::w[0]) * q;
  sfor<0, (Q - 1) / 2>([&](auto p) {
    constexpr int i = 2 * decltype(p)::value + 1;
    const T e = dotc<L::c[i][0], L::c[i][1], L::c[i][2]>(mx, my, mz);
    const T A = mad(T(L::w[i]) * nine, e * e, T(L::w[i]) * q);
    const T B = T(3.0 * L::w[i]) * e;
    n[i] = (f[i] - A) - B;
    n[i + 1] = (f[i + 1] - A) + B;
  });
  if constexpr (EXACT) {
    T s0 = n[0], sx = T(0), sy = T(0), sz = T(0);
    sfor<0, (Q - 1) / 2>([&](auto p) {
      constexpr int i = 2 * decltype(p)::value + 1;
      const T dd = n[i] - n[i + 1];
      s0 = s0 + (n[i] + n[i + 1]);
      sx = addc<L::c[i][0]>(sx, dd);
      sy = addc<L::c[i][1]>(sy, dd);
      sz = addc<L::c[i][2]>(sz, dd);
    });
    sx = T(3) * sx;
    sy = T(3) * sy;
    sz = T(3) * sz;
    n[0] = mad(T(-L::w[0]), s0, n[0]);
    sfor<0, (Q - 1) / 2>([&](auto p) {
      constexpr int i = 2 * decltype(p)::value + 1;
      const T e = dotc<L::c[i][0], L::c[i][1], L::c[i][2]>(sx, sy, sz);
      n[i] = mad(T(-L::w[i]), s0 + e, n[i]);
      n[i + 1] = mad(T(-L::w[i + 1]), s0 - e, n[i + 1]);
    });
  } else {
    // systematic mass of f_neq: drho - (W q + (9/2) G m^2/rho)
    n[0] = n[0] - mad(T(1.0 - W), r, T(1.5 * W - 4.5 * G) * (m2 * inv));
    // systematic momentum of f_neq: (1 - K) m, half on each axis direction
    constexpr double kHalf = 0.5 * (1.0 - K);
    sfor<0, (Q - 1) / 2>([&](auto p) {
      constexpr int i = 2 * decltype(p)::value + 1;
      constexpr int cx = L::c[i][0], cy = L::c[i][1], cz = L::c[i][2];
      if constexpr (cx * cx + cy * cy + cz * cz == 1) {
        const T k = T(kHalf) * (cx != 0 ? mx : cy != 0 ? my : mz) * T(cx + cy + cz);
        n[i] = n[i] - k;
        n[i + 1] = n[i + 1] + k;
      }
    });
  }
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    f[d] = mad(om, n[d], f[d]);
  });
  return h;
}

// MRT relaxation of the shifted storage forms in binary32 (these follow no
// reference rounding): the same m_neq = M f_neq and f* = f - sum_k (S_k N_kd)
// m_neq_k as the binary64 form, with the rows of the d'Humieres basis
// grouped by their parity under inversion.  An even row needs the rest value
// and the pair sums of f_neq, an odd row the pair differences; the
// relaxation of pair (d, d+1) is E + O on d and E - O on d+1, with E the
// even moments' part and O the odd moments'.  About half the operations of
// the row-by-column form.
template <int Q, typename T>
__device__ __forceinline__ void mrt_relax_pairs(const T (&fneq)[Q], const StepArgs& a,
                                                T (&f)[Q]) {
  using L = Lat<Q>;
  static_assert(pairs_opposite<Q>() && mrt_rows_have_parity<Q>(),
                "MRT pair form: opposite direction pairs and rows of definite parity");
  constexpr int NM = L::nmom;
  T sg[Q], df[Q];  // pair sums and differences, at the pair's first direction
  sfor<1, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    if constexpr (d % 2 == 1) {
      sg[d] = fneq[d] + fneq[d + 1];
      df[d] = fneq[d] - fneq[d + 1];
    }
  });
  T mneq[NM];
  sfor<0, NM>([&](auto ki) {
    constexpr int k = decltype(ki)::value;
    constexpr bool even = mrt_parity<Q>(k) == 1;
    T acc = T(0.);
    if constexpr (even && L::M[k][0] != 0) acc = T(L::M[k][0]) * fneq[0];
    sfor<1, Q>([&](auto di) {
      constexpr int d = decltype(di)::value;
      constexpr int m = L::M[k][d];
      if constexpr (d % 2 == 1 && m != 0) {
        const T v = even ? sg[d] : df[d];
        if constexpr (m == 1) acc = acc + v;
        else if constexpr (m == -1) acc = acc - v;
        else acc = mad(T(m), v, acc);
      }
    });
    mneq[k] = acc;
  });
  // S_k N_kd as in the binary64 form (the 1/tau moments from the runtime rate)
  const double s_tau = a.mrt_s_tau;
  const auto coef = [&](auto ki, auto di) {
    constexpr int k = decltype(ki)::value, d = decltype(di)::value;
    constexpr double N = (double)L::M[k][d] / mrt_diag<Q>(k);
    constexpr double rate = mrt_rate(Q, k);
    if constexpr (rate != 0.0) {
      constexpr double cc = rate * N;
      return T(cc);
    } else {
      return T(s_tau * N);
    }
  };
  {
    T e0 = T(0.);
    sfor<0, NM>([&](auto ki) {
      constexpr int k = decltype(ki)::value;
      if constexpr (mrt_parity<Q>(k) == 1 && L::M[k][0] != 0)
        e0 = mad(coef(ki, std::integral_constant<int, 0>{}), mneq[k], e0);
    });
    f[0] = f[0] - e0;
  }
  sfor<1, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    if constexpr (d % 2 == 1) {
      T ev = T(0.), od = T(0.);
      sfor<0, NM>([&](auto ki) {
        constexpr int k = decltype(ki)::value;
        if constexpr (L::M[k][d] != 0) {
          if constexpr (mrt_parity<Q>(k) == 1) ev = mad(coef(ki, di), mneq[k], ev);
          else od = mad(coef(ki, di), mneq[k], od);
        }
      });
      f[d] = f[d] - (ev + od);
      f[d + 1] = f[d + 1] - (ev - od);
    }
  });
}

// Collide in place: f (post-stream, possibly shifted) -> f* ; returns the
// moments the streamers of the next step need.  Binary64 LBGK and MRT in
// the reference's evaluation order, MRT of the shifted forms below; LBGK of
// the shifted forms in collide_lbgk_shifted.
template <int Q, int KERNEL, typename S, typename T = typename Store<S>::T>
__device__ __forceinline__ Hydro<Q, T> collide(T (&f)[Q], const StepArgs& a) {
  constexpr bool SHIFT = kShifted<S>;
  if constexpr (SHIFT && KERNEL == 0) {
    return collide_lbgk_shifted<Q, T, std::is_same<S, float>::value>(f, a);
  } else {
    using L = Lat<Q>;
    Hydro<Q, T> h;
    T r;
    moments<Q, T>(f, r, h.mx, h.my, h.mz);
    T fneq[Q];
    if constexpr (SHIFT) {
      const T rho = T(a.rho0) + r;
      h.rho = rho;
      FeqShifted<T> fe(r, rho, h.mx, h.my, h.mz);
      sfor<0, Q>([&](auto di) {
        constexpr int d = decltype(di)::value;
        fneq[d] = f[d] - fe.template eq<Q, d>();
      });
    } else {
      h.rho = r;
      FeqCoef<T> fe(r, h.mx, h.my, h.mz);
      sfor<0, Q>([&](auto di) {
        constexpr int d = decltype(di)::value;
        fneq[d] = f[d] - fe.template eq<Q, d>();
      });
    }
    if constexpr (KERNEL == 0) {
      // LBGK::Collide: f + f_neq * omega (LBGK.h:167-174)
      const T omega = std::is_same<T, double>::value ? T(a.omega) : T(a.omega_f);
      sfor<0, Q>([&](auto di) {
        constexpr int d = decltype(di)::value;
        f[d] = mad(fneq[d], omega, f[d]);
      });
    } else if constexpr (SHIFT) {
      mrt_relax_pairs<Q, T>(fneq, a, f);
    } else {
      // MRT: m_neq = M f_neq (MRT.h:123-135); f* = f - sum_k (S_k N_kd) m_neq_k
      // with N = M / diag(M M^T) (MRT.h:139-152).  S_k N_kd is a compile-time
      // binary64 product except for the 1/tau moments, where it is formed from
      // the runtime 1/tau exactly as the reference forms it.
      constexpr int NM = L::nmom;
      T mneq[NM];
      sfor<0, NM>([&](auto ki) {
        constexpr int k = decltype(ki)::value;
        T acc = T(0.);
        sfor<0, Q>([&](auto ii) {
          constexpr int i = decltype(ii)::value;
          constexpr int m = L::M[k][i];
          if constexpr (m == 1) acc = acc + fneq[i];
          else if constexpr (m == -1) acc = acc - fneq[i];
          else if constexpr (m != 0) acc = acc + T(m) * fneq[i];
        });
        mneq[k] = acc;
      });
      const double s_tau = a.mrt_s_tau;
      sfor<0, Q>([&](auto di) {
        constexpr int d = decltype(di)::value;
        T coll = T(0.);
        sfor<0, NM>([&](auto ki) {
          constexpr int k = decltype(ki)::value;
          if constexpr (L::M[k][d] != 0) {
            constexpr double N = (double)L::M[k][d] / mrt_diag<Q>(k);
            constexpr double rate = mrt_rate(Q, k);
            double c;
            if constexpr (rate != 0.0) {
              constexpr double cc = rate * N;
              c = cc;
            } else {
              c = s_tau * N;
            }
            coll = mad(T(c), mneq[k], coll);
          }
        });
        f[d] = f[d] - coll;
      });
    }
    return h;
  }
}

// ---------------------------------------------------------------------------
// Layouts: where a thread's site lives and where its neighbours are.
// ---------------------------------------------------------------------------
struct SiteRef {
  int64_t x;      // index into every per-direction array
  uint32_t cut;   // wall|iolet link mask of the site (0: bulk site)
  uint32_t rec;   // boundary record (valid when cut != 0)
  uint32_t wall, iolet;  // the record's words (0 for a bulk site)
  int32_t io;
  uint32_t qoff;
  uint32_t w;     // block layout: wave index (block * 8 + x plane)
  uint32_t lane;  // block layout: lane = y * 8 + z inside the plane
  int32_t tb[27]; // block layout: neighbour blocks of this wave's block
};

// The site's boundary record, or none: one load, so that the cut distances,
// the iolet's values and the pulls all start from here instead of one after
// the other.  A launch is as long as its slowest wave's chain of loads: with
// the neighbour table loaded beside the masks and the stash formed after the
// stores, a step of 43 k sites (D3Q19 BFL) takes 9.0 instead of 9.7 us, of the
// 7.93 M-site tree 507, 285 and 183 instead of 513, 290 and 190 us (binary64,
// 32, 16).
__device__ __forceinline__ void load_record(const DevDomain& D, bool boundary, SiteRef& r) {
  r.wall = r.iolet = r.qoff = 0;
  r.io = -1;
  if (boundary) {
    const uint4 v = *reinterpret_cast<const uint4*>(D.b_rec + r.rec);
    r.wall = v.x;
    r.iolet = v.y;
    r.io = (int32_t)v.z;
    r.qoff = v.w;
  }
  r.cut = r.wall | (r.iolet & BoundaryRecord::kLinks);
}

__device__ __forceinline__ uint32_t logical_workgroup() {
  // XCD-aware remap: hardware dispatches workgroup b to XCD b % 8; give
  // every XCD one contiguous range of logical workgroups.
  const uint32_t nwg = gridDim.x, b = blockIdx.x;
  const uint32_t xcd = b & 7u, k = b >> 3;
  const uint32_t base = nwg >> 3, rem = nwg & 7u;
  const uint32_t start = xcd * base + (xcd < rem ? xcd : rem);
  return start + k;
}

// Logical workgroup of the step kernels.  remap 0: the hardware order
// (consecutive workgroups on different XCDs); 1: one contiguous range per
// XCD; run >= 2: XCD x takes runs of `run` consecutive logical workgroups
// and the eight XCDs work on eight adjacent runs at a time, so the planes
// of a block and of its Morton neighbours stay in one XCD's L2 while the
// whole chip sweeps one region.  The grid is a multiple of 8 * run (the
// launcher pads it), which makes the map a bijection.
__device__ __forceinline__ uint32_t step_workgroup(uint32_t remap) {
  if (remap == 0) return blockIdx.x;
  if (remap == 1) return logical_workgroup();
  const uint32_t b = blockIdx.x, x = b & 7u, j = b >> 3;
  const uint32_t r = j / remap, o = j - r * remap;
  return (r * 8u + x) * remap + o;
}

// Compact layout: sites packed in Morton-block order.  The 32-bit pull
// table holds, per direction e, the offset (inside array e) of the value
// that streams into slot e: the source site for a fluid link, or the site's
// own slot of the inverse direction (x + (inv(e) - e) * np) for a cut link.
struct SparseLayout {
  static __device__ __forceinline__ bool locate(const DevDomain& D, SiteRef& r) {
    const int64_t x = (int64_t)logical_workgroup() * blockDim.x + threadIdx.x;
    if (x >= D.n) return false;
    at(D, x, r);
    return true;
  }
  // Compact site x (x < D.n).
  static __device__ __forceinline__ void at(const DevDomain& D, int64_t x, SiteRef& r) {
    r.x = x;
    const uint32_t bi = D.binfo[x];
    r.rec = bi - 1;
    load_record(D, bi != 0, r);
  }
  // State index of direction d of slot x, and of the value streaming into
  // slot E of the lane's site.
  template <int Q>
  static __device__ __forceinline__ int64_t at(const DevDomain& D, int d, int64_t x) {
    return (int64_t)d * D.np + x;
  }
  template <int Q, int E, bool M>
  static __device__ __forceinline__ int64_t index(const DevDomain& D, const SiteRef& r) {
    return (int64_t)E * D.np + (int64_t)D.src[(int64_t)(E - 1) * D.np + r.x];
  }
  static __device__ __forceinline__ int64_t compact(const DevDomain&, const SiteRef& r) {
    return r.x;
  }
  static __device__ __forceinline__ void relax(const DevDomain&, const SiteRef&, StepArgs&) {}
};

// In-plane order of the block layouts (the lane of a site inside its x
// plane, slot & 63):
// * binary64 storage: the bits of (y, z) inside the block interleaved, z in
//   bits 0, 2, 4 and y in bits 1, 3, 5 (a 2-D Morton order).  A 32-byte
//   sector then holds a 2 x 2 tile of the plane, so the column of a
//   neighbour block that a pull across a z face reads touches 4 sectors
//   instead of 8; the step reads 4 % fewer bytes and runs 2 % faster.
// * binary32 and binary16: rows of z (y in bits 3-5, z in bits 0-2).  The
//   interleaved order saved them no bytes, and binary16 ran 6 % slower with
//   it (its shifted gathers touch more distinct lines per quarter wave).
template <typename S> constexpr bool kMortonLanes = std::is_same<S, double>::value;
template <bool M> struct LaneBits {
  static constexpr uint32_t Y = M ? 0x2Au : 0x38u, Z = M ? 0x15u : 0x07u;
  static constexpr uint32_t UY = M ? 2u : 8u;  // lowest bit of Y
};
// Lane of (y - CY, z - CZ) mod 8: the decrement or increment of one
// coordinate's bits, with the carry or borrow run through the other's.
template <int CY, int CZ, bool M>
__device__ __forceinline__ uint32_t lane_shift(uint32_t lane) {
  using B = LaneBits<M>;
  uint32_t y = lane & B::Y, z = lane & B::Z;
  if constexpr (CY > 0) y = (y - B::UY) & B::Y;
  if constexpr (CY < 0) y = ((y | B::Z) + B::UY) & B::Y;
  if constexpr (CZ > 0) z = (z - 1u) & B::Z;
  if constexpr (CZ < 0) z = ((z | B::Y) + 1u) & B::Z;
  return y | z;
}
// Whether x - c leaves the block across its y (z) face: y == 0 for CY > 0,
// y == 7 for CY < 0.
template <int CY, bool M>
__device__ __forceinline__ bool lane_cross_y(uint32_t lane) {
  if constexpr (CY == 0) return false;
  else return (lane & LaneBits<M>::Y) == (CY > 0 ? 0u : LaneBits<M>::Y);
}
template <int CZ, bool M>
__device__ __forceinline__ bool lane_cross_z(uint32_t lane) {
  if constexpr (CZ == 0) return false;
  else return (lane & LaneBits<M>::Z) == (CZ > 0 ? 0u : LaneBits<M>::Z);
}

// The same as a mask: all ones where x - c leaves the block across its y (z)
// face, else zero.  Bit 6 of (coordinate bits - 1), or of (coordinate bits +
// 64 - all of them), is set exactly there.  (The empty statement keeps the
// compiler from turning the mask back into a compare and selects.)
template <int C, uint32_t BITS>
__device__ __forceinline__ uint32_t lane_cross_mask(uint32_t lane) {
  if constexpr (C == 0) return 0u;
  else {
    uint32_t m = (uint32_t)__builtin_amdgcn_sbfe(
        (int)((lane & BITS) + (C > 0 ? 0xFFFFFFFFu : 64u - BITS)), 6u, 1u);
    asm("" : "+v"(m));
    return m;
  }
}

// Block layout: every 8^3 block holding fluid owns 512 slots (x-plane major,
// lanes in the storage's in-plane order above) and its Q directions are stored together, block after block
// ([block][direction][512 slots]), so that one block's distributions are
// one contiguous run of memory; a wave covers one x plane of one block.  Neighbours come from
// slot arithmetic and the block's 27-entry neighbour table, which each wave
// loads once; per-wave 64-bit masks say which lanes are fluid and which carry
// a boundary record, whose wall and iolet masks mark the cut links.
struct BlockLayout {
  static __device__ __forceinline__ bool locate(const DevDomain& D, SiteRef& r) {
    const int64_t slot = (int64_t)logical_workgroup() * blockDim.x + threadIdx.x;
    return locate_wave(D, __builtin_amdgcn_readfirstlane((uint32_t)(slot >> 6)), r);
  }
  // The lane's site in wave (x plane) w; false for lanes without a fluid
  // site and for w beyond the domain.
  static __device__ __forceinline__ bool locate_wave(const DevDomain& D, uint32_t w,
                                                     SiteRef& r) {
    r.w = w;
    r.lane = threadIdx.x & 63u;
    r.x = ((int64_t)r.w << 6) + r.lane;
    if (r.w >= D.nwaves) return false;
    const uint64_t fm = D.wave_fluid[r.w];
    const uint64_t bm = D.wave_bnd[r.w];
    const uint32_t rb = D.wave_rec[r.w];
    // (before the exit of the lanes without a site, so that the table is on
    // its way while the masks are)
    const int32_t* nbt = D.bnbr + (int64_t)(r.w >> 3) * 27;
    sfor<0, 27>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      r.tb[i] = nbt[i];
    });
    if (!((fm >> r.lane) & 1ull)) return false;
    r.rec = rb + (uint32_t)__popcll(bm & ((1ull << r.lane) - 1ull));
    load_record(D, (bm >> r.lane) & 1ull, r);
    return true;
  }
  template <int Q>
  static __device__ __forceinline__ int64_t at(const DevDomain&, int d, int64_t slot) {
    return ((slot >> 9) * Q + d) * 512 + (slot & 511);
  }
  template <int Q, int E, bool M>
  static __device__ __forceinline__ int64_t index(const DevDomain& D, const SiteRef& r) {
    constexpr int CX = Lat<Q>::c[E][0], CY = Lat<Q>::c[E][1], CZ = Lat<Q>::c[E][2];
    const int lx = (int)(r.w & 7u);
    // source = x - c_E; crossing a block face moves to the neighbour block
    // at offset -c_E along that axis.
    const bool bx = CX != 0 && (CX > 0 ? lx == 0 : lx == 7);  // wave-uniform
    const bool by = lane_cross_y<CY, M>(r.lane);
    const bool bz = lane_cross_z<CZ, M>(r.lane);
    constexpr int i000 = 13, i100 = 13 - 9 * CX, i010 = 13 - 3 * CY, i001 = 13 - CZ;
    constexpr int i110 = 13 - 9 * CX - 3 * CY, i101 = 13 - 9 * CX - CZ;
    constexpr int i011 = 13 - 3 * CY - CZ, i111 = 13 - 9 * CX - 3 * CY - CZ;
    const int32_t n00 = bx ? r.tb[i100] : r.tb[i000];
    const int32_t n10 = bx ? r.tb[i110] : r.tb[i010];
    const int32_t n01 = bx ? r.tb[i101] : r.tb[i001];
    const int32_t n11 = bx ? r.tb[i111] : r.tb[i011];
    const int32_t nb = by ? (bz ? n11 : n10) : (bz ? n01 : n00);
    const int64_t src = ((int64_t)nb * Q + E) * 512 +
                        ((((lx - CX) & 7) << 6) | lane_shift<CY, CZ, M>(r.lane));
    constexpr int DP = inv_dir(E);
    const int64_t own = at<Q>(D, DP, r.x);
    return ((r.cut >> (DP - 1)) & 1u) ? own : src;
  }
  static __device__ __forceinline__ int64_t compact(const DevDomain& D, const SiteRef& r) {
    const uint64_t fm = D.wave_fluid[r.w];
    return (int64_t)D.wave_cbase[r.w] + __popcll(fm & ((1ull << r.lane) - 1ull));
  }
  // Ensembles relax each block with its instance's rates (one scalar load
  // per wave); otherwise the StepArgs values hold everywhere.
  static __device__ __forceinline__ void relax(const DevDomain& D, const SiteRef& r,
                                               StepArgs& a) {
    if (D.blk_omega) {
      const uint32_t b = r.w >> 3;
      a.omega = D.blk_omega[b];
      a.omega_f = D.blk_omega_f[b];
      a.mrt_s_tau = D.blk_s_tau[b];
    }
  }
};

// Compact-block layout: the waves, masks and neighbour-block table of the
// block layout, but the distributions are stored densely by compact site
// (Morton block order, then planes, then the in-plane order), so that no cache line carries empty
// slots.  The site of lane s of plane w is wave_cbase[w] + popcount of the
// plane's fluid mask below s; a neighbour's index comes from the same count
// on the source plane, whose mask and base are wave-uniform scalar loads.
struct CompactBlockLayout {
  static __device__ __forceinline__ int64_t site_of(uint64_t mask, uint32_t base,
                                                    uint32_t lane) {
    return (int64_t)base + __popcll(mask & ((1ull << lane) - 1ull));
  }
  static __device__ __forceinline__ bool locate(const DevDomain& D, SiteRef& r) {
    const int64_t slot = (int64_t)logical_workgroup() * blockDim.x + threadIdx.x;
    return locate_wave(D, __builtin_amdgcn_readfirstlane((uint32_t)(slot >> 6)), r);
  }
  static __device__ __forceinline__ bool locate_wave(const DevDomain& D, uint32_t w,
                                                     SiteRef& r) {
    r.w = w;
    r.lane = threadIdx.x & 63u;
    if (r.w >= D.nwaves) return false;
    const uint64_t fm = D.wave_fluid[r.w];
    const uint64_t bm = D.wave_bnd[r.w];
    const uint32_t rb = D.wave_rec[r.w];
    if (!((fm >> r.lane) & 1ull)) return false;
    r.x = site_of(fm, D.wave_cbase[r.w], r.lane);
    const int32_t* nbt = D.bnbr + (int64_t)(r.w >> 3) * 27;
    sfor<0, 27>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      r.tb[i] = nbt[i];
    });
    r.rec = rb + (uint32_t)__popcll(bm & ((1ull << r.lane) - 1ull));
    load_record(D, (bm >> r.lane) & 1ull, r);
    return true;
  }
  // Fluid mask and compact base of x plane px of block nb (nb < 0: absent,
  // and then no lane reads it).
  static __device__ __forceinline__ void plane(const DevDomain& D, int32_t nb, int px,
                                               uint64_t& m, uint32_t& b) {
    if (nb >= 0) {
      const uint32_t pw = ((uint32_t)nb << 3) | (uint32_t)px;
      m = D.wave_fluid[pw];
      b = D.wave_cbase[pw];
    } else {
      m = 0;
      b = 0;
    }
  }
  template <int Q>
  static __device__ __forceinline__ int64_t at(const DevDomain& D, int d, int64_t x) {
    return (int64_t)d * D.np + x;
  }
  template <int Q, int E, bool M>
  static __device__ __forceinline__ int64_t index(const DevDomain& D, const SiteRef& r) {
    constexpr int CX = Lat<Q>::c[E][0], CY = Lat<Q>::c[E][1], CZ = Lat<Q>::c[E][2];
    const int lx = (int)(r.w & 7u);
    const bool bx = CX != 0 && (CX > 0 ? lx == 0 : lx == 7);  // wave-uniform
    const bool by = lane_cross_y<CY, M>(r.lane);
    const bool bz = lane_cross_z<CZ, M>(r.lane);
    constexpr int i000 = 13, i100 = 13 - 9 * CX, i010 = 13 - 3 * CY, i001 = 13 - CZ;
    constexpr int i110 = 13 - 9 * CX - 3 * CY, i101 = 13 - 9 * CX - CZ;
    constexpr int i011 = 13 - 3 * CY - CZ, i111 = 13 - 9 * CX - 3 * CY - CZ;
    const int px = (lx - CX) & 7;
    uint64_t m00, m10 = 0, m01 = 0, m11 = 0;
    uint32_t b00, b10 = 0, b01 = 0, b11 = 0;
    plane(D, bx ? r.tb[i100] : r.tb[i000], px, m00, b00);
    if constexpr (CY != 0) plane(D, bx ? r.tb[i110] : r.tb[i010], px, m10, b10);
    if constexpr (CZ != 0) plane(D, bx ? r.tb[i101] : r.tb[i001], px, m01, b01);
    if constexpr (CY != 0 && CZ != 0) plane(D, bx ? r.tb[i111] : r.tb[i011], px, m11, b11);
    const uint64_t m = by ? (bz ? m11 : m10) : (bz ? m01 : m00);
    const uint32_t b = by ? (bz ? b11 : b10) : (bz ? b01 : b00);
    const uint32_t sl = lane_shift<CY, CZ, M>(r.lane);
    const int64_t src = site_of(m, b, sl);
    constexpr int DP = inv_dir(E);
    return ((r.cut >> (DP - 1)) & 1u) ? at<Q>(D, DP, r.x) : at<Q>(D, E, src);
  }
  static __device__ __forceinline__ int64_t compact(const DevDomain&, const SiteRef& r) {
    return r.x;
  }
  static __device__ __forceinline__ void relax(const DevDomain& D, const SiteRef& r,
                                               StepArgs& a) {
    BlockLayout::relax(D, r, a);
  }
};

// The block layout addressed by 32-bit byte offsets from the state buffer's
// base, for states of every direction below 4 GiB.  A load or store is then
// the kernel argument's 64-bit base (a scalar register pair) plus one 32-bit
// lane offset, which the global instructions add themselves: the wave-uniform
// parts (block, direction, plane, and the neighbour blocks' offsets) are
// scalar arithmetic, and a gather costs a select and an add per lane instead
// of 64-bit multiply-adds.  Same elements, same order as BlockLayout.
struct BlockLayout32 : BlockLayout {
  // byte offset of slot `lane` of direction d in this wave's plane
  template <int Q, typename P>
  static __device__ __forceinline__ uint32_t own_off(const SiteRef& r, uint32_t d) {
    constexpr uint32_t ES = sizeof(P);
    return (((r.w >> 3) * (uint32_t)Q + d) * 512u + ((r.w & 7u) << 6)) * ES + r.lane * ES;
  }
  template <int Q, typename P>
  static __device__ __forceinline__ P* own_ptr(const SiteRef& r, P* base, int d) {
    constexpr uint32_t ES = sizeof(P);
    // wave-uniform part first (scalar), then the lane's offset
    const uint32_t uni = (((r.w >> 3) * (uint32_t)Q + (uint32_t)d) * 512u + ((r.w & 7u) << 6)) * ES;
    using C = std::conditional_t<std::is_const<P>::value, const char, char>;
    return (P*)(((C*)base + uni) + r.lane * ES);
  }
  // Byte offset of the value at x - c_E, where `pick(t)` gives the block of
  // neighbour-table entry t.  The lanes that leave the block across its y or
  // z face add the difference of two blocks' offsets under a mask (modulo
  // 2^32): one `and` with a scalar and a part of one three-way add.  A select
  // between two scalar offsets needs both moved to vector registers first, as
  // a vector instruction takes one scalar operand.  The D3Q19 LBGK pull's
  // vector instructions a wave: 185 -> 138 (binary64, binary32), 113 -> 84
  // (binary16).  It shows where a wave's latency counts (1280 sites BFL
  // binary64 7.63 -> 7.45 us a step, 43 k sites 8.21 -> 7.97) and not where
  // memory does (trees within 0.2 %; binary16, 7.9 M sites, 182.4 -> 181.7).
  template <int Q, int E, typename P, class Pick>
  static __device__ __forceinline__ uint32_t src_off(const SiteRef& r, Pick pick) {
    constexpr int CX = Lat<Q>::c[E][0], CY = Lat<Q>::c[E][1], CZ = Lat<Q>::c[E][2];
    constexpr uint32_t ES = sizeof(P), BS = (uint32_t)Q * 512u * ES;
    constexpr bool M = kMortonLanes<std::remove_const_t<P>>;
    using B = LaneBits<M>;
    const int lx = (int)(r.w & 7u);
    const bool bx = CX != 0 && (CX > 0 ? lx == 0 : lx == 7);  // wave-uniform
    constexpr int i000 = 13, i100 = 13 - 9 * CX, i010 = 13 - 3 * CY, i001 = 13 - CZ;
    constexpr int i110 = 13 - 9 * CX - 3 * CY, i101 = 13 - 9 * CX - CZ;
    constexpr int i011 = 13 - 3 * CY - CZ, i111 = 13 - 9 * CX - 3 * CY - CZ;
    // wave-uniform: direction E's array in each candidate block, source plane
    // (readfirstlane keeps the products scalar: without it the compiler moves
    // the multiply into a vector multiply)
    const uint32_t uni = ((uint32_t)E * 512u + ((uint32_t)((lx - CX) & 7) << 6)) * ES;
    const auto blk = [&](int32_t t) {
      return __builtin_amdgcn_readfirstlane((uint32_t)pick(t) * BS);
    };
    const uint32_t n00 = blk(bx ? r.tb[i100] : r.tb[i000]);
    uint32_t off = lane_shift<CY, CZ, M>(r.lane) * ES;
    const uint32_t my = lane_cross_mask<CY, B::Y>(r.lane), mz = lane_cross_mask<CZ, B::Z>(r.lane);
    uint32_t n10 = 0, n01 = 0;
    if constexpr (CY != 0) {
      n10 = blk(bx ? r.tb[i110] : r.tb[i010]);
      off += my & (n10 - n00);
    }
    if constexpr (CZ != 0) {
      n01 = blk(bx ? r.tb[i101] : r.tb[i001]);
      off += mz & (n01 - n00);
    }
    if constexpr (CY != 0 && CZ != 0) {
      const uint32_t n11 = blk(bx ? r.tb[i111] : r.tb[i011]);
      off += (my & mz) & (n11 - n10 - n01 + n00);
    }
    return off + __builtin_amdgcn_readfirstlane(n00 + uni);
  }
  template <int Q, int E, typename P>
  static __device__ __forceinline__ P* src_ptr(const SiteRef& r, P* base) {
    constexpr int DP = inv_dir(E);
    // a cut link reads the site's own slot of the inverse direction (both
    // offsets are formed first so that the choice is a bit select, not a
    // divergent branch)
    const uint32_t own = own_off<Q, P>(r, DP);
    const uint32_t src = src_off<Q, E, P>(r, [](int32_t t) { return t; });
    uint32_t off = src;
    if constexpr (DP > 0) {
      uint32_t cut = (uint32_t)__builtin_amdgcn_sbfe((int)r.cut, DP - 1, 1u);
      asm("" : "+v"(cut));
      off = (cut & own) | (~cut & src);
    }
    using C = std::conditional_t<std::is_const<P>::value, const char, char>;
    return (P*)((C*)base + off);
  }
  // The value at x - c_E whether or not link E is cut (the gather then
  // replaces a cut link's value): a neighbour block that does not exist is
  // replaced by the own block, so that the address stays inside the state.
  template <int Q, int E, typename P>
  static __device__ __forceinline__ P* src_any_ptr(const SiteRef& r, P* base) {
    const int32_t self = (int32_t)(r.w >> 3);
    const uint32_t off =
        src_off<Q, E, P>(r, [&](int32_t t) { return t < 0 ? self : t; });
    using C = std::conditional_t<std::is_const<P>::value, const char, char>;
    return (P*)((C*)base + off);
  }
  // Streamed store of slot d of the lane's site: a buffer store whose scalar
  // offset carries the wave-uniform part and whose vector offset is the
  // lane's (the same register for every direction), with the non-temporal
  // bit, as the 64-bit layouts' non-temporal stores.
  template <int Q, typename S>
  static __device__ __forceinline__ void store(const DevDomain& D, const SiteRef& r, S* base,
                                               int d, S v) {
    constexpr uint32_t ES = sizeof(S);
    const uint32_t uni = (((r.w >> 3) * (uint32_t)Q + (uint32_t)d) * 512u + ((r.w & 7u) << 6)) * ES;
    const uint32_t bytes = (uint32_t)D.np * (uint32_t)Q * ES;  // below 4 GiB
    // word 3 of a raw buffer resource on gfx9 parts: 32-bit data format
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000);
    constexpr int kNonTemporal = 2;
    const int voff = (int)(r.lane * ES);
    if constexpr (ES == 2)
      __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), rs, voff,
                                            (int)uni, kNonTemporal);
    else if constexpr (ES == 4)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), rs, voff,
                                            (int)uni, kNonTemporal);
    else {
      using U2 = unsigned int __attribute__((ext_vector_type(2)));
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), rs, voff, (int)uni,
                                            kNonTemporal);
    }
  }
};

template <class Lay>
constexpr bool kWaveLayout = std::is_same<Lay, BlockLayout>::value ||
                             std::is_same<Lay, BlockLayout32>::value ||
                             std::is_same<Lay, CompactBlockLayout>::value;

// Own slot E of the lane's site where pick_e, else its own slot DP (a
// per-lane choice between two directions).  BlockLayout32: the wave-uniform
// offset of the lower direction plus a per-lane choice of two non-negative
// constants.
template <int Q, int E, int DP, class Lay, typename P>
__device__ __forceinline__ P* own_pick_ptr(const DevDomain& D, const SiteRef& r, P* base,
                                           bool pick_e) {
  if constexpr (std::is_same<Lay, BlockLayout32>::value) {
    constexpr uint32_t ES = sizeof(P);
    constexpr int LO = E < DP ? E : DP;
    constexpr uint32_t dE = (uint32_t)(E - LO) * 512u * ES, dP = (uint32_t)(DP - LO) * 512u * ES;
    const uint32_t uni = (((r.w >> 3) * (uint32_t)Q + (uint32_t)LO) * 512u + ((r.w & 7u) << 6)) * ES;
    using C = std::conditional_t<std::is_const<P>::value, const char, char>;
    return (P*)(((C*)base + uni) + (r.lane * ES + (pick_e ? dE : dP)));
  } else {
    return base + Lay::template at<Q>(D, pick_e ? E : DP, r.x);
  }
}

// Addresses of state elements: slot d of the lane's own site, and the value
// streaming into slot E of it (its source, or its own inverse slot across a
// cut link).  Element indices for the 64-bit layouts, byte offsets for
// BlockLayout32.
template <int Q, class Lay, typename P>
__device__ __forceinline__ P* own_ptr(const DevDomain& D, const SiteRef& r, P* base, int d) {
  if constexpr (std::is_same<Lay, BlockLayout32>::value)
    return Lay::template own_ptr<Q>(r, base, d);
  else
    return base + Lay::template at<Q>(D, d, r.x);
}
template <int Q, int E, class Lay, typename P>
__device__ __forceinline__ P* src_ptr(const DevDomain& D, const SiteRef& r, P* base) {
  if constexpr (std::is_same<Lay, BlockLayout32>::value)
    return Lay::template src_ptr<Q, E>(r, base);
  else
    return base + Lay::template index<Q, E, kMortonLanes<std::remove_const_t<P>>>(D, r);
}

// ---------------------------------------------------------------------------
// Streaming (pull) with boundary links
// ---------------------------------------------------------------------------
// Ghost equilibrium of the Nash zeroth-order pressure links of iolet-site
// record io on iolet k (NashZerothOrderPressure.h:27-60): density of the
// iolet, momentum = (n_float * (m.n_float / rho)) * rho_ghost; a link's value
// is one component of Lattice::CalculateFeq.  Always binary64.
__device__ __forceinline__ FeqCoef<double> nash_ghost(const DevDomain& D, const StepArgs& A,
                                                      int io, int k) {
  const double rho_g = A.bv[2 * k];
  const double comp = D.io_stash[io];
  const double gx = (double)D.iolet_nf[3 * k + 0] * comp * rho_g;
  const double gy = (double)D.iolet_nf[3 * k + 1] * comp * rho_g;
  const double gz = (double)D.iolet_nf[3 * k + 2] * comp * rho_g;
  return FeqCoef<double>(rho_g, gx, gy, gz);
}

// The Ladd links of an iolet site (LaddIolet.h:29-66): what all of them share,
// and the correction 2 w_d (rho u_w . c_d)/Cs2 of link DP with u_w the iolet
// velocity half way along it.
struct LaddSite {
  double rho, nx, ny, nz, a, b;
  const double* coef;   // two per link
  bool womersley;
  template <int Q>
  static __device__ __forceinline__ LaddSite of(const DevDomain& D, const StepArgs& A, int io,
                                                int k) {
    return LaddSite{D.io_stash[io],
                    D.iolet_n[3 * k],
                    D.iolet_n[3 * k + 1],
                    D.iolet_n[3 * k + 2],
                    A.bv[2 * k],
                    A.bv[2 * k + 1],
                    D.io_ladd + (int64_t)io * (Q - 1) * 2,
                    D.iolet_kind[k] == 2};
  }
  template <int Q, int DP>
  __device__ __forceinline__ double correction() const {
    using L = Lat<Q>;
    const double* lc = coef + (DP - 1) * 2;
    // InOutLetWomersleyVelocity::GetVelocity: Re[A e^{i w t}], u = n * -vm;
    // InOutLetParabolicVelocity::GetVelocity: n * (max * (1 - r^2/R^2))
    const double s = womersley ? -(lc[0] * a - lc[1] * b) : a * lc[0];
    double ux = nx * s, uy = ny * s, uz = nz * s;
    ux *= rho;
    uy *= rho;
    uz *= rho;
    const double dot = dotc<L::c[DP][0], L::c[DP][1], L::c[DP][2]>(ux, uy, uz);
    return 2. * L::w[DP] * dot / kCs2;
  }
};

// Cut distances of links 1..Q-1 from 16-bit fixed-point records (the
// reduced-precision forms): QS16 = Q - 1 rounded up to a multiple of 8.
template <int Q> constexpr int kQS16 = (Q - 1 + 7) / 8 * 8;
template <int Q>
__device__ __forceinline__ void decode_q16(const uint4 (&v)[kQS16<Q> / 8], float (&q)[kQS16<Q>]) {
  sfor<0, kQS16<Q> / 8>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
    sfor<0, 4>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      q[8 * i + 2 * j] = (float)(w[j] & 0xFFFFu) * (1.0f / 65535.0f);
      q[8 * i + 2 * j + 1] = (float)(w[j] >> 16) * (1.0f / 65535.0f);
    });
  });
}

// BouzidiFirdaousLallemandLink::StreamLink (BouzidiFirdaousLallemand.h:41-66):
// with q >= 0.5 and a fluid opposite link the slot gets
// (f*_d + (2q - 1) f*_inv(d)) / (2q); both values are the site's own
// (opp[e] = f*_e of the site).  Slot e is a candidate (bit e-1 of cand) when
// the inverse link is a wall link and not an iolet link, and link e itself
// is not a wall link.  A link outside `plane` (the union of cand over the
// wave's lanes, a scalar) is passed over by one scalar branch.
template <int Q, typename S, typename T>
__device__ __forceinline__ void bfl_stream_links(const float (&q)[kQS16<Q>], uint32_t cand,
                                                 const T (&opp)[Q], T (&f)[Q],
                                                 uint32_t plane = ~0u) {
  sfor<1, Q>([&](auto ei) {
    constexpr int e = decltype(ei)::value;
    constexpr int dp = inv_dir(e);
    if (!((plane >> (e - 1)) & 1u)) return;
    const T qd = (T)(double)q[dp - 1];
    if (((cand >> (e - 1)) & 1u) && !(qd < T(0.5))) {
      if constexpr (kShifted<S>)
        f[e] = mad(T(2.0) * qd - T(1), opp[e], f[e]) * recip(T(2.0) * qd);
      else
        f[e] = (f[e] + (T(2.0) * qd - T(1)) * opp[e]) / (T(2.0) * qd);
    }
  });
}

// Iolet links of a boundary site: the Nash ghost equilibrium or the
// Ladd correction of the bounce-back value.  What a site's links share (the
// iolet's values, the ghost's two divisions) is formed once: with all of it
// in each link's own branch, these waves were the last of every step, and the
// step of a small vessel as long as they are (1280 sites, D3Q15: 7.2 us a step
// with, 6.3 without; an 819 k-site tree 69.1 and 67.3 us in binary64, 32.3 and
// 30.3 in binary16).
template <int Q, typename S, typename T>
__device__ __forceinline__ void iolet_links(const DevDomain& D, const StepArgs& A,
                                            const SiteRef& r, T (&f)[Q]) {
  const int io = r.io;
  const uint32_t im = r.iolet;
  const int k = (int)(r.iolet >> BoundaryRecord::kIndexBit);
  if (!((r.iolet >> BoundaryRecord::kBcBit) & 1u)) {
    const FeqCoef<double> ghost = nash_ghost(D, A, io, k);
    sfor<1, Q>([&](auto ei) {
      constexpr int e = decltype(ei)::value;
      constexpr int dp = inv_dir(e);
      if ((im >> (dp - 1)) & 1u) {
        double v = ghost.template eq<Q, e>();
        if constexpr (kShifted<S>) v -= Lat<Q>::w[e] * A.rho0;
        f[e] = (T)v;
      }
    });
  } else {
    const LaddSite site = LaddSite::of<Q>(D, A, io, k);
    sfor<1, Q>([&](auto ei) {
      constexpr int e = decltype(ei)::value;
      constexpr int dp = inv_dir(e);
      if ((im >> (dp - 1)) & 1u) f[e] = f[e] - (T)site.template correction<Q, dp>();
    });
  }
}

// BouzidiFirdaousLallemandLink::PostStepLink: links d with a wall and no
// wall on the inverse link, q < 0.5 (`plane`: the union of those links over
// the wave's lanes, as for bfl_stream_links)
template <int Q, typename S, typename T>
__device__ __forceinline__ void bfl_post_links(const float (&q)[kQS16<Q>], uint32_t wm,
                                               T (&f)[Q], uint32_t plane = ~0u) {
  const uint32_t post = wm & ~pair_swap(wm);
  sfor<1, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    constexpr int id = inv_dir(d);
    if (!((plane >> (d - 1)) & 1u)) return;
    const T qd = (T)(double)q[d - 1];
    if (((post >> (d - 1)) & 1u) && qd < T(0.5)) {
      if constexpr (kShifted<S>)
        f[id] = mad(T(2.0) * qd, f[id] - f[d], f[d]);
      else
        f[id] = T(2.0) * qd * f[id] + (T(1.0) - T(2.0) * qd) * f[d];
    }
  });
}

// Binary16 with 32-bit offsets: every load of a site is issued in one batch
// after the plane's tables, none waits for the boundary record.  The pulls
// read x - c_e whether or not link e is cut (an absent neighbour block is
// replaced by the own block, so the address stays in the state), and lanes
// with a boundary record also load their own Q-1 values and cut distances;
// the bounce-back value of a cut link and the BFL value f*_e are then picked
// from the own values.  The same values and arithmetic as gather's other
// path: binary16 loads every own value that path picks from anyway.
template <int Q, typename S, typename T>
__device__ __forceinline__ void gather_early(const DevDomain& D, const StepArgs& A,
                                             const S* __restrict__ fin, const SiteRef& r,
                                             T (&f)[Q]) {
  using St = Store<S>;
  using Lay = BlockLayout32;
  const bool bnd = (D.wave_bnd[r.w] >> r.lane) & 1ull;
  f[0] = St::ld(own_ptr<Q, Lay>(D, r, fin, 0));
  sfor<1, Q>([&](auto ei) {
    constexpr int e = decltype(ei)::value;
    f[e] = St::ld(Lay::template src_any_ptr<Q, e>(r, fin));
  });
  T own[Q];
  uint4 qv[kQS16<Q> / 8];
  if (bnd) {
    sfor<1, Q>([&](auto ei) {
      constexpr int e = decltype(ei)::value;
      own[e] = St::ld(own_ptr<Q, Lay>(D, r, fin, e));
    });
    if (A.wall == 1) {
      const uint4* q8 = reinterpret_cast<const uint4*>(D.b_q16 + (int64_t)r.rec * kQS16<Q>);
      sfor<0, kQS16<Q> / 8>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        qv[i] = q8[i];
      });
    }
  }
  if (!bnd) return;
  sfor<1, Q>([&](auto ei) {
    constexpr int e = decltype(ei)::value;
    constexpr int dp = inv_dir(e);
    if ((r.cut >> (dp - 1)) & 1u) f[e] = own[dp];
  });
  const uint32_t wm = r.wall, im = r.iolet & BoundaryRecord::kLinks;
  // the plane's BFL links: formulas of links no lane has are skipped
  const uint64_t wl = D.wave_links[r.w];
  float q[kQS16<Q>];
  if (A.wall == 1 && wm) {
    decode_q16<Q>(qv, q);
    bfl_stream_links<Q, S, T>(q, pair_swap(wm) & ~pair_swap(im) & ~wm, own, f, (uint32_t)wl);
  }
  if (im) iolet_links<Q, S, T>(D, A, r, f);
  if (A.wall == 1 && wm) bfl_post_links<Q, S, T>(q, wm, f, (uint32_t)(wl >> 32));
}

// Post-stream distributions of a site (the reference's fNew after
// StreamAndCollide and PostStep) from the post-collision state `fin`.
// All Q loads are issued first: a cut link reads the site's own value of the
// inverse direction (the bounce-back value); the wall and iolet formulas are
// applied afterwards.
template <int Q, typename S, typename T, class Lay, bool BULK = false>
__device__ __forceinline__ void gather(const DevDomain& D, const StepArgs& A,
                                       const S* __restrict__ fin, const SiteRef& r,
                                       T (&f)[Q]) {
  if constexpr (!BULK && sizeof(S) == 2 && std::is_same<Lay, BlockLayout32>::value) {
    gather_early<Q, S, T>(D, A, fin, r, f);
    return;
  }
  using St = Store<S>;
  f[0] = St::ld(own_ptr<Q, Lay>(D, r, fin, 0));
  sfor<1, Q>([&](auto ei) {
    constexpr int e = decltype(ei)::value;
    f[e] = St::ld(src_ptr<Q, e, Lay>(D, r, fin));
  });
  if constexpr (BULK) return;  // a wave without boundary sites
  if (!r.cut) return;
  const uint32_t wm = r.wall, im = r.iolet & BoundaryRecord::kLinks;
  // cut distances of links 1..Q-1 (only the wall links' are read): 16-bit
  // fixed-point records for the shifted forms, binary32 values of the wall
  // links alone, packed, for binary64 storage
  float q[kQS16<Q>];
  if (A.wall == 1 && wm) {
    if constexpr (kShifted<S>) {
      const uint4* q8 = reinterpret_cast<const uint4*>(D.b_q16 + (int64_t)r.rec * kQS16<Q>);
      uint4 qv[kQS16<Q> / 8];
      sfor<0, kQS16<Q> / 8>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        qv[i] = q8[i];
      });
      decode_q16<Q>(qv, q);
    } else {
      // 4.6 wall links per wall site on the vessel tree: 18 bytes instead
      // of an 80-byte record of every link
      const float* qp = D.b_q + r.qoff;
      sfor<0, Q - 1>([&](auto kk) {
        constexpr int k = decltype(kk)::value;
        q[k] = -1.0f;
        if ((wm >> k) & 1u) q[k] = qp[__popc(wm & ((1u << k) - 1u))];
      });
    }
  }
  // The iolet links of a site and its interpolated wall links write different
  // slots, so the iolet ones go first, while the cut distances are on their
  // way.
  if (im) iolet_links<Q, S, T>(D, A, r, f);
  if (A.wall == 1 && wm) {
    // The links that take the interpolated form need the site's own f*_e.
    // Binary64 and binary32: only those lanes load (the rest are masked
    // off; measured 0.3-0.6 % faster on the vessel tree).  Binary16 (64-bit
    // addressing): every lane loads, the unused ones their already-fetched
    // bounce-back slot (predicated 16-bit loads measured 10 % slower).
    const uint32_t cand = pair_swap(wm) & ~pair_swap(im) & ~wm;
    T opp[Q];
    sfor<1, Q>([&](auto ei) {
      constexpr int e = decltype(ei)::value;
      constexpr int dp = inv_dir(e);
      const bool link = (cand >> (e - 1)) & 1u;
      if constexpr (sizeof(S) >= 4) {
        opp[e] = T(0);
        if (link && !((T)(double)q[dp - 1] < T(0.5)))
          opp[e] = St::ld(own_ptr<Q, Lay>(D, r, fin, e));
      } else {
        opp[e] = St::ld(own_pick_ptr<Q, e, dp, Lay>(D, r, fin, link));
      }
    });
    bfl_stream_links<Q, S, T>(q, cand, opp, f);
    bfl_post_links<Q, S, T>(q, wm, f);
  }
}

template <int Q, typename T, bool BULK = false>
__device__ __forceinline__ void update_stash(const DevDomain& D, const SiteRef& r,
                                             const Hydro<Q, T>& h) {
  if constexpr (BULK) return;
  const int io = r.io;
  if (io < 0) return;
  const double rho = (double)h.rho;
  if (!((r.iolet >> BoundaryRecord::kBcBit) & 1u)) {
    // component = Dot(momentum, n_float) / density (NashZerothOrderPressure.h:43)
    const int k = (int)(r.iolet >> BoundaryRecord::kIndexBit);
    double acc = 0.0;
    acc = acc + (double)h.mx * (double)D.iolet_nf[3 * k];
    acc = acc + (double)h.my * (double)D.iolet_nf[3 * k + 1];
    acc = acc + (double)h.mz * (double)D.iolet_nf[3 * k + 2];
    D.io_stash[io] = acc / rho;
  } else {
    D.io_stash[io] = rho;  // LaddIolet.h:55-58 (compressible lattice)
  }
}

template <typename S>
__device__ __forceinline__ void store_out(S* p, typename Store<S>::T v) {
  // Written once per step and read only by the next launch: stream it past
  // the caches.
  __builtin_nontemporal_store((S)v, p);
}


inline dim3 grid_for(int64_t n, int threads = 256) {
  return dim3((unsigned)((n + threads - 1) / threads));
}

// Threads launched for a per-site kernel: compact sites or all slots.
inline int64_t thread_count(const DevDomain& d) {
  return d.layout == 0 ? d.n : (int64_t)d.nwaves * 64;  // sites, or lanes of all planes
}

// (lattice, kernel, storage) -> instantiation, for one layout
template <int LAYOUT, typename Fn>
int dispatch_in(const StepArgs& a, Fn&& fn) {
  using Lay = std::conditional_t<LAYOUT == 0, SparseLayout,
                                 std::conditional_t<LAYOUT == 1, BlockLayout, CompactBlockLayout>>;
#define HLB_CASE(Q_, K_, S_, SC_)                                                    \
  if (a.Q == Q_ && a.kernel == K_ && a.storage == SC_)                                \
    return fn(std::integral_constant<int, Q_>{}, std::integral_constant<int, K_>{}, \
              (S_*)nullptr, (Lay*)nullptr);
  HLB_CASE(15, 0, double, 0) HLB_CASE(15, 1, double, 0)
  HLB_CASE(19, 0, double, 0) HLB_CASE(19, 1, double, 0)
  HLB_CASE(15, 0, float, 1) HLB_CASE(15, 1, float, 1)
  HLB_CASE(19, 0, float, 1) HLB_CASE(19, 1, float, 1)
  HLB_CASE(15, 0, _Float16, 2) HLB_CASE(15, 1, _Float16, 2)
  HLB_CASE(19, 0, _Float16, 2) HLB_CASE(19, 1, _Float16, 2)
#undef HLB_CASE
  return (int)hipErrorInvalidValue;
}

// (layout, lattice, kernel, storage) -> instantiation
template <typename Fn>
int dispatch(const DevDomain& d, const StepArgs& a, Fn&& fn) {
  if (d.layout == 0) return dispatch_in<0>(a, fn);
  if (d.layout == 1) return dispatch_in<1>(a, fn);
  return dispatch_in<2>(a, fn);
}

// Whether every state element of the block layout is reachable by a 32-bit
// byte offset (and the launch shape does not ask for 64-bit addressing).
inline bool narrow_offsets(const DevDomain& d, const StepArgs& a, size_t esize) {
  return !a.wide && (uint64_t)a.Q * (uint64_t)d.np * esize <= 0xFFFFFFFFull;
}

// As dispatch, with BlockLayout32 in the place of BlockLayout where its
// offsets reach the whole state.
template <typename Fn>
int dispatch_narrow(const DevDomain& d, const StepArgs& a, Fn&& fn) {
  return dispatch(d, a, [&](auto q, auto k, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    if constexpr (std::is_same<Lay, BlockLayout>::value)
      if (narrow_offsets(d, a, sizeof(S))) return fn(q, k, s, (BlockLayout32*)nullptr);
    return fn(q, k, s, lay);
  });
}

}  // namespace

// The timestep's launches for one layout (lbm_kernels.hip, compiled once per
// layout).
template <int LAYOUT>
int step_in(const DevDomain& d, const StepArgs& a, const void* fin, void* fout, void* stream);
template <int LAYOUT>
int collide_only_in(const DevDomain& d, const StepArgs& a, const void* fin, void* fout,
                    void* stream);

}  // namespace hlb
