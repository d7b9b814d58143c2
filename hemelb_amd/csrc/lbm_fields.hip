// Kernels around the timestep: initialisation and import, exports of the
// post-stream distributions and of the fields derived from them, monitors
// and reductions, halo exchange, and the device-copy ceiling.
#include "lbm_device.h"

// Static scratch of the allocation-free monitor: kMonitorGroups * 5
// workgroup partials, then (rho, u) of up to kStaticIoletSites iolet sites.
// Host code never names this array (its name is only a host-side stand-in);
// it uses the per-device address from hlb::scratch_address.
static __device__ __align__(256) double scratch[hlb::kStaticScratchDoubles];

namespace hlb {
namespace {

// Post-stream distributions in binary64, compact SoA [Q][npc].
template <int Q, typename S, class Lay>
__global__ __launch_bounds__(256) void k_stream_only(DevDomain D, StepArgs A,
                                                     const S* __restrict__ fin,
                                                     double* __restrict__ out,
                                                     int from_post_stream) {
  using T = typename Store<S>::T;
  SiteRef r;
  if (!Lay::locate(D, r)) return;
  T f[Q];
  if (from_post_stream) {
    sfor<0, Q>([&](auto di) {
      constexpr int d = decltype(di)::value;
      f[d] = Store<S>::ld(fin + Lay::template at<Q>(D, d, r.x));
    });
  } else {
    gather<Q, S, T, Lay>(D, A, fin, r, f);
  }
  const int64_t c = Lay::compact(D, r);
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    double v = (double)f[d];
    if constexpr (kShifted<S>) v += Lat<Q>::w[d] * A.rho0;
    out[(int64_t)d * D.npc + c] = v;
  });
}

// Device-copy ceiling of the step's traffic: the Q state arrays (stride
// `stride` words of type W) copied from `in` to `out`, `words` per array,
// one word per thread and array, all loads issued before the streamed
// stores, workgroups mapped to XCDs as the step maps them.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <int Q, typename W>
__global__ __launch_bounds__(256) void k_copy_arrays(int64_t stride, int64_t words, int64_t run,
                                                     const W* __restrict__ in,
                                                     W* __restrict__ out, uint32_t remap) {
  const int64_t i = (int64_t)step_workgroup(remap) * blockDim.x + threadIdx.x;
  if (i >= words) return;
  // run > 0: the block layout's order, runs of `run` words per direction
  // and block; else arrays of `stride` words per direction
  const int64_t base = run ? (i / run) * Q * run + (i % run) : i;
  const int64_t step = run ? run : stride;
  W v[Q];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    v[d] = __builtin_nontemporal_load(in + base + d * step);
  });
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    __builtin_nontemporal_store(v[d], out + base + d * step);
  });
}

// Halo exchange between subdomains: stored values copied as raw words
// (E = the storage's 8-, 4- or 2-byte word), from state to a buffer (pack)
// or from a buffer to state (unpack), at precomputed state indices.
template <typename E>
__global__ void k_halo_pack(int64_t count, const int64_t* __restrict__ idx,
                            const E* __restrict__ state, E* __restrict__ buf) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < count) buf[k] = state[idx[k]];
}
template <typename E>
__global__ void k_halo_unpack(int64_t count, const int64_t* __restrict__ idx,
                              const E* __restrict__ buf, E* __restrict__ state) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < count) state[idx[k]] = buf[k];
}

// Caller-order AoS [n][Q] -> state, perm[compact] = caller index.
template <int Q, typename S, class Lay>
__global__ __launch_bounds__(256) void k_import(DevDomain D, const double* aos,
                                                const int64_t* perm, S* state,
                                                double rho0) {
  SiteRef r;
  if (!Lay::locate(D, r)) return;
  const int64_t c = perm[Lay::compact(D, r)];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    double v = aos[c * Q + d];
    if constexpr (kShifted<S>) v -= Lat<Q>::w[d] * rho0;
    Store<S>::st(state + Lay::template at<Q>(D, d, r.x), (typename Store<S>::T)v);
  });
}

// Equilibrium of a per-site (density, momentum) field, caller's site order
// (perm maps the layout's compact index to it), with the collision's own
// Lattice::CalculateFeq arithmetic.
template <int Q, typename S, class Lay>
__global__ __launch_bounds__(256) void k_import_equilibrium(DevDomain D, const double* rho,
                                                            const double* mom,
                                                            const int64_t* perm, S* state,
                                                            double rho0) {
  SiteRef r;
  if (!Lay::locate(D, r)) return;
  const int64_t c = perm[Lay::compact(D, r)];
  const FeqCoef<double> fe(rho[c], mom[3 * c], mom[3 * c + 1], mom[3 * c + 2]);
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    double v = fe.template eq<Q, d>();
    if constexpr (kShifted<S>) v -= Lat<Q>::w[d] * rho0;
    Store<S>::st(state + Lay::template at<Q>(D, d, r.x), (typename Store<S>::T)v);
  });
}

template <int Q, typename S>
__global__ void k_fill(int64_t nslots, int64_t np, int blockwise, const double* vals,
                       S* state, double rho0) {
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= nslots) return;
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    double v = vals[d];
    if constexpr (kShifted<S>) v -= Lat<Q>::w[d] * rho0;
    const int64_t i = blockwise ? ((x >> 9) * Q + d) * 512 + (x & 511) : (int64_t)d * np + x;
    Store<S>::st(state + i, (typename Store<S>::T)v);
  });
}

__global__ void k_soa_to_aos(int Q, int64_t n, int64_t np, const double* soa,
                             const int64_t* perm, double* aos) {
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  const int64_t c = perm[x];
  for (int d = 0; d < Q; ++d) aos[c * Q + d] = soa[(int64_t)d * np + x];
}

template <int Q>
__global__ void k_moments(int64_t n, int64_t np, const double* soa, double* rho,
                          double* u) {
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  double f[Q];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    f[d] = soa[(int64_t)d * np + x];
  });
  double r, mx, my, mz;
  moments<Q, double>(f, r, mx, my, mz);
  rho[x] = r;
  u[x] = mx / r;
  u[np + x] = my / r;
  u[2 * np + x] = mz / r;
}

// Per-block binary64 reductions in a fixed tree order: [mass, min rho,
// max rho, max |u|, unstable] per block.
template <int Q>
__global__ __launch_bounds__(256) void k_reduce(int64_t n, int64_t np,
                                                const double* soa,
                                                const double* rho,
                                                const double* u,
                                                double* partials) {
  __shared__ double s_sum[256], s_min[256], s_max[256], s_u[256], s_bad[256];
  const int t = threadIdx.x;
  double sum = 0.0, mn = 1.7976931348623157e308, mx = -1.7976931348623157e308,
         um = 0.0, bad = 0.0;
  for (int64_t x = (int64_t)blockIdx.x * blockDim.x + t; x < n;
       x += (int64_t)gridDim.x * blockDim.x) {
    const double r = rho[x];
    sum += r;
    mn = r < mn ? r : mn;
    mx = r > mx ? r : mx;
    const double a = u[x], b = u[np + x], c = u[2 * np + x];
    const double m = sqrt(((0.0 + a * a) + b * b) + c * c);
    um = m > um ? m : um;
    for (int d = 0; d < Q; ++d)
      if (!(soa[(int64_t)d * np + x] > 0.0)) bad = 1.0;
  }
  s_sum[t] = sum; s_min[t] = mn; s_max[t] = mx; s_u[t] = um; s_bad[t] = bad;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) {
      s_sum[t] += s_sum[t + w];
      s_min[t] = s_min[t + w] < s_min[t] ? s_min[t + w] : s_min[t];
      s_max[t] = s_max[t + w] > s_max[t] ? s_max[t + w] : s_max[t];
      s_u[t] = s_u[t + w] > s_u[t] ? s_u[t + w] : s_u[t];
      s_bad[t] = s_bad[t + w] > s_bad[t] ? s_bad[t + w] : s_bad[t];
    }
    __syncthreads();
  }
  if (t == 0) {
    double* p = partials + 5 * blockIdx.x;
    p[0] = s_sum[0]; p[1] = s_min[0]; p[2] = s_max[0]; p[3] = s_u[0]; p[4] = s_bad[0];
  }
}

// The monitor's statistics straight from the state, without an exported
// copy: every site's fOld (the state itself when it is post-stream, else the
// pull of k_stream_only), its density and velocity as k_moments computes
// them, and per workgroup [mass, min rho, max rho, max |u|, unstable] as
// k_reduce combines them.  Workgroup g visits the x planes g*W + k*W*grid
// (W waves per workgroup) of the block layouts, or the compact sites
// g*256 + t + k*256*grid of the pull table, so the partials depend on the
// grid size only.  The density and velocity of every iolet site go to
// io_vals[4*record..] (rho, u_x, u_y, u_z) for the iolet fluxes.
template <int Q, typename S, class Lay>
__global__ __launch_bounds__(256) void k_monitor(DevDomain D, StepArgs A,
                                                 const S* __restrict__ fin,
                                                 int from_post_stream,
                                                 double* __restrict__ partials,
                                                 double* __restrict__ io_vals) {
  using T = typename Store<S>::T;
  __shared__ double s_sum[256], s_min[256], s_max[256], s_u[256], s_bad[256];
  const int t = threadIdx.x;
  double sum = 0.0, mn = 1.7976931348623157e308, mx = -1.7976931348623157e308,
         um = 0.0, bad = 0.0;
  auto visit = [&](const SiteRef& r) {
    T f[Q];
    if (from_post_stream) {
      sfor<0, Q>([&](auto di) {
        constexpr int d = decltype(di)::value;
        f[d] = Store<S>::ld(fin + Lay::template at<Q>(D, d, r.x));
      });
    } else {
      gather<Q, S, T, Lay>(D, A, fin, r, f);
    }
    double g[Q];
    sfor<0, Q>([&](auto di) {
      constexpr int d = decltype(di)::value;
      double v = (double)f[d];
      if constexpr (kShifted<S>) v += Lat<Q>::w[d] * A.rho0;
      g[d] = v;
      if (!(v > 0.0)) bad = 1.0;
    });
    double rho, m0, m1, m2;
    moments<Q, double>(g, rho, m0, m1, m2);
    const double ux = m0 / rho, uy = m1 / rho, uz = m2 / rho;
    sum += rho;
    mn = rho < mn ? rho : mn;
    mx = rho > mx ? rho : mx;
    const double m = sqrt(((0.0 + ux * ux) + uy * uy) + uz * uz);
    um = m > um ? m : um;
    if (r.cut) {
      const int io = D.b_io[r.rec];
      if (io >= 0) {
        io_vals[4 * (int64_t)io] = rho;
        io_vals[4 * (int64_t)io + 1] = ux;
        io_vals[4 * (int64_t)io + 2] = uy;
        io_vals[4 * (int64_t)io + 3] = uz;
      }
    }
  };
  if constexpr (kWaveLayout<Lay>) {
    const uint32_t wpg = blockDim.x >> 6;
    for (uint32_t base = blockIdx.x * wpg; base < D.nwaves; base += gridDim.x * wpg) {
      const uint32_t w = __builtin_amdgcn_readfirstlane(base + ((uint32_t)t >> 6));
      SiteRef r;
      if (Lay::locate_wave(D, w, r)) visit(r);
    }
  } else {
    for (int64_t x = (int64_t)blockIdx.x * blockDim.x + t; x < D.n;
         x += (int64_t)gridDim.x * blockDim.x) {
      SiteRef r;
      Lay::at(D, x, r);
      visit(r);
    }
  }
  s_sum[t] = sum; s_min[t] = mn; s_max[t] = mx; s_u[t] = um; s_bad[t] = bad;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) {
      s_sum[t] += s_sum[t + w];
      s_min[t] = s_min[t + w] < s_min[t] ? s_min[t + w] : s_min[t];
      s_max[t] = s_max[t + w] > s_max[t] ? s_max[t + w] : s_max[t];
      s_u[t] = s_u[t + w] > s_u[t] ? s_u[t + w] : s_u[t];
      s_bad[t] = s_bad[t + w] > s_bad[t] ? s_bad[t + w] : s_bad[t];
    }
    __syncthreads();
  }
  if (t == 0) {
    double* p = partials + 5 * blockIdx.x;
    p[0] = s_sum[0]; p[1] = s_min[0]; p[2] = s_max[0]; p[3] = s_u[0]; p[4] = s_bad[0];
  }
}

// The same statistics per chunk of sites [range[2b], range[2b+1]) (one
// workgroup per chunk; chunks never mix instances of an ensemble).
template <int Q>
__global__ __launch_bounds__(256) void k_reduce_ranges(int64_t np, const int64_t* range,
                                                       const double* soa,
                                                       const double* rho,
                                                       const double* u,
                                                       double* partials) {
  __shared__ double s_sum[256], s_min[256], s_max[256], s_u[256], s_bad[256];
  const int t = threadIdx.x;
  double sum = 0.0, mn = 1.7976931348623157e308, mx = -1.7976931348623157e308,
         um = 0.0, bad = 0.0;
  const int64_t end = range[2 * blockIdx.x + 1];
  for (int64_t x = range[2 * blockIdx.x] + t; x < end; x += blockDim.x) {
    const double r = rho[x];
    sum += r;
    mn = r < mn ? r : mn;
    mx = r > mx ? r : mx;
    const double a = u[x], b = u[np + x], c = u[2 * np + x];
    const double m = sqrt(((0.0 + a * a) + b * b) + c * c);
    um = m > um ? m : um;
    for (int d = 0; d < Q; ++d)
      if (!(soa[(int64_t)d * np + x] > 0.0)) bad = 1.0;
  }
  s_sum[t] = sum; s_min[t] = mn; s_max[t] = mx; s_u[t] = um; s_bad[t] = bad;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) {
      s_sum[t] += s_sum[t + w];
      s_min[t] = s_min[t + w] < s_min[t] ? s_min[t + w] : s_min[t];
      s_max[t] = s_max[t + w] > s_max[t] ? s_max[t + w] : s_max[t];
      s_u[t] = s_u[t + w] > s_u[t] ? s_u[t + w] : s_u[t];
      s_bad[t] = s_bad[t + w] > s_bad[t] ? s_bad[t + w] : s_bad[t];
    }
    __syncthreads();
  }
  if (t == 0) {
    double* p = partials + 5 * blockIdx.x;
    p[0] = s_sum[0]; p[1] = s_min[0]; p[2] = s_max[0]; p[3] = s_u[0]; p[4] = s_bad[0];
  }
}

__global__ __launch_bounds__(256) void k_velocity_change_ranges(
    int64_t np, const int64_t* range, const double* u, const double* u0,
    const double* inv_ref, double* partials) {
  __shared__ double s[256];
  const int t = threadIdx.x;
  double m = 0.0;
  const double ir = inv_ref[blockIdx.x];
  const int64_t end = range[2 * blockIdx.x + 1];
  for (int64_t x = range[2 * blockIdx.x] + t; x < end; x += blockDim.x) {
    const double a = u[x] - u0[x], b = u[np + x] - u0[np + x],
                 c = u[2 * np + x] - u0[2 * np + x];
    const double v = sqrt(((0.0 + a * a) + b * b) + c * c) * ir;
    m = v > m ? v : m;
  }
  s[t] = m;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) s[t] = s[t + w] > s[t] ? s[t + w] : s[t];
    __syncthreads();
  }
  if (t == 0) partials[blockIdx.x] = s[0];
}

__global__ __launch_bounds__(256) void k_velocity_change(int64_t n, int64_t np,
                                                         const double* u,
                                                         const double* u0,
                                                         double inv_ref,
                                                         double* partials) {
  __shared__ double s[256];
  const int t = threadIdx.x;
  double m = 0.0;
  for (int64_t x = (int64_t)blockIdx.x * blockDim.x + t; x < n;
       x += (int64_t)gridDim.x * blockDim.x) {
    const double a = u[x] - u0[x], b = u[np + x] - u0[np + x],
                 c = u[2 * np + x] - u0[2 * np + x];
    const double v = sqrt(((0.0 + a * a) + b * b) + c * c) * inv_ref;
    m = v > m ? v : m;
  }
  s[t] = m;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) s[t] = s[t + w] > s[t] ? s[t + w] : s[t];
    __syncthreads();
  }
  if (t == 0) partials[blockIdx.x] = s[0];
}

// Wall shear stress magnitude at the wall sites (Lattice.h:652-727) from the
// post-stream binary64 distributions: f_neq = f - f_eq with the SSE3-order
// equilibrium; Pi_ab = sum_l f_neq_l c_la c_lb accumulated in direction
// order (terms with c_la c_lb = 0 add nothing); t_a = sum_b (Pi_ab n_b) temp;
// result sqrt(|t|^2 - (t . n)^2).
template <int Q, int A, int B>
__device__ __forceinline__ double second_moment(const double (&fneq)[Q]) {
  using L = Lat<Q>;
  double acc = 0.0;
  sfor<0, Q>([&](auto li) {
    constexpr int l = decltype(li)::value;
    constexpr int c = L::c[l][A] * L::c[l][B];
    if constexpr (c == 1) acc = acc + fneq[l];
    else if constexpr (c == -1) acc = acc - fneq[l];
  });
  return acc;
}

template <int Q>
__global__ __launch_bounds__(256) void k_wall_shear_stress(
    int64_t nw, int64_t np, const double* __restrict__ soa,
    const int64_t* __restrict__ site, const float* __restrict__ nrm,
    const double* __restrict__ temp_of, double* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nw) return;
  const int64_t x = site[i];
  double f[Q];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    f[d] = soa[(int64_t)d * np + x];
  });
  double r, mx, my, mz;
  moments<Q, double>(f, r, mx, my, mz);
  const FeqCoef<double> fe(r, mx, my, mz);
  double fneq[Q];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    fneq[d] = f[d] - fe.template eq<Q, d>();
  });
  const double p00 = second_moment<Q, 0, 0>(fneq), p10 = second_moment<Q, 1, 0>(fneq),
               p11 = second_moment<Q, 1, 1>(fneq), p20 = second_moment<Q, 2, 0>(fneq),
               p21 = second_moment<Q, 2, 1>(fneq), p22 = second_moment<Q, 2, 2>(fneq);
  const double pi[3][3] = {{p00, p10, p20}, {p10, p11, p21}, {p20, p21, p22}};
  const double n[3] = {(double)nrm[3 * i], (double)nrm[3 * i + 1], (double)nrm[3 * i + 2]};
  const double temp = temp_of[i];
  double sq = 0.0, nn = 0.0;
  for (int a = 0; a < 3; ++a) {
    double t = 0.0;
    for (int b = 0; b < 3; ++b) t += pi[a][b] * n[b] * temp;
    sq += t * t;
    nn += t * n[a];
  }
  out[i] = sqrt(sq - nn * nn);
}

// The other stress outputs of the reference's property cache (Lattice.h):
// f_neq = f - f_eq (SSE3 order), Pi_ab = sum_l f_neq_l c_la c_lb in direction
// order.  Stress tensor (CalculateStressTensor, 630-645): Pi * (1 - 1/(2 tau))
// plus (rho - 1) Cs2 on the diagonal, upper triangle xx xy xz yy yz zz;
// von Mises stress (508-552); shear rate (728-753, 890-907).  The tau of
// each site is tau_site[x] when given.
template <int Q>
__global__ __launch_bounds__(256) void k_stress_fields(
    int64_t n, int64_t np, const double* __restrict__ soa, double tau,
    const double* __restrict__ tau_site, double* __restrict__ t6,
    double* __restrict__ vm, double* __restrict__ sr) {
  using L = Lat<Q>;
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  const double ts = tau_site ? tau_site[x] : tau;
  double f[Q];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    f[d] = soa[(int64_t)d * np + x];
  });
  double r, mx, my, mz;
  moments<Q, double>(f, r, mx, my, mz);
  const FeqCoef<double> fe(r, mx, my, mz);
  double fneq[Q];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    fneq[d] = f[d] - fe.template eq<Q, d>();
  });
  const double p00 = second_moment<Q, 0, 0>(fneq), p10 = second_moment<Q, 1, 0>(fneq),
               p11 = second_moment<Q, 1, 1>(fneq), p20 = second_moment<Q, 2, 0>(fneq),
               p21 = second_moment<Q, 2, 1>(fneq), p22 = second_moment<Q, 2, 2>(fneq);
  if (t6) {
    const double fac = 1 - 1 / (2 * ts);
    const double pr = (r - 1) * kCs2;
    t6[x] = p00 * fac + pr;
    t6[np + x] = p10 * fac;
    t6[2 * np + x] = p20 * fac;
    t6[3 * np + x] = p11 * fac + pr;
    t6[4 * np + x] = p21 * fac;
    t6[5 * np + x] = p22 * fac + pr;
  }
  if (vm) {
    // sums of f_neq (cx^2 - cy^2) etc. in direction order
    double xx_yy = 0.0, yy_zz = 0.0, xx_zz = 0.0, xy = 0.0, xz = 0.0, yz = 0.0;
    sfor<0, Q>([&](auto li) {
      constexpr int l = decltype(li)::value;
      constexpr int cx = L::c[l][0], cy = L::c[l][1], cz = L::c[l][2];
      constexpr int a = cx * cx - cy * cy, b = cy * cy - cz * cz, c = cx * cx - cz * cz;
      if constexpr (a != 0) xx_yy += fneq[l] * (double)a;
      if constexpr (b != 0) yy_zz += fneq[l] * (double)b;
      if constexpr (c != 0) xx_zz += fneq[l] * (double)c;
      if constexpr (cx * cy != 0) xy += fneq[l] * (double)cx * (double)cy;
      if constexpr (cx * cz != 0) xz += fneq[l] * (double)cx * (double)cz;
      if constexpr (cy * cz != 0) yz += fneq[l] * (double)cy * (double)cz;
    });
    const double a = xx_yy * xx_yy + yy_zz * yy_zz + xx_zz * xx_zz;
    const double b = xy * xy + xz * xz + yz * yz;
    const double sp = (1.0 - 1.0 / (2.0 * ts)) / sqrt(2.0);
    vm[x] = sp * sqrt(a + 6.0 * b);
  }
  if (sr) {
    const double k = -1.0 / (2.0 * ts * r * kCs2);
    const double e[6] = {p00 * k, p10 * k, p20 * k, p11 * k, p21 * k, p22 * k};
    // rows: (0,0) (0,1) (0,2) (1,1) (1,2) (2,2)
    double acc = 0.0;
    acc += e[0] * e[0];
    acc += 2 * e[1] * e[1];
    acc += 2 * e[2] * e[2];
    acc += e[3] * e[3];
    acc += 2 * e[4] * e[4];
    acc += e[5] * e[5];
    sr[x] = sqrt(2 * acc);
  }
}

// Traction sigma n and its tangential projection t - n (t . n) at the wall
// sites (CalculateTractionOnAPoint / CalculateTangentialProjectionTraction,
// Lattice.h:560-602); tau_of[i] is the tau of wall site i.
template <int Q>
__global__ __launch_bounds__(256) void k_traction(
    int64_t nw, int64_t np, const double* __restrict__ soa,
    const int64_t* __restrict__ site, const float* __restrict__ nrm,
    const double* __restrict__ tau_of, double* __restrict__ tr, double* __restrict__ tg) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nw) return;
  const int64_t x = site[i];
  double f[Q];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    f[d] = soa[(int64_t)d * np + x];
  });
  double r, mx, my, mz;
  moments<Q, double>(f, r, mx, my, mz);
  const FeqCoef<double> fe(r, mx, my, mz);
  double fneq[Q];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    fneq[d] = f[d] - fe.template eq<Q, d>();
  });
  const double fac = 1 - 1 / (2 * tau_of[i]);
  const double pr = (r - 1) * kCs2;
  const double p00 = second_moment<Q, 0, 0>(fneq), p10 = second_moment<Q, 1, 0>(fneq),
               p11 = second_moment<Q, 1, 1>(fneq), p20 = second_moment<Q, 2, 0>(fneq),
               p21 = second_moment<Q, 2, 1>(fneq), p22 = second_moment<Q, 2, 2>(fneq);
  const double sg[3][3] = {{p00 * fac + pr, p10 * fac, p20 * fac},
                           {p10 * fac, p11 * fac + pr, p21 * fac},
                           {p20 * fac, p21 * fac, p22 * fac + pr}};
  const double n[3] = {(double)nrm[3 * i], (double)nrm[3 * i + 1], (double)nrm[3 * i + 2]};
  double t[3];
  for (int a = 0; a < 3; ++a) {
    t[a] = 0.0;
    for (int b = 0; b < 3; ++b) t[a] += sg[a][b] * n[b];
  }
  double tn = 0.0;
  for (int a = 0; a < 3; ++a) tn = tn + t[a] * n[a];
  for (int a = 0; a < 3; ++a) {
    tr[3 * i + a] = t[a];
    tg[3 * i + a] = t[a] - n[a] * tn;
  }
}

template <typename S>
__global__ void k_gather_pairs(int64_t count, int64_t np, int Q, int blockwise,
                               const int64_t* slot, const S* state, double rho0,
                               const double* w, double* out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int64_t sidx = slot[i];
  double v = (double)Store<S>::ld(state + sidx);
  const int d = blockwise ? (int)((sidx >> 9) % Q) : (int)(sidx / np);
  if constexpr (kShifted<S>) v += w[d] * rho0;
  out[i] = v;
}

// Halo unpack: state[slot[i]] = in[i] (shifted storage stores in - w rho0).
template <typename S>
__global__ void k_scatter_pairs(int64_t count, int64_t np, int Q, int blockwise,
                                const int64_t* slot, const double* in, double rho0,
                                const double* w, S* state) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int64_t sidx = slot[i];
  double v = in[i];
  const int d = blockwise ? (int)((sidx >> 9) % Q) : (int)(sidx / np);
  if constexpr (kShifted<S>) v -= w[d] * rho0;
  Store<S>::st(state + sidx, (typename Store<S>::T)v);
}

}  // namespace

int launch_fill(const DevDomain& d, const StepArgs& a, const double* vals, void* state,
                void* stream) {
  return dispatch(d, a, [&](auto q, auto, auto* s, auto*) {
    using S = std::remove_pointer_t<decltype(s)>;
    constexpr int Q = decltype(q)::value;
    hipLaunchKernelGGL((k_fill<Q, S>), grid_for(d.np), dim3(256), 0, (hipStream_t)stream,
                       d.np, d.np, d.layout == 1 ? 1 : 0, vals, (S*)state, a.rho0);
    return (int)hipGetLastError();
  });
}

int launch_step(const DevDomain& d, const StepArgs& a, const void* fin, void* fout,
                void* stream) {
  return d.layout == 0   ? step_in<0>(d, a, fin, fout, stream)
         : d.layout == 1 ? step_in<1>(d, a, fin, fout, stream)
                         : step_in<2>(d, a, fin, fout, stream);
}

int launch_collide_only(const DevDomain& d, const StepArgs& a, const void* fin,
                        void* fout, void* stream) {
  return d.layout == 0   ? collide_only_in<0>(d, a, fin, fout, stream)
         : d.layout == 1 ? collide_only_in<1>(d, a, fin, fout, stream)
                         : collide_only_in<2>(d, a, fin, fout, stream);
}

int launch_stream_only(const DevDomain& d, const StepArgs& a, const void* fin,
                       double* s_out, int from_post_stream, void* stream) {
  return dispatch(d, a, [&](auto q, auto, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    hipLaunchKernelGGL((k_stream_only<decltype(q)::value, S, Lay>), grid_for(thread_count(d)),
                       dim3(256), 0, (hipStream_t)stream, d, a, (const S*)fin, s_out,
                       from_post_stream);
    return (int)hipGetLastError();
  });
}

int launch_import(const DevDomain& d, const StepArgs& a, const double* aos,
                  const int64_t* perm, void* state, void* stream) {
  return dispatch(d, a, [&](auto q, auto, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    hipLaunchKernelGGL((k_import<decltype(q)::value, S, Lay>), grid_for(thread_count(d)),
                       dim3(256), 0, (hipStream_t)stream, d, aos, perm, (S*)state, a.rho0);
    return (int)hipGetLastError();
  });
}

int launch_import_equilibrium(const DevDomain& d, const StepArgs& a, const double* rho,
                              const double* mom, const int64_t* perm, void* state,
                              void* stream) {
  return dispatch(d, a, [&](auto q, auto, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    hipLaunchKernelGGL((k_import_equilibrium<decltype(q)::value, S, Lay>),
                       grid_for(thread_count(d)), dim3(256), 0, (hipStream_t)stream, d, rho,
                       mom, perm, (S*)state, a.rho0);
    return (int)hipGetLastError();
  });
}

int launch_soa_to_aos(int Q, int64_t n, int64_t np, const double* soa,
                      const int64_t* perm, double* aos, void* stream) {
  hipLaunchKernelGGL(k_soa_to_aos, grid_for(n), dim3(256), 0, (hipStream_t)stream,
                     Q, n, np, soa, perm, aos);
  return (int)hipGetLastError();
}

int launch_moments(int Q, int64_t n, int64_t np, const double* soa, double* rho,
                   double* u, void* stream) {
  if (Q == 15)
    hipLaunchKernelGGL(k_moments<15>, grid_for(n), dim3(256), 0,
                       (hipStream_t)stream, n, np, soa, rho, u);
  else
    hipLaunchKernelGGL(k_moments<19>, grid_for(n), dim3(256), 0,
                       (hipStream_t)stream, n, np, soa, rho, u);
  return (int)hipGetLastError();
}

int launch_wall_shear_stress(int Q, int64_t nw, int64_t np, const double* soa,
                             const int64_t* site, const float* normal, const double* temp,
                             double* out, void* stream) {
  if (nw == 0) return 0;
  if (Q == 15)
    hipLaunchKernelGGL(k_wall_shear_stress<15>, grid_for(nw), dim3(256), 0,
                       (hipStream_t)stream, nw, np, soa, site, normal, temp, out);
  else
    hipLaunchKernelGGL(k_wall_shear_stress<19>, grid_for(nw), dim3(256), 0,
                       (hipStream_t)stream, nw, np, soa, site, normal, temp, out);
  return (int)hipGetLastError();
}

int launch_reduce(int Q, int64_t n, int64_t np, const double* soa,
                  const double* rho, const double* u, double* partials,
                  int nblocks, void* stream) {
  if (Q == 15)
    hipLaunchKernelGGL(k_reduce<15>, dim3(nblocks), dim3(256), 0,
                       (hipStream_t)stream, n, np, soa, rho, u, partials);
  else
    hipLaunchKernelGGL(k_reduce<19>, dim3(nblocks), dim3(256), 0,
                       (hipStream_t)stream, n, np, soa, rho, u, partials);
  return (int)hipGetLastError();
}

int launch_copy_arrays(int Q, int64_t stride_bytes, int64_t bytes, int64_t run_bytes,
                       int width, const void* in, void* out, uint32_t threads, uint32_t remap,
                       void* stream) {
  if (width != 4 && width != 8 && width != 16) return (int)hipErrorInvalidValue;
  if (stride_bytes % width || bytes % width || run_bytes % width)
    return (int)hipErrorInvalidValue;
  if (run_bytes && bytes % run_bytes) return (int)hipErrorInvalidValue;
  const int64_t run = run_bytes / width;
  if (threads != 64 && threads != 128 && threads != 256) return (int)hipErrorInvalidValue;
  const int64_t words = bytes / width, stride = stride_bytes / width;
  uint64_t groups = ((uint64_t)words + threads - 1) / threads;
  if (remap >= 2) {
    const uint64_t m = 8ull * remap;
    groups = (groups + m - 1) / m * m;
  }
  const dim3 grid((unsigned)std::max<uint64_t>(groups, 1)), block(threads);
  auto go = [&](auto q, auto* w) {
    using W = std::remove_pointer_t<decltype(w)>;
    hipLaunchKernelGGL((k_copy_arrays<decltype(q)::value, W>), grid, block, 0,
                       (hipStream_t)stream, stride, words, run, (const W*)in, (W*)out, remap);
  };
  if (Q == 15) {
    if (width == 4) go(std::integral_constant<int, 15>{}, (unsigned int*)nullptr);
    else if (width == 8) go(std::integral_constant<int, 15>{}, (u32x2*)nullptr);
    else go(std::integral_constant<int, 15>{}, (u32x4*)nullptr);
  } else if (Q == 19) {
    if (width == 4) go(std::integral_constant<int, 19>{}, (unsigned int*)nullptr);
    else if (width == 8) go(std::integral_constant<int, 19>{}, (u32x2*)nullptr);
    else go(std::integral_constant<int, 19>{}, (u32x4*)nullptr);
  } else {
    return (int)hipErrorInvalidValue;
  }
  return (int)hipGetLastError();
}

int launch_halo(int64_t count, const int64_t* idx, int esize, const void* from, void* to,
                int pack, void* stream) {
  if (count == 0) return 0;
  const dim3 grid = grid_for(count), block(256);
  auto go = [&](auto* e) {
    using E = std::remove_pointer_t<decltype(e)>;
    if (pack)
      hipLaunchKernelGGL(k_halo_pack<E>, grid, block, 0, (hipStream_t)stream, count, idx,
                         (const E*)from, (E*)to);
    else
      hipLaunchKernelGGL(k_halo_unpack<E>, grid, block, 0, (hipStream_t)stream, count, idx,
                         (const E*)from, (E*)to);
  };
  if (esize == 8) go((uint64_t*)nullptr);
  else if (esize == 4) go((uint32_t*)nullptr);
  else if (esize == 2) go((uint16_t*)nullptr);
  else return (int)hipErrorInvalidValue;
  return (int)hipGetLastError();
}

int scratch_address(int device, double** out) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static double* addr[kMaxDevices] = {};
  if (device < 0 || device >= kMaxDevices) return (int)hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[device]) {
    // the caller has made `device` current: this is its copy of the array
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    addr[device] = (double*)p;
  }
  *out = addr[device];
  return 0;
}

int launch_monitor(const DevDomain& d, const StepArgs& a, const void* fin,
                   int from_post_stream, double* partials, double* io_vals, void* stream) {
  return dispatch(d, a, [&](auto q, auto, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    hipLaunchKernelGGL((k_monitor<decltype(q)::value, S, Lay>), dim3(kMonitorGroups),
                       dim3(256), 0, (hipStream_t)stream, d, a, (const S*)fin,
                       from_post_stream, partials, io_vals);
    return (int)hipGetLastError();
  });
}

int launch_stress_fields(int Q, int64_t n, int64_t np, const double* soa, double tau,
                         const double* tau_site, double* t6, double* vm, double* sr,
                         void* stream) {
  if (n == 0) return 0;
  if (Q == 15)
    hipLaunchKernelGGL(k_stress_fields<15>, grid_for(n), dim3(256), 0, (hipStream_t)stream, n,
                       np, soa, tau, tau_site, t6, vm, sr);
  else
    hipLaunchKernelGGL(k_stress_fields<19>, grid_for(n), dim3(256), 0, (hipStream_t)stream, n,
                       np, soa, tau, tau_site, t6, vm, sr);
  return (int)hipGetLastError();
}

int launch_traction(int Q, int64_t nw, int64_t np, const double* soa, const int64_t* site,
                    const float* normal, const double* tau_of, double* tr, double* tg,
                    void* stream) {
  if (nw == 0) return 0;
  if (Q == 15)
    hipLaunchKernelGGL(k_traction<15>, grid_for(nw), dim3(256), 0, (hipStream_t)stream, nw, np,
                       soa, site, normal, tau_of, tr, tg);
  else
    hipLaunchKernelGGL(k_traction<19>, grid_for(nw), dim3(256), 0, (hipStream_t)stream, nw, np,
                       soa, site, normal, tau_of, tr, tg);
  return (int)hipGetLastError();
}

int launch_reduce_ranges(int Q, int64_t nchunks, int64_t np, const int64_t* range,
                         const double* soa, const double* rho, const double* u,
                         double* partials, void* stream) {
  if (nchunks == 0) return 0;
  if (Q == 15)
    hipLaunchKernelGGL(k_reduce_ranges<15>, dim3((unsigned)nchunks), dim3(256), 0,
                       (hipStream_t)stream, np, range, soa, rho, u, partials);
  else
    hipLaunchKernelGGL(k_reduce_ranges<19>, dim3((unsigned)nchunks), dim3(256), 0,
                       (hipStream_t)stream, np, range, soa, rho, u, partials);
  return (int)hipGetLastError();
}

int launch_velocity_change_ranges(int64_t nchunks, int64_t np, const int64_t* range,
                                  const double* u, const double* u_ref,
                                  const double* inv_ref, double* partials, void* stream) {
  if (nchunks == 0) return 0;
  hipLaunchKernelGGL(k_velocity_change_ranges, dim3((unsigned)nchunks), dim3(256), 0,
                     (hipStream_t)stream, np, range, u, u_ref, inv_ref, partials);
  return (int)hipGetLastError();
}

int launch_velocity_change(int64_t n, int64_t np, const double* u,
                           const double* u_ref, double inv_ref, double* partials,
                           int nblocks, void* stream) {
  hipLaunchKernelGGL(k_velocity_change, dim3(nblocks), dim3(256), 0,
                     (hipStream_t)stream, n, np, u, u_ref, inv_ref, partials);
  return (int)hipGetLastError();
}

int launch_gather_pairs(int64_t count, int64_t np, int Q, int blockwise,
                        const int64_t* slot_index, const void* state, int storage, double rho0,
                        const double* w, double* out, void* stream) {
  if (storage == 0)
    hipLaunchKernelGGL(k_gather_pairs<double>, grid_for(count), dim3(256), 0,
                       (hipStream_t)stream, count, np, Q, blockwise, slot_index,
                       (const double*)state, rho0, w, out);
  else if (storage == 1)
    hipLaunchKernelGGL(k_gather_pairs<float>, grid_for(count), dim3(256), 0,
                       (hipStream_t)stream, count, np, Q, blockwise, slot_index,
                       (const float*)state, rho0, w, out);
  else
    hipLaunchKernelGGL(k_gather_pairs<_Float16>, grid_for(count), dim3(256), 0,
                       (hipStream_t)stream, count, np, Q, blockwise, slot_index,
                       (const _Float16*)state, rho0, w, out);
  return (int)hipGetLastError();
}

int launch_scatter_pairs(int64_t count, int64_t np, int Q, int blockwise,
                         const int64_t* slot_index, const double* in, int storage, double rho0,
                         const double* w, void* state, void* stream) {
  if (storage == 0)
    hipLaunchKernelGGL(k_scatter_pairs<double>, grid_for(count), dim3(256), 0,
                       (hipStream_t)stream, count, np, Q, blockwise, slot_index, in, rho0, w,
                       (double*)state);
  else if (storage == 1)
    hipLaunchKernelGGL(k_scatter_pairs<float>, grid_for(count), dim3(256), 0,
                       (hipStream_t)stream, count, np, Q, blockwise, slot_index, in, rho0, w,
                       (float*)state);
  else
    hipLaunchKernelGGL(k_scatter_pairs<_Float16>, grid_for(count), dim3(256), 0,
                       (hipStream_t)stream, count, np, Q, blockwise, slot_index, in, rho0, w,
                       (_Float16*)state);
  return (int)hipGetLastError();
}

}  // namespace hlb
