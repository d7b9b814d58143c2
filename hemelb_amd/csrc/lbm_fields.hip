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

// Post-stream distributions of a site (the reference's fOld) in binary64:
// the state itself when it already is post-stream, else the pull.
template <int Q, typename S, class Lay>
__device__ __forceinline__ void post_stream_site(const DevDomain& D, const StepArgs& A,
                                                 const S* __restrict__ fin,
                                                 int from_post_stream, const SiteRef& r,
                                                 double (&g)[Q]) {
  using T = typename Store<S>::T;
  T f[Q];
  if (from_post_stream) {
    sfor<0, Q>([&](auto di) {
      constexpr int d = decltype(di)::value;
      f[d] = Store<S>::ld(own_ptr<Q, Lay>(D, r, fin, d));
    });
  } else {
    gather<Q, S, T, Lay>(D, A, fin, r, f);
  }
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    double v = (double)f[d];
    if constexpr (kShifted<S>) v += Lat<Q>::w[d] * A.rho0;
    g[d] = v;
  });
}

// Calls visit(site) for every site of workgroup blockIdx.x: without `range`
// the x planes g*W + k*W*grid (W waves per workgroup) of the block layouts, or
// the compact sites g*256 + t + k*256*grid of the pull table, so that a
// reduction's partials depend on the grid size only; with it, the planes (or
// sites) range[2g] .. range[2g+1].
template <class Lay, typename V>
__device__ __forceinline__ void visit_sites(const DevDomain& D, const int64_t* range, V&& visit) {
  const int t = threadIdx.x;
  if constexpr (kWaveLayout<Lay>) {
    const uint32_t wpg = blockDim.x >> 6;
    const uint32_t step = range ? wpg : gridDim.x * wpg;
    const uint32_t end = range ? (uint32_t)range[2 * blockIdx.x + 1] : D.nwaves;
    for (uint32_t base = range ? (uint32_t)range[2 * blockIdx.x] : blockIdx.x * wpg; base < end;
         base += step) {
      const uint32_t w = __builtin_amdgcn_readfirstlane(base + ((uint32_t)t >> 6));
      SiteRef r;
      if (w < end && Lay::locate_wave(D, w, r)) visit(r);
    }
  } else {
    const int64_t step = range ? blockDim.x : (int64_t)gridDim.x * blockDim.x;
    const int64_t end = range ? range[2 * blockIdx.x + 1] : D.n;
    for (int64_t x = (range ? range[2 * blockIdx.x] : (int64_t)blockIdx.x * blockDim.x) + t;
         x < end; x += step) {
      SiteRef r;
      Lay::at(D, x, r);
      visit(r);
    }
  }
}

// The monitor's statistics straight from the state, without an exported
// copy: every site's fOld (the state itself when it is post-stream, else its
// pull), its density and velocity, and per workgroup [mass, min rho,
// max rho, max |u|, unstable] in a fixed tree order.  The density and
// velocity of every iolet site go to io_vals[4*record..] (rho, u_x, u_y,
// u_z) for the iolet fluxes, when given.  Bound by the state's read.  The
// outputs may be pinned host memory: a few KB and 32 bytes per iolet site,
// written once, cost less over the bus than a copy after the kernel (1.13 M
// sites, 141 k of them at an iolet: 0.61 -> 0.36 ms).  Monitor, velocity change and
// snapshot together on an 819 k-site binary64 tree: 0.38 ms before (two
// exported copies of the distributions, four copies), 0.22 ms now.
template <int Q, typename S, class Lay>
__global__ __launch_bounds__(256) void k_monitor(DevDomain D, StepArgs A,
                                                 const S* __restrict__ fin,
                                                 int from_post_stream, const int64_t* range,
                                                 double* __restrict__ partials,
                                                 double* __restrict__ io_vals) {
  __shared__ double s_sum[256], s_min[256], s_max[256], s_u[256], s_bad[256];
  const int t = threadIdx.x;
  double sum = 0.0, mn = 1.7976931348623157e308, mx = -1.7976931348623157e308,
         um = 0.0, bad = 0.0;
  visit_sites<Lay>(D, range, [&](const SiteRef& r) {
    double g[Q];
    post_stream_site<Q, S, Lay>(D, A, fin, from_post_stream, r, g);
    sfor<0, Q>([&](auto di) {
      if (!(g[decltype(di)::value] > 0.0)) bad = 1.0;
    });
    double rho, m0, m1, m2;
    moments<Q, double>(g, rho, m0, m1, m2);
    const double ux = m0 / rho, uy = m1 / rho, uz = m2 / rho;
    sum += rho;
    mn = rho < mn ? rho : mn;
    mx = rho > mx ? rho : mx;
    const double m = sqrt(((0.0 + ux * ux) + uy * uy) + uz * uz);
    um = m > um ? m : um;
    if (io_vals) {
      const int io = r.io;
      if (io >= 0) {
        io_vals[4 * (int64_t)io] = rho;
        io_vals[4 * (int64_t)io + 1] = ux;
        io_vals[4 * (int64_t)io + 2] = uy;
        io_vals[4 * (int64_t)io + 3] = uz;
      }
    }
  });
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

// The velocity of fOld, u[3][npc] by compact site (the convergence monitor's
// snapshot), straight from the state.
template <int Q, typename S, class Lay>
__global__ __launch_bounds__(256) void k_snapshot_velocity(DevDomain D, StepArgs A,
                                                           const S* __restrict__ fin,
                                                           int from_post_stream,
                                                           double* __restrict__ u) {
  SiteRef r;
  if (!Lay::locate(D, r)) return;
  double g[Q];
  post_stream_site<Q, S, Lay>(D, A, fin, from_post_stream, r, g);
  double rho, mx, my, mz;
  moments<Q, double>(g, rho, mx, my, mz);
  const int64_t c = Lay::compact(D, r);
  u[c] = mx / rho;
  u[D.npc + c] = my / rho;
  u[2 * D.npc + c] = mz / rho;
}

// Per workgroup max |u - u0| * inv_ref over its sites, u from the state.
template <int Q, typename S, class Lay>
__global__ __launch_bounds__(256) void k_velocity_change(
    DevDomain D, StepArgs A, const S* __restrict__ fin, int from_post_stream,
    const int64_t* range, const double* __restrict__ u0, const double* __restrict__ inv_refs,
    double inv_ref, double* __restrict__ partials) {
  __shared__ double s[256];
  const int t = threadIdx.x;
  double m = 0.0;
  const double ir = inv_refs ? inv_refs[blockIdx.x] : inv_ref;
  visit_sites<Lay>(D, range, [&](const SiteRef& r) {
    const int64_t x = Lay::compact(D, r);
    const double v0 = u0[x], v1 = u0[D.npc + x], v2 = u0[2 * D.npc + x];
    double g[Q];
    post_stream_site<Q, S, Lay>(D, A, fin, from_post_stream, r, g);
    double rho, mx, my, mz;
    moments<Q, double>(g, rho, mx, my, mz);
    const double a = mx / rho - v0, b = my / rho - v1, c = mz / rho - v2;
    const double v = sqrt(((0.0 + a * a) + b * b) + c * c) * ir;
    m = v > m ? v : m;
  });
  s[t] = m;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) s[t] = s[t + w] > s[t] ? s[t + w] : s[t];
    __syncthreads();
  }
  if (t == 0) partials[blockIdx.x] = s[0];
}

// fOld as the caller's AoS [n][Q].  The lane's Q values go through LDS so
// that the wave writes each site's Q values as one run of memory (the perm
// of neighbouring sites is mostly consecutive) instead of 19 stores of 64
// scattered values.
template <int Q, typename S, class Lay>
__global__ __launch_bounds__(256) void k_export_distributions(
    DevDomain D, StepArgs A, const S* __restrict__ fin, int from_post_stream,
    const int64_t* __restrict__ perm, double* __restrict__ out) {
  __shared__ double rows[4][64 * Q];
  __shared__ int64_t site[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  SiteRef r;
  const bool live = Lay::locate(D, r);
  const uint64_t mask = __ballot(live);
  if (live) {
    double g[Q];
    post_stream_site<Q, S, Lay>(D, A, fin, from_post_stream, r, g);
    const int k = __popcll(mask & ((1ull << lane) - 1ull));
    site[wv][k] = perm[Lay::compact(D, r)];
    sfor<0, Q>([&](auto di) {
      constexpr int d = decltype(di)::value;
      rows[wv][k * Q + d] = g[d];
    });
  }
  __syncthreads();
  const int count = __popcll(mask) * Q;
  for (int j = lane; j < count; j += 64) {
    const int k = j / Q;
    out[site[wv][k] * Q + (j - k * Q)] = rows[wv][j];
  }
}

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

// The property fields of fOld in the caller's site order, straight from the
// state: one pull per site, no exported distributions in between (they cost
// 2 Q 8 bytes a site and a second kernel per field), and no permutation on
// the host.  Bound by the host link: with both gone, all 19 output doubles of
// a 2.76 M-site tree take 42 ms instead of 109, and density and velocity of a
// 7.93 M-site tree 25 ms instead of 95.
//
// Density and velocity: Lattice::CalculateDensityAndMomentum (SSE3 order) and
// momentum / density.  With STRESS, from f_neq = f - f_eq (SSE3 order) and
// Pi_ab = sum_l f_neq_l c_la c_lb in direction order (terms with
// c_la c_lb = 0 add nothing):
// * wall shear stress magnitude (Lattice.h:652-727): t_a = sum_b (Pi_ab n_b)
//   temp, sqrt(|t|^2 - (t . n)^2) at wall sites, the largest double (the
//   reference's NO_VALUE) elsewhere;
// * stress tensor (CalculateStressTensor, 630-645): Pi * (1 - 1/(2 tau))
//   plus (rho - 1) Cs2 on the diagonal, upper triangle xx xy xz yy yz zz;
// * von Mises stress (508-552) and shear rate (728-753, 890-907);
// * traction sigma n and its tangential projection t - n (t . n) (560-602)
//   at wall sites, zero elsewhere (Common.h:107-121).
template <int Q, typename S, class Lay, bool STRESS>
__global__ __launch_bounds__(256) void k_export_fields(DevDomain D, StepArgs A,
                                                       const S* __restrict__ fin,
                                                       int from_post_stream, FieldPtrs F) {
  using L = Lat<Q>;
  SiteRef r;
  if (!Lay::locate(D, r)) return;
  if (STRESS && F.by_record && !r.wall) return;
  double f[Q];
  post_stream_site<Q, S, Lay>(D, A, fin, from_post_stream, r, f);
  double rho, mx, my, mz;
  moments<Q, double>(f, rho, mx, my, mz);
  const int64_t c = STRESS && F.by_record ? (int64_t)r.rec : F.perm[Lay::compact(D, r)];
  if constexpr (!STRESS) {
    if (F.density) F.density[c] = rho;
    if (F.velocity) {
      F.velocity[3 * c] = mx / rho;
      F.velocity[3 * c + 1] = my / rho;
      F.velocity[3 * c + 2] = mz / rho;
    }
    return;
  }
  const FeqCoef<double> fe(rho, mx, my, mz);
  double fneq[Q];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    fneq[d] = f[d] - fe.template eq<Q, d>();
  });
  const double p00 = second_moment<Q, 0, 0>(fneq), p10 = second_moment<Q, 1, 0>(fneq),
               p11 = second_moment<Q, 1, 1>(fneq), p20 = second_moment<Q, 2, 0>(fneq),
               p21 = second_moment<Q, 2, 1>(fneq), p22 = second_moment<Q, 2, 2>(fneq);
  double ts = F.tau;
  if constexpr (kWaveLayout<Lay>)
    if (D.blk_tau) ts = D.blk_tau[r.w >> 3];
  const bool wall = r.wall != 0;
  double n[3] = {0.0, 0.0, 0.0};
  if (wall && F.rec_normal)
    for (int a = 0; a < 3; ++a) n[a] = (double)F.rec_normal[3 * (int64_t)r.rec + a];
  if (F.wss) {
    double v = 1.7976931348623157e308;  // NO_VALUE, constants.h:47
    if (wall) {
      // -sqrt(2) * the stress parameter of LbmParameters
      // (LbmParameters.h:34-39), as Lattice.h:669 uses it
      const double temp = (1.0 - 1.0 / (2.0 * ts)) / sqrt(2.0) * (-sqrt(2.0));
      const double pi[3][3] = {{p00, p10, p20}, {p10, p11, p21}, {p20, p21, p22}};
      double sq = 0.0, nn = 0.0;
      for (int a = 0; a < 3; ++a) {
        double t = 0.0;
        for (int b = 0; b < 3; ++b) t += pi[a][b] * n[b] * temp;
        sq += t * t;
        nn += t * n[a];
      }
      v = sqrt(sq - nn * nn);
    }
    F.wss[c] = v;
  }
  const double fac = 1 - 1 / (2 * ts);
  const double pr = (rho - 1) * kCs2;
  const double s00 = p00 * fac + pr, s10 = p10 * fac, s20 = p20 * fac, s11 = p11 * fac + pr,
               s21 = p21 * fac, s22 = p22 * fac + pr;
  if (F.tensor) {
    double* t6 = F.tensor + 6 * c;
    t6[0] = s00;
    t6[1] = s10;
    t6[2] = s20;
    t6[3] = s11;
    t6[4] = s21;
    t6[5] = s22;
  }
  if (F.von_mises) {
    // sums of f_neq (cx^2 - cy^2) etc. in direction order
    double xx_yy = 0.0, yy_zz = 0.0, xx_zz = 0.0, xy = 0.0, xz = 0.0, yz = 0.0;
    sfor<0, Q>([&](auto li) {
      constexpr int l = decltype(li)::value;
      constexpr int cx = L::c[l][0], cy = L::c[l][1], cz = L::c[l][2];
      constexpr int a = cx * cx - cy * cy, b = cy * cy - cz * cz, d = cx * cx - cz * cz;
      if constexpr (a != 0) xx_yy += fneq[l] * (double)a;
      if constexpr (b != 0) yy_zz += fneq[l] * (double)b;
      if constexpr (d != 0) xx_zz += fneq[l] * (double)d;
      if constexpr (cx * cy != 0) xy += fneq[l] * (double)cx * (double)cy;
      if constexpr (cx * cz != 0) xz += fneq[l] * (double)cx * (double)cz;
      if constexpr (cy * cz != 0) yz += fneq[l] * (double)cy * (double)cz;
    });
    const double a = xx_yy * xx_yy + yy_zz * yy_zz + xx_zz * xx_zz;
    const double b = xy * xy + xz * xz + yz * yz;
    const double sp = (1.0 - 1.0 / (2.0 * ts)) / sqrt(2.0);
    F.von_mises[c] = sp * sqrt(a + 6.0 * b);
  }
  if (F.shear_rate) {
    const double k = -1.0 / (2.0 * ts * rho * kCs2);
    const double e[6] = {p00 * k, p10 * k, p20 * k, p11 * k, p21 * k, p22 * k};
    // rows: (0,0) (0,1) (0,2) (1,1) (1,2) (2,2)
    double acc = 0.0;
    acc += e[0] * e[0];
    acc += 2 * e[1] * e[1];
    acc += 2 * e[2] * e[2];
    acc += e[3] * e[3];
    acc += 2 * e[4] * e[4];
    acc += e[5] * e[5];
    F.shear_rate[c] = sqrt(2 * acc);
  }
  if (F.traction || F.tangential) {
    double t[3] = {0.0, 0.0, 0.0}, tn = 0.0;
    if (wall) {
      const double sg[3][3] = {{s00, s10, s20}, {s10, s11, s21}, {s20, s21, s22}};
      for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) t[a] += sg[a][b] * n[b];
      for (int a = 0; a < 3; ++a) tn = tn + t[a] * n[a];
    }
    // by record: consecutive lanes on consecutive words
    const int64_t at = F.by_record ? c : 3 * c, next = F.by_record ? D.nb : 1;
    for (int a = 0; a < 3; ++a) {
      if (F.traction) F.traction[at + a * next] = t[a];
      if (F.tangential) F.tangential[at + a * next] = wall ? t[a] - n[a] * tn : 0.0;
    }
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

int launch_export_distributions(const DevDomain& d, const StepArgs& a, const void* fin,
                                int from_post_stream, const int64_t* perm, double* out,
                                void* stream) {
  return dispatch_narrow(d, a, [&](auto q, auto, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    hipLaunchKernelGGL((k_export_distributions<decltype(q)::value, S, Lay>),
                       grid_for(thread_count(d)), dim3(256), 0, (hipStream_t)stream, d, a,
                       (const S*)fin, from_post_stream, perm, out);
    return (int)hipGetLastError();
  });
}

int launch_export_fields(const DevDomain& d, const StepArgs& a, const void* fin,
                         int from_post_stream, const FieldPtrs& fields, void* stream) {
  const bool stress = fields.wss || fields.tensor || fields.von_mises || fields.shear_rate ||
                      fields.traction || fields.tangential;
  return dispatch_narrow(d, a, [&](auto q, auto, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    constexpr int Q = decltype(q)::value;
    const dim3 grid = grid_for(thread_count(d)), block(256);
    if (stress)
      hipLaunchKernelGGL((k_export_fields<Q, S, Lay, true>), grid, block, 0,
                         (hipStream_t)stream, d, a, (const S*)fin, from_post_stream, fields);
    else
      hipLaunchKernelGGL((k_export_fields<Q, S, Lay, false>), grid, block, 0,
                         (hipStream_t)stream, d, a, (const S*)fin, from_post_stream, fields);
    return (int)hipGetLastError();
  });
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

int monitor_groups(const DevDomain& d) {
  const int64_t units = d.layout == 0 ? (d.n + 255) / 256 : ((int64_t)d.nwaves + 3) / 4;
  return (int)std::min<int64_t>(kMonitorGroups, std::max<int64_t>(units, 1));
}

int launch_monitor(const DevDomain& d, const StepArgs& a, const void* fin,
                   int from_post_stream, const int64_t* range, int groups, double* partials,
                   double* io_vals, void* stream) {
  return dispatch_narrow(d, a, [&](auto q, auto, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    hipLaunchKernelGGL((k_monitor<decltype(q)::value, S, Lay>), dim3(groups), dim3(256), 0,
                       (hipStream_t)stream, d, a, (const S*)fin, from_post_stream, range,
                       partials, io_vals);
    return (int)hipGetLastError();
  });
}

int launch_snapshot_velocity(const DevDomain& d, const StepArgs& a, const void* fin,
                             int from_post_stream, double* u, void* stream) {
  return dispatch_narrow(d, a, [&](auto q, auto, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    hipLaunchKernelGGL((k_snapshot_velocity<decltype(q)::value, S, Lay>),
                       grid_for(thread_count(d)), dim3(256), 0, (hipStream_t)stream, d, a,
                       (const S*)fin, from_post_stream, u);
    return (int)hipGetLastError();
  });
}

int launch_velocity_change(const DevDomain& d, const StepArgs& a, const void* fin,
                           int from_post_stream, const int64_t* range, int groups,
                           const double* u0, const double* inv_refs, double inv_ref,
                           double* partials, void* stream) {
  return dispatch_narrow(d, a, [&](auto q, auto, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    hipLaunchKernelGGL((k_velocity_change<decltype(q)::value, S, Lay>), dim3(groups), dim3(256),
                       0, (hipStream_t)stream, d, a, (const S*)fin, from_post_stream, range, u0,
                       inv_refs, inv_ref, partials);
    return (int)hipGetLastError();
  });
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
