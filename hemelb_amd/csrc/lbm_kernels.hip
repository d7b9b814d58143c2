// The timestep's kernels and their launches.  The build compiles this file
// once per layout (HLB_LAYOUT 0, 1, 2), in parallel.
#include "lbm_device.h"

#ifndef HLB_LAYOUT
#error "compile with -DHLB_LAYOUT=0, 1 or 2"
#endif

namespace hlb {
namespace {

template <int Q, int KERNEL, typename S, class Lay, bool BULK = false>
__device__ __forceinline__ void step_site(const DevDomain& D, const StepArgs& A,
                                          const S* __restrict__ fin,
                                          S* __restrict__ fout, const SiteRef& r) {
  using T = typename Store<S>::T;
  T f[Q];
  gather<Q, S, T, Lay, BULK>(D, A, fin, r, f);
  // Stability (every f > 0) is tested on the state by the monitor's
  // reduction, as the reference's StabilityTester tests fNew
  // (StabilityTester.h:97-113), not inside the step.
  StepArgs a = A;
  Lay::relax(D, r, a);
  const Hydro<Q, T> h = collide<Q, KERNEL, S>(f, a);
  // The stash's loads and division come after the stores, which need not wait
  // for them (binary16: before, where its registers suffice; 4 % faster).
  if constexpr (sizeof(S) == 2) update_stash<Q, T, BULK>(D, r, h);
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    if constexpr (std::is_same<Lay, BlockLayout32>::value)
      Lay::template store<Q, S>(D, r, fout, d, (S)f[d]);
    else
      store_out<S>(own_ptr<Q, Lay>(D, r, fout, d), f[d]);
  });
  if constexpr (sizeof(S) != 2) update_stash<Q, T, BULK>(D, r, h);
}

// One timestep, one site per thread.  Block layout: one x plane per wave,
// workgroups of A.threads, optionally remapped to XCD-contiguous ranges.
template <int Q, int KERNEL, typename S, class Lay>
__device__ __forceinline__ void step_wave(const DevDomain& D, const StepArgs& A,
                                          const S* __restrict__ fin, S* __restrict__ fout) {
  SiteRef r;
  if constexpr (kWaveLayout<Lay>) {
    const uint32_t g = step_workgroup(A.xcd_remap);
    const uint32_t w = __builtin_amdgcn_readfirstlane(g * (blockDim.x >> 6) + (threadIdx.x >> 6));
    // (A wave-uniform branch to the boundary-free code for planes without
    // boundary sites cuts their instructions by a third but measured slower:
    // the kernel then needs more registers and the two paths more
    // instruction cache.)
    if (!Lay::locate_wave(D, w, r)) return;
  } else {
    if (!Lay::locate(D, r)) return;
  }
  step_site<Q, KERNEL, S, Lay>(D, A, fin, fout, r);
}
template <int Q, int KERNEL, typename S, class Lay>
__global__ __launch_bounds__(256) void k_step(DevDomain D, StepArgs A,
                                              const S* __restrict__ fin,
                                              S* __restrict__ fout) {
  step_wave<Q, KERNEL, S, Lay>(D, A, fin, fout);
}
// The same step held to kStepWaves waves per SIMD: binary16 to 7 (at most 72
// VGPRs; it is bound by the issue and latency of its vector instructions rather
// than by bytes, and the seventh wave measured 3 % faster on the vessel tree),
// binary32 to 6 (80 VGPRs; left to itself it takes 86, 5 waves, and the step of
// a 4 M-site tree 168.5 instead of 163.2 us).  Only the D3Q19 binary16 forms
// with 64-bit addresses and of the compact layout spill for it, one register (8
// bytes of scratch a lane; 109.4 and 167.9 us on that tree).  Binary64 takes
// its natural 4: held to 5 it spills.
template <typename S> constexpr int kStepWaves = sizeof(S) == 2 ? 7 : 6;
template <int Q, int KERNEL, typename S, class Lay>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kStepWaves<S>)))
void k_step_held(DevDomain D, StepArgs A, const S* __restrict__ fin, S* __restrict__ fout) {
  step_wave<Q, KERNEL, S, Lay>(D, A, fin, fout);
}

// The timestep over a list of waves (x planes).  The solver splits the
// planes of the block layouts into those without any boundary site, run by
// the BULK instantiation (no boundary code, so far fewer registers and more
// waves in flight), and those with one, run by the full one; together the
// two launches update every site exactly as k_step does.
template <int Q, int KERNEL, typename S, class Lay, bool BULK>
__global__ __launch_bounds__(256) void k_step_list(DevDomain D, StepArgs A,
                                                   const S* __restrict__ fin,
                                                   S* __restrict__ fout,
                                                   const uint32_t* __restrict__ waves,
                                                   uint32_t count) {
  const uint32_t g = step_workgroup(A.xcd_remap);
  const uint32_t i = __builtin_amdgcn_readfirstlane(g * (blockDim.x >> 6) + (threadIdx.x >> 6));
  if (i >= count) return;
  const uint32_t w = __builtin_amdgcn_readfirstlane(waves[i]);
  SiteRef r;
  if (!Lay::locate_wave(D, w, r)) return;
  if constexpr (BULK) r.cut = 0;  // known: no boundary sites in these planes
  step_site<Q, KERNEL, S, Lay, BULK>(D, A, fin, fout, r);
}

// The same timestep for the block layout with a wave loop: each wave takes
// A.planes consecutive x planes and a grid of A.groups workgroups strides
// over the domain (a persistent launch).  The loop keeps lane-derived
// offsets live across iterations, so it needs more registers than k_step;
// the launch-shape tuner measures both.
template <int Q, int KERNEL, typename S, class Lay>
__global__ __launch_bounds__(256) void k_step_loop(DevDomain D, StepArgs A,
                                                   const S* __restrict__ fin,
                                                   S* __restrict__ fout) {
  const uint32_t wpg = blockDim.x >> 6;
  const uint32_t g = step_workgroup(A.xcd_remap);
  const uint32_t gw = __builtin_amdgcn_readfirstlane(g * wpg + (threadIdx.x >> 6));
  const uint32_t stride = gridDim.x * wpg * A.planes;
  for (uint32_t base = gw * A.planes; base < D.nwaves; base += stride) {
    for (uint32_t i = 0; i < A.planes; ++i) {
      SiteRef r;
      if (Lay::locate_wave(D, base + i, r))
        step_site<Q, KERNEL, S, Lay>(D, A, fin, fout, r);
    }
  }
}

template <int Q, int KERNEL, typename S, class Lay>
__global__ __launch_bounds__(256) void k_collide_only(DevDomain D, StepArgs A,
                                                      const S* __restrict__ fin,
                                                      S* __restrict__ fout) {
  using T = typename Store<S>::T;
  SiteRef r;
  if (!Lay::locate(D, r)) return;
  T f[Q];
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    f[d] = Store<S>::ld(fin + Lay::template at<Q>(D, d, r.x));
  });
  StepArgs a = A;
  Lay::relax(D, r, a);
  const Hydro<Q, T> h = collide<Q, KERNEL, S>(f, a);
  update_stash<Q, T>(D, r, h);
  sfor<0, Q>([&](auto di) {
    constexpr int d = decltype(di)::value;
    Store<S>::st(fout + Lay::template at<Q>(D, d, r.x), f[d]);
  });
}


// One step on the launch shape in `a` with layout Lay.
template <int Q, int K, typename S, class Lay>
int step_launch(const DevDomain& d, const StepArgs& a, const void* fin, void* fout,
                void* stream) {
  if constexpr (kWaveLayout<Lay>) {
    // launch shape: a.threads per workgroup, a.planes per wave, a grid of
    // a.groups workgroups (0: enough to cover every plane once)
    const uint32_t wpg = a.threads / 64u;
    const uint64_t need = ((uint64_t)d.nwaves + (uint64_t)wpg * a.planes - 1) /
                          ((uint64_t)wpg * a.planes);
    uint64_t groups = a.groups ? std::min<uint64_t>(a.groups, need) : need;
    const bool one_pass = a.planes == 1 && groups == need;
    if (one_pass && a.split && d.bulk_waves && d.bnd_waves) {
      // bulk planes first, then the planes with boundary sites
      const uint32_t counts[2] = {d.n_bulk_waves, d.n_bnd_waves};
      const uint32_t* lists[2] = {d.bulk_waves, d.bnd_waves};
      for (int part = 0; part < 2; ++part) {
        if (!counts[part]) continue;
        uint64_t gp = ((uint64_t)counts[part] + wpg - 1) / wpg;
        if (a.xcd_remap >= 2) {
          const uint64_t m = 8ull * a.xcd_remap;
          gp = (gp + m - 1) / m * m;
        }
        const dim3 gridp((unsigned)gp), blockp(a.threads);
        if (part == 0)
          hipLaunchKernelGGL((k_step_list<Q, K, S, Lay, true>),
                             gridp, blockp, 0, (hipStream_t)stream, d, a, (const S*)fin,
                             (S*)fout, lists[part], counts[part]);
        else
          hipLaunchKernelGGL((k_step_list<Q, K, S, Lay, false>),
                             gridp, blockp, 0, (hipStream_t)stream, d, a, (const S*)fin,
                             (S*)fout, lists[part], counts[part]);
      }
      return (int)hipGetLastError();
    }
    if (a.xcd_remap >= 2) {
      // runs of a.xcd_remap workgroups per XCD: pad the grid to whole
      // groups of 8 runs; padded workgroups see planes >= nwaves and exit
      const uint64_t m = 8ull * a.xcd_remap;
      groups = (groups + m - 1) / m * m;
    }
    const dim3 grid((unsigned)std::max<uint64_t>(groups, 1)), block(a.threads);
    if (one_pass) {
      if constexpr (kShifted<S>)
        hipLaunchKernelGGL((k_step_held<Q, K, S, Lay>), grid,
                           block, 0, (hipStream_t)stream, d, a, (const S*)fin, (S*)fout);
      else
        hipLaunchKernelGGL((k_step<Q, K, S, Lay>), grid,
                           block, 0, (hipStream_t)stream, d, a, (const S*)fin, (S*)fout);
    } else
      hipLaunchKernelGGL((k_step_loop<Q, K, S, Lay>), grid,
                         block, 0, (hipStream_t)stream, d, a, (const S*)fin, (S*)fout);
  } else {
    hipLaunchKernelGGL((k_step<Q, K, S, Lay>),
                       grid_for(thread_count(d)), dim3(256), 0, (hipStream_t)stream, d, a,
                       (const S*)fin, (S*)fout);
  }
  return (int)hipGetLastError();
}

}  // namespace

template <>
int step_in<HLB_LAYOUT>(const DevDomain& d, const StepArgs& a, const void* fin, void* fout,
                        void* stream) {
  return dispatch_in<HLB_LAYOUT>(a, [&](auto q, auto k, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    constexpr int Q = decltype(q)::value, K = decltype(k)::value;
    if constexpr (std::is_same<Lay, BlockLayout>::value) {
      if (narrow_offsets(d, a, sizeof(S)))
        return step_launch<Q, K, S, BlockLayout32>(d, a, fin, fout, stream);
    }
    return step_launch<Q, K, S, Lay>(d, a, fin, fout, stream);
  });
}

template <>
int collide_only_in<HLB_LAYOUT>(const DevDomain& d, const StepArgs& a, const void* fin,
                                void* fout, void* stream) {
  return dispatch_in<HLB_LAYOUT>(a, [&](auto q, auto k, auto* s, auto* lay) {
    using S = std::remove_pointer_t<decltype(s)>;
    using Lay = std::remove_pointer_t<decltype(lay)>;
    hipLaunchKernelGGL((k_collide_only<decltype(q)::value, decltype(k)::value, S, Lay>),
                       grid_for(thread_count(d)), dim3(256), 0, (hipStream_t)stream, d, a,
                       (const S*)fin, (S*)fout);
    return (int)hipGetLastError();
  });
}

}  // namespace hlb
