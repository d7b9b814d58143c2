// Scenarios of the solver's host code (csrc/solver.cpp) on the fake HIP
// runtime, with the kernels replaced by stand-ins that note their arguments.
// argv[1] chooses one; prints what happened.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <string>
#include <vector>

#include "fake_hip_memory.h"
#include "hemelb_amd.h"
#include "lbm_internal.h"

// Host memory: allocations of at least so many bytes fail.
static size_t refused_bytes = SIZE_MAX;
void* operator new(size_t n, const std::nothrow_t&) noexcept {
  return n < refused_bytes ? std::malloc(n ? n : 1) : nullptr;
}
void* operator new(size_t n) {
  if (void* p = operator new(n, std::nothrow)) return p;
  throw std::bad_alloc();
}
void* operator new[](size_t n) { return operator new(n); }
void* operator new[](size_t n, const std::nothrow_t&) noexcept { return operator new(n, std::nothrow); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }
void operator delete[](void* p) noexcept { std::free(p); }
void operator delete[](void* p, size_t) noexcept { std::free(p); }

namespace {

std::vector<int64_t> seen_range;      // of the last monitor launch
bool monitor_had_range = false, launch_fails = false;
struct { uint32_t threads, planes, xcd_remap; } fast_shape{0, 0, 0};  // 1 ms a step, others 2
std::vector<float> seen_normals;      // of the last field export
bool seen_by_record = false;

}  // namespace

namespace hlb {

int monitor_groups(const DevDomain&) { return 1; }
int launch_fill(const DevDomain&, const StepArgs&, const double*, void*, void*) { return 0; }
int launch_step(const DevDomain&, const StepArgs& a, const void*, void*, void* stream) {
  const bool fast = a.threads == fast_shape.threads && a.planes == fast_shape.planes &&
                    a.xcd_remap == fast_shape.xcd_remap && a.split == 0 && a.groups == 0;
  static_cast<hipStream_t>(stream)->push([fast] { fake::clock_ms += fast ? 1.0 : 2.0; });
  return 0;
}
int launch_collide_only(const DevDomain&, const StepArgs&, const void*, void*, void*) { return 0; }
int launch_export_distributions(const DevDomain&, const StepArgs&, const void*, int,
                                const int64_t*, double*, void*) {
  return 0;
}
int launch_export_fields(const DevDomain& d, const StepArgs&, const void*, int,
                         const FieldPtrs& f, void*) {
  seen_by_record = f.by_record;
  seen_normals.clear();
  if (f.rec_normal) seen_normals.assign(f.rec_normal, f.rec_normal + 3 * d.nb);
  return 0;
}
int launch_import(const DevDomain&, const StepArgs&, const double*, const int64_t*, void*, void*) {
  return 0;
}
int launch_import_equilibrium(const DevDomain&, const StepArgs&, const double*, const double*,
                              const int64_t*, void*, void*) {
  return 0;
}
int launch_copy_arrays(int, int64_t, int64_t, int64_t, int, const void*, void*, uint32_t, uint32_t,
                       void*) {
  return 0;
}
int launch_halo(int64_t, const int64_t*, int, const void*, void*, int, void*) { return 0; }
int launch_monitor(const DevDomain&, const StepArgs&, const void*, int, const int64_t* range,
                   int groups, double* partials, double*, void*) {
  monitor_had_range = range != nullptr;
  seen_range.clear();
  if (range) seen_range.assign(range, range + 2 * groups);
  std::fill(partials, partials + 5 * groups, 0.0);
  return 0;
}
int launch_snapshot_velocity(const DevDomain&, const StepArgs&, const void*, int, double*, void*) {
  return launch_fails ? 1 : 0;
}
int launch_velocity_change(const DevDomain&, const StepArgs&, const void*, int, const int64_t*,
                           int groups, const double*, const double*, double, double* partials,
                           void*) {
  std::fill(partials, partials + groups, 0.0);
  return 0;
}
int scratch_address(int, double** out) {
  static std::vector<double> scratch(kStaticScratchDoubles);
  *out = scratch.data();
  return 0;
}
int launch_scatter_pairs(int64_t, int64_t, int, int, const int64_t*, const double*, int, double,
                         const double*, void*, void*) {
  return 0;
}
int launch_gather_pairs(int64_t, int64_t, int, int, const int64_t*, const void*, int, double,
                        const double*, double*, void*) {
  return 0;
}

}  // namespace hlb

namespace {

// Isolated sites (every link a wall) in blocks of their own, one vessel each.
struct Sites {
  std::vector<int32_t> coords, ids, instance;
  std::vector<uint32_t> type, wall, iolet;
  std::vector<float> normals;
  std::vector<double> tau;
  hlb_solver* s = nullptr;

  explicit Sites(int n) {
    for (int i = 0; i < n; ++i) {
      coords.insert(coords.end(), {32 * i, 0, 0});
      normals.insert(normals.end(), {1.0f + i, 2.0f + i, 3.0f + i});
      instance.push_back(i);
    }
    ids.assign(n, 0);
    type.assign(n, HLB_SITE_FLUID);
    wall.assign(n, (1u << 18) - 1);
    iolet.assign(n, 0);
    tau.assign(n, 0.8);
    hlb_params p{};
    p.lattice = 19;
    p.tau = 0.8;
    p.rho0 = 1.0;
    hlb_domain d{n, coords.data(), type.data(), wall.data(), iolet.data(), ids.data(), nullptr,
                 normals.data()};
    const double rest[3] = {0.0, 0.0, 0.0};
    if (hlb_create_ensemble(&p, &d, instance.data(), n, tau.data(), nullptr, 0, nullptr, 0, &s) ||
        hlb_set_equilibrium(s, 1.0, rest)) {
      std::printf("create: %s\n", hlb_last_error());
      std::exit(1);
    }
  }
  ~Sites() { hlb_destroy(s); }
};

// A failure while the per-vessel list of planes is sent to the device, then the
// same call again.
int instances_after(int& countdown) {
  Sites v(3);
  std::vector<hlb_instance_monitor> m(3);
  countdown = 1;
  const int first = hlb_reduce_instances(v.s, m.data());
  countdown = 0;
  const int second = hlb_reduce_instances(v.s, m.data());
  std::printf("first %d second %d ranges %d", first, second, (int)seen_range.size() / 2);
  bool ordered = monitor_had_range && seen_range.size() == 12;
  for (size_t k = 0; k + 1 < seen_range.size(); ++k)
    ordered = ordered && 0 <= seen_range[k] && seen_range[k] <= seen_range[k + 1] &&
              seen_range[k + 1] <= 24;
  std::printf(" ordered %d\n", (int)ordered);
  return 0;
}

// The same for the wall normals of the stress outputs.
int normals_after(int& countdown) {
  Sites v(3);
  std::vector<double> wss(3);
  countdown = 1;
  const int first = hlb_get_wall_shear_stress(v.s, wss.data());
  countdown = 0;
  const int second = hlb_get_wall_shear_stress(v.s, wss.data());
  std::sort(seen_normals.begin(), seen_normals.end());
  std::printf("first %d second %d normals %d\n", first, second,
              (int)(seen_normals == std::vector<float>{1, 2, 2, 3, 3, 3, 4, 4, 5}));
  return 0;
}

// A first snapshot that fails, the velocity change after it, and the two again.
int snapshot_fails() {
  Sites v(2);
  double change = -1;
  launch_fails = true;
  const int failed = hlb_snapshot_velocity(v.s), without = hlb_velocity_change(v.s, 1.0, &change);
  launch_fails = false;
  const int taken = hlb_snapshot_velocity(v.s), with = hlb_velocity_change(v.s, 1.0, &change);
  std::printf("failed %d without %d taken %d with %d\n", failed, without, taken, with);
  return 0;
}

// Both tractions of a closed box of 1.2 M sites, 215 k of them at a wall: their
// values take 10 MB of host memory on the way, which there is not at first.
int tractions_without_memory() {
  const int nx = 316, nz = 12, n = nx * nx * nz;
  const int c[19][3] = {{0, 0, 0},   {1, 0, 0},   {-1, 0, 0},  {0, 1, 0},   {0, -1, 0},
                        {0, 0, 1},   {0, 0, -1},  {1, 1, 0},   {-1, -1, 0}, {1, -1, 0},
                        {-1, 1, 0},  {1, 0, 1},   {-1, 0, -1}, {1, 0, -1},  {-1, 0, 1},
                        {0, 1, 1},   {0, -1, -1}, {0, 1, -1},  {0, -1, 1}};
  std::vector<int32_t> coords, ids(n, 0);
  std::vector<uint32_t> type(n, HLB_SITE_FLUID), wall(n, 0), iolet(n, 0);
  std::vector<float> normals;
  for (int i = 0; i < n; ++i) {
    const int x = i / (nx * nz), y = i / nz % nx, z = i % nz;
    coords.insert(coords.end(), {x, y, z});
    for (int q = 1; q < 19; ++q) {
      const int X = x + c[q][0], Y = y + c[q][1], Z = z + c[q][2];
      if (X < 0 || Y < 0 || Z < 0 || X >= nx || Y >= nx || Z >= nz) wall[i] |= 1u << (q - 1);
    }
    normals.insert(normals.end(), {0.0f, 0.0f, 1.0f});
  }
  hlb_params p{};
  p.lattice = 19;
  p.tau = 0.8;
  p.rho0 = 1.0;
  hlb_domain d{n, coords.data(), type.data(), wall.data(), iolet.data(), ids.data(), nullptr,
               normals.data()};
  const double rest[3] = {0.0, 0.0, 0.0};
  hlb_solver* s = nullptr;
  if (hlb_create(&p, &d, nullptr, 0, nullptr, 0, &s) || hlb_set_equilibrium(s, 1.0, rest)) {
    std::printf("create: %s\n", hlb_last_error());
    return 1;
  }
  std::vector<double> a(3 * n), b(3 * n);
  refused_bytes = 8 << 20;
  const int first = hlb_get_stress(s, nullptr, nullptr, nullptr, a.data(), b.data());
  refused_bytes = SIZE_MAX;
  const int second = hlb_get_stress(s, nullptr, nullptr, nullptr, a.data(), b.data());
  std::printf("first %d second %d by_record %d\n", first, second, (int)seen_by_record);
  hlb_destroy(s);
  return 0;
}

// The tuner where one shape takes half the time of all others: the one held on
// entry, or another (`held` null: the default shape).
int tune(uint32_t threads, uint32_t planes, uint32_t remap, const hlb_launch_shape* held) {
  Sites v(2);
  fake::on_event = [](hipEvent_t e) {
    std::lock_guard<std::mutex> lock(fake::mu);
    fake::event_ms[e] = fake::clock_ms;
  };
  if (held && hlb_set_launch_shape(v.s, held)) return 1;
  fast_shape = {threads, planes, remap};
  hlb_launch_shape best{}, now{};
  double ms = 0;
  const int rc = hlb_autotune(v.s, 4, &best, &ms);
  hlb_get_launch_shape(v.s, &now);
  std::printf("error %d ms %g threads %d planes %d remap %d kept %d\n", rc, ms, best.threads,
              best.planes, best.xcd_remap,
              (int)(now.threads == best.threads && now.planes == best.planes &&
                    now.xcd_remap == best.xcd_remap));
  return 0;
}

}  // namespace

int main(int, char** argv) {
  const std::string what = argv[1];
  if (what == "instances_after_malloc") return instances_after(fake::fail_malloc);
  if (what == "instances_after_memcpy") return instances_after(fake::fail_memcpy);
  if (what == "normals_after_malloc") return normals_after(fake::fail_malloc);
  if (what == "normals_after_memcpy") return normals_after(fake::fail_memcpy);
  if (what == "snapshot_fails") return snapshot_fails();
  if (what == "tractions_without_memory") return tractions_without_memory();
  if (what == "tune_default_fastest") return tune(64, 1, 16, nullptr);
  if (what == "tune_held_fastest") {
    const hlb_launch_shape held{256, 4, 0, 1, 0, 0};
    return tune(256, 4, 1, &held);
  }
  if (what == "tune_other_default_fastest") return tune(128, 1, 2, nullptr);
  return 2;
}
