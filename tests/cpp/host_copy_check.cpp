// Scenarios of hlb::copy_to_host on the fake HIP runtime, chosen by argv[1];
// prints what happened and returns 0, or 1 after a wrong result.
#include <chrono>
#include <cstdio>
#include <string>
#include <vector>

#include "fake_hip.h"
#include "host_copy.h"

namespace {

constexpr size_t kLarge = (size_t(64) << 20) + 12345, kSmall = size_t(1) << 20;

std::vector<char> pattern(size_t n, unsigned seed) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (char)((i * 2654435761u + seed) >> 11);
  return v;
}
void nap(double s) { std::this_thread::sleep_for(std::chrono::duration<double>(s)); }

// A small copy waits for its stream while another solver's large one starts.
int small_beside_large() {
  ihipStream_t a(0), b(0);
  const auto small = pattern(kSmall, 1), large = pattern(kLarge, 2);
  std::vector<char> small_out(kSmall), large_out(kLarge);
  a.gate(false);
  std::thread t([&] { (void)hlb::copy_to_host({{small_out.data(), small.data(), kSmall}}, &a); });
  while (fake::direct == 0) nap(0.001);   // its copy is queued
  const hipError_t e = hlb::copy_to_host({{large_out.data(), large.data(), kLarge}}, &b);
  const int staged = fake::staged;
  a.gate(true);
  t.join();
  std::printf("staged %d\n", staged);
  return e == hipSuccess && small_out == small && large_out == large ? 0 : 1;
}

// A copy behind half a second of work on its stream: the processor time the
// process uses in the last 0.4 of it.
int waiting() {
  ihipStream_t s(0);
  const auto data = pattern(kLarge, 3);
  std::vector<char> out(kLarge);
  s.gate(false);
  hipError_t e = hipSuccess;
  std::thread t([&] { e = hlb::copy_to_host({{out.data(), data.data(), kLarge}}, &s); });
  auto cpu = [] {
    timespec ts;
    clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &ts);
    return ts.tv_sec + 1e-9 * ts.tv_nsec;
  };
  nap(0.1);
  const double before = cpu();
  nap(0.4);
  const double used = cpu() - before;
  s.gate(true);
  t.join();
  std::printf("cpu %g\n", used);
  return e == hipSuccess && out == data ? 0 : 1;
}

// While one solver's large export waits for its steps, another's is ready.
int large_beside_waiting() {
  ihipStream_t a(0), b(0);
  const auto first = pattern(kLarge, 4), second = pattern(kLarge, 5);
  std::vector<char> out1(kLarge), out2(kLarge);
  a.gate(false);
  hipError_t e1 = hipSuccess;
  std::thread t([&] { e1 = hlb::copy_to_host({{out1.data(), first.data(), kLarge}}, &a); });
  nap(0.1);
  const int before = fake::staged;
  const hipError_t e2 = hlb::copy_to_host({{out2.data(), second.data(), kLarge}}, &b);
  const int staged = fake::staged - before;
  a.gate(true);
  t.join();
  std::printf("staged %d\n", staged);
  return e1 == hipSuccess && e2 == hipSuccess && out1 == first && out2 == second ? 0 : 1;
}

// A solver on another device than the thread's current one.
int other_device() {
  ihipStream_t s(1);
  const auto data = pattern(kLarge, 6);
  std::vector<char> out(kLarge);
  const hipError_t e = hlb::copy_to_host({{out.data(), data.data(), kLarge}}, &s);
  std::printf("error %d current %d staged %d\n", (int)e, fake::device, (int)fake::staged);
  return e != hipSuccess || out == data ? 0 : 1;
}

}  // namespace

int main(int, char** argv) {
  const std::string what = argv[1];
  if (what == "small_beside_large") return small_beside_large();
  if (what == "waiting") return waiting();
  if (what == "large_beside_waiting") return large_beside_waiting();
  if (what == "other_device") return other_device();
  return 2;
}
