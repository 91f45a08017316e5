// The pinned slots that sizes are reported in (csrc/common.h): every call that
// takes one gives the same without (all slots held, so that it copies instead),
// and a slot is free again only after the kernels of its call, also where the
// call ends early with an error.
#include <dlfcn.h>

#include <cstdint>
#include <memory>
#include <vector>

#include "../../daxtoolkit_amd/csrc/common.h"
#include "Testing.h"

// The library's launch checks, of which the test can make one fail.
namespace {
int g_checks = 0, g_fail_at = 0;
}
extern "C" hipError_t hipGetLastError(void) {
  static auto real = reinterpret_cast<hipError_t (*)()>(dlsym(RTLD_NEXT, "hipGetLastError"));
  const hipError_t e = real();
  return ++g_checks == g_fail_at ? hipErrorLaunchFailure : e;
}

namespace {
using daxhip::HostSlot;

#define HIP_OK(e) DAX_TEST_ASSERT((e) == hipSuccess, "HIP call failed")

constexpr int kN = 24;  // points per axis
constexpr int64_t kPoints = (int64_t)kN * kN * kN, kCells = (int64_t)(kN - 1) * (kN - 1) * (kN - 1);

template <class T>
struct Device {
  T* p = nullptr;
  size_t n;
  explicit Device(size_t count) : n(count) { HIP_OK(hipMalloc((void**)&p, n * sizeof(T))); }
  explicit Device(const std::vector<T>& v) : Device(v.size()) {
    HIP_OK(hipMemcpy(p, v.data(), n * sizeof(T), hipMemcpyHostToDevice));
  }
  ~Device() { (void)hipFree(p); }
  std::vector<T> host() const {
    std::vector<T> v(n);
    HIP_OK(hipMemcpy(v.data(), p, n * sizeof(T), hipMemcpyDeviceToHost));
    return v;
  }
};

// Holds the stream for about 10 ms of the 100 MHz clock.
__global__ void k_hold() {
  const long long t0 = wall_clock64();
  for (int i = 0; i < (1 << 20) && wall_clock64() - t0 < 1000000; ++i) __builtin_amdgcn_s_sleep(8);
}

struct Inputs {
  std::vector<float> field, points;
  std::vector<int32_t> cells;
  Inputs() {
    for (int k = 0; k < kN; ++k)
      for (int j = 0; j < kN; ++j)
        for (int i = 0; i < kN; ++i) {
          const float x = i - 11.3f, y = j - 10.9f, z = k - 11.7f;
          field.push_back(std::sqrt(x * x + y * y + z * z));
          points.insert(points.end(), {(float)i, (float)j, (float)k});
        }
    const int32_t sy = kN, sz = kN * kN;
    for (int k = 0; k + 1 < kN; ++k)
      for (int j = 0; j + 1 < kN; ++j)
        for (int i = 0; i + 1 < kN; ++i) {
          const int32_t p = i + sy * j + sz * k;
          cells.insert(cells.end(),
                       {p, p + 1, p + 1 + sy, p + sy, p + sz, p + 1 + sz, p + 1 + sy + sz, p + sy + sz});
        }
  }
};

// One of the calls that report sizes; its sizes and what it wrote.
struct Calls {
  Inputs in;
  Device<float> field{in.field}, points{in.points};
  Device<int32_t> cells{in.cells};
  hipStream_t s = nullptr;
  Calls() { HIP_OK(hipStreamCreate(&s)); }
  ~Calls() { (void)hipStreamDestroy(s); }
  static constexpr int kCount = 5;

  // After a call that ended with an error: nothing writes any more into the
  // slot that the next call would get.
  int ended(int rc) {
    if (rc) {
      HostSlot next(s);
      DAX_TEST_ASSERT(next.p, "no slot");
      for (int i = 0; i < 8; ++i) ((volatile int64_t*)next.p)[i] = -77;
      HIP_OK(hipStreamSynchronize(s));
      for (int i = 0; i < 8; ++i)
        DAX_TEST_ASSERT(((volatile int64_t*)next.p)[i] == -77, "a slot was written after its call");
    }
    HIP_OK(hipStreamSynchronize(s));
    return rc;
  }

  int run(int which, std::vector<int64_t>& out) {
    out.clear();
    int64_t a = 0, b = 0, plan[8] = {};
    int rc = 0;
    const float o[3] = {11.0f, 11.0f, 11.0f}, n[3] = {0.3f, 0.2f, 1.0f};
    if (which < 2) {
      Device<char> ws(dax_hip_mc_workspace_bytes(kN, kN, kN));
      rc = which == 0 ? dax_hip_mc_count(field.p, kN, kN, kN, 8.0f, ws.p, ws.n, &a, &b, s)
                      : dax_hip_mc_slice_count(kN, kN, kN, nullptr, nullptr, o, n, ws.p, ws.n, &a,
                                               &b, s);
      out = {a, b};
      return ended(rc);
    } else if (which < 4) {
      Device<char> ws(dax_hip_topology_workspace_bytes(kCells, kPoints));
      Device<int32_t> counts(kCells), mask(kPoints);
      rc = which == 2 ? dax_hip_threshold_plan_uniform(field.p, kN, kN, kN, 2.0f, 9.0f,
                                                       DAX_HIP_MC_DEDUP, counts.p, ws.p, ws.n,
                                                       mask.p, plan, s)
                      : dax_hip_threshold_plan_cells(cells.p, 8, kCells, field.p, kPoints, 2.0f,
                                                     9.0f, DAX_HIP_MC_DEDUP, counts.p, ws.p, ws.n,
                                                     mask.p, plan, s);
      out = {plan[2], plan[3]};
      if (!ended(rc))
        for (int32_t m : mask.host()) out.push_back(m);
    } else {  // a count and a generate
      Device<char> ws(dax_hip_cells_workspace_bytes(kCells));
      rc = dax_hip_mc_hex_count_cells(cells.p, kCells, field.p, kPoints, 8.0f, ws.p, ws.n, &a, s);
      if (ended(rc)) return rc;
      Device<char> scratch(dax_hip_mc_hex_scratch_bytes(a));
      Device<float> v(9 * a), w(3 * a);
      Device<int32_t> conn(3 * a), first(3 * a), second(3 * a);
      rc = dax_hip_mc_hex_generate_cells(cells.p, kCells, field.p, points.p, kPoints, 8.0f,
                                         DAX_HIP_MC_DEDUP, ws.p, ws.n, a, scratch.p, scratch.n, v.p,
                                         conn.p, first.p, second.p, w.p, &b, s);
      out = {a, b};
      if (!ended(rc))
        for (int32_t c : conn.host()) out.push_back(c);
    }
    return rc;
  }
};

void TestWithoutSlots() {
  Calls calls;
  for (int which = 0; which < Calls::kCount; ++which) {
    std::vector<int64_t> want, got;
    DAX_TEST_ASSERT(calls.run(which, want) == 0, "call failed");
    DAX_TEST_ASSERT(want[0] > 0 && want[1] > 0, "nothing found");
    std::vector<std::unique_ptr<HostSlot>> held;
    do {
      held.emplace_back(new HostSlot(calls.s));
      DAX_TEST_ASSERT(held.size() <= 65, "more slots than there are");
    } while (held.back()->p);
    DAX_TEST_ASSERT(held.size() > 1, "no pinned slots");
    DAX_TEST_ASSERT(calls.run(which, got) == 0, "call without a slot failed");
    DAX_TEST_ASSERT(got == want, "call without a slot differs");
    std::printf("call %d without slots: same\n", which);
  }
}

void TestErrorsKeepTheSlot() {
  Calls calls;
  for (int which = 0; which < Calls::kCount; ++which) {
    std::vector<int64_t> want, got;
    g_checks = g_fail_at = 0;
    DAX_TEST_ASSERT(calls.run(which, want) == 0, "call failed");
    const int checks = g_checks;
    for (int fail = 1; fail <= checks; ++fail) {
      k_hold<<<1, 64, 0, calls.s>>>();
      HIP_OK(hipPeekAtLastError());
      g_checks = 0;
      g_fail_at = fail;
      const int rc = calls.run(which, got);
      g_fail_at = 0;
      DAX_TEST_ASSERT(rc != 0, "the failed check went unnoticed");
    }
    DAX_TEST_ASSERT(calls.run(which, got) == 0 && got == want, "call after errors differs");
    std::printf("call %d: %d checks failed in turn\n", which, checks);
  }
}

void TestHostSlots() {
  TestWithoutSlots();
  TestErrorsKeepTheSlot();
}
}  // namespace

int main() { return RunTest(TestHostSlots); }
