// Unique points of unstructured cells (csrc/unstructured.hip) where there is no
// memory for the tables that number the edges: they are sorted instead, in less,
// and the grid is the same.
#include <dlfcn.h>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "../../include/dax_hip.h"
#include "Testing.h"

// The library's temporaries, of which the test can refuse the large ones.
namespace {
size_t g_limit = 0;
int g_refused = 0;
}  // namespace
extern "C" hipError_t hipMallocFromPoolAsync(void** p, size_t bytes, hipMemPool_t pool,
                                             hipStream_t s) {
  using Fn = hipError_t (*)(void**, size_t, hipMemPool_t, hipStream_t);
  static auto real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "hipMallocFromPoolAsync"));
  if (g_limit && bytes > g_limit) {
    ++g_refused;
    return hipErrorOutOfMemory;
  }
  return real(p, bytes, pool, s);
}

namespace {
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
  void append(std::vector<float>& out, size_t count) const {
    std::vector<T> v(count);
    HIP_OK(hipMemcpy(v.data(), p, count * sizeof(T), hipMemcpyDeviceToHost));
    out.insert(out.end(), v.begin(), v.end());
  }
};

// Counts, then generates with temporaries of up to limit bytes a triangle (0:
// any), on a stream of its own; everything that came out.
std::vector<float> Grid(size_t limit) {
  std::vector<float> f, x;
  std::vector<int32_t> c;
  for (int k = 0; k < kN; ++k)
    for (int j = 0; j < kN; ++j)
      for (int i = 0; i < kN; ++i) {
        f.push_back((i - 11.3f) * (i - 11.3f) + (j - 10.9f) * (j - 10.9f) + (k - 11.7f) * (k - 11.7f));
        x.insert(x.end(), {(float)i, (float)j, (float)k});
      }
  const int32_t sy = kN, sz = kN * kN;
  for (int k = 0; k + 1 < kN; ++k)
    for (int j = 0; j + 1 < kN; ++j)
      for (int i = 0; i + 1 < kN; ++i) {
        const int32_t p = i + sy * j + sz * k;
        c.insert(c.end(),
                 {p, p + 1, p + 1 + sy, p + sy, p + sz, p + 1 + sz, p + 1 + sy + sz, p + sy + sz});
      }
  const Device<float> field(f), points(x);
  const Device<int32_t> cells(c);
  hipStream_t s = nullptr;
  HIP_OK(hipStreamCreate(&s));
  Device<char> ws(dax_hip_cells_workspace_bytes(kCells));
  int64_t tris = 0, n = 0;
  DAX_TEST_ASSERT(dax_hip_mc_hex_count_cells(cells.p, kCells, field.p, kPoints, 64.0f, ws.p, ws.n,
                                             &tris, s) == 0 && tris > 0, "count failed");
  Device<char> scratch(dax_hip_mc_hex_scratch_bytes(tris));
  Device<float> v(9 * tris), w(3 * tris);
  Device<int32_t> conn(3 * tris), first(3 * tris), second(3 * tris);
  g_limit = limit * tris;
  g_refused = 0;
  const int rc = dax_hip_mc_hex_generate_cells(
      cells.p, kCells, field.p, points.p, kPoints, 64.0f, DAX_HIP_MC_DEDUP, ws.p, ws.n, tris,
      scratch.p, scratch.n, v.p, conn.p, first.p, second.p, w.p, &n, s);
  g_limit = 0;
  DAX_TEST_ASSERT(rc == 0, dax_hip_last_error());
  DAX_TEST_ASSERT((g_refused > 0) == (limit > 0), "temporaries of another size");
  HIP_OK(hipStreamSynchronize(s));
  DAX_TEST_ASSERT(n > 0 && n < 3 * tris, "no unique points");
  std::vector<float> out{(float)tris, (float)n};
  v.append(out, 3 * n);
  w.append(out, n);
  first.append(out, n);
  second.append(out, n);
  conn.append(out, 3 * tris);
  HIP_OK(hipStreamDestroy(s));
  return out;
}

void TestCellsDedup() {
  const std::vector<float> want = Grid(0);
  DAX_TEST_ASSERT(Grid(48) == want, "the sorted grid differs");
}
}  // namespace

int main() { return RunTest(TestCellsDedup); }
