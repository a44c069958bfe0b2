// Device memory under a small limit, on the CPU: the mirrors (mirror.cpp) and
// the run memory (runspace.hpp) against HIP calls that only count bytes.
//   device_memory mirror  a matrix whose mirror fits without its packed columns
//                         is mirrored, and packed where there is room
//   device_memory spaces  memory kept between runs gives way to what is needed,
//                         and is bounded over all matrices
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <numeric>
#include <vector>

#include <tbsla/cpp/MatrixCOO.hpp>
#include <tbsla/cpp/MatrixCSR.hpp>

#include "../../tbsla_amd/csrc/device/kernels.hpp"
#include "../../tbsla_amd/csrc/device/mirror.hpp"

static std::size_t g_limit = ~std::size_t(0), g_used = 0;
static std::map<void *, std::size_t> g_live;
static hipError_t g_last = hipSuccess;

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  if (n > g_limit || g_used > g_limit - n) return g_last = hipErrorOutOfMemory;
  *p = std::malloc(n > (1u << 20) ? 1 : n);  // (large blocks are never touched)
  g_live[*p] = n;
  g_used += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (p) g_used -= g_live.at(p), g_live.erase(p), std::free(p);
  return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) {
  if (n <= 1u << 20) std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free(e);
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "error"; }
}

namespace tbsla {
namespace hip {
// the packing kernels, as far as memory goes (three words for four entries)
void pack_columns(DeviceMatrix &d, bool pairs) {
  (void)(pairs ? d.col24_pairs : d.col24).try_reserve(static_cast<std::size_t>((d.entries + 255) / 256 * 64) * 12);
}
void pack_ell_columns(DeviceMatrix &) {}
}  // namespace hip
}  // namespace tbsla

using namespace tbsla;

static int fails = 0;
#define CHECK(c)                                                      \
  do {                                                                \
    if (!(c)) std::printf("line %d: %s\n", __LINE__, #c), fails++;    \
  } while (0)

template <class F>
static bool throws(F f) {
  try {
    f();
  } catch (const std::exception &) {
    return true;
  }
  return false;
}

static void mirrors() {
  const int n = 3000, k = 8;
  std::vector<int> ptr(n + 1), row(n * k), col(n * k);
  for (int i = 0; i <= n; i++) ptr[i] = i * k;
  for (int e = 0; e < n * k; e++) row[e] = e / k, col[e] = (e * 37) % n;
  std::vector<double> val(n * k, 0.5);
  const auto bytes = [&](const cpp::Matrix &m, bool transposed) {  // without and with the packed columns
    const hip::DeviceMatrix &d = transposed ? hip::transpose_mirror(m) : hip::mirror(m, hip::Dtype::F64);
    const std::size_t packed = (d.col24.get() ? d.col24.bytes() + 256 : 0) +
                               (d.col24_pairs.get() ? d.col24_pairs.bytes() + 256 : 0);
    CHECK(packed > 0);
    return std::pair<std::size_t, std::size_t>(g_used - packed, g_used);
  };
  for (int what = 0; what < 3; what++) {
    const auto make = [&]() -> std::unique_ptr<cpp::Matrix> {
      if (what == 1) return std::unique_ptr<cpp::Matrix>(new cpp::MatrixCOO(n, n, val, row, col));
      return std::unique_ptr<cpp::Matrix>(new cpp::MatrixCSR(n, n, val, ptr, col));
    };
    const auto build = [&](const cpp::Matrix &m) {
      if (what == 2)
        (void)hip::transpose_mirror(m);
      else
        (void)hip::mirror(m, hip::Dtype::F64);
    };
    std::pair<std::size_t, std::size_t> need;
    {
      auto m = make();
      need = bytes(*m, what == 2);
    }
    CHECK(g_used == 0);
    for (std::size_t limit = need.first; limit < need.second; limit += 4 * 1009) {
      g_limit = limit;
      auto m = make();
      CHECK(!throws([&] { build(*m); }));
    }
    g_limit = need.first - 1;
    {
      auto m = make();
      CHECK(throws([&] { build(*m); }));
    }
    g_limit = ~std::size_t(0);
  }
  CHECK(g_used == 0);
}

static void spaces() {
  const std::size_t MB = 1 << 20;
  {
    hip::RunSpaces a, b;
    g_limit = 100 * MB;
    a.give(a.take(60 * MB));
    CHECK(g_used > 60 * MB);       // kept
    auto s = a.take(50 * MB);      // the idle one serves
    CHECK(g_used < 61 * MB);
    a.give(std::move(s));
    s = a.take(80 * MB);           // too small: it gives way
    CHECK(s && s->mem.bytes() >= 80 * MB);
    a.give(std::move(s));
    s = b.take(70 * MB);           // another matrix's gives way
    CHECK(s && g_used < 71 * MB);
    b.give(std::move(s));
    hip::DevBuf buf;               // and so it does to any other buffer
    buf.alloc(60 * MB);
    CHECK(g_used < 61 * MB);
    CHECK(throws([&] { (void)a.take(50 * MB); }));  // held memory does not
    CHECK(hipGetLastError() == hipSuccess);        // and no failure is left for a later check
    g_limit = ~std::size_t(0);
    a.give(a.take(10 * MB));
    a.give(a.take(20 * MB));
  }
  CHECK(g_used == 0);
  {  // bounded over all matrices, the oldest goes first
    std::vector<std::unique_ptr<hip::RunSpaces>> all;
    const std::size_t some = hip::kIdleBytes / 16;
    for (int k = 0; k < 40; k++) {
      all.emplace_back(new hip::RunSpaces());
      all.back()->give(all.back()->take(some));
    }
    CHECK(g_used <= hip::kIdleBytes + MB);
    CHECK(g_used > hip::kIdleBytes - 2 * some);
    const std::size_t before = g_used;
    all.back()->give(all.back()->take(some));  // the youngest is there
    CHECK(g_used == before);
    all.front()->give(all.front()->take(some));  // the oldest is not, and takes another's place
    CHECK(g_used == before);
    hip::RunSpaces big;  // more than the bound is not kept, and the others stay
    big.give(big.take(hip::kIdleBytes + MB));
    CHECK(g_used == before);
  }
  CHECK(g_used == 0);
}

int main(int argc, char **argv) {
  if (argc > 1 && !std::strcmp(argv[1], "mirror")) mirrors();
  if (argc > 1 && !std::strcmp(argv[1], "spaces")) spaces();
  return fails ? 1 : 0;
}
