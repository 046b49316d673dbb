// Host check of the library's device-memory bookkeeping
// (hom3_amd/csrc/memory.hpp) over a stand-in device of a given size: hipMalloc
// fails past it, as on a GPU.  Each check prints a line when it fails; exit
// status 0 when none does.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>
#include <set>
#include <hip/hip_runtime.h>

// ---- the stand-in device ------------------------------------------------------
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
using hipStream_t = int;
constexpr int hipHostMallocDefault = 0;
static size_t device_size = 0, device_used = 0, device_peak = 0;
static std::map<char*, size_t> device_live;
static hipError_t last_error = hipSuccess;
// addresses only: nothing is written to them
static char* next_address = reinterpret_cast<char*>(size_t(1) << 40);
inline hipError_t hipMalloc(void** p, size_t n) {
  if (device_used + n > device_size) return last_error = hipErrorOutOfMemory;
  device_used += n;
  if (device_used > device_peak) device_peak = device_used;
  *p = next_address;
  device_live[next_address] = n;
  next_address += (n + 4095) & ~size_t(4095);
  return hipSuccess;
}
inline hipError_t hipFree(void* p) {
  auto i = device_live.find(static_cast<char*>(p));
  if (i == device_live.end()) { std::printf("free of unknown memory\n"); std::abort(); }
  device_used -= i->second;
  device_live.erase(i);
  return hipSuccess;
}
inline hipError_t hipGetLastError() { hipError_t e = last_error; last_error = hipSuccess; return e; }
inline const char* hipGetErrorString(hipError_t e) { return e ? "out of memory" : "success"; }
inline hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) { *p = std::malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipDeviceSynchronize() { return hipSuccess; }

#include "memory.hpp"
using namespace hom3g;

static int failures = 0;
#define CHECK(cond, ...)                                 \
  do {                                                   \
    if (!(cond)) {                                       \
      ++failures;                                        \
      std::printf("line %d: %s ", __LINE__, #cond);      \
      std::printf(__VA_ARGS__);                          \
      std::printf("\n");                                 \
    }                                                    \
  } while (0)

constexpr size_t MB = size_t(1) << 20;

// pieces handed out lie in live allocations and do not overlap
struct Pieces {
  std::map<char*, size_t> at;
  void add(void* q, size_t n) {
    char* p = static_cast<char*>(q);
    CHECK(reinterpret_cast<size_t>(p) % 256 == 0, "alignment");
    auto a = device_live.upper_bound(p);
    bool in = a != device_live.begin();
    if (in) {
      --a;
      in = p >= a->first && p + n <= a->first + a->second;
    }
    CHECK(in, "%zu bytes outside the allocations", n);
    auto b = at.lower_bound(p);
    CHECK(b == at.end() || p + n <= b->first, "overlap");
    if (b != at.begin()) {
      --b;
      CHECK(b->first + b->second <= p, "overlap");
    }
    at[p] = n;
  }
};

// the buffers of one call: steps x stages states of a fluid and a solid and a
// few small ones; returns the bytes asked for
static size_t call(Workspace& w, size_t nc, size_t nh, int buffers) {
  Pieces P;
  size_t sum = 0;
  auto take = [&](size_t n) {
    P.add(w.take(n), n);
    sum += n;
  };
  for (int k = 0; k < buffers; ++k) {
    take(nc);
    take(nh);
  }
  for (size_t n : {size_t(8), size_t(600), size_t(100000)}) take(n);
  w.give_back();
  return sum;
}

// A call fits a device that its buffers fit (with 10% left, as the sweeps
// check): one chunk of small buffers and one partly used chunk of each size
// are all that it takes beyond them.
static void at_the_limit(size_t nc, size_t nh, int buffers) {
  device_size = (size_t)((nc + nh) * (double)buffers / 0.9) + 3 * Workspace::kChunk;
  Workspace w;
  for (int pass = 0; pass < 3; ++pass) {
    device_peak = device_used;
    try {
      const size_t sum = call(w, nc, nh, buffers);
      CHECK(device_peak <= 1.05 * sum + 3 * Workspace::kChunk, "%zu + %zu bytes: %zu for %zu", nc, nh, device_peak, sum);
    } catch (const Error& e) {
      CHECK(false, "%zu + %zu bytes, pass %d: %s", nc, nh, pass, e.what());
    }
    CHECK(device_used <= Workspace::kKeep, "%zu bytes kept", device_used);
  }
}

int main() {
  // states of the uniform channels (fluid and solid) at several levels, and
  // sizes around the chunk's and the shared buffers' limits
  const size_t sizes[][2] = {{33 * MB, 1 * MB + 64}, {20 * MB, 160000}, {2 * MB + 4096, 20000}, {160 * MB, 5 * MB},
                             {64 * MB, 64 * MB}, {64 * MB + 1, 2 * MB}, {43 * MB, 43 * MB}, {40 * MB, 30 * MB},
                             {2 * MB, 2 * MB + 1}, {1200 * MB, 40 * MB}, {300000, 10000}};
  for (auto& s : sizes)
    for (int n : {1, 7, 60}) at_the_limit(s[0], s[1], n);

  // calls of other sizes after one another in one workspace, at random
  std::mt19937 rng(5);
  for (int round = 0; round < 200; ++round) {
    device_size = size_t(64) << 30;
    Workspace w;
    for (int k = 0; k < 6; ++k) {
      const size_t nc = size_t(1) << std::uniform_int_distribution<int>(10, 29)(rng);
      call(w, nc + rng() % 5000, nc / (1 + rng() % 64) + 8, 1 + rng() % 12);
      CHECK(device_used <= Workspace::kKeep, "%zu bytes kept", device_used);
    }
    // a large call on a device that only fits it once the rest has gone
    device_size = size_t(3) << 30;
    try {
      call(w, 900 * MB, 20 * MB, 3);
    } catch (const Error& e) {
      CHECK(false, "after other calls: %s", e.what());
    }
  }
  CHECK(device_used == 0, "%zu bytes lost", device_used);
  std::printf("%d failures\n", failures);
  return failures ? 1 : 0;
}
