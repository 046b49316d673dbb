// Host check of the library's device-memory bookkeeping
// (hom3_amd/csrc/memory.hpp) over a stand-in device of a given size: hipMalloc
// fails past it, as on a GPU.  Each check prints a line when it fails; exit
// status 0 when none does.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>
#include <thread>
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
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
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
static size_t call(Pool& pool, size_t nc, size_t nh, int buffers) {
  Pool::Use use(pool, 0, 1);
  Workspace& w = pool.ws;
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
  return sum;
}

// A call fits a device that its buffers fit (with 10% left, as the sweeps
// check): one chunk of small buffers and one partly used chunk of each size
// are all that it takes beyond them.
static void at_the_limit(size_t nc, size_t nh, int buffers) {
  device_size = (size_t)((nc + nh) * (double)buffers / 0.9) + 3 * Workspace::kChunk;
  Pool w;
  w.enlist(0);
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

// What a pool keeps goes when an allocation runs short, also one of another
// context; a pool that a call of another thread holds is left alone, and a
// call's own keeps what the call uses.
static void short_of_memory() {
  device_size = 4096 * MB;
  Pool a, b, other;
  a.enlist(0);
  b.enlist(0);
  other.enlist(1);
  auto object = [](size_t n) {
    auto p = std::make_shared<DevBuf<char>>();
    p->alloc(n);
    return p;
  };
  auto adjoint = [&](Pool& p, int cns, int heat, size_t list) {
    Pool::Use use(p, cns, heat);
    for (int id : {cns, heat})
      if (!p.find(id, cns + heat - id)) p.keep(id, cns + heat - id, list, object(list));
    for (int k = 0; k < 4; ++k) p.ws.take(100 * MB);
  };
  adjoint(a, 0, 1, 300 * MB);
  adjoint(b, 0, 1, 300 * MB);
  adjoint(other, 0, 1, 300 * MB);
  CHECK(device_used == 3000 * MB, "%zu", device_used);
  DevBuf<char> big;
  big.alloc(2900 * MB);  // both pools of device 0 go, device 1's stays
  CHECK(device_used == 3900 * MB && hipGetLastError() == hipSuccess, "%zu", device_used);
  big.release();
  // a call of another thread holds b
  adjoint(a, 0, 1, 300 * MB);
  {
    Pool::Use use(b, 4, 5);
    b.keep(4, 5, 300 * MB, object(300 * MB));
    b.ws.take(100 * MB);
    std::thread([&] {
      DevBuf<char> x;
      x.alloc(2600 * MB);  // a's 1000 MB go
      CHECK(device_used == 4000 * MB, "%zu", device_used);
      bool failed = false;
      try {
        DevBuf<char> y;
        y.alloc(200 * MB);
      } catch (const OutOfMemory& e) {
        failed = e.code == HOM3G_ERR_HIP;
      }
      CHECK(failed && hipGetLastError() == hipSuccess, "no error, or one left for the next launch");
    }).join();
    CHECK(b.find(4, 5) != nullptr, "an object in use");
    // the call's own: what it uses stays, the rest goes
    b.keep(7, 8, 300 * MB, object(300 * MB));
    DevBuf<char> x;
    x.alloc(2600 * MB);
    CHECK(b.find(4, 5) && !b.find(7, 8), "objects of the call");
  }
  CHECK(b.find(4, 5) != nullptr, "kept after the call");
  b.forget(5);
  CHECK(!b.find(4, 5), "the object of a destroyed partner");
  CHECK(b.release() && !b.release() && device_used == 1000 * MB, "%zu", device_used);
  CHECK(other.release() && device_used == 0, "%zu", device_used);
  // the bound, over the workspace and the objects of all solvers
  device_size = size_t(64) << 30;
  for (int k = 0; k < 20; ++k) {
    adjoint(a, 2 * k, 2 * k + 1, (k % 7 + 1) * 150 * MB);
    CHECK(device_used <= Workspace::kKeep, "%zu bytes kept after call %d", device_used, k);
    CHECK(a.find(2 * k, 2 * k + 1) != nullptr, "the last call's object");
  }
  adjoint(a, 100, 101, 3000 * MB);
  CHECK(!a.find(100, 101) && device_used <= Workspace::kKeep, "an object above the bound");
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
    Pool w;
    w.enlist(0);
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
  short_of_memory();
  CHECK(device_used == 0, "%zu bytes lost", device_used);
  std::printf("%d failures\n", failures);
  return failures ? 1 : 0;
}
