// Device and pinned host memory of the library: owning buffers and the
// workspace of the adjoint sweeps.  Host code only.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/hom3g.h"

namespace hom3g {

struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

// device memory ran out (after what is kept between calls was freed)
struct OutOfMemory : Error {
  explicit OutOfMemory(size_t bytes) : Error(HOM3G_ERR_HIP, "out of device memory: " + std::to_string(bytes) + " bytes") {}
};

#define H3_HIP(expr)                                                                        \
  do {                                                                                      \
    hipError_t e_ = (expr);                                                                 \
    if (e_ != hipSuccess)                                                                   \
      throw ::hom3g::Error(HOM3G_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

#define H3_REQUIRE(cond, msg) \
  do {                        \
    if (!(cond)) throw ::hom3g::Error(HOM3G_ERR_ARG, msg); \
  } while (0)

#define H3_LAUNCH_CHECK() H3_HIP(hipGetLastError())

// What the contexts of a device keep between calls (Pool) and nobody uses
// now, freed; true if there was something.
inline bool release_idle(int device);

// hipMalloc; short of memory, what is kept goes first
inline void device_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    int device = 0;
    if (hipGetDevice(&device) == hipSuccess && release_idle(device)) e = hipMalloc(p, bytes);
  }
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();  // reported here and not by the next launch
    throw OutOfMemory(bytes);
  }
  H3_HIP(e);
}

template <class T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { release(); }
  void alloc(size_t count) {
    if (count == n && p) return;
    release();
    if (count) device_malloc((void**)&p, count * sizeof(T));
    n = count;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  void upload(const T* h, size_t count, hipStream_t s, size_t off = 0) {
    H3_HIP(hipMemcpyAsync(p + off, h, count * sizeof(T), hipMemcpyHostToDevice, s));
  }
  void download(T* h, size_t count, hipStream_t s, size_t off = 0) const {
    H3_HIP(hipMemcpyAsync(h, p + off, count * sizeof(T), hipMemcpyDeviceToHost, s));
  }
};

// Pinned host buffer (hipHostMalloc) for stream-ordered copies out of and
// back into device memory; released only after the device has finished the
// copies that may still read or write it.
template <class T>
struct PinnedBuf {
  T* p = nullptr;
  size_t n = 0;
  PinnedBuf() = default;
  PinnedBuf(const PinnedBuf&) = delete;
  PinnedBuf& operator=(const PinnedBuf&) = delete;
  ~PinnedBuf() { release(); }
  void alloc(size_t count) {
    if (count == n && p) return;
    release();
    if (count) H3_HIP(hipHostMalloc((void**)&p, count * sizeof(T), hipHostMallocDefault));
    n = count;
  }
  void release() {
    if (p) {
      (void)hipDeviceSynchronize();
      (void)hipHostFree(p);
    }
    p = nullptr;
    n = 0;
  }
};

// Device workspace handed out in pieces and kept between calls (Pool): the
// adjoint takes some hundred buffers per call, and allocating and freeing
// each cost more than the sweeps.
//
// Buffers above kShare come from chunks that hold a whole number of them (the
// states of one solver are all of one size), so that at the limit of the
// device's memory a call needs what its buffers need: 33 MB states from
// plain 64 MB chunks took almost twice as much.
struct Workspace {
  static constexpr size_t kChunk = size_t(64) << 20, kShare = kChunk / 32, kKeep = size_t(2) << 30;
  struct Chunk {
    DevBuf<char> buf;
    size_t used = 0, unit = 0;  // unit: the size it was made for, 0: buffers up to kShare
    size_t left() const { return buf.n - used; }
    void* take(size_t bytes) {
      void* p = buf.p + used;
      used += bytes;
      return p;
    }
  };
  std::vector<std::unique_ptr<Chunk>> chunks;
  void* take(size_t bytes) {
    bytes = (bytes + 255) & ~size_t(255);
    const size_t unit = bytes > kShare ? bytes : 0;
    for (auto& c : chunks)
      if (c->unit == unit && c->left() >= bytes) return c->take(bytes);
    // a chunk made for another size, the one that it fills best
    Chunk* best = nullptr;
    for (auto& c : chunks)
      if (unit && c->unit && c->left() >= bytes && (!best || c->left() < best->left())) best = c.get();
    if (best) return best->take(bytes);
    auto c = std::make_unique<Chunk>();
    const size_t want = unit ? (kChunk / bytes > 1 ? kChunk / bytes * bytes : bytes) : kChunk;
    c->buf.alloc(want);
    c->unit = unit;
    chunks.push_back(std::move(c));
    return chunks.back()->take(bytes);
  }
  bool drop_unused() {
    const size_t n = chunks.size();
    chunks.erase(std::remove_if(chunks.begin(), chunks.end(), [](auto& c) { return c->used == 0; }), chunks.end());
    return chunks.size() < n;
  }
  // bytes kept and not handed out
  size_t spare() const {
    size_t n = 0;
    for (auto& c : chunks) n += c->left();
    return n;
  }
  // end of a call: nothing handed out is in use any more; up to `keep` bytes
  // stay, returned
  size_t give_back(size_t keep = kKeep) {
    size_t total = 0;
    for (size_t k = 0; k < chunks.size();) {
      chunks[k]->used = 0;
      if (total + chunks[k]->buf.n > keep) {
        chunks.erase(chunks.begin() + k);
      } else {
        total += chunks[k]->buf.n;
        ++k;
      }
    }
    return total;
  }
};

// What a context keeps between its adjoint calls: the workspace, and objects
// of its solvers (their reverse lists and buffers), together up to
// Workspace::kKeep.  It goes when its owner does, when release_idle is
// called, or when any allocation of the library on its device runs short.
//
// A call holds the pool with a Use; while it does, the workspace and the
// objects of the call's two solvers stay, and other threads leave the pool
// alone.
struct Pool {
  struct Item {
    int owner, partner;  // solver ids
    size_t bytes;
    std::shared_ptr<void> p;
  };
  Workspace ws;

  Pool() = default;
  Pool(const Pool&) = delete;
  Pool& operator=(const Pool&) = delete;
  ~Pool() { delist(); }

  // from here on release_idle reaches it
  void enlist(int dev) {
    std::lock_guard<std::mutex> g(registry_lock());
    device = dev;
    registry().push_back(this);
  }
  void delist() {
    std::lock_guard<std::mutex> g(registry_lock());
    auto& r = registry();
    r.erase(std::remove(r.begin(), r.end(), this), r.end());
  }

  struct Use {
    Pool& P;
    std::unique_lock<std::mutex> call;
    Use(Pool& p, int a, int b) : P(p), call(p.call_lock) {
      std::lock_guard<std::mutex> g(P.lock);
      P.users[0] = a;
      P.users[1] = b;
      P.in_use = true;
      held() = &P;
    }
    // (the call's work on the device has ended)
    ~Use() {
      std::lock_guard<std::mutex> g(P.lock);
      P.in_use = false;
      held() = nullptr;
      // the objects of the call's solvers first, then the workspace, then
      // those of the others
      size_t n = 0;
      auto fits = [&](const Item& i) {
        if (n + i.bytes > Workspace::kKeep) return false;
        n += i.bytes;
        return true;
      };
      P.drop([&](const Item& i) { return P.user(i) && !fits(i); });
      n += P.ws.give_back(Workspace::kKeep - n);
      P.drop([&](const Item& i) { return !P.user(i) && !fits(i); });
    }
  };

  // an object kept for a solver and its partner, or null (by a call that
  // holds the pool)
  std::shared_ptr<void> find(int owner, int partner) const {
    for (const Item& i : items)
      if (i.owner == owner && i.partner == partner) return i.p;
    return nullptr;
  }
  // (one object per solver)
  void keep(int owner, int partner, size_t bytes, std::shared_ptr<void> p) {
    std::lock_guard<std::mutex> g(lock);
    drop([&](const Item& i) { return i.owner == owner; });
    items.push_back(Item{owner, partner, bytes, std::move(p)});
  }
  // the objects of a solver that is destroyed
  void forget(int solver) {
    std::lock_guard<std::mutex> g(lock);
    drop([&](const Item& i) { return i.owner == solver || i.partner == solver; });
  }
  // Frees what no call uses; all: also the objects of the calling thread's
  // own call (before it has taken them)
  bool release(bool all = false) {
    std::lock_guard<std::mutex> g(lock);
    if (in_use && held() != this) return false;
    const bool w = ws.drop_unused();
    return drop([&](const Item& i) { return all || !in_use || !user(i); }) || w;
  }

 private:
  friend bool release_idle(int device);
  int device = -1;
  int users[2] = {-1, -1};
  bool in_use = false;
  std::vector<Item> items;
  std::mutex lock;       // the members above
  std::mutex call_lock;  // held by a call

  bool user(const Item& i) const { return i.owner == users[0] || i.owner == users[1]; }
  template <class F>
  bool drop(F&& f) {
    const size_t n = items.size();
    items.erase(std::remove_if(items.begin(), items.end(), f), items.end());
    return items.size() < n;
  }
  static Pool*& held() {
    static thread_local Pool* p = nullptr;
    return p;
  }
  static std::mutex& registry_lock() {
    static std::mutex& m = *new std::mutex;  // (outlives the static contexts)
    return m;
  }
  static std::vector<Pool*>& registry() {
    static std::vector<Pool*>& r = *new std::vector<Pool*>;
    return r;
  }
};

inline bool release_idle(int device) {
  std::lock_guard<std::mutex> g(Pool::registry_lock());
  bool any = false;
  for (Pool* p : Pool::registry())
    if (p->device == device) any = p->release() || any;
  return any;
}

}  // namespace hom3g
