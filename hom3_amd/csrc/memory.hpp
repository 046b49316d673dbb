// Device and pinned host memory of the library: owning buffers and the
// workspace of the adjoint sweeps.  Host code only.
#pragma once
#include <hip/hip_runtime.h>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/hom3g.h"

namespace hom3g {

struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
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
    if (count) H3_HIP(hipMalloc((void**)&p, count * sizeof(T)));
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

// Device workspace handed out in pieces and kept between calls: the adjoint
// takes some hundred buffers per call, and allocating and freeing each cost
// more than the sweeps.  What exceeds kKeep is given back at the end of a
// call, the rest with its owner.
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
    try {
      c->buf.alloc(want);
    } catch (const Error&) {
      // short of memory: what lies unused goes first
      (void)hipGetLastError();
      drop_unused();
      c->buf.alloc(want);
    }
    c->unit = unit;
    chunks.push_back(std::move(c));
    return chunks.back()->take(bytes);
  }
  void drop_unused() {
    for (size_t k = 0; k < chunks.size();)
      if (chunks[k]->used == 0) chunks.erase(chunks.begin() + k);
      else ++k;
  }
  // bytes kept and not handed out
  size_t spare() const {
    size_t n = 0;
    for (auto& c : chunks) n += c->left();
    return n;
  }
  // end of a call: nothing handed out is in use any more
  void give_back() {
    size_t total = 0;
    for (size_t k = 0; k < chunks.size();) {
      chunks[k]->used = 0;
      if (total + chunks[k]->buf.n > kKeep) {
        chunks.erase(chunks.begin() + k);
      } else {
        total += chunks[k]->buf.n;
        ++k;
      }
    }
  }
};

}  // namespace hom3g
