// common.hpp -- shared helpers of the nosh_amd HIP library (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

namespace nosh {

// Error carrying a C-ABI status code; converted at the ABI boundary.
struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

enum Status : int {
  kOk = 0,
  kInvalid = 1,
  kUnsupported = 2,
  kMissingParam = 3,
  kHip = 4,
  kNotBuilt = 5,
  kNotConverged = 6,
};

#define NOSH_HIP(call)                                                                   \
  do {                                                                                   \
    hipError_t e_ = (call);                                                              \
    if (e_ != hipSuccess)                                                                \
      throw ::nosh::Error(::nosh::kHip, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

#define NOSH_CHECK(cond, code, msg)                 \
  do {                                              \
    if (!(cond)) throw ::nosh::Error((code), (msg)); \
  } while (0)

// Device allocation: owned, or a part of a Slab that outlives it.
template <class T>
struct DBuf {
  T* p = nullptr;
  size_t n = 0;
  bool owned = true;
  DBuf() = default;
  explicit DBuf(size_t count) { alloc(count); }
  DBuf(const DBuf&) = delete;
  DBuf& operator=(const DBuf&) = delete;
  DBuf(DBuf&& o) noexcept : p(o.p), n(o.n), owned(o.owned) {
    o.p = nullptr;
    o.n = 0;
    o.owned = true;
  }
  DBuf& operator=(DBuf&& o) noexcept {
    if (this != &o) {
      release();
      p = o.p;
      n = o.n;
      owned = o.owned;
      o.p = nullptr;
      o.n = 0;
      o.owned = true;
    }
    return *this;
  }
  ~DBuf() { release(); }
  void alloc(size_t count) {
    release();
    n = count;
    if (count) NOSH_HIP(hipMalloc(&p, count * sizeof(T)));
  }
  void release() {
    if (p && owned) (void)hipFree(p);
    p = nullptr;
    n = 0;
    owned = true;
  }
  void view(T* part, size_t count) {
    release();
    p = part;
    n = count;
    owned = false;
  }
  void upload(const T* h, size_t count, hipStream_t s) {
    NOSH_HIP(hipMemcpyAsync(p, h, count * sizeof(T), hipMemcpyHostToDevice, s));
  }
  void download(T* h, size_t count, hipStream_t s) const {
    NOSH_HIP(hipMemcpyAsync(h, p, count * sizeof(T), hipMemcpyDeviceToHost, s));
  }
  void zero(hipStream_t s) {
    if (n) NOSH_HIP(hipMemsetAsync(p, 0, n * sizeof(T), s));
  }
  size_t bytes() const { return n * sizeof(T); }
};

// Device memory handed out in order from one allocation (an allocation costs
// 30-100 us, its release with everything it waits for 100-150). mark / reset
// give parts back, last taken first: work on one stream may reuse them at
// once. What does not fit the estimate gets an allocation of its own.
class Slab {
 public:
  explicit Slab(size_t bytes) : buf_(bytes) {}
  template <class T>
  T* take(size_t count) {
    const size_t bytes = (std::max<size_t>(count, 1) * sizeof(T) + 255) / 256 * 256;
    if (off_ + bytes <= buf_.n) {
      T* r = reinterpret_cast<T*>(buf_.p + off_);
      off_ += bytes;
      return r;
    }
    more_.emplace_back(bytes);
    return reinterpret_cast<T*>(more_.back().p);
  }
  template <class T>
  void take(DBuf<T>& b, size_t count) {
    b.view(take<T>(count), count);
  }
  size_t mark() const { return off_; }
  void reset(size_t m) { off_ = m; }

 private:
  DBuf<char> buf_;
  size_t off_ = 0;
  std::vector<DBuf<char>> more_;
};
// Bytes `count` entries of T take in a Slab.
template <class T>
size_t slab_bytes(size_t count) {
  return (std::max<size_t>(count, 1) * sizeof(T) + 255) / 256 * 256;
}

inline unsigned grid_for(int64_t work, int block) {
  int64_t g = (work + block - 1) / block;
  return unsigned(g < 1 ? 1 : g);
}

// Library-wide stream: one per process, default priority.
hipStream_t default_stream();

}  // namespace nosh
