// hes_host.hpp -- host-side helpers shared by the libhes translation units:
// error reporting, HIP error checks and material constants.
#pragma once
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>

#include "hes_device.hpp"
#include "hes_units.hpp"
#include "../../include/hes.h"

namespace hes {

inline thread_local std::string g_err;

inline int fail(int code, const char* msg) {
  g_err = msg;
  return code;
}

#define HIP_TRY(expr)                                                              \
  do {                                                                             \
    hipError_t e__ = (expr);                                                       \
    if (e__ != hipSuccess) {                                                       \
      ::hes::g_err = std::string(#expr) + ": " + hipGetErrorString(e__);           \
      return HES_ERR_HIP;                                                          \
    }                                                                              \
  } while (0)

// Barton2009 constants (rho0, c0, cv, t0, b0, alpha, beta, gamma) -> MatDev
// with the derived quantities (EquationsOfState.jl:90-115).
inline MatDev make_mat(const double* p) {
  MatDev m;
  std::memset(&m, 0, sizeof(m));
  m.rho0 = p[0];
  m.irho0 = 1.0 / p[0];
  m.cv = p[2];
  m.t0 = p[3];
  double b0 = p[4];
  m.alpha = p[5];
  m.beta = p[6];
  m.gamma = p[7];
  m.b0sq = b0 * b0;  // EquationsOfState.jl:111-112
  m.k0 = p[1] * p[1] - (4.0 / 3.0) * (b0 * b0);
  m.hk0a2 = 0.5 * m.k0 / (m.alpha * m.alpha);
  m.k0_2a = m.k0 / (2.0 * m.alpha);
  m.k0_a = m.k0 / m.alpha;
  m.cvt0 = m.cv * m.t0;
  m.icvt0 = 1.0 / m.cvt0;
  m.hb0sq = 0.5 * m.b0sq;
  m.half_a = 0.5 * m.alpha;
  m.half_b = 0.5 * m.beta;
  m.half_g = 0.5 * m.gamma;
  m.ac_t = 3.0 + 2.0 * m.beta;
  m.ac_s = 2.0 + m.beta;
  m.ac_e = m.gamma * (1.0 + m.gamma);
  m.ac_w = m.beta * (1.0 + m.beta);
  m.fast = (m.alpha == 1.0 && m.beta == 3.0 && m.gamma == 2.0) ? 1 : 0;
  return m;
}

inline bool mat_ok(const double* p) {
  for (int k = 0; k < 8; ++k)
    if (!std::isfinite(p[k])) return false;
  return p[0] > 0 && p[2] > 0 && p[3] > 0 && p[5] != 0;
}

// Copies and fills that belong to a handle run on the handle's stream and are
// waited for: a plain hipMemcpy / hipMemset goes to the null stream, which is
// not ordered with the handle's non-blocking stream.
inline hipError_t copy_on(hipStream_t s, void* dst, const void* src, size_t bytes,
                          hipMemcpyKind kind) {
  hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  return e;
}

inline hipError_t zero_on(hipStream_t s, void* dst, size_t bytes) {
  hipError_t e = hipMemsetAsync(dst, 0, bytes, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  return e;
}

// What a call works in: page-locked host memory that the kernels read and
// write themselves (small calls: no copies), device memory (larger ones), and
// a stream of its own.  Allocated for every call they cost one on a single
// state 90 of its 100 us.  One per call that is under way; a few are kept for
// the next, with at most Space::DEVICE bytes each.
struct Space {
  static constexpr size_t HOST = 128 * 1024, DEVICE = 96 << 20;
  int dev = 0;
  char* host = nullptr;
  char* device = nullptr;
  size_t device_bytes = 0;
  hipStream_t stream = nullptr;
};
// What finished calls leave for the next ones, at most PER_DEVICE of it for each
// device (T::dev).  A fixed array: taking and giving allocate nothing.
template <class T, int PER_DEVICE>
class Kept {
 public:
  bool take(int dev, T* t) {
    std::lock_guard<std::mutex> lock(mutex_);
    for (int k = 0; k < n_; ++k)
      if (kept_[k].dev == dev) {
        *t = kept_[k];
        kept_[k] = kept_[--n_];
        return true;
      }
    return false;
  }
  bool give(const T& t) {  // false: there is enough of it
    std::lock_guard<std::mutex> lock(mutex_);
    int here = 0;
    for (int k = 0; k < n_; ++k) here += kept_[k].dev == t.dev;
    if (here == PER_DEVICE || n_ == ROOM) return false;
    kept_[n_++] = t;
    return true;
  }
  template <class F>
  void each(F f) {
    std::lock_guard<std::mutex> lock(mutex_);
    for (int k = 0; k < n_; ++k) f(kept_[k]);
  }

 private:
  static constexpr int ROOM = 8 * PER_DEVICE;
  std::mutex mutex_;
  T kept_[ROOM];
  int n_ = 0;
};
using KeptSpaces = Kept<Space, 4>;
inline KeptSpaces& spaces() {
  static KeptSpaces s;
  static_assert(std::is_trivially_destructible<KeptSpaces>::value, "outlives the runtime's own end");
  return s;
}

// Device memory.  Where it is short, that of kept spaces is given back first.
template <class T>
hipError_t device_alloc(T** p, size_t bytes) {
  hipError_t e = hipMalloc((void**)p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  bool freed = false;
  spaces().each([&](Space& s) {
    if (!s.device) return;
    freed = true;
    (void)hipFree(s.device);
    s.device = nullptr;
    s.device_bytes = 0;
  });
  if (!freed) return e;
  (void)hipGetLastError();  // of the first attempt
  return hipMalloc((void**)p, bytes);
}

// After an allocation that can be done without: whether there was no room for it.
inline bool no_room(hipError_t e) {
  if (e != hipErrorOutOfMemory) return false;
  (void)hipGetLastError();
  return true;
}

inline void space_free(Space& s) {
  if (s.stream) (void)hipStreamDestroy(s.stream);
  if (s.host) (void)hipHostFree(s.host);
  if (s.device) (void)hipFree(s.device);
}
inline hipError_t space_take(Space* s) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (spaces().take(dev, s)) return hipSuccess;
  s->dev = dev;
  e = hipHostMalloc((void**)&s->host, Space::HOST);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    space_free(*s);
    *s = Space();
  }
  return e;
}
inline void space_give(Space& s, bool keep) {
  if (!keep || s.device_bytes > Space::DEVICE || !spaces().give(s)) space_free(s);
}

// Device memory of at least `bytes` in s (its contents are lost when it grows).
inline hipError_t space_device(Space& s, size_t bytes) {
  if (s.device_bytes >= bytes) return hipSuccess;
  hipError_t e = s.device ? hipFree(s.device) : hipSuccess;
  s.device = nullptr;
  s.device_bytes = 0;
  if (e == hipSuccess) e = device_alloc(&s.device, bytes);
  if (e == hipSuccess) s.device_bytes = bytes;
  return e;
}

}  // namespace hes
