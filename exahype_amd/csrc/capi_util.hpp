// capi_util.hpp -- helpers shared by the C-ABI translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <memory>
#include <new>

#include "../../include/exahype_amd.h"
#include "aderdg.hpp"

using exa::FaceDesc;
using exa::SolverDesc;

namespace {

// PNPM[order], stableTimeStepSize.cpph:33-34
const double kPNPM[10] = {1.0, 0.33, 0.17, 0.1, 0.069, 0.045, 0.038, 0.03, 0.02, 0.015};

int from_hip(hipError_t e) {
  if (e == hipSuccess) return EXA_OK;
  if (e == hipErrorNotSupported) return EXA_E_UNSUPPORTED;
  if (e == hipErrorOutOfMemory) return EXA_E_NOMEM;
  return EXA_E_HIP;
}

#define EXA_TRY(expr)                     \
  do {                                    \
    const hipError_t e_ = (expr);         \
    if (e_ != hipSuccess) return from_hip(e_); \
  } while (0)

bool to_desc(const exa_solver* s, SolverDesc* d) {
  if (!s) return false;
  d->pde = s->pde;
  d->order = s->order;
  d->nvar = s->num_variables;
  d->npar = s->num_parameters;
  d->terms = s->terms;
  d->no_time_averaging = s->no_time_averaging;
  d->cfl = s->cfl;
  d->precision = s->precision;
  d->linear = s->linear;
  return s->order >= 0 && s->order <= 9 && s->num_variables > 0 && s->num_parameters >= 0;
}

// Device buffer owned for the duration of one synchronous call.
struct DevBuf {
  void* p = nullptr;
  hipError_t alloc(size_t bytes) { return hipMalloc(&p, bytes ? bytes : 8); }
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
  double* d() const { return static_cast<double*>(p); }
};

// The device buffers of one call: inputs copied up, results copied down, the
// rest scratch, in one allocation.  A call on one cell spends its time on the
// host path (each allocation, copy and synchronisation of the runtime takes 3
// to 10 us, the kernel 2 to 25), so small calls make one copy each way, through
// a host buffer that the parts are packed in; a large batch copies its arrays
// directly.  Single-cell calls of order 3 (predictor with temporaries, volume
// integral, three Riemann problems, surface integral, update, time step):
// 954 -> 399 us.
class CallBuffers {
 public:
  // Results first and inputs after, with in and out arrays in between, so that
  // either direction is one range; zero: cleared before the call.
  int in(const void* host, size_t bytes) { return add(host, nullptr, bytes, kIn); }
  int inout(const void* from, void* to, size_t bytes) { return add(from, to, bytes, kInOut); }
  int out(void* host, size_t bytes, bool zero = false) { return add(nullptr, host, bytes, zero ? kInOut : kOut); }
  int zeroed(size_t bytes) { return add(nullptr, nullptr, bytes, kIn); }
  int scratch(size_t bytes) { return add(nullptr, nullptr, bytes, kScratch); }
  double* d(int i) const { return static_cast<double*>(at(i)); }
  template <typename T>
  T* as(int i) const {
    return static_cast<T*>(at(i));
  }
  // Allocates, lays the parts out and copies the inputs up.
  hipError_t up() {
    if (full_) return hipErrorInvalidValue;
    size_t end = 0;
    for (int k = 0; k < kKinds; ++k) {
      begin_[k] = end;
      for (int i = 0; i < n_; ++i)
        if (part_[i].kind == k) {
          part_[i].offset = end;
          end += (std::max<size_t>(part_[i].bytes, 8) + 255) / 256 * 256;
        }
    }
    begin_[kKinds] = end;
    if (hipError_t e = mem_.alloc(end); e != hipSuccess) return e;
    const size_t lo = begin_[kInOut], hi = begin_[kScratch];  // kInOut and kIn; scratch is not packed
    if (hi <= kPackBytes) host_.reset(new (std::nothrow) char[hi]);
    for (int i = 0; i < n_; ++i) {
      const Part& p = part_[i];
      if (p.kind != kIn && p.kind != kInOut) continue;
      hipError_t e = hipSuccess;
      if (host_) {
        if (p.from)
          std::memcpy(host_.get() + p.offset, p.from, p.bytes);
        else
          std::memset(host_.get() + p.offset, 0, p.bytes);
      } else if (p.from) {
        e = hipMemcpy(at(i), p.from, p.bytes, hipMemcpyHostToDevice);
      } else {
        e = hipMemset(at(i), 0, p.bytes);
      }
      if (e != hipSuccess) return e;
    }
    if (!host_ || hi == lo) return hipSuccess;
    return hipMemcpy(static_cast<char*>(mem_.p) + lo, host_.get() + lo, hi - lo, hipMemcpyHostToDevice);
  }
  // Waits for the call's kernels and copies the results down.
  hipError_t down() {
    const size_t hi = begin_[kIn];  // kOut and kInOut
    if (host_) {
      hipError_t e = hi > 0 ? hipMemcpy(host_.get(), mem_.p, hi, hipMemcpyDeviceToHost) : hipDeviceSynchronize();
      if (e != hipSuccess) return e;
    } else if (hipError_t e = hipDeviceSynchronize(); e != hipSuccess) {
      return e;
    }
    for (int i = 0; i < n_; ++i) {
      const Part& p = part_[i];
      if (!p.to) continue;
      if (host_) {
        std::memcpy(p.to, host_.get() + p.offset, p.bytes);
      } else if (hipError_t e = hipMemcpy(p.to, at(i), p.bytes, hipMemcpyDeviceToHost); e != hipSuccess) {
        return e;
      }
    }
    return hipSuccess;
  }

 private:
  static constexpr size_t kPackBytes = 1 << 20;
  enum Kind { kOut, kInOut, kIn, kScratch, kKinds };
  struct Part {
    const void* from;
    void* to;
    size_t bytes, offset;
    Kind kind;
  };
  int add(const void* from, void* to, size_t bytes, Kind kind) {
    if (n_ == kParts) {  // reported by up()
      full_ = true;
      return n_ - 1;
    }
    part_[n_] = {from, to, bytes, 0, kind};
    return n_++;
  }
  void* at(int i) const { return static_cast<char*>(mem_.p) + part_[i].offset; }
  static constexpr int kParts = 16;
  Part part_[kParts];
  int n_ = 0;
  bool full_ = false;
  size_t begin_[kKinds + 1] = {};
  DevBuf mem_;
  std::unique_ptr<char[]> host_;
};

struct Sizes {
  long B, B2, B3, B4, D, V;
  explicit Sizes(const SolverDesc& sd)
      : B(sd.order + 1), B2(B * B), B3(B2 * B), B4(B3 * B), D(sd.nvar + sd.npar), V(sd.nvar) {}
};

uint64_t splitmix64(uint64_t& x) {
  uint64_t z = (x += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// The formula fields of ICArgs from an exa_euler_ic: the seeded Fourier
// modes draw integer wave vectors in [-3,3]^3 (not all zero) and four phases
// in [0, 2 pi) each from splitmix64.
void fill_euler_ic(const exa_euler_ic* ic, exa::ICArgs* a) {
  for (int d = 0; d < 3; ++d) {
    a->k[d] = ic->k[d];
    a->vel[d] = ic->vel[d];
  }
  a->rho0 = ic->rho0;
  a->amp = ic->amp;
  a->p = ic->p;
  a->nmodes = ic->nmodes;
  a->mode_amp = ic->mode_amp;
  uint64_t state = ic->seed;
  for (int m = 0; m < ic->nmodes; ++m) {
    int kk[3];
    do {
      for (int d = 0; d < 3; ++d) kk[d] = (int)(splitmix64(state) % 7) - 3;
    } while (kk[0] == 0 && kk[1] == 0 && kk[2] == 0);
    for (int d = 0; d < 3; ++d) a->mode_k[m][d] = kk[d];
    for (int c = 0; c < 4; ++c)
      a->mode_phase[m][c] = 6.283185307179586476925286766559 * (double)(splitmix64(state) >> 11) * 0x1.0p-53;
  }
}

}  // namespace
