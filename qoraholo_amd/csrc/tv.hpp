// FGP total-variation proximal step on the device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "runtime.hpp"

namespace qh {

// d[0, n) = v, by a kernel (safe inside captured graphs, unlike a memset node).
void fill(float* d, long n, float v, hipStream_t s);

// Dual state of the TV prox, kept across calls (FISTA warm start): four rotating dual buffers
// of three components each. Steps run up to four per pass, the last of which forms the output
// where it has at most three (set_fused(false) runs them one per pass and the output in a kernel
// of its own, for comparisons; the results are the same bits).
class TvState {
 public:
  // The dual buffers in device memory of its own, for up to `batch` volumes proxed together.
  TvState(int nz, int ny, int nx, int batch = 1);
  // The dual buffers in `workspace` (`floats` of device memory, at least workspace_floats(nz, ny,
  // nx), 256-byte aligned, not owned: it must outlive the state).
  TvState(int nz, int ny, int nx, float* workspace, std::size_t floats);
  static std::size_t workspace_floats(int nz, int ny, int nx);
  // Zero duals for the next `batch` volumes (at most the capacity), which every prox until the
  // next reset takes together: b and out then hold that many volumes one after another.
  void reset(hipStream_t s, int batch = 1);
  // out = prox_{lambda TV, x >= 0}(b) by `inner` FGP steps from the current dual.
  // out may be b itself. Events t0 and t1, when given, bracket the passes of FGP steps.
  void prox(const float* b, float* out, float lambda, int inner, hipStream_t s,
            bool to_index = false, float nm2 = 0.0f, float inv_k02 = 0.0f, Event* t0 = nullptr,
            Event* t1 = nullptr);
  std::size_t bytes() const;
  void set_fused(bool on) { fused_ = on; }
  // Whether every operation of a step rounds on its own (the default), or multiply-adds are fused.
  void set_exact(bool on) { exact_ = on; }
  // Kernel passes of the last prox call.
  int launches() const { return launches_; }

 private:
  int nz_, ny_, nx_;
  long vol_;
  long rows_;      // of a plane of the dual: ny, in whole groups of four where the buffers have room
  int cap_ = 1;    // volumes the buffers hold
  int batch_ = 1;  // volumes of the current solve
  DeviceBuffer<float> owned_;
  float* p_[4];  // dual buffers of three components each, inside owned_ or the workspace
  int cur_ = 0;
  bool fused_ = true;
  bool exact_ = true;
  int launches_ = 0;
};

}  // namespace qh
