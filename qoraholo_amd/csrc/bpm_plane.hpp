// Beam propagation of planes that fit one block, all slices in one launch (see bpm_plane.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "runtime.hpp"

namespace qh {

struct BpmPlaneArgs {
  const float2* tw;      // exp(-2 pi i t / n)
  int nz;
  const float2* screen;  // exp(i phase x), (nz, n, n)
  const float2* step;    // tables of the chunk's illuminations, (count, n, n)
  const float2* last;
  const float* q;
  float2* w;             // envelopes, slices w_slice apart: written by the forward pass (null:
                         // not kept), replaced by the gradient terms in the adjoint
  long w_slice;
  const float2* in;      // adjoint: forward x transform of the residual, (count, n, n)
  float2* out;           // forward: inverse y transform of the last spectrum, (count, n, n)
  float inv;             // 1 / n^2
  float phase;
};

// Whether a plane of side n fits one block.
bool bpm_plane_supported(int n);
// Slices 0 .. nz-1 of `count` illuminations.
void bpm_plane_forward(int n, int count, const BpmPlaneArgs& a, hipStream_t s);
// Slices nz-1 .. 0, and grad (+)= the gradient terms in illumination order.
void bpm_plane_adjoint(int n, int count, const BpmPlaneArgs& a, float* grad, bool init,
                       hipStream_t s);

}  // namespace qh
