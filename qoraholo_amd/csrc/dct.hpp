// Cosine transforms of the phase unwrapping on the register engines (see dct.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace qh {

// Divergence of the wrapped phase differences of image psi (ny, nx) at (y, x).
__device__ __forceinline__ float wrapped_divergence(const float* psi, int y, int x, int ny, int nx) {
  const float* const at = psi + static_cast<long>(y) * nx + x;
  const float p = *at;
  float r = 0.0f;
  if (x + 1 < nx) r += wrap_phase(at[1] - p);
  if (x > 0) r -= wrap_phase(p - at[-1]);
  if (y + 1 < ny) r += wrap_phase(at[nx] - p);
  if (y > 0) r -= wrap_phase(p - at[-nx]);
  return r;
}

// Both sides have an engine: the solve below takes these kernels.
bool dct_supported(int ny, int nx);
// phi (images, ny, nx): least-squares phase of psi up to a constant per image: divergence, DCT-II
// along x and y, division by the Neumann eigenvalues (DC set to 0), inverse DCTs.
void dct_poisson(const float* psi, float* phi, int images, int ny, int nx, hipStream_t s);

}  // namespace qh
