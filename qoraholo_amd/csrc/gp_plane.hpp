// The part of a Gerchberg-Papoulis step within the planes of a half spectrum (see gp_plane.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace qh {

// Planes (n, n/2 + 1) of e, in place: inverse y transform, inverse real x transform times scale,
// max(., 0), real x transform, y transform. False, with nothing done, for sides without a kernel.
bool gp_plane(float2* e, long planes, int n, float scale, hipStream_t s);

}  // namespace qh
