// Gerchberg-Papoulis passes on full spectra (see gp_complex.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace qh {

// Rows (contiguous, of n) of p, in place: inverse transform times scale, the real part's max(., 0),
// forward transform.
void gp_complex_rows(float2* p, long rows, int n, float scale, hipStream_t s);
// Rows of p: inverse transform times scale, to the refractive index.
void gp_complex_index(const float2* p, long rows, int n, float scale, float nm2, float inv_k02,
                      float* ri, hipStream_t s);
// z lines of p (nz, plane), in place: forward transform, the measured bins (counts > 0) restored,
// inverse transform.
void gp_complex_z(float2* p, const float2* measured, const std::uint16_t* counts, int nz,
                  long plane, hipStream_t s);

}  // namespace qh
