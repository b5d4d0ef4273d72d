// Arguments of the transform kernels, and the launchers of the lengths of split_lines.hpp.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "fft.hpp"

namespace qh {

__device__ __forceinline__ long line_base(long l, const Lines& g) {
  return (l / g.inner) * g.outer + (l % g.inner) * g.inner_stride;
}

struct LinesArgs {
  const float2* in;
  float2* out;
  Lines g;
  int n;
  int lines_per_block;
  FftFactors f;
  const float2* tw;
  int inverse;
  float scale;
  int alt_mod;
};

struct RowsArgs {
  const float* x;
  const float* x2;
  float* xo;
  long x_pitch;
  float2* c;
  long c_pitch;
  long rows;
  int n;
  int rows_per_block;
  FftFactors f;      // of n / 2
  const float2* tw;  // exp(-2 pi i t / n), t in [0, n)
  RealOp op;
};

struct ZArgs {
  float2* e;
  const float2* a;
  const std::uint8_t* hits;
  long lines;
  long plane;
  int nz;
  int lines_per_block;
  FftFactors f;
  const float2* tw;
  long vol;  // elements between the volumes of a batch (0: one volume, lines == plane)
};

// First element of z line l: lines past a plane's belong to the next volumes of the batch.
__device__ __forceinline__ long z_line_base(const ZArgs& a, long l) {
  return a.vol == 0 ? l : (l / a.plane) * a.vol + l % a.plane;
}

// The kernel for a length of split_lines.hpp (lines and z: n; rows: n / 2); false for other lengths.
bool split_fft_lines(const LinesArgs& a, bool contig, hipStream_t s);
bool split_rfft_rows(const RowsArgs& a, bool inverse, hipStream_t s);
bool split_z_roundtrip(const ZArgs& a, hipStream_t s);

}  // namespace qh
