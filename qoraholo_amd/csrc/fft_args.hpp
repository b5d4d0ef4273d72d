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

// Bin k of a real row of 2m samples from bins k and m - k (k = 0, m: bin 0 twice) of its packed
// transform: X[k] = (Z[k] + conj Z[m-k]) / 2 - i/2 w (Z[k] - conj Z[m-k]), w = exp(-i pi k / m).
__device__ __forceinline__ float2 real_bin(float2 zk, float2 zmk, float2 w, int k, int m) {
  const float2 zm = cconj(zmk);
  const float2 ev = {0.5f * (zk.x + zm.x), 0.5f * (zk.y + zm.y)};
  const float2 d = {0.5f * (zk.x - zm.x), 0.5f * (zk.y - zm.y)};
  const float2 od = cmul(w, d);
  const float2 o = {od.y, -od.x};
  return (k == 0 || k == m) ? float2{ev.x + o.x, 0.0f} : cadd(ev, o);
}

// The way back: Z[k] = (X[k] + conj X[m-k]) + i conj(w) (X[k] - conj X[m-k]); imaginary parts of
// X[0] and X[m] are dropped.
__device__ __forceinline__ float2 real_pack(float2 xk, float2 xm, float2 w, int k) {
  if (k == 0) {
    xk.y = 0.0f;
    xm.y = 0.0f;
  }
  const float2 s = cadd(xk, cconj(xm));
  const float2 d = csub(xk, cconj(xm));
  const float2 wd = cmul(cconj(w), d);
  return cadd(s, float2{-wd.y, wd.x});
}

__device__ __forceinline__ float2 scale_nonneg(float2 v, float scale) {
  const float x = v.x * scale;
  const float y = v.y * scale;
  return {x < 0.0f ? 0.0f : x, y < 0.0f ? 0.0f : y};
}

// First element of z line l: lines past a plane's belong to the next volumes of the batch.
__device__ __forceinline__ long z_line_base(const ZArgs& a, long l) {
  return a.vol == 0 ? l : (l / a.plane) * a.vol + l % a.plane;
}

// The kernel for a length of split_lines.hpp (lines and z: n; rows: n / 2); false for other lengths.
bool split_fft_lines(const LinesArgs& a, bool contig, hipStream_t s);
bool split_rfft_rows(const RowsArgs& a, bool inverse, hipStream_t s);
bool split_rows_roundtrip(const RowsArgs& a, hipStream_t s);
bool split_z_roundtrip(const ZArgs& a, hipStream_t s);

}  // namespace qh
