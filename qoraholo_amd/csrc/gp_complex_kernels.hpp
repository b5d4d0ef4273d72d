// Kernels of the Gerchberg-Papoulis passes on full spectra (see gp_complex.hip), which two source
// files instantiate: a process loads the code of a file with its first launch from it (three kernels
// for 41 lengths in one file: 5 ms of the first reconstruction).
#pragma once

#include <cstdint>
#include <type_traits>

#include "common.hpp"
#include "fft.hpp"
#include "fft_engine.hpp"
#include "runtime.hpp"

namespace qh::gp {

struct RowArgs {
  LineGeom g;
  float2* p;
  float scale;
};

struct IndexArgs {
  LineGeom g;
  const float2* p;
  float scale;
  float nm2;
  float inv_k02;
  float* ri;
};

struct ZLineArgs {
  LineGeom g;
  float2* p;
  const float2* measured;
  const std::uint16_t* counts;
  long plane;
};

template <class E>
__global__ void __launch_bounds__(E::kBlock) k_gp_rows(RowArgs a) {
  E e(a.g);
  const long n = a.g.n;
  e.load([&](long l, int i) { return a.p[l * n + i]; });
  e.first(true);
  e.mid([&](long, int, float2& v) {
    const float x = v.x * a.scale;
    v = {x < 0.0f ? 0.0f : x, 0.0f};
  });
  e.second(false);
  e.store2([&](long l, int k, float2 v) { a.p[l * n + k] = v; });
}

template <class E>
__global__ void __launch_bounds__(E::kBlock) k_gp_index(IndexArgs a) {
  E e(a.g);
  const long n = a.g.n;
  e.load([&](long l, int i) { return a.p[l * n + i]; });
  e.first(true);
  e.store1([&](long l, int x, float2 v) {
    const float2 p = cscale(v, a.scale);
    a.ri[l * n + x] = index_from_potential(p.x, p.y, a.nm2, a.inv_k02);
  });
}

// Most bins are not measured: their counts come first (ahead of the transform where the engine
// numbers its bins) and the measured values only where they say so.
template <class E>
__global__ void __launch_bounds__(E::kBlock) k_gp_z(ZLineArgs a) {
  E e(a.g);
  e.load([&](long l, int i) { return a.p[i * a.plane + l]; });
  if constexpr (requires { E::kBins; }) {
    std::uint16_t c[E::kBins];
    e.bins([&](int i, long l, int k, float2&) { c[i] = a.counts[k * a.plane + l]; });
    e.first(false);
    e.bins([&](int i, long l, int k, float2& v) {
      if (c[i] > 0) v = a.measured[k * a.plane + l];
    });
  } else {
    e.first(false);
    e.mid([&](long l, int k, float2& v) {
      if (a.counts[k * a.plane + l] > 0) v = a.measured[k * a.plane + l];
    });
  }
  e.second(true);
  e.store2([&](long l, int i, float2 v) { a.p[i * a.plane + l] = v; });
}

template <class E>
void launch(RowArgs a, unsigned grid, std::size_t lds, hipStream_t s) {
  hipLaunchKernelGGL(k_gp_rows<E>, dim3(grid), dim3(E::kBlock), lds, s, a);
}
template <class E>
void launch(IndexArgs a, unsigned grid, std::size_t lds, hipStream_t s) {
  hipLaunchKernelGGL(k_gp_index<E>, dim3(grid), dim3(E::kBlock), lds, s, a);
}
template <class E>
void launch(ZLineArgs a, unsigned grid, std::size_t lds, hipStream_t s) {
  hipLaunchKernelGGL(k_gp_z<E>, dim3(grid), dim3(E::kBlock), lds, s, a);
}

// Rows: about 256 threads a block. Adjacent lines: 16, a whole 128-byte segment of each block row.
template <class A>
constexpr bool kAdjacent = std::is_same_v<A, ZLineArgs>;

// The kernel for a length of split_lines.hpp; false for other lengths.
bool split(const RowArgs& a, hipStream_t s);
bool split(const IndexArgs& a, hipStream_t s);
bool split(const ZLineArgs& a, hipStream_t s);

}  // namespace qh::gp
