// Kernels of the cosine transforms of the phase unwrapping (see dct.hip), which two source files
// instantiate: a process loads the code of a file with its first launch from it (three kernels for
// 41 lengths in one file: 6.5 ms of the first unwrapping).
#pragma once

#include <type_traits>

#include "common.hpp"
#include "dct.hpp"
#include "fft.hpp"
#include "fft_engine.hpp"
#include "runtime.hpp"

namespace qh::dct {

struct RowsForward {
  LineGeom g;
  const float2* dtw;  // exp(-i pi k / (2 n))
  const float* psi;
  float* a;
  int ny;
};

struct RowsInverse {
  LineGeom g;
  const float2* dtw;
  float* a;
  float inv_n;
};

struct Columns {
  LineGeom g;
  const float2* dtw;
  float* a;
  int nx;
  const float* eig_y;
  const float* eig_x;
  float inv_n;
};

// Element of a line that is element i of its transform's input.
__device__ __forceinline__ int source(int i, int n) {
  return 2 * i < n ? 2 * i : 2 * (n - 1 - i) + 1;
}

// Cosine coefficients k of lines a and b from bins k and n - k of the transform of a + i b.
__device__ __forceinline__ float2 cosine_pair(float2 z, float2 zm, float2 w) {
  const float2 a = {0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y)};
  const float2 b = {0.5f * (z.y + zm.y), 0.5f * (zm.x - z.x)};
  return {w.x * a.x - w.y * a.y, w.x * b.x - w.y * b.y};
}

// Bin k of a + i b from the coefficients k and n - k (k = 0: zero) of both lines.
__device__ __forceinline__ float2 bin_pair(float2 x, float2 m, float2 w) {
  return cmul(cconj(w), float2{x.x + m.y, x.y - m.x});
}

// Line l is rows 2 l and 2 l + 1.
template <class E>
__global__ void __launch_bounds__(E::kBlock) k_dct_rows_forward(RowsForward a) {
  constexpr int N = E::N;
  E e(a.g);
  const int half = a.ny / 2;
  e.load([&](long l, int i) {
    const long image = l / half;
    const int y = 2 * static_cast<int>(l - image * half);
    const float* const psi = a.psi + image * a.ny * N;
    const int x = source(i, N);
    return float2{wrapped_divergence(psi, y, x, a.ny, N), wrapped_divergence(psi, y + 1, x, a.ny, N)};
  });
  e.first(false);
  // Natural order in the engine's exchange buffer, which holds more than n of a line.
  float2* const row = e.t + e.line * (N + 1);
  __syncthreads();
  e.store1([&](long, int k, float2 v) { row[k] = v; });
  __syncthreads();
  e.store1([&](long l, int k, float2 v) {
    const float2 c = cosine_pair(v, row[k == 0 ? 0 : N - k], a.dtw[k]);
    float* const out = a.a + 2 * l * N + k;
    out[0] = c.x;
    out[N] = c.y;
  });
}

template <class E>
__global__ void __launch_bounds__(E::kBlock) k_dct_rows_inverse(RowsInverse a) {
  constexpr int N = E::N;
  E e(a.g);
  e.load([&](long l, int k) {
    const float* const row = a.a + 2 * l * N;
    const float2 x = {row[k], row[N + k]};
    const float2 m = k == 0 ? float2{0.0f, 0.0f} : float2{row[N - k], row[2 * N - k]};
    return bin_pair(x, m, a.dtw[k]);
  });
  e.first(true);
  e.store1([&](long l, int i, float2 v) {
    float* const row = a.a + 2 * l * N + source(i, N);
    row[0] = v.x * a.inv_n;
    row[N] = v.y * a.inv_n;
  });
}

// Line l of an image is columns 2 l and 2 l + 1.
template <class E>
__global__ void __launch_bounds__(E::kBlock) k_dct_columns(Columns a) {
  constexpr int N = E::N;
  E e(a.g);
  const int half = a.nx / 2;
  const auto at = [&](long l, int i) {
    const long image = l / half;
    return reinterpret_cast<float2*>(a.a) + (image * N + i) * half + (l - image * half);
  };
  e.load([&](long l, int i) { return *at(l, source(i, N)); });
  e.first(false);
  // Coefficient k of the block's lines at t[k LINES + line].
  float2* const t = e.t + e.line;
  __syncthreads();
  e.store1([&](long, int k, float2 v) { t[k * E::LINES] = v; });
  __syncthreads();
  e.bins([&](int, long l, int k, float2& v) {
    const int kx = 2 * static_cast<int>(l % half);
    const float2 c = cosine_pair(v, t[(k == 0 ? 0 : N - k) * E::LINES], a.dtw[k]);
    v = {(k == 0 && kx == 0) ? 0.0f : c.x / (a.eig_y[k] + a.eig_x[kx] - 4.0f),
         c.y / (a.eig_y[k] + a.eig_x[kx + 1] - 4.0f)};
  });
  __syncthreads();
  e.store1([&](long, int k, float2 v) { t[k * E::LINES] = v; });
  __syncthreads();
  e.load([&](long, int k) {
    const float2 m = k == 0 ? float2{0.0f, 0.0f} : t[(N - k) * E::LINES];
    return bin_pair(t[k * E::LINES], m, a.dtw[k]);
  });
  e.first(true);
  e.store1([&](long l, int i, float2 v) {
    *at(l, source(i, N)) = float2{v.x * a.inv_n, v.y * a.inv_n};
  });
}

template <class E>
void launch(const RowsForward& a, hipStream_t s) {
  hipLaunchKernelGGL(k_dct_rows_forward<E>, dim3(E::grid(a.g.lines)), dim3(E::kBlock), 0, s, a);
}
template <class E>
void launch(const RowsInverse& a, hipStream_t s) {
  hipLaunchKernelGGL(k_dct_rows_inverse<E>, dim3(E::grid(a.g.lines)), dim3(E::kBlock), 0, s, a);
}
template <class E>
void launch(const Columns& a, hipStream_t s) {
  hipLaunchKernelGGL(k_dct_columns<E>, dim3(E::grid(a.g.lines)), dim3(E::kBlock), 0, s, a);
}

// Rows: about 256 threads a block. Columns: 16 pairs, a whole 128-byte segment of each row.
template <class A>
constexpr bool kColumns = std::is_same_v<A, Columns>;

// The kernel for a length of split_lines.hpp; false for other lengths.
bool split(const RowsForward& a, hipStream_t s);
bool split(const RowsInverse& a, hipStream_t s);
bool split(const Columns& a, hipStream_t s);

}  // namespace qh::dct
