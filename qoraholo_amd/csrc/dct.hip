// Cosine transforms of the phase unwrapping on the register engines.
//
// A DCT-II of a real line is an FFT of the line with its even elements first and its odd ones
// reversed (Makhoul). Two lines go as the real and imaginary part of one, two rows of an image or
// two adjacent columns: half the transforms, and columns load as whole complex values. The rows
// form the divergence they transform, the columns divide by the eigenvalues between their two
// transforms, so that the solve is three passes over the images. 49 images of 256^2: 31.0, 15.3 and
// 9.4 us, against 16.9 (divergence), 24.3, 48.5 and 23.8 us with LDS transforms of single lines; the
// 26 MB a pass moves take 5 us. What bounds the first: the eight wrapped differences of a pair of
// rows, each with a division; the others: the exchanges of a block.
#include "dct.hpp"

#include <algorithm>
#include <type_traits>

#include "fft.hpp"
#include "fft_engine.hpp"
#include "runtime.hpp"
#include "split_lines.hpp"

namespace qh {

namespace {

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

constexpr int floor_pow2(int v) { return v < 2 ? 1 : 2 * floor_pow2(v / 2); }

template <int N1, int N2, class A>
bool launch_reg(const A& a, hipStream_t s) {
  constexpr int kT = N1 > N2 ? N1 : N2;
  constexpr int kLines = kColumns<A> ? std::max(16, floor_pow2(256 / kT)) : floor_pow2(256 / kT);
  launch<RegLines<N1, N2, kColumns<A>, kLines * kT>>(a, s);
  return true;
}

template <int N>
struct Split {
  template <class A>
  static void run(const A& a, hipStream_t s) {
    constexpr int kT = SplitLines<N, false, 1>::T;
    launch<SplitLines<N, kColumns<A>, kColumns<A> ? 16 : std::max(1, 256 / kT)>>(a, s);
  }
};

template <class A>
void run(const A& a, const char* what, hipStream_t s) {
  const auto go = [&] {
    switch (a.g.n) {
      case 32: return launch_reg<8, 4>(a, s);
      case 48: return launch_reg<8, 6>(a, s);
      case 64: return launch_reg<8, 8>(a, s);
      case 96: return launch_reg<16, 6>(a, s);
      case 128: return launch_reg<16, 8>(a, s);
      case 192: return launch_reg<16, 12>(a, s);
      case 256: return launch_reg<16, 16>(a, s);
      case 384: return launch_reg<16, 24>(a, s);
      case 512: return launch_reg<32, 16>(a, s);
      default: return with_split<Split>(a.g.n, a, s);
    }
  };
  require(go(), "dct: no kernel for this length");
  check_launch(what);
}

template <int N>
struct Any {
  static void run() {}
};

bool length_supported(int n) {
  for (int m : {32, 48, 64, 96, 128, 192, 256, 384, 512}) {
    if (n == m) return true;
  }
  return with_split<Any>(n);
}

LineGeom geometry(int n, long lines) { return {fft_twiddles(n), FftFactors{}, n, lines, 0}; }

}  // namespace

bool dct_supported(int ny, int nx) { return length_supported(ny) && length_supported(nx); }

void dct_poisson(const float* psi, float* phi, int images, int ny, int nx, hipStream_t s) {
  const LineGeom rows = geometry(nx, static_cast<long>(images) * (ny / 2));
  const LineGeom columns = geometry(ny, static_cast<long>(images) * (nx / 2));
  run(RowsForward{rows, dct_twiddles(nx), psi, phi, ny}, "dct_rows", s);
  run(Columns{columns, dct_twiddles(ny), phi, nx, neumann_terms(ny), neumann_terms(nx),
              1.0f / static_cast<float>(ny)},
      "dct_columns", s);
  run(RowsInverse{rows, dct_twiddles(nx), phi, 1.0f / static_cast<float>(nx)}, "dct_rows", s);
}

}  // namespace qh
