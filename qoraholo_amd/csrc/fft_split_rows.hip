// Real row transforms for the lengths without a four-step kernel, on the register engine of
// split_lines.hpp: the operations and bits of the LDS kernels of fft.hip, which remain for the
// lengths whose groups do not fit.
#include <algorithm>

#include "common.hpp"
#include "fft_args.hpp"
#include "fft_rows_roundtrip.hpp"
#include "runtime.hpp"
#include "split_lines.hpp"

namespace qh {

namespace {

// Real rows of n = 2 M (see k_rfft_rows and k_irfft_rows of fft.hip). The bins of a row lie in the
// engine's exchange buffer, which holds more than M + 1 of them.
template <class E>
__global__ void __launch_bounds__(E::kBlock) k_split_rfft_rows(RowsArgs a, LineGeom g) {
  constexpr int M = E::N;
  E e(g);
  // All loads of a thread before the first use (the operation is uniform over the grid).
  e.load([&](long l, int i) { return *reinterpret_cast<const float2*>(a.x + l * a.x_pitch + 2 * i); });
  if (a.op.in == RealIn::momentum) {
    float2 q[E::N1];
#pragma unroll
    for (int i = 0; i < E::N1; ++i) {
      q[i] = (e.valid && e.j < E::N2)
                 ? *reinterpret_cast<const float2*>(a.x2 + e.l * a.x_pitch + 2 * (e.j + E::N2 * i))
                 : float2{0.0f, 0.0f};
    }
#pragma unroll
    for (int i = 0; i < E::N1; ++i) {
      e.v[i].x = e.v[i].x + a.op.a * (e.v[i].x - q[i].x);
      e.v[i].y = e.v[i].y + a.op.a * (e.v[i].y - q[i].y);
    }
  }
  e.first(false);
  float2* const row = e.t + e.line * E::kLine;
  __syncthreads();
  e.store1([&](long, int k, float2 v) { row[k] = v; });
  __syncthreads();
  if (!e.valid) return;
  for (int k = e.j; k <= M; k += E::T) {
    a.c[e.l * a.c_pitch + k] =
        real_bin(row[k == M ? 0 : k], row[k == 0 ? 0 : M - k], a.tw[k], k, M);
  }
}

template <class E>
__global__ void __launch_bounds__(E::kBlock) k_split_irfft_rows(RowsArgs a, LineGeom g) {
  constexpr int M = E::N;
  E e(g);
  float2* const row = e.t + e.line * E::kLine;
  if (e.valid) {
    for (int k = e.j; k <= M; k += E::T) row[k] = a.c[e.l * a.c_pitch + k];
  }
  __syncthreads();
  e.load([&](long, int k) {
    return real_pack(row[k], row[M - k], a.tw[k], k);
  });
  e.first(true);
  e.store1([&](long l, int m, float2 v) {
    float u0 = v.x * a.op.a;
    float u1 = v.y * a.op.a;
    if (a.op.out == RealOut::index) {
      u0 = index_from_real(u0, a.op.nm2, a.op.inv_k02);
      u1 = index_from_real(u1, a.op.nm2, a.op.inv_k02);
    }
    *reinterpret_cast<float2*>(a.xo + l * a.x_pitch + 2 * m) = float2{u0, u1};
  });
}

// About 256 threads a block.
template <int N>
using RowEngine = SplitLines<N, false, std::max(1, 256 / SplitLines<N, false, 1>::T)>;

template <int N>
struct LaunchRows {
  static void run(const RowsArgs& a, bool inverse, hipStream_t s) {
    using E = RowEngine<N>;
    const LineGeom g = row_geometry(N, a.rows);
    if (inverse) {
      hipLaunchKernelGGL(k_split_irfft_rows<E>, dim3(E::grid(g.lines)), dim3(E::kBlock), 0, s, a, g);
    } else {
      hipLaunchKernelGGL(k_split_rfft_rows<E>, dim3(E::grid(g.lines)), dim3(E::kBlock), 0, s, a, g);
    }
  }
};

template <int N>
struct LaunchRoundtrip {
  static void run(const RowsArgs& a, hipStream_t s) { launch_rows_roundtrip<RowEngine<N>>(a, s); }
};

// F<M>::run(args...) for half lengths M with an engine; false for the others. Odd halves are row
// lengths alone: 50, 54, 90, ... have them.
template <template <int> class F, class... Args>
bool with_half(int m, Args&&... args) {
  switch (m) {
#define QH_SPLIT_CASE(N) \
  case N:                \
    F<N>::run(args...);  \
    return true;
    QH_SPLIT_CASE(25) QH_SPLIT_CASE(27) QH_SPLIT_CASE(30) QH_SPLIT_CASE(45) QH_SPLIT_CASE(75)
    QH_SPLIT_CASE(81) QH_SPLIT_CASE(125) QH_SPLIT_CASE(135) QH_SPLIT_CASE(225) QH_SPLIT_CASE(243)
#undef QH_SPLIT_CASE
    default: return with_split<F>(m, args...);
  }
}

}  // namespace

bool split_rfft_rows(const RowsArgs& a, bool inverse, hipStream_t s) {
  return with_half<LaunchRows>(a.n / 2, a, inverse, s);
}

bool split_rows_roundtrip(const RowsArgs& a, hipStream_t s) {
  return with_half<LaunchRoundtrip>(a.n / 2, a, s);
}

}  // namespace qh
