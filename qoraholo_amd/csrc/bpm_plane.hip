// Beam propagation of small planes: one block per illumination marches all slices.
//
// The slice kernels of bpm_kernels.hpp take two dependent launches per slice, of 4.5 to 6 us each
// up to 64^2 however little there is to do. Here a block keeps the plane of its illumination in
// LDS and the propagation state of each bin in the registers of the thread that holds it, and goes
// through the slices with barriers only. The lines run on the same engines with the same
// operations, so the results are those of the slice kernels bit for bit. What bounds it: the
// vector work of a plane on one CU. 64 slices of 64^2: forward 610 -> 319 us, vjp 1221 -> 687 us
// with 1 illumination, 625 -> 318 and 1339 -> 713 us with 49; 20 slices with 700 (three rounds of
// the CUs): forward 611 -> 328, vjp 1870 -> 860 us; 36^2 with 9: 219 -> 116 and 426 -> 220 us.
#include "bpm_plane.hpp"

#include <algorithm>

#include "common.hpp"
#include "fft.hpp"
#include "fft_engine.hpp"
#include "split_lines.hpp"

namespace qh {

namespace {

// Row and column engines of a whole plane, and the LDS they share: the plane in natural order
// lies in the engines' exchange buffer, which is free between transforms.
template <class R, class C>
struct PlaneEngines {
  using Rows = R;
  using Cols = C;
  static constexpr int N = R::N;
  static constexpr int kBlock = R::kBlock;
  static_assert(R::kBlock == C::kBlock && R::LINES == N && C::LINES == N, "one plane per block");
  static constexpr int kLds = std::max(std::max(R::kLds, C::kLds), N * N);
};

template <class E>
__device__ __forceinline__ void store_plane(E& e, float2* plane, bool rows) {
  __syncthreads();
  e.store2([&](long l, int m, float2 v) { plane[rows ? l * E::N + m : m * E::N + l] = v; });
  __syncthreads();
}

template <class P>
__global__ void __launch_bounds__(P::kBlock) k_bpm_plane_fwd(BpmPlaneArgs a) {
  constexpr int N = P::N;
  constexpr long kPlane = static_cast<long>(N) * N;
  __shared__ float2 plane[P::kLds];
  __shared__ float2 tw_rows[P::Rows::kTw];
  __shared__ float2 tw_cols[P::Cols::kTw];
  typename P::Rows er(plane, tw_rows, a.tw);
  typename P::Cols ec(plane, tw_cols, a.tw);
  const long image = static_cast<long>(blockIdx.x) * kPlane;
  constexpr int KC = P::Cols::kBins;
  constexpr int KR = P::Rows::kBins;
  // The state, propagator and weight of the thread's bins.
  float2 s[KC], c[KC];
  float q[KC];
  ec.bins([&](int i, long l, int ky, float2&) {
    const long x = image + static_cast<long>(ky) * N + l;
    s[i] = (ky == 0 && l == 0) ? float2{static_cast<float>(kPlane), 0.0f} : float2{0.0f, 0.0f};
    c[i] = a.step[x];
    q[i] = a.q[x];
  });
  __syncthreads();
  for (int k = 0; k < a.nz; ++k) {
    const float2* const screen = a.screen + k * kPlane;
    float2* const w = a.w ? a.w + k * a.w_slice + image : nullptr;
    if (k == 0) {
      er.load([&](long l, int i) {
        if (w) w[l * N + i] = float2{1.0f, 0.0f};
        return screen[l * N + i];
      });
      er.first(false);
      __syncthreads();
      er.store1([&](long l, int m, float2 v) { plane[l * N + m] = v; });
      __syncthreads();
    } else {
      float2 t[KR];
      er.bins([&](int i, long l, int x, float2&) { t[i] = screen[l * N + x]; });
      er.load([&](long l, int i) { return plane[l * N + i]; });
      er.first(true);
      er.bins([&](int i, long l, int x, float2& v) {
        const float2 e = cscale(v, a.inv);
        if (w) w[l * N + x] = e;
        v = cmul(t[i], e);
      });
      er.second(false);
      store_plane(er, plane, true);
    }
    if (k == a.nz - 1) {
      ec.bins([&](int i, long l, int ky, float2&) { c[i] = a.last[image + static_cast<long>(ky) * N + l]; });
    }
    ec.load([&](long l, int i) { return plane[i * N + l]; });
    ec.first(false);
    ec.bins([&](int i, long, int, float2& v) {
      bpm_step(c[i].x, c[i].y, q[i], v.x, v.y, s[i].x, s[i].y);
      v = s[i];
    });
    ec.second(true);
    if (k == a.nz - 1) {
      ec.store2([&](long l, int m, float2 v) { a.out[image + static_cast<long>(m) * N + l] = v; });
    } else {
      store_plane(ec, plane, false);
    }
  }
}

// The adjoint from the forward x transform of the residual. The gradient term of a voxel replaces
// its envelope (the real part of the pair), for k_bpm_plane_reduce.
template <class P>
__global__ void __launch_bounds__(P::kBlock) k_bpm_plane_adj(BpmPlaneArgs a) {
  constexpr int N = P::N;
  constexpr long kPlane = static_cast<long>(N) * N;
  __shared__ float2 plane[P::kLds];
  __shared__ float2 tw_rows[P::Rows::kTw];
  __shared__ float2 tw_cols[P::Cols::kTw];
  typename P::Rows er(plane, tw_rows, a.tw);
  typename P::Cols ec(plane, tw_cols, a.tw);
  const long image = static_cast<long>(blockIdx.x) * kPlane;
  constexpr int KC = P::Cols::kBins;
  constexpr int KR = P::Rows::kBins;
  float2 g[KC], c[KC];
  float q[KC];
  ec.bins([&](int i, long l, int ky, float2&) {
    const long x = image + static_cast<long>(ky) * N + l;
    c[i] = a.last[x];
    q[i] = a.q[x];
  });
  __syncthreads();
  for (int k = a.nz - 1; k >= 0; --k) {
    const bool first = k == a.nz - 1;
    const float2* const screen = a.screen + k * kPlane;
    float2* const w = a.w + k * a.w_slice + image;
    float2 t[KR], e[KR];
    er.bins([&](int i, long l, int x, float2&) {
      t[i] = screen[l * N + x];
      e[i] = w[l * N + x];
    });
    if (first) {
      ec.load([&](long l, int i) { return a.in[image + static_cast<long>(i) * N + l]; });
    } else {
      ec.load([&](long l, int i) { return plane[i * N + l]; });
    }
    ec.first(false);
    ec.bins([&](int i, long, int, float2& v) {
      float gre = v.x;
      float gim = v.y;
      if (!first) {
        gre = g[i].x + v.x;
        gim = g[i].y + v.y;
      }
      float are = 0.0f;
      float aim = 0.0f;
      bpm_step_adjoint(c[i].x, c[i].y, q[i], gre, gim, are, aim);
      g[i] = float2{gre, gim};
      v = float2{are, aim};
    });
    if (first) {
      ec.bins([&](int i, long l, int ky, float2&) { c[i] = a.step[image + static_cast<long>(ky) * N + l]; });
    }
    ec.second(true);
    store_plane(ec, plane, false);
    er.load([&](long l, int i) { return plane[l * N + i]; });
    er.first(true);
    er.bins([&](int i, long l, int x, float2& v) {
      const float2 b = cscale(v, a.inv);
      const float2 tw = cmul(t[i], e[i]);
      w[l * N + x].x = a.phase * (tw.x * b.y - tw.y * b.x);
      v = cmul(cconj(t[i]), b);
    });
    if (k > 0) {
      er.second(false);
      store_plane(er, plane, true);
    }
  }
}

// grad[k][i] += the terms of illuminations 0 .. chunk-1 in order (from 0 with init).
__global__ void __launch_bounds__(256) k_bpm_plane_reduce(const float2* w, int chunk, long plane,
                                                          long w_slice, long total, float* grad,
                                                          int init) {
  const long o = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (o >= total) return;
  const long k = o / plane;
  const float2* const p = w + k * w_slice + (o - k * plane);
  float g = init ? 0.0f : grad[o];
  int b = 0;
  for (; b + 8 <= chunk; b += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[(b + u) * plane].x;
#pragma unroll
    for (int u = 0; u < 8; ++u) g += v[u];
  }
  for (; b < chunk; ++b) g += p[b * plane].x;
  grad[o] = g;
}

// The engines of a side: four-step lines where the slice kernels have them.
template <int N>
struct Engines {
  using type = PlaneEngines<SplitLines<N, false, N>, SplitLines<N, true, N>>;
};
template <int N1, int N2>
using FourStep = PlaneEngines<RegLines<N1, N2, false, (N1 > N2 ? N1 : N2) * N1 * N2>,
                              RegLines<N1, N2, true, (N1 > N2 ? N1 : N2) * N1 * N2>>;
template <>
struct Engines<32> { using type = FourStep<8, 4>; };
template <>
struct Engines<48> { using type = FourStep<8, 6>; };
template <>
struct Engines<64> { using type = FourStep<8, 8>; };

// f.template operator()<P>() with the engines of side n; false for the other sides. Planes up to
// 64^2: those of 72 and 80 take 648 and 800 threads, whose registers spill (20 slices with 9
// illuminations: 250 against 244 us and 356 against 242 us with the slice kernels).
template <class F>
bool with_plane(int n, F f) {
  switch (n) {
#define QH_PLANE(N) \
  case N: f.template operator()<typename Engines<N>::type>(); return true;
    QH_PLANE(32) QH_PLANE(36) QH_PLANE(40) QH_PLANE(48) QH_PLANE(50) QH_PLANE(54) QH_PLANE(60)
    QH_PLANE(64)
#undef QH_PLANE
    default: return false;
  }
}

}  // namespace

bool bpm_plane_supported(int n) {
  return with_plane(n, []<class P>() {});
}

void bpm_plane_forward(int n, int count, const BpmPlaneArgs& a, hipStream_t s) {
  require(with_plane(n, [&]<class P>() {
            hipLaunchKernelGGL(k_bpm_plane_fwd<P>, dim3(count), dim3(P::kBlock), 0, s, a);
          }),
          "bpm: no plane kernel for this side");
  check_launch("bpm_plane_fwd");
}

void bpm_plane_adjoint(int n, int count, const BpmPlaneArgs& a, float* grad, bool init,
                       hipStream_t s) {
  require(with_plane(n, [&]<class P>() {
            hipLaunchKernelGGL(k_bpm_plane_adj<P>, dim3(count), dim3(P::kBlock), 0, s, a);
          }),
          "bpm: no plane kernel for this side");
  check_launch("bpm_plane_adj");
  const long plane = static_cast<long>(n) * n;
  const long total = plane * a.nz;
  hipLaunchKernelGGL(k_bpm_plane_reduce, dim3(blocks_for(total)), dim3(256), 0, s, a.w, count,
                     plane, a.w_slice, total, grad, init ? 1 : 0);
  check_launch("bpm_plane_reduce");
}

}  // namespace qh
