// The part of a Gerchberg-Papoulis step within a z plane, for planes that fit one block.
//
// Between two z passes every plane of the half spectrum goes through the inverse y transform, the
// inverse real x transform, max(., 0), and both transforms forward: four dependent passes over the
// plane (three launches of 7 us each at 128^3). Here one block keeps the plane in LDS and takes all
// of them with barriers only; the lines run on the engines of the separate passes.
//
// The columns of bins 0 and m = n / 2 go through the y transforms as one. The x transform takes the
// real parts of both and returns real values for both, so the inverse transform of
// H(X_0) + i H(X_m), with H the part of a column whose inverse transform is real, holds the one in
// its real and the other in its imaginary part, and the forward transform of such a pair splits the
// same way. That leaves m columns of n points and n rows of m packed points, the same number of
// threads for both at 64, 96 and 128.
#include "gp_plane.hpp"

#include <algorithm>

#include "common.hpp"
#include "fft.hpp"
#include "fft_args.hpp"
#include "fft_engine.hpp"
#include "runtime.hpp"

namespace qh {

namespace {

struct PlaneArgs {
  float2* e;         // (planes, n, m + 1)
  const float2* tw;  // exp(-2 pi i t / n)
  const float2* twm; // exp(-2 pi i t / m)
  float scale;
};

// Column engine C (n points), row engine R (m = n / 2 packed points), of the same block size.
template <class C_, class R_>
struct Engines {
  using C = C_;
  using R = R_;
  static constexpr int N = C::N;
  static constexpr int M = R::N;
  static constexpr int kBlock = C::kBlock;
  static_assert(N == 2 * M && C::LINES >= M && R::LINES == N && R::kBlock == kBlock, "one plane");
  // The plane in LDS between transforms: n rows of m bins, whose start moves 8 bins over the 32
  // bin-wide banks from row to row, so that the 8 rows of a wave's 8 threads each use them all.
  static constexpr int kPitch = M + 8;
  static constexpr int kLds = std::max({C::kLds, R::kLds, N * kPitch});
};

// real_pack and real_bin of the bins between 0 and m, without their tests (bin 0 reads the unset
// element m of its row for them, and drops the result).
__device__ __forceinline__ float2 packed(float2 xk, float2 xm, float2 w) {
  const float2 d = csub(xk, cconj(xm));
  const float2 wd = cmul(cconj(w), d);
  return cadd(cadd(xk, cconj(xm)), float2{-wd.y, wd.x});
}
__device__ __forceinline__ float2 bin(float2 zk, float2 zmk, float2 w) {
  const float2 zm = cconj(zmk);
  const float2 d = {0.5f * (zk.x - zm.x), 0.5f * (zk.y - zm.y)};
  const float2 od = cmul(w, d);
  return cadd(float2{0.5f * (zk.x + zm.x), 0.5f * (zk.y + zm.y)}, float2{od.y, -od.x});
}

template <class P>
__global__ void __launch_bounds__(P::kBlock) k_gp_plane(PlaneArgs a) {
  constexpr int N = P::N;
  constexpr int M = P::M;
  constexpr int kPitch = P::kPitch;
  using C = typename P::C;
  using R = typename P::R;
  __shared__ float2 lds[P::kLds];
  __shared__ float2 tw_cols[C::kTw];
  __shared__ float2 tw_rows[R::kTw];
  __shared__ float2 twn[M];
  __shared__ float2 pair[N];
  float2* const e = a.e + static_cast<long>(blockIdx.x) * N * (M + 1);
  C ec(lds, tw_cols, a.tw);
  R er(lds, tw_rows, a.twm);
  ec.valid = ec.line < M;
  for (int i = static_cast<int>(threadIdx.x); i < M; i += P::kBlock) twn[i] = a.tw[i];
  // Column 0 with column m: ((A + conj A(-k)) + i (B + conj B(-k))) / 2.
  const auto negative = [](int k) { return k == 0 ? 0 : N - k; };
  ec.load([&](long l, int i) { return e[i * (M + 1) + l]; });
  if (ec.line == 0 && ec.j < C::kFirst) {
    float2 b[C::kSamples], an[C::kSamples], bn[C::kSamples];
#pragma unroll
    for (int u = 0; u < C::kSamples; ++u) {
      const int i = ec.j + C::kFirst * u;
      b[u] = e[i * (M + 1) + M];
      an[u] = e[negative(i) * (M + 1)];
      bn[u] = e[negative(i) * (M + 1) + M];
    }
#pragma unroll
    for (int u = 0; u < C::kSamples; ++u) {
      const float2 p = {ec.v[u].x + an[u].x, ec.v[u].y - an[u].y};
      const float2 q = {b[u].x + bn[u].x, b[u].y - bn[u].y};
      ec.v[u] = {0.5f * (p.x - q.y), 0.5f * (p.y + q.x)};
    }
  }
  ec.first(true);
  __syncthreads();
  ec.store1([&](long l, int y, float2 v) { lds[y * kPitch + l] = v; });
  __syncthreads();
  er.load([&](long y, int k) {
    const float2* const row = lds + y * kPitch;
    const float2 x = row[k];
    const float2 p = packed(x, row[M - k], twn[k]);
    return k == 0 ? float2{x.x + x.y, x.x - x.y} : p;
  });
  er.first(true);
  er.mid([&](long, int, float2& v) { v = scale_nonneg(v, a.scale); });
  er.second(false);
  __syncthreads();
  er.store2([&](long y, int k, float2 v) { lds[y * kPitch + k] = v; });
  __syncthreads();
  ec.load([&](long l, int y) {
    const int k = static_cast<int>(l);
    const float2* const row = lds + y * kPitch;
    const float2 z = row[k];
    const float2 x = bin(z, row[M - k], twn[k]);
    return k == 0 ? float2{z.x + z.y, z.x - z.y} : x;
  });
  ec.first(false);
  ec.store1([&](long l, int k, float2 v) {
    if (l == 0) {
      pair[k] = v;
    } else {
      e[k * (M + 1) + l] = v;
    }
  });
  __syncthreads();
  for (int k = static_cast<int>(threadIdx.x); k < N; k += P::kBlock) {
    const float2 c = pair[k];
    const float2 d = pair[negative(k)];
    e[k * (M + 1)] = {0.5f * (c.x + d.x), 0.5f * (c.y - d.y)};
    e[k * (M + 1) + M] = {0.5f * (c.y + d.y), 0.5f * (d.x - c.x)};
  }
}

// f.template operator()<P>() with the engines of side n; false for other sides. Both engines of a
// side here take the same number of threads. Those of 72, 80, 90, 108 and 120 do not (72: 324 for
// the columns, 648 for the rows), and 100 (1000 for both) has not been tried: these sides go through
// the three launches, at about the time of their neighbours (an iteration at 72^3 / 80^3 / 96^3 22 /
// 23 / 23 us, at 100^3 / 108^3 / 120^3 / 128^3 33 / 32 / 38 / 33 us).
template <class F>
bool with_plane(int n, F f) {
  switch (n) {
    case 64: f.template operator()<Engines<RegLines<8, 8, true, 512>, RegLines<8, 4, false, 512>>>(); return true;
    case 96: f.template operator()<Engines<RegLines<16, 6, true, 768>, RegLines<8, 6, false, 768>>>(); return true;
    case 128: f.template operator()<Engines<RegLines<16, 8, true, 1024>, RegLines<8, 8, false, 1024>>>(); return true;
    default: return false;
  }
}

}  // namespace

bool gp_plane(float2* e, long planes, int n, float scale, hipStream_t s) {
  const bool ran = with_plane(n, [&]<class P>() {
    const PlaneArgs a{e, fft_twiddles(n), fft_twiddles(n / 2), scale};
    hipLaunchKernelGGL(k_gp_plane<P>, dim3(static_cast<unsigned>(planes)), dim3(P::kBlock), 0, s, a);
  });
  if (ran) check_launch("gp_plane");
  return ran;
}

}  // namespace qh
