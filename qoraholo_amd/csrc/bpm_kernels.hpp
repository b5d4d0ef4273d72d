// The line kernels of the beam propagation model, written once over the line engines
// (fft_engine.hpp, split_lines.hpp), and their launch with one of them. See bpm.hip.
#pragma once

#include "bpm.hpp"
#include "common.hpp"
#include "fft.hpp"
#include "fft_engine.hpp"

namespace qh {

struct BpmModel::Args {
  LineGeom g;
  const float2* in;
  float2* out;
  const float2* screen;  // exp(i phase x) of the slice, (n, n)
  float2* w;             // envelopes of the chunk for this slice, or null
  const float2* data;    // measured fields of the chunk (residual), or null
  double* loss;          // per-line data term of the chunk
  const float2* s_in;    // spectrum in front of the slice; null: the unit envelope
  float2* s_out;
  float2* g_state;       // adjoint state, (chunk, n, n)
  float* p;              // per-illumination gradient terms, (chunk, n, n)
  const float2* c;       // propagator of the slice from the chunk's first illumination
  const float* q;
  float inv;             // 1 / n^2
  float phase;
  int first;             // adjoint: the first slice processed (no state yet)
  int s_zero;            // columns with s_in == null: the state in front of slice 0 is zero
                         // (the tangent), not the unit envelope
  const float* h;        // tangent direction of the slice, (n, n)
  // Adjoint columns also sum the gradient terms of the slice processed before (red_p, left by
  // the previous rows launch) into red_grad, in blocks after the line blocks; red_init: the
  // first chunk, whose sum starts from zero rather than from red_grad.
  const float* red_p;
  float* red_grad;
  int red_chunk;
  int red_blocks;
  int red_init;
  int line_blocks;  // with red_blocks: the grid's first line_blocks blocks run the lines
};

enum class BpmKind { rows_fwd, rows_out, rows_adj, rows_jvp, cols_fwd, cols_adj };

// The kernel for lines of a length of with_split (split_lines.hpp); false for other lengths.
bool bpm_split_rows(BpmKind k, const BpmModel::Args& a, hipStream_t s);
bool bpm_split_cols(BpmKind k, const BpmModel::Args& a, hipStream_t s);

namespace {

using Args = BpmModel::Args;

// Side of the lines of engine E: a compile-time constant for the register engines, so that the
// line arithmetic below compiles to multiplications; the LDS engine's lines have any length.
template <class E>
__device__ __forceinline__ int line_side(int n) {
  if constexpr (requires { E::N; }) {
    return E::N;
  } else {
    return n;
  }
}

// Row (or column) r of line l = b n + r within its illumination's plane, in 32-bit arithmetic
// (a chunk holds far fewer than 2^31 lines; 64-bit remainders by a runtime n had been expanded
// once per element).
template <class E>
__device__ __forceinline__ int line_in_plane(long l, int n) {
  return static_cast<int>(static_cast<unsigned>(l) % static_cast<unsigned>(line_side<E>(n)));
}

// Envelopes are stored for the adjoint, which reads them back only after the rest of their
// segment has been recomputed and every other plane of it has passed through the caches:
// written non-temporally they displace nothing that the next kernels read (384/81 gradient
// 189 -> 184 ms, 256/49 30.8 -> 30.4 ms; the same hint on the propagation state, which the
// next slice reads, was slower at 256, where that state stays in the MALL).
__device__ __forceinline__ void store_envelope(float2* p, float2 v) {
  typedef float vec2 __attribute__((ext_vector_type(2)));
  __builtin_nontemporal_store(vec2{v.x, v.y}, reinterpret_cast<vec2*>(p));
}

// Bins whose operands the slice kernels load together before using any of them (mid_loaded):
// 8 for lines of 384 and more (384/81 gradient 210 -> 191 ms; its column blocks hold one block
// per CU either way), 4 for shorter lines, where 8 would take the 256-point column kernels past
// 128 registers and one of their two blocks per CU (256/49 gradient 32.4 -> 30.7 ms with 4, 32.8
// with 8). Same results bit for bit.
template <class E>
constexpr int mid_group() {
  if constexpr (requires { E::N; }) {
    return E::N >= 384 ? 8 : 4;
  } else {
    return 1;
  }
}

// Whether the adjoint rows load their operands, from memory that no recent kernel has touched
// (the envelopes), before the first transform: up to 192, where that fits the registers of four
// waves per SIMD (adjoint of 96 slices of 128^2 with 9 illuminations 1370 -> 1275 us, with 25 1535
// -> 1466 us; 64 of 192^2 with 49 2055 -> 2000 us; of 256^2 with 49 3077 -> 3139 us). The other
// kernels, whose operands the caches hold, gained nothing by it or lost waves to the registers
// (columns at 256: 2317 -> 2715 us). Nor did the two-group lines, whose threads hold more bins: a
// gradient at 72^2 x 48 1.22 -> 1.25 ms, at 120^2 1.58 -> 1.57, at 160^2 2.00 -> 2.26, at 240^2 2.96
// -> 3.35.
template <class E>
constexpr bool operands_ahead() {
  if constexpr (requires { E::kMatrix; }) {  // the four-step engine
    return E::N <= 192;
  } else {
    return false;
  }
}

// Rows (line l = b n + y, element i at l n + i): inverse x transform of T, envelope, screen,
// forward x transform. in == null: the unit envelope of the first slice. out == null: store the
// envelope only.
template <class E>
__global__ void __launch_bounds__(E::kBlock) k_bpm_rows_fwd(Args a) {
  E e(a.g);
  const int n = a.g.n;
  if (a.in == nullptr) {
    e.load([&](long l, int i) {
      if (a.w) a.w[l * n + i] = float2{1.0f, 0.0f};
      return a.screen[line_in_plane<E>(l, n) * n + i];
    });
    if (a.out == nullptr) return;
    e.first(false);
    e.store1([&](long l, int k, float2 v) { a.out[l * n + k] = v; });
    return;
  }
  e.load([&](long l, int i) { return a.in[l * n + i]; });
  e.first(true);
  e.template mid_loaded<mid_group<E>()>(
      [&](long l, int k) { return a.screen[line_in_plane<E>(l, n) * n + k]; },
      [&](long l, int k, float2& v, float2 t) {
        const float2 w = cscale(v, a.inv);
        if (a.w) store_envelope(a.w + l * n + k, w);
        v = cmul(t, w);
      });
  if (a.out == nullptr) return;
  e.second(false);
  e.store2([&](long l, int m, float2 v) { a.out[l * n + m] = v; });
}

// Tangent rows (bpm_jvp, src/cpu/bpm.cpp:141-176): inverse x transform of the tangent dT,
// dw = dT / n^2, dv = t (dw + i phase h w) with the envelope w the primal rows stored for this
// slice, forward x transform. in == null: dw = 0 (the first slice).
template <class E>
__global__ void __launch_bounds__(E::kBlock) k_bpm_rows_jvp(Args a) {
  E e(a.g);
  const int n = a.g.n;
  // The complex operations of the reference, in its order: (0, phase h) w, + dw, t times that.
  const auto tangent = [&](long l, int k, float2 dw) {
    const float2 w = a.w[l * n + k];
    const float p = a.phase * a.h[line_in_plane<E>(l, n) * n + k];
    const float2 d{dw.x + (0.0f * w.x - p * w.y), dw.y + (0.0f * w.y + p * w.x)};
    return cmul(a.screen[line_in_plane<E>(l, n) * n + k], d);
  };
  if (a.in == nullptr) {
    e.load([&](long l, int i) { return tangent(l, i, float2{0.0f, 0.0f}); });
    e.first(false);
    e.store1([&](long l, int k, float2 v) { a.out[l * n + k] = v; });
    return;
  }
  e.load([&](long l, int i) { return a.in[l * n + i]; });
  e.first(true);
  e.mid([&](long l, int k, float2& v) { v = tangent(l, k, cscale(v, a.inv)); });
  e.second(false);
  e.store2([&](long l, int m, float2 v) { a.out[l * n + m] = v; });
}

// Column lines: element i of line l = b n + c at b n^2 + i n + c. The division takes the runtime
// n: with the compile-time side the 384-point column kernel ran 10% slower (measured).
template <class E>
__device__ __forceinline__ long col_at(long l, int i, int n, long plane) {
  const unsigned m = static_cast<unsigned>(n);
  const unsigned lu = static_cast<unsigned>(l);
  const unsigned b = lu / m;
  return static_cast<long>(b) * plane + static_cast<long>(i) * m + (lu - b * m);
}

// Columns (line l = b n + kx, element i at b n^2 + i n + kx): forward y transform, propagation
// step S = c (q A + (1 - q) S) (src/common.hpp:158-163), inverse y transform.
template <class E>
__global__ void __launch_bounds__(E::kBlock) k_bpm_cols_fwd(Args a) {
  E e(a.g);
  const int n = a.g.n;
  const long plane = static_cast<long>(n) * n;
  e.load([&](long l, int i) { return a.in[col_at<E>(l, i, n, plane)]; });
  e.first(false);
  // Operands of a bin: the state S in front of the slice, the propagator c and the weight q.
  struct Ops {
    float2 s, c;
    float q;
  };
  e.template mid_loaded<mid_group<E>()>(
      [&](long l, int ky) {
        const long x = col_at<E>(l, ky, n, plane);
        Ops o;
        if (a.s_in) {
          o.s = a.s_in[x];
        } else if (a.s_zero) {
          o.s = float2{0.0f, 0.0f};
        } else {
          o.s = (ky == 0 && line_in_plane<E>(l, n) == 0) ? float2{static_cast<float>(plane), 0.0f}
                                                          : float2{0.0f, 0.0f};
        }
        o.c = a.c[x];
        o.q = a.q[x];
        return o;
      },
      [&](long l, int ky, float2& v, Ops o) {
        bpm_step(o.c.x, o.c.y, o.q, v.x, v.y, o.s.x, o.s.y);
        a.s_out[col_at<E>(l, ky, n, plane)] = o.s;
        v = o.s;
      });
  if (a.out == nullptr) return;
  e.second(true);
  e.store2([&](long l, int m, float2 v) { a.out[col_at<E>(l, m, n, plane)] = v; });
}

// Rows after the last slice: y = inverse x transform / n^2. Without data, y is the output;
// with data, r = y - d, the per-row data term, and the forward x transform of r, the first
// half of the transform that starts the adjoint.
template <class E>
__global__ void __launch_bounds__(E::kBlock) k_bpm_rows_out(Args a) {
  E e(a.g);
  const int n = a.g.n;
  e.load([&](long l, int i) { return a.in[l * n + i]; });
  e.first(true);
  if (a.data == nullptr) {
    e.store1([&](long l, int k, float2 v) { a.out[l * n + k] = cscale(v, a.inv); });
    return;
  }
  e.mid([&](long l, int k, float2& v) {
    const float2 y = cscale(v, a.inv);
    const float2 d = a.data[l * n + k];
    v = float2{y.x - d.x, y.y - d.y};
  });
  e.reduce_lines(
      [&](long, int, const float2& v) {
        const double re = v.x;
        const double im = v.y;
        return re * re + im * im;
      },
      a.loss);
  e.second(false);
  e.store2([&](long l, int m, float2 v) { a.out[l * n + m] = v; });
}

// grad[i] += p[b][i] for b = 0 .. chunk-1 in order (from 0 instead of grad[i] with init, the
// same bits as adding to a zeroed grad); the loads of eight illuminations are issued together
// so that each thread keeps several in flight.
__device__ __forceinline__ void reduce_terms(const float* p, int chunk, long plane, float* grad,
                                             bool init, long i) {
  float g = init ? 0.0f : grad[i];
  int b = 0;
  for (; b + 8 <= chunk; b += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[(b + u) * plane + i];
#pragma unroll
    for (int u = 0; u < 8; ++u) g += v[u];
  }
  for (; b < chunk; ++b) g += p[b * plane + i];
  grad[i] = g;
}

// Adjoint columns: forward y transform completes back = FFT2(conj(t) b) of the slice above (or
// FFT2(r) on the first slice processed); with the carried g, U = conj(c) (g + back), g <- (1-q) U,
// b = q U (src/common.hpp:168-176); inverse y transform of b.
template <class E>
__global__ void __launch_bounds__(E::kBlock) k_bpm_cols_adj(Args a) {
  const int nb = a.red_blocks > 0 ? a.line_blocks : static_cast<int>(gridDim.x);
  if (static_cast<int>(blockIdx.x) >= nb) {
    // A reduction block (the last red_blocks of the grid, dealt to the XCDs in turn after the
    // line blocks): the previous slice's gradient terms, one plane element per thread.
    const long plane = static_cast<long>(a.g.n) * a.g.n;
    const long i = static_cast<long>(static_cast<int>(blockIdx.x) - nb) * E::kBlock + threadIdx.x;
    if (i < plane) reduce_terms(a.red_p, a.red_chunk, plane, a.red_grad, a.red_init != 0, i);
    return;
  }
  E e(a.g, nb);
  const int n = a.g.n;
  const long plane = static_cast<long>(n) * n;
  e.load([&](long l, int i) { return a.in[col_at<E>(l, i, n, plane)]; });
  e.first(false);
  // Operands of a bin: the carried adjoint state g, the propagator c and the weight q.
  struct Ops {
    float2 g, c;
    float q;
  };
  e.template mid_loaded<mid_group<E>()>(
      [&](long l, int ky) {
        const long x = col_at<E>(l, ky, n, plane);
        Ops o;
        o.g = a.first ? float2{0.0f, 0.0f} : a.g_state[x];
        o.c = a.c[x];
        o.q = a.q[x];
        return o;
      },
      [&](long l, int ky, float2& v, Ops o) {
        float gre = v.x;
        float gim = v.y;
        if (!a.first) {
          gre = o.g.x + v.x;
          gim = o.g.y + v.y;
        }
        float are = 0.0f;
        float aim = 0.0f;
        bpm_step_adjoint(o.c.x, o.c.y, o.q, gre, gim, are, aim);
        a.g_state[col_at<E>(l, ky, n, plane)] = float2{gre, gim};
        v = float2{are, aim};
      });
  e.second(true);
  e.store2([&](long l, int m, float2 v) { a.out[col_at<E>(l, m, n, plane)] = v; });
}

// Adjoint rows: b = inverse x transform / n^2; gradient term phase Im(conj(t w) b) per
// illumination; back = conj(t) b and its forward x transform (skipped on slice 0). Four waves
// per SIMD: the 384-point kernel otherwise takes 129 registers, one over the limit for four.
template <class E>
__global__ void __launch_bounds__(E::kBlock) __attribute__((amdgpu_waves_per_eu(4)))
k_bpm_rows_adj(Args a) {
  E e(a.g);
  const int n = a.g.n;
  e.load([&](long l, int i) { return a.in[l * n + i]; });
  // Operands of a bin: the screen t and the stored envelope w.
  struct Ops {
    float2 t, w;
  };
  const auto operands = [&](long l, int k) {
    return Ops{a.screen[line_in_plane<E>(l, n) * n + k], a.w[l * n + k]};
  };
  const auto term = [&](long l, int k, float2& v, Ops o) {
    const float2 b = cscale(v, a.inv);
    const float2 tw = cmul(o.t, o.w);
    a.p[l * n + k] = a.phase * (tw.x * b.y - tw.y * b.x);
    v = cmul(cconj(o.t), b);
  };
  if constexpr (operands_ahead<E>()) {
    Ops o[E::kBins];
    e.bins([&](int i, long l, int k, float2&) { o[i] = operands(l, k); });
    e.first(true);
    e.bins([&](int i, long l, int k, float2& v) { term(l, k, v, o[i]); });
  } else {
    e.first(true);
    e.template mid_loaded<mid_group<E>()>(operands, term);
  }
  if (a.out == nullptr) return;
  e.second(false);
  e.store2([&](long l, int m, float2 v) { a.out[l * n + m] = v; });
}

template <bool ROWS, class E>
void launch_with(BpmKind k, Args a, unsigned grid, std::size_t lds, hipStream_t s) {
  if constexpr (ROWS) {
    switch (k) {
      case BpmKind::rows_fwd: hipLaunchKernelGGL(k_bpm_rows_fwd<E>, dim3(grid), dim3(E::kBlock), lds, s, a); break;
      case BpmKind::rows_out: hipLaunchKernelGGL(k_bpm_rows_out<E>, dim3(grid), dim3(E::kBlock), lds, s, a); break;
      case BpmKind::rows_jvp: hipLaunchKernelGGL(k_bpm_rows_jvp<E>, dim3(grid), dim3(E::kBlock), lds, s, a); break;
      default: hipLaunchKernelGGL(k_bpm_rows_adj<E>, dim3(grid), dim3(E::kBlock), lds, s, a); break;
    }
  } else {
    if (k == BpmKind::cols_adj && a.red_grad != nullptr) {
      const long plane = static_cast<long>(a.g.n) * a.g.n;
      a.line_blocks = static_cast<int>(grid);
      a.red_blocks = static_cast<int>((plane + E::kBlock - 1) / E::kBlock);
      grid += static_cast<unsigned>(a.red_blocks);
    }
    switch (k) {
      case BpmKind::cols_fwd: hipLaunchKernelGGL(k_bpm_cols_fwd<E>, dim3(grid), dim3(E::kBlock), lds, s, a); break;
      default: hipLaunchKernelGGL(k_bpm_cols_adj<E>, dim3(grid), dim3(E::kBlock), lds, s, a); break;
    }
  }
}

}  // namespace

}  // namespace qh
