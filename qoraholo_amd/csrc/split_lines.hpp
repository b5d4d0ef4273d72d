// Register engine for the lengths without a four-step kernel: the Stockham passes of lds_fft,
// run in registers in two groups.
//
// lds_fft transforms a line of n = R_1 ... R_m by m passes between two LDS buffers, 4 or 5 for
// most lengths, each with a barrier and an integer division per butterfly. The passes of a
// prefix R_1 ... R_c of the factors, N1 = R_1 ... R_c, only combine elements b + N2 i (N2 = n / N1)
// for a fixed b < N2, and those of the rest only elements k + N1 i for a fixed k < N1. So thread b
// runs the first c passes on its N1 elements in registers, the line is exchanged through LDS once,
// and thread k runs the others on its N2 elements: the same butterflies on the same operands with
// the same twiddles in the same order, so the results are those of lds_fft bit for bit, with one
// exchange per transform instead of a round trip per pass. The cut makes the larger of N1 and N2
// least (240 = 8 2 | 3 5, 500 = 4 5 | 5 5); a thread holds at most kSplitMost elements.
//
// What bounds it: at 240^2 with 31 illuminations the slice kernels of the BPM took 26-29 us in LDS
// passes and take 12.3 (rows) and 15.5 us (columns) forward, 14.5 and 16.7 us in the adjoint, 4 TB/s
// on the bytes they must move, against 13.5 and 21.5 us of the four-step kernels on twice the
// pixels at 256: the chain of passes in a thread and the second exchange. Real rows of 200 (160
// planes of 200 rows, momentum fused): 35 -> 29 us; z round trips of 160: 38 -> 28 us.
#pragma once

#include <hip/hip_runtime.h>

#include "fft_core.hpp"
#include "fft_engine.hpp"

namespace qh {

// The factors of n in the order of fft_factors, at compile time.
struct SplitFactors {
  int r[kMaxFactors] = {};
  int count = 0;
};
constexpr SplitFactors split_factors(int n) {
  SplitFactors f;
  constexpr int kOrder[] = {8, 4, 2, 3, 5};
  for (int r : kOrder) {
    while (n % r == 0) {
      f.r[f.count++] = r;
      n /= r;
    }
  }
  return f;
}
constexpr int split_product(const SplitFactors& f, int from, int to) {
  int p = 1;
  for (int i = from; i < to; ++i) p *= f.r[i];
  return p;
}
// How many factors the first group takes: the cut with the least larger group.
constexpr int split_cut(int n) {
  const SplitFactors f = split_factors(n);
  int best = 1;
  int best_most = n;
  for (int c = 1; c < f.count; ++c) {
    const int a = split_product(f, 0, c);
    const int b = split_product(f, c, f.count);
    const int most = a > b ? a : b;
    if (most < best_most) {
      best_most = most;
      best = c;
    }
  }
  return best;
}

// Passes P .. P1-1 of an N-point transform on the LEN elements a thread holds; NS is the product
// of the group's earlier factors. tw(kk, s, step) is the twiddle of sub-transform position kk.
template <int N, int LEN, int P, int P1, int NS, class TW>
__device__ __forceinline__ void split_passes(float2 (&v)[LEN], TW tw, bool inv) {
  if constexpr (P < P1) {
    constexpr int R = split_factors(N).r[P];
    constexpr int Q = LEN / R;
    float2 u[LEN];
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      const int kk = j % NS;
      float2 x[R];
#pragma unroll
      for (int s = 0; s < R; ++s) x[s] = v[j + s * Q];
#pragma unroll
      for (int s = 1; s < R; ++s) tw(x[s], kk, s, LEN / (NS * R));
      bfly<R>(x, inv);
#pragma unroll
      for (int s = 0; s < R; ++s) u[(j - kk) * R + kk + s * NS] = x[s];
    }
#pragma unroll
    for (int i = 0; i < LEN; ++i) v[i] = u[i];
    split_passes<N, LEN, P + 1, P1, NS * R>(v, tw, inv);
  }
}

// Line engine (see fft_engine.hpp) of lines of length N, LINES_ of them per block.
template <int N_, bool LINE_FAST, int LINES_>
struct SplitLines {
  static constexpr int N = N_;
  static constexpr SplitFactors kF = split_factors(N);
  static constexpr int kCut = split_cut(N);
  static constexpr int N1 = split_product(kF, 0, kCut);
  static constexpr int N2 = N / N1;
  static constexpr int T = N1 > N2 ? N1 : N2;
  static constexpr int LINES = LINES_;
  static constexpr int kBlock = T * LINES;
  static_assert(kBlock <= 1024, "a block holds whole lines");
  // Threads that walk along lines write the exchange with a stride of N1, padded by one.
  static constexpr int kPitch = LINE_FAST ? N1 : N1 + 1;
  static constexpr int kLine = N2 * kPitch;  // elements of a line in LDS, at least N

  float2* t;
  float2* tw;
  int line;
  int j;
  long l;
  bool valid;
  float2 v[N1];
  float2 w[N2];

  __device__ static float2* lds_t() {
    __shared__ float2 s[kLine * LINES];
    return s;
  }
  __device__ static float2* lds_tw() {
    __shared__ float2 s[N];
    return s;
  }
  __device__ static double* lds_red() {
    __shared__ double s[kBlock];
    return s;
  }
  static unsigned grid(long lines) { return static_cast<unsigned>((lines + LINES - 1) / LINES); }

  __device__ explicit SplitLines(const LineGeom& g) { init<false>(g, 0); }
  // The grid's first nb blocks run the lines (its later blocks run other work).
  __device__ SplitLines(const LineGeom& g, int nb) { init<true>(g, nb); }
  // The block's own LINES lines, numbered from 0, with LDS of the caller's (kLds and kTw values);
  // table is exp(-2 pi i t / N). The caller synchronises before the first transform.
  static constexpr int kLds = kLine * LINES;
  static constexpr int kTw = N;
  static constexpr int kBins = N2;  // bins a thread holds after a transform
  __device__ SplitLines(float2* lds, float2* lds_table, const float2* table)
      : t(lds), tw(lds_table) {
    fill(table);
    l = line;
    valid = true;
  }
  template <bool PART>
  __device__ void init(const LineGeom& g, int nb) {
    t = lds_t();
    tw = lds_tw();
    fill(g.tw);
    l = (PART ? xcd_block(nb) : xcd_block()) * LINES + line;
    valid = l < g.lines;
  }
  __device__ __forceinline__ void fill(const float2* table) {
    const int tid = static_cast<int>(threadIdx.x);
    for (int i = tid; i < N; i += kBlock) tw[i] = table[i];
    line = LINE_FAST ? tid % LINES : tid / T;
    j = LINE_FAST ? tid / LINES : tid % T;
  }
  // f(i, l, k, v&) for the thread's i-th bin k.
  template <class F>
  __device__ void bins(F f) {
    if (valid && j < N1) {
#pragma unroll
      for (int i = 0; i < N2; ++i) f(i, l, j + N1 * i, w[i]);
    }
  }
  __device__ __forceinline__ float2& at(int i) { return LINE_FAST ? t[i * LINES + line] : t[line * kLine + i]; }

  // Both groups on v, with the exchange between them; the result in w: element j + N1 i in w[i].
  __device__ __forceinline__ void transform(bool inv) {
    if (j < N2) {
      split_passes<N, N1, 0, kCut, 1>(
          v,
          [&](float2& x, int kk, int s, int step) {
            if (kk == 0) return;
            float2 c = tw[kk * s * step * N2];
            if (inv) c.y = -c.y;
            x = cmul(x, c);
          },
          inv);
#pragma unroll
      for (int k = 0; k < N1; ++k) at(j * kPitch + k) = v[k];
    }
    __syncthreads();
    if (j < N1) {
#pragma unroll
      for (int i = 0; i < N2; ++i) w[i] = at(j + kPitch * i);
      split_passes<N, N2, kCut, kF.count, 1>(
          w,
          [&](float2& x, int kk, int s, int step) {
            float2 c = tw[(j + N1 * kk) * s * step];
            if (inv) c.y = -c.y;
            // Position 0 takes no twiddle (as in lds_fft).
            const float2 y = cmul(x, c);
            x = (kk == 0 && j == 0) ? x : y;
          },
          inv);
    }
  }

  template <class F>
  __device__ void load(F f) {
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      v[i] = (valid && j < N2) ? f(l, j + N2 * i) : float2{0.0f, 0.0f};
    }
    __syncthreads();
  }
  __device__ void first(bool inverse) { transform(inverse); }
  template <class F>
  __device__ void mid(F f) {
    if (valid && j < N1) {
#pragma unroll
      for (int i = 0; i < N2; ++i) f(l, j + N1 * i, w[i]);
    }
  }
  template <int G, class L, class F>
  __device__ void mid_loaded(L ld, F f) {
    if (valid && j < N1) {
#pragma unroll
      for (int i0 = 0; i0 < N2; i0 += G) {
        decltype(ld(l, 0)) ops[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          if (i0 + g < N2) ops[g] = ld(l, j + N1 * (i0 + g));
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          if (i0 + g < N2) f(l, j + N1 * (i0 + g), w[i0 + g], ops[g]);
        }
      }
    }
  }
  template <class F>
  __device__ void reduce_lines(F f, double* out) {
    double* red = lds_red();
    double s = 0.0;
    if (valid && j < N1) {
#pragma unroll
      for (int i = 0; i < N2; ++i) s += f(l, j + N1 * i, w[i]);
    }
    red[line * T + j] = s;
    __syncthreads();
    if (valid && j == 0) {
      double total = 0.0;
      for (int jj = 0; jj < N1; ++jj) total += red[line * T + jj];
      out[l] = total;
    }
  }
  // The line in natural order through LDS (the first transform leaves every N1-th element with a
  // thread, the second starts from every N2-th), then the same again.
  __device__ void second(bool inverse) {
    __syncthreads();
    if (j < N1) {
#pragma unroll
      for (int i = 0; i < N2; ++i) at(j + N1 * i) = w[i];
    }
    __syncthreads();
    if (j < N2) {
#pragma unroll
      for (int i = 0; i < N1; ++i) v[i] = at(j + N2 * i);
    }
    __syncthreads();
    transform(inverse);
  }
  template <class F>
  __device__ void store1(F f) {
    if (valid && j < N1) {
#pragma unroll
      for (int i = 0; i < N2; ++i) f(l, j + N1 * i, w[i]);
    }
  }
  template <class F>
  __device__ void store2(F f) { store1(f); }
};

// Elements a thread may hold, and the lengths that gives, except those with a four-step kernel.
inline constexpr int kSplitMost = 40;
constexpr bool split_length(int n) {
  const SplitFactors f = split_factors(n);
  if (split_product(f, 0, f.count) != n || f.count < 2) return false;
  const int a = split_product(f, 0, split_cut(n));
  return a <= kSplitMost && n / a <= kSplitMost;
}

// F<N>::run(args...) for the even lengths above 32 without a four-step kernel whose two groups
// fit, up to 512; false for the others. The list is what split_length admits there.
#define QH_SPLIT_LENGTHS(X)                                                                     \
  X(36) X(40) X(50) X(54) X(60) X(72) X(80) X(90) X(100) X(108) X(120) X(144) X(150) X(160)   \
  X(162) X(180) X(200) X(216) X(240) X(250) X(270) X(288) X(300) X(320) X(324) X(360) X(400)    \
  X(432) X(450) X(480) X(486) X(500)
template <template <int> class F, class... Args>
bool with_split(int n, Args&&... args) {
  switch (n) {
#define QH_SPLIT_CASE(N)                                \
  case N:                                               \
    static_assert(split_length(N), "two groups fit");   \
    F<N>::run(args...);                                 \
    return true;
    QH_SPLIT_LENGTHS(QH_SPLIT_CASE)
#undef QH_SPLIT_CASE
    default: return false;
  }
}

}  // namespace qh
