// Complex transforms for the lengths without a four-step kernel, on the register engine of
// split_lines.hpp: the operations and bits of the LDS kernels of fft.hip, which remain for the
// lengths whose groups do not fit.
#include <algorithm>

#include "common.hpp"
#include "fft_args.hpp"
#include "runtime.hpp"
#include "split_lines.hpp"

namespace qh {

namespace {

template <class E>
__global__ void __launch_bounds__(E::kBlock) k_split_lines(LinesArgs a, LineGeom g) {
  E e(g);
  e.load([&](long l, int i) { return a.in[line_base(l, a.g) + i * a.g.stride]; });
  e.first(a.inverse != 0);
  e.store1([&](long l, int k, float2 v) {
    if (a.scale != 1.0f) v = cscale(v, a.scale);
    if (a.alt_mod > 0 && ((k + l % a.alt_mod) & 1)) v = {-v.x, -v.y};
    a.out[line_base(l, a.g) + k * a.g.stride] = v;
  });
}

LineGeom geometry(int n, long lines) { return LineGeom{fft_twiddles(n), FftFactors{}, n, lines, 0}; }

// About 256 threads a block.
template <int N>
using RowEngine = SplitLines<N, false, std::max(1, 256 / SplitLines<N, false, 1>::T)>;
// Adjacent lines: 16, so that each block row is a whole 128-byte segment.
template <int N>
using ColumnEngine = SplitLines<N, true, 16>;

template <int N>
struct LaunchLines {
  static void run(const LinesArgs& a, bool contig, hipStream_t s) {
    const LineGeom g = geometry(N, a.g.count);
    if (contig) {
      using E = RowEngine<N>;
      hipLaunchKernelGGL(k_split_lines<E>, dim3(E::grid(g.lines)), dim3(E::kBlock), 0, s, a, g);
    } else {
      using E = ColumnEngine<N>;
      hipLaunchKernelGGL(k_split_lines<E>, dim3(E::grid(g.lines)), dim3(E::kBlock), 0, s, a, g);
    }
  }
};

}  // namespace

bool split_fft_lines(const LinesArgs& a, bool contig, hipStream_t s) {
  return with_split<LaunchLines>(a.n, a, contig, s);
}

}  // namespace qh
