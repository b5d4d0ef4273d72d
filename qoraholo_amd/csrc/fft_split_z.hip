// The z round trip for the lengths without a four-step kernel, on the register engine of
// split_lines.hpp: the operations and bits of the LDS kernels of fft.hip, which remain for the
// lengths whose groups do not fit.
#include <algorithm>

#include "common.hpp"
#include "fft_args.hpp"
#include "runtime.hpp"
#include "split_lines.hpp"

namespace qh {

namespace {

template <class E, bool BATCH>
__global__ void __launch_bounds__(E::kBlock) k_split_zrt(ZArgs a, LineGeom g) {
  E e(g);
  const auto at = [&](long l, int i) {
    return static_cast<long>(i) * a.plane + (BATCH ? z_line_base(a, l) : l);
  };
  e.load([&](long l, int i) { return a.e[at(l, i)]; });
  e.first(false);
  struct Ops {
    float2 d;
    int hits;
  };
  e.template mid_loaded<4>(
      [&](long l, int k) {
        const long x = at(l, k);
        return Ops{a.a[x], a.hits[x]};
      },
      [&](long, int, float2& v, Ops o) { hermitian_restore(o.d.x, o.d.y, o.hits, v.x, v.y); });
  e.second(true);
  e.store2([&](long l, int i, float2 v) { a.e[at(l, i)] = v; });
}

LineGeom geometry(int n, long lines) { return LineGeom{fft_twiddles(n), FftFactors{}, n, lines, 0}; }

// Adjacent lines: 16, so that each block row is a whole 128-byte segment.
template <int N>
using ColumnEngine = SplitLines<N, true, 16>;

template <int N>
struct LaunchZ {
  static void run(const ZArgs& a, hipStream_t s) {
    using E = ColumnEngine<N>;
    const LineGeom g = geometry(N, a.lines);
    if (a.vol != 0) {
      hipLaunchKernelGGL((k_split_zrt<E, true>), dim3(E::grid(g.lines)), dim3(E::kBlock), 0, s, a, g);
    } else {
      hipLaunchKernelGGL((k_split_zrt<E, false>), dim3(E::grid(g.lines)), dim3(E::kBlock), 0, s, a, g);
    }
  }
};

}  // namespace

bool split_z_roundtrip(const ZArgs& a, hipStream_t s) { return with_split<LaunchZ>(a.nz, a, s); }

}  // namespace qh
