// Gerchberg-Papoulis passes on full spectra for the lengths of split_lines.hpp.
#include <algorithm>

#include "gp_complex_kernels.hpp"
#include "split_lines.hpp"

namespace qh::gp {

namespace {

template <int N>
struct Split {
  template <class A>
  static void run(const A& a, hipStream_t s) {
    constexpr int kT = SplitLines<N, false, 1>::T;
    using E = SplitLines<N, kAdjacent<A>, kAdjacent<A> ? 16 : std::max(1, 256 / kT)>;
    launch<E>(a, E::grid(a.g.lines), 0, s);
  }
};

}  // namespace

bool split(const RowArgs& a, hipStream_t s) { return with_split<Split>(a.g.n, a, s); }
bool split(const IndexArgs& a, hipStream_t s) { return with_split<Split>(a.g.n, a, s); }
bool split(const ZLineArgs& a, hipStream_t s) { return with_split<Split>(a.g.n, a, s); }

}  // namespace qh::gp
