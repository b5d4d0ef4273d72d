// Cosine transforms of the phase unwrapping for the lengths of split_lines.hpp.
#include <algorithm>

#include "dct_kernels.hpp"
#include "split_lines.hpp"

namespace qh::dct {

namespace {

template <int N>
struct Split {
  template <class A>
  static void run(const A& a, hipStream_t s) {
    constexpr int kT = SplitLines<N, false, 1>::T;
    launch<SplitLines<N, kColumns<A>, kColumns<A> ? 16 : std::max(1, 256 / kT)>>(a, s);
  }
};

}  // namespace

bool split(const RowsForward& a, hipStream_t s) { return with_split<Split>(a.g.n, a, s); }
bool split(const RowsInverse& a, hipStream_t s) { return with_split<Split>(a.g.n, a, s); }
bool split(const Columns& a, hipStream_t s) { return with_split<Split>(a.g.n, a, s); }

}  // namespace qh::dct
