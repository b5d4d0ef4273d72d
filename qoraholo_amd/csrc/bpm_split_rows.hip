// Row kernels of the beam propagation model for the lengths of split_lines.hpp.
#include "bpm_kernels.hpp"
#include "split_lines.hpp"

namespace qh {

namespace {

// Blocks of 8 rows, as the four-step lengths have.
template <int N>
struct Launch {
  static void run(BpmKind k, BpmModel::Args a, hipStream_t s) {
    using E = SplitLines<N, false, 8>;
    launch_with<true, E>(k, a, E::grid(a.g.lines), 0, s);
  }
};

}  // namespace

bool bpm_split_rows(BpmKind k, const BpmModel::Args& a, hipStream_t s) {
  if (!with_split<Launch>(a.g.n, k, a, s)) return false;
  check_launch("bpm");
  return true;
}

}  // namespace qh
