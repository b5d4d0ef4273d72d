// Column kernels of the beam propagation model for the lengths of split_lines.hpp.
#include "bpm_kernels.hpp"
#include "split_lines.hpp"

namespace qh {

namespace {

// Blocks of 16 columns: each block row is a whole 128-byte segment.
template <int N>
struct Launch {
  static void run(BpmKind k, BpmModel::Args a, hipStream_t s) {
    using E = SplitLines<N, true, 16>;
    launch_with<false, E>(k, a, E::grid(a.g.lines), 0, s);
  }
};

}  // namespace

bool bpm_split_cols(BpmKind k, const BpmModel::Args& a, hipStream_t s) {
  if (!with_split<Launch>(a.g.n, k, a, s)) return false;
  check_launch("bpm");
  return true;
}

}  // namespace qh
