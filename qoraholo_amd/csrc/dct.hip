// Cosine transforms of the phase unwrapping on the register engines.
//
// A DCT-II of a real line is an FFT of the line with its even elements first and its odd ones
// reversed (Makhoul). Two lines go as the real and imaginary part of one, two rows of an image or
// two adjacent columns: half the transforms, and columns load as whole complex values. The rows
// form the divergence they transform, the columns divide by the eigenvalues between their two
// transforms, so that the solve is three passes over the images. 49 images of 256^2: 31.0, 15.3 and
// 9.4 us, against 16.9 (divergence), 24.3, 48.5 and 23.8 us with LDS transforms of single lines; the
// 26 MB a pass moves take 5 us. What bounds the first: the eight wrapped differences of a pair of
// rows, each with a division; the others: the exchanges of a block.
#include "dct.hpp"

#include <algorithm>

#include "dct_kernels.hpp"
#include "split_lines.hpp"

namespace qh {

namespace {

using namespace dct;

constexpr int floor_pow2(int v) { return v < 2 ? 1 : 2 * floor_pow2(v / 2); }

template <int N1, int N2, class A>
bool launch_reg(const A& a, hipStream_t s) {
  constexpr int kT = N1 > N2 ? N1 : N2;
  constexpr int kLines = kColumns<A> ? std::max(16, floor_pow2(256 / kT)) : floor_pow2(256 / kT);
  launch<RegLines<N1, N2, kColumns<A>, kLines * kT>>(a, s);
  return true;
}

template <class A>
void run(const A& a, const char* what, hipStream_t s) {
  const auto go = [&] {
    switch (a.g.n) {
      case 32: return launch_reg<8, 4>(a, s);
      case 48: return launch_reg<8, 6>(a, s);
      case 64: return launch_reg<8, 8>(a, s);
      case 96: return launch_reg<16, 6>(a, s);
      case 128: return launch_reg<16, 8>(a, s);
      case 192: return launch_reg<16, 12>(a, s);
      case 256: return launch_reg<16, 16>(a, s);
      case 384: return launch_reg<16, 24>(a, s);
      case 512: return launch_reg<32, 16>(a, s);
      default: return split(a, s);
    }
  };
  require(go(), "dct: no kernel for this length");
  check_launch(what);
}

template <int N>
struct Any {
  static void run() {}
};

bool length_supported(int n) {
  for (int m : {32, 48, 64, 96, 128, 192, 256, 384, 512}) {
    if (n == m) return true;
  }
  return with_split<Any>(n);
}

LineGeom geometry(int n, long lines) { return {fft_twiddles(n), FftFactors{}, n, lines, 0}; }

}  // namespace

bool dct_supported(int ny, int nx) { return length_supported(ny) && length_supported(nx); }

void dct_poisson(const float* psi, float* phi, int images, int ny, int nx, hipStream_t s) {
  const LineGeom rows = geometry(nx, static_cast<long>(images) * (ny / 2));
  const LineGeom columns = geometry(ny, static_cast<long>(images) * (nx / 2));
  run(RowsForward{rows, dct_twiddles(nx), psi, phi, ny}, "dct_rows", s);
  run(Columns{columns, dct_twiddles(ny), phi, nx, neumann_terms(ny), neumann_terms(nx),
              1.0f / static_cast<float>(ny)},
      "dct_columns", s);
  run(RowsInverse{rows, dct_twiddles(nx), phi, 1.0f / static_cast<float>(nx)}, "dct_rows", s);
}

}  // namespace qh
