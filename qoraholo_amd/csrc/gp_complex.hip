// Gerchberg-Papoulis on full spectra (gp_transform c2c): the steps between two transforms along one
// axis, in one pass with them.
//
// An iteration forms max(Re p, 0) of the volume, transforms it, restores the measured bins and
// transforms back. Both steps work on single elements, so the x transforms go around the first and
// the z transforms around the second: with the y transforms between them an iteration is 4 passes
// over the volume instead of 8: requests of 20 iterations 1801 -> 1032 us at 128^3, 6723 -> 4125 us
// at 256^3, 5957 -> 2659 us at 200^2 x 160 (there with faster lines too). What bounds them: a read
// and a write of the volume each (128^3, 34 MB: rows 8.9, y 9.7 us), and for the z pass the hit
// counts with the measured bins (13.5 us).
#include "gp_complex.hpp"

#include <algorithm>

#include "gp_complex_kernels.hpp"

namespace qh {

namespace {

using namespace gp;

constexpr int floor_pow2(int v) { return v < 2 ? 1 : 2 * floor_pow2(v / 2); }

template <int N1, int N2, class A>
void launch_reg(const A& a, hipStream_t s) {
  constexpr int kT = N1 > N2 ? N1 : N2;
  constexpr int kLines = kAdjacent<A> ? std::max(16, floor_pow2(256 / kT)) : floor_pow2(256 / kT);
  using E = RegLines<N1, N2, kAdjacent<A>, kLines * kT>;
  launch<E>(a, E::grid(a.g.lines), 0, s);
}

template <class A>
void run(A a, const char* what, hipStream_t s) {
  if (a.g.lines == 0) return;
  switch (a.g.n) {
    case 32: launch_reg<8, 4>(a, s); break;
    case 48: launch_reg<8, 6>(a, s); break;
    case 64: launch_reg<8, 8>(a, s); break;
    case 96: launch_reg<16, 6>(a, s); break;
    case 128: launch_reg<16, 8>(a, s); break;
    case 192: launch_reg<16, 12>(a, s); break;
    case 256: launch_reg<16, 16>(a, s); break;
    case 384: launch_reg<16, 24>(a, s); break;
    case 512: launch_reg<32, 16>(a, s); break;
    default: {
      if (split(a, s)) break;
      using E = LdsLines<!kAdjacent<A>>;
      a.g.lines_per_block = E::lines_per_block(a.g.n);
      launch<E>(a, E::grid(a.g.lines, a.g.lines_per_block), E::dynamic_lds(a.g.n), s);
      break;
    }
  }
  check_launch(what);
}

LineGeom geometry(int n, long lines) { return {fft_twiddles(n), fft_factors(n), n, lines, 0}; }

}  // namespace

void gp_complex_rows(float2* p, long rows, int n, float scale, hipStream_t s) {
  run(RowArgs{geometry(n, rows), p, scale}, "gp_rows", s);
}

void gp_complex_index(const float2* p, long rows, int n, float scale, float nm2, float inv_k02,
                      float* ri, hipStream_t s) {
  run(IndexArgs{geometry(n, rows), p, scale, nm2, inv_k02, ri}, "gp_index", s);
}

void gp_complex_z(float2* p, const float2* measured, const std::uint16_t* counts, int nz,
                  long plane, hipStream_t s) {
  run(ZLineArgs{geometry(nz, plane), p, measured, counts, plane}, "gp_z", s);
}

}  // namespace qh
