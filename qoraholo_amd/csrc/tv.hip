// Total-variation proximal step by fast gradient projection on the dual (FGP), the inner loop
// of FISTA-TV, on gfx950.
//
// k_fgp_steps runs up to four FGP steps per pass over the volume. The extrapolated dual
// r_k = p_k + m_{k-1} (p_k - p_{k-1}) is not stored: a pass of T steps reads b and the two latest
// dual iterates p_k, p_{k-1} and writes p_{k+T-1} and p_{k+T}, 7 volumes in and 6 out. The first
// pass of a prox starts from r = p_k (src/cpu/tv.cpp:10) and reads no p_{k-1}; the last one forms
// the prox output as it goes and writes no p_{k+T-1}.
//
// The dual is the library's own, laid out for these accesses: within each plane of a component,
// rows go in groups of four ("quads"), stored column by column, so that the four rows of a column
// are 16 consecutive bytes and a 128-byte line holds 4 rows of 8 columns. A wave loads or stores
// its 64 columns x 4 rows as one 16-byte access per lane, and tiles cut at multiples of 8 columns
// and 4 rows share no line they write. With plain rows a tile of 64 columns wrote parts of lines
// and the 256^3 pass of three steps took 290-350 us against 220 us (a kernel that only moves the
// same data in that pattern took 326 us cut at 58 columns, 231 us cut at 48, and 186-202 us in
// quads). Planes of the dual hold whole quads: rows past the last of the volume are zero and stay
// zero.
//
// Per prox of 10 steps, output included (4 + 3 + 3 steps), against two steps per pass and a kernel
// for the output before: 671 against 837 us at 256^3, 1131 against 2635 us at 320^3, 1952 against
// 3183 us at 384^3, 158 against 184 us at 128^3 and 73 against 131 us at 64^3. What bounds it: the
// middle pass moves 978 MB with the halo re-reads, at 4.6 TB/s (a device copy reaches 4.9). The first
// and last are bound by neither traffic nor vector work alone: of their 206 and 222 us the 722 and 820
// MB would take 147 and 167, and the vector units of the CUs that hold a block (220 of 256 at 256^3)
// are busy 64 and 52% of the cycles (48% in the middle pass; 33 instructions a point and step in the
// first, 47 in its exact form, and only 24 of 32 rows and 56 of 64 columns of a tile are its own). Two
// waves a SIMD hide the one behind the other in part.
#include <algorithm>
#include <atomic>

#include "common.hpp"
#include "fft_core.hpp"
#include "runtime.hpp"
#include "tv.hpp"

namespace qh {

namespace {

// The arithmetic of a step, in two forms. EXACT: every operation rounded on its own, in the order
// of the reference's expressions (src/common.hpp:121-141), and the projection's 1 / sqrt(n) the
// float nearest to 1 / (float nearest to sqrt(n)); the bits of the reference's expressions, which
// the data terms of the BPM inversion are compared by. Otherwise multiply-adds are fused and
// 1 / sqrt(n) takes one Newton step from the hardware's: nearer to real arithmetic by itself and 11%
// faster over a 256^3 prox of 10 steps (744 -> 670 us).
template <bool EXACT>
__device__ __forceinline__ float multiply_add(float a, float x, float y) {
  return EXACT ? y + a * x : fmaf(a, x, y);
}

// max(b - lambda L(r), 0) from the components of r at a point and at its lower neighbours, added
// in the order of the negative divergence L(r)(i) = sum_a r_a(i) - r_a(i - e_a), axes z, y, x. A
// component is zero on the last plane, row or column along its axis (its difference is), and the
// neighbour before the first counts as zero, so the faces need no case of their own.
template <bool EXACT>
__device__ __forceinline__ float primal_value(float b, float lambda, float rz, float rz_below,
                                              float ry, float ry_up, float rx, float rx_left) {
  float s = rz - rz_below;
  s += ry;
  s -= ry_up;
  s += rx;
  s -= rx_left;
  return fmaxf(multiply_add<EXACT>(-lambda, s, b), 0.0f);
}

// 1 / max(1, sqrt(norm2)) from the hardware's reciprocal square root y. EXACT: g = n y corrected
// once is the nearest float to sqrt(n), and y corrected once against that the nearest to its
// reciprocal, except where every mantissa bit of the root is set: there the correction ends on the
// tie between two floats and rounds to the even one, and the nearest is the next (the one exception
// to a reciprocal corrected with fused operations). With it these are the bits of 1.0f / sqrtf(n)
// for every float n from 1 to infinity (all 2^30 compared on the device), in 11 operations instead
// of the compiler's 25. The bounds keep the limits of the division: 0 for an infinite norm, whose
// residuals are NaN; a NaN norm counts as below one, as in norm2 > 1 ? ... : 1.
template <bool EXACT>
__device__ __forceinline__ float ball_scale(float norm2) {
  const float n = fmaxf(norm2, 1.0f);
  const float y = __builtin_amdgcn_rsqf(n);
  const float g = n * y;
  const float h = 0.5f * y;
  if constexpr (EXACT) {
    const float root = fmaf(fmaf(-g, g, n), h, g);
    const float even = fmaf(fmaf(-root, y, 1.0f), y, y);
    const unsigned up = __builtin_amdgcn_frexp_mantf(root) == 0x1.fffffep-1f ? 1u : 0u;
    return fmaxf(__uint_as_float(__float_as_uint(even) + up), 0.0f);
  } else {
    return fmaf(h, fmaxf(fmaf(-g, y, 1.0f), -1.0f), y);
  }
}

// The value of the lane below (lane 0: zero) and of the lane above (lane 63: zero).
__device__ __forceinline__ float lane_below(float v) {
  constexpr int kWaveShr1 = 0x138;
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), kWaveShr1, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_above(float v) {
  constexpr int kWaveShl1 = 0x130;
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), kWaveShl1, 0xf, 0xf, true));
}

// A window of device memory in scalar registers: an access at a byte offset past its end loads
// zero or stores nothing. So faces, halos and arrays that a pass does without need no branch, and
// the compiler knows how many accesses are in flight (with stores in branches it waits for all of
// them where it needs the loads before them).
constexpr unsigned kOutside = 0x80000000u;  // past the end of every window
struct Window {
  typedef unsigned quad __attribute__((ext_vector_type(4)));
  static constexpr int kNonTemporal = 2;
  __amdgpu_buffer_rsrc_t rsrc;
  // `bytes` from p, or nothing where not `on` (the same for the whole wave).
  __device__ __forceinline__ Window(const float* p, int bytes, bool on)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, on ? bytes : 0,
                                               0x00020000)) {}
  __device__ __forceinline__ float load(unsigned at) const {
    return __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, at, 0, 0));
  }
  __device__ __forceinline__ void store(float v, unsigned at) const {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v), rsrc, at, 0, 0);
  }
  __device__ __forceinline__ void load4(float (&v)[4], unsigned at) const {
    const quad q = __builtin_amdgcn_raw_buffer_load_b128(rsrc, at, 0, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = __uint_as_float(q[j]);
  }
  // Non-temporal: the dual iterates are all written before the next pass reads them.
  __device__ __forceinline__ void stream4(const float (&v)[4], unsigned at) const {
    quad q;
#pragma unroll
    for (int j = 0; j < 4; ++j) q[j] = __float_as_uint(v[j]);
    __builtin_amdgcn_raw_buffer_store_b128(q, rsrc, at, 0, kNonTemporal);
  }
  __device__ __forceinline__ void stream(float v, unsigned at) const {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v), rsrc, at, 0, kNonTemporal);
  }
};

// A block of NW waves holds a tile of 64 columns (one per lane) by NW quads of rows (one per
// wave) and marches z. Stage s = 0 .. T-1 runs step k+s+1 on the planes as they come: with plane f
// of the inputs loaded, stage s forms z_{k+s} on plane f - s from r_{k+s} there, then p_{k+s+1} and
// r_{k+s+1} on plane f - s - 1, which stage s + 1 takes. Each stage keeps one plane of r, p and z of
// the tile in registers (7 floats a point); the last planes of b wait in LDS. x neighbours come
// by DPP from the next lane, y neighbours from the thread's own registers except at the edges of
// a wave's quad (a row of r_y and one of z per wave and stage through LDS), z neighbours from the
// registers of the plane before. Every step makes one column, row and plane on either side of the
// tile invalid, so tiles overlap by kHalo columns and rows on each side and a chunk of planes
// starts T planes early. FINAL adds a stage that forms max(b - lambda L(p_{k+T}), 0), which takes
// one more of each on the lower side (L reads p at x - 1, y - 1 and z - 1): T + FINAL of them lie
// within kHalo, so that a pass with the output has at most three steps.
//
// Eight waves of up to 256 registers make one block per CU. Twelve waves (48 rows a tile) leave 168
// registers, which T = 3 just fits and the other passes spill: 209 against 220 us for a 256^3 pass
// of three steps but 330 against 232 us for one with the output, and no gain at 384^3 (665 against
// 643 us) or 128^3 (56 against 44 us), where fewer, larger tiles fill the CUs less evenly.
constexpr int kRows = 4;   // rows of a quad
constexpr int kWaves = 8;  // quads of a tile
constexpr int kHalo = 4;   // columns and rows of a tile, on each side, that are not its own
constexpr int kMaxSteps = 4;

struct StepArgs {
  const float* b;
  const float* p_k;    // p_k (r_k is formed from it)
  const float* p_km1;  // p_{k-1} (not read on the first step of a prox)
  float* p_prev;       // out: p_{k+T-1}, or null
  float* p_last;       // out: p_{k+T}, or null
  float* x;            // out with FINAL: the prox output
  long vol;
  int nz, ny, nx;
  float lambda;
  float step;
  float m[kMaxSteps];  // m[s]: momentum of r_{k+s}; 0 on the first step of a prox
  int first;
  int zlen;              // planes per chunk
  int tiles_x, tiles_y;
  int tile_x, tile_y;    // columns and rows a tile writes
  int halo_x, halo_y;    // kHalo, or 0 where one tile holds the volume's side
  int to_index;          // the output as refractive index
  float nm2, inv_k02;
  long dual_plane, dual_vol;  // floats of a plane and of a component of the dual
};

// The march, unrolled over T + 1 planes: the r and p a stage hands on take the registers of the
// plane it has done with, so the register sets rotate through the T stages and the loads, and after
// T + 1 planes are back in place (a rolled loop moves 7 floats a point and stage back by v_mov). The
// unrolled planes are numbered U = 0 .. T; without steps two planes, for two exchange buffers.
//
// FIRST: the first pass of a prox, which needs no p_{k-1}.
//
// ROWS: how the volume's rows fill the quads of the dual. whole: ny is a multiple of 4. filled: the
// dual's planes hold the rest of the last quad as well (a variant of its own: the sizes that then
// differ between the dual and b are values to hold, 2% of a 256^3 request, 16.72 against 16.33 ms).
// cut: the dual's planes end with the volume's last row (a fixed workspace without room for more), and
// the rows of the last quad are stored column by column like the others (h floats a column for h
// rows), which takes accesses of 4 bytes: 206 against 128 us for a prox of 10 steps at 90^3, 590
// against 359 us at 270^2 x 90.
enum class Rows { whole, filled, cut };

template <int T, bool FIRST, bool FINAL, Rows ROWS, bool EXACT>
struct StepMarch {
  static constexpr int NW = kWaves;
  static constexpr int HL = T + (FINAL ? 1 : 0);  // planes in front of a chunk
  static_assert(HL <= kHalo, "the points a tile writes are out of reach of its edges");
  static constexpr int S = T + (FINAL ? 1 : 0);   // stages that exchange rows
  static constexpr int TS = T > 0 ? T : 1;
  static constexpr int kUnroll = T > 0 ? T + 1 : 2;
  // Row exchange buffers: planes that follow one another use different ones, as a wave may be one
  // barrier ahead of its neighbours, never a plane. With a single buffer a wave could overwrite the
  // row of a plane that the next wave has yet to read.
  static constexpr int kBufs = kUnroll % 2 == 0 ? 2 : 3;
  static constexpr int buf(int u) { return u == kUnroll - 1 && kBufs == 3 ? 2 : u % 2; }
  static constexpr bool bufs_alternate() {
    for (int u = 0; u < kUnroll; ++u) {
      if (buf(u) == buf((u + 1) % kUnroll) || buf(u) >= kBufs) return false;
    }
    return true;
  }
  static_assert(bufs_alternate(), "consecutive planes exchange rows through different buffers");

  struct Lds {
    float ry[kBufs][S][NW + 1][64];  // r_y of the last row of wave w at w + 1; zero at 0
    float z[kBufs][TS][NW + 1][64];  // z of the first row of wave w at w; zero at NW
    float4 b[kUnroll][NW][64];       // the last planes of b; read back by the thread that wrote
  };

  const StepArgs& a;
  Lds& l;
  int w, lane, z0, z1, yw, last_plane;
  bool gx_on;
  long plane, wave_row;
  int rows;      // of the wave's quad inside the volume (0: none)
  bool wave_on;  // the wave's rows are the tile's to write
  // Byte offsets of the thread's column in a quad of the dual and in a row of b, or kOutside; and
  // the same where the column is the tile's to write. (Rows outside the volume end past a window.)
  unsigned xq, xr, xq_out, xr_out;
  float R[TS][kRows][3], P[TS][kRows][3], Z[TS][kRows], PZ[kRows];
  // p_k, p_{k-1} (zero on the first step of a prox, whose m[0] is zero: r = p) and b of the next
  // plane, loaded a plane ahead.
  float pk[3][kRows], pm[3][kRows], bb[kRows];

  // Floats of a plane and of a component of the dual, and bytes of the wave's quad in a plane.
  __device__ __forceinline__ long dual_plane() const {
    return ROWS == Rows::filled ? a.dual_plane : plane;
  }
  __device__ __forceinline__ long dual_vol() const {
    return ROWS == Rows::filled ? a.dual_vol : a.vol;
  }
  __device__ __forceinline__ int dual_bytes() const {
    return ROWS == Rows::filled && rows > 0 ? 4 * kRows * a.nx : 4 * rows * a.nx;
  }

  __device__ __forceinline__ void load_dual(float (&v)[3][kRows], const float* p, long at,
                                            bool on) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const Window q(p + c * dual_vol() + at, dual_bytes(), on);
      if constexpr (ROWS != Rows::cut) {
        q.load4(v[c], xq);
      } else {
#pragma unroll
        for (int j = 0; j < kRows; ++j) v[c][j] = q.load(j < rows ? xq + 4u * j : kOutside);
      }
    }
  }
  __device__ __forceinline__ void load(int f) {
    const long z = static_cast<long>(min(f, a.nz - 1));
    const long at = z * plane + wave_row;
    const long dual_at = z * dual_plane() + wave_row;
    load_dual(pk, a.p_k, dual_at, true);
    if constexpr (!FIRST) load_dual(pm, a.p_km1, dual_at, a.first == 0);
    const Window b(a.b + at, 4 * rows * a.nx, true);
#pragma unroll
    for (int j = 0; j < kRows; ++j) bb[j] = b.load(xr + 4u * static_cast<unsigned>(j * a.nx));
  }

  // Component-wise rows of p on plane z, where that is the tile's to write.
  __device__ __forceinline__ void store(float* p, int z, const float (&v)[kRows][3]) {
    const bool on = p != nullptr && wave_on && z >= z0 && z < z1;
    const long at = static_cast<long>(max(z, 0)) * dual_plane() + wave_row;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const Window q(p + c * dual_vol() + at, dual_bytes(), on);
      if constexpr (ROWS != Rows::cut) {
        const float r[kRows] = {v[0][c], v[1][c], v[2][c], v[3][c]};
        q.stream4(r, xq_out);
      } else {
#pragma unroll
        for (int j = 0; j < kRows; ++j) q.stream(v[j][c], j < rows ? xq_out + 4u * j : kOutside);
      }
    }
  }

  __device__ __forceinline__ void planes_of_b(int u, float (&v)[kRows]) {
    const float4 q = l.b[u][w][lane];
    v[0] = q.x;
    v[1] = q.y;
    v[2] = q.z;
    v[3] = q.w;
  }

  // Stage s on plane f - s: takes r and p of that plane, leaves p and r of the step on the plane
  // below it.
  template <int U, int s>
  __device__ __forceinline__ void stage(int f, float (&rn)[kRows][3], float (&pn)[kRows][3]) {
    constexpr int kBuf = buf(U);
    constexpr int kLast = buf((U + kUnroll - 1) % kUnroll);  // of the plane before
    float bs[kRows];
    planes_of_b((U + kUnroll - s) % kUnroll, bs);
    l.ry[kBuf][s][w + 1][lane] = rn[kRows - 1][1];
    __syncthreads();
    const float ry_edge = l.ry[kBuf][s][w][lane];
    const float z_edge = l.z[kLast][s][w + 1][lane];
    const int zo = f - s - 1;  // plane of p_{k+s+1}
    const bool gz_on = zo >= 0 && zo < a.nz - 1;
    float z_first = 0.0f;
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      const float ry_up = j > 0 ? R[s][j > 0 ? j - 1 : 0][1] : ry_edge;
      const float zn = primal_value<EXACT>(bs[j], a.lambda, rn[j][0], R[s][j][0], rn[j][1],
                                           ry_up, rn[j][2], lane_below(rn[j][2]));
      const float zc = Z[s][j];
      const float z_dn = j < kRows - 1 ? Z[s][j < kRows - 1 ? j + 1 : j] : z_edge;
      const float qz = multiply_add<EXACT>(a.step, zc - zn, R[s][j][0]);
      const float qy = multiply_add<EXACT>(a.step, zc - z_dn, R[s][j][1]);
      const float qx = multiply_add<EXACT>(a.step, zc - lane_above(zc), R[s][j][2]);
      // A point outside the volume differs from one inside only in that no step updates its
      // component along the axis it is outside of, so it never reaches a point inside.
      const float q[3] = {gz_on ? qz : 0.0f,
                          yw + j >= 0 && yw + j < a.ny - 1 ? qy : 0.0f, gx_on ? qx : 0.0f};
      const float scale = ball_scale<EXACT>(multiply_add<EXACT>(
          q[2], q[2], multiply_add<EXACT>(q[1], q[1], q[0] * q[0])));
      if (j == 0) z_first = zn;
      Z[s][j] = zn;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const float next = q[c] * scale;
        const float old = P[s][j][c];
        R[s][j][c] = rn[j][c];
        P[s][j][c] = pn[j][c];
        pn[j][c] = next;
        if constexpr (s + 1 < T) rn[j][c] = multiply_add<EXACT>(a.m[s + 1], next - old, next);
      }
    }
    l.z[kBuf][s][w][lane] = z_first;
    if constexpr (s == T - 2) store(a.p_prev, zo, pn);
    if constexpr (s == T - 1) store(a.p_last, zo, pn);
    if constexpr (s + 1 < T) stage<U, s + 1>(f, rn, pn);
  }

  // The prox output on plane f - T from p_{k+T} there.
  template <int U>
  __device__ __forceinline__ void output(int f, const float (&pn)[kRows][3]) {
    constexpr int kBuf = buf(U);
    float bs[kRows];
    planes_of_b((U + kUnroll - T) % kUnroll, bs);
    l.ry[kBuf][S - 1][w + 1][lane] = pn[kRows - 1][1];
    __syncthreads();
    const float py_edge = l.ry[kBuf][S - 1][w][lane];
    const int zp = f - T;
    const Window x(a.x + static_cast<long>(max(zp, 0)) * plane + wave_row, 4 * rows * a.nx,
                   wave_on && zp >= z0 && zp < z1);
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      const float py_up = j > 0 ? pn[j > 0 ? j - 1 : 0][1] : py_edge;
      float v = primal_value<EXACT>(bs[j], a.lambda, pn[j][0], PZ[j], pn[j][1], py_up, pn[j][2],
                                    lane_below(pn[j][2]));
      PZ[j] = pn[j][0];
      if (a.to_index) v = index_from_real(v, a.nm2, a.inv_k02);
      x.store(v, xr_out + 4u * static_cast<unsigned>(j * a.nx));
    }
  }

  template <int U>
  __device__ __forceinline__ void planes(int f) {
    float rn[kRows][3], pn[kRows][3];
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        pn[j][c] = pk[c][j];
        rn[j][c] = FIRST ? pk[c][j]
                         : multiply_add<EXACT>(a.m[0], pk[c][j] - pm[c][j], pk[c][j]);
      }
    }
    l.b[U][w][lane] = float4{bb[0], bb[1], bb[2], bb[3]};
    load(f + 1);
    if constexpr (T > 0) stage<U, 0>(f, rn, pn);
    if constexpr (FINAL) output<U>(f, pn);
    if constexpr (U + 1 < kUnroll) {
      // The longer passes with the output end within a turn (128^3: 53 against 61 us); in the others
      // the test costs more, in scheduling across planes, than the planes it saves (256^3: 236
      // against 218 us).
      if (FINAL && f >= last_plane) return;
      planes<U + 1>(f + 1);
    }
  }
};

template <int T, bool FIRST, bool FINAL, Rows ROWS, bool EXACT>
__global__ void __launch_bounds__(kWaves * 64)
    __attribute__((amdgpu_waves_per_eu(kWaves / 4, kWaves / 4))) k_fgp_steps(StepArgs a) {
  using M = StepMarch<T, FIRST, FINAL, ROWS, EXACT>;
  __shared__ typename M::Lds lds;
  // Volume blockIdx.y of a batch of volumes that lie one after another.
  const long batch = static_cast<long>(blockIdx.y);
  a.b += batch * a.vol;
  const long dual_vol = ROWS == Rows::filled ? a.dual_vol : a.vol;
  a.p_k += 3 * batch * dual_vol;
  if (a.p_km1) a.p_km1 += 3 * batch * dual_vol;
  if (a.p_prev) a.p_prev += 3 * batch * dual_vol;
  if (a.p_last) a.p_last += 3 * batch * dual_vol;
  if (a.x) a.x += batch * a.vol;
  M m{a, lds};
  // The wave index is uniform across the wave: as a scalar it keeps the row arithmetic, the
  // windows and the y tests off the vector ALU.
  m.w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  m.lane = static_cast<int>(threadIdx.x) & 63;
  // Tiles of one chunk are consecutive (x fastest), so that tiles that share halos run on one
  // XCD and share its L2.
  const int tile = static_cast<int>(xcd_block());
  const int tx = tile % a.tiles_x;
  const int rest = tile / a.tiles_x;
  const int ty = rest % a.tiles_y;
  m.z0 = (rest / a.tiles_y) * a.zlen;
  m.z1 = min(m.z0 + a.zlen, a.nz);
  const int x = tx * a.tile_x - a.halo_x + m.lane;
  m.yw = ty * a.tile_y - a.halo_y + m.w * kRows;
  m.rows = m.yw < 0 ? 0 : max(0, min(kRows, a.ny - m.yw));
  m.wave_on = m.yw >= ty * a.tile_y && m.yw < (ty + 1) * a.tile_y;
  m.gx_on = x >= 0 && x < a.nx - 1;
  m.plane = static_cast<long>(a.ny) * a.nx;
  m.wave_row = m.rows > 0 ? static_cast<long>(m.yw) * a.nx : 0;
  const bool in_x = x >= 0 && x < a.nx;
  const bool out_x = in_x && x >= tx * a.tile_x && x < (tx + 1) * a.tile_x;
  m.xq = in_x ? 4u * static_cast<unsigned>(x * (ROWS == Rows::filled ? kRows : m.rows)) : kOutside;
  m.xr = in_x ? 4u * static_cast<unsigned>(x) : kOutside;
  m.xq_out = out_x ? m.xq : kOutside;
  m.xr_out = out_x ? m.xr : kOutside;
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    m.PZ[j] = 0.0f;
#pragma unroll
    for (int s = 0; s < T; ++s) {
      m.Z[s][j] = 0.0f;
#pragma unroll
      for (int c = 0; c < 3; ++c) m.R[s][j][c] = m.P[s][j][c] = 0.0f;
    }
  }
  float* const words = reinterpret_cast<float*>(&lds);
  for (int i = static_cast<int>(threadIdx.x); i < static_cast<int>(sizeof(lds) / 4);
       i += kWaves * 64) {
    words[i] = 0.0f;
  }
  __syncthreads();
  const int first_plane = max(m.z0 - M::HL, 0);
  m.last_plane = m.z1 - 1 + T;
  m.load(first_plane);
  for (int f = first_plane; f <= m.last_plane; f += M::kUnroll) m.template planes<0>(f);
}

__global__ void k_fill(float* d, long n, float v) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) d[i] = v;
}

}  // namespace

void fill(float* d, long n, float v, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_fill, dim3(blocks_for(n)), dim3(256), 0, s, d, n, v);
  check_launch("fill");
}

namespace {

// CUs of the current device, queried once per device.
int device_cus() {
  static std::atomic<int> cache[64];
  int dev = 0;
  check(hipGetDevice(&dev), "hipGetDevice");
  require(dev >= 0 && dev < 64, "tv: device index above 63");
  int cus = cache[dev].load(std::memory_order_relaxed);
  if (cus == 0) {
    check(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev),
          "hipDeviceGetAttribute");
    cus = std::max(cus, 1);
    cache[dev].store(cus, std::memory_order_relaxed);
  }
  return cus;
}

// Planes per z chunk for a grid of `tiles` tiles (one block per CU): the length that minimises the
// rounds of blocks per CU times the planes a block marches (its chunk and a halo of planes on
// either side, in turns of `turn` planes); the longest on ties.
int step_chunk(int steps, int halo, int turn, long tiles, int nz) {
  const long slots = device_cus();
  int best = nz;
  long best_cost = -1;
  for (int zl = nz; zl >= 1; --zl) {
    const long chunks = (nz + zl - 1) / zl;
    const long planes = (std::min(zl + halo, nz + steps) + turn - 1) / turn * turn;
    const long cost = (tiles * chunks + slots - 1) / slots * planes;
    if (best_cost < 0 || cost < best_cost) {
      best_cost = cost;
      best = zl;
    }
  }
  return best;
}

// Rows of a plane of the dual that holds whole quads.
long whole_quads(int ny) { return (static_cast<long>(ny) + kRows - 1) / kRows * kRows; }

// Volumes whose rows do not fill their last quad round every operation, as their results always have.
template <int T, bool FIRST, bool FINAL>
void launch_steps(StepArgs a, hipStream_t s, int batch, bool exact) {
  const auto cut = [](int n, int width, int& own, int& halo) {
    halo = n <= width ? 0 : kHalo;
    own = width - 2 * halo;
    return (n + own - 1) / own;
  };
  a.tiles_x = cut(a.nx, 64, a.tile_x, a.halo_x);
  a.tiles_y = cut(a.ny, kWaves * kRows, a.tile_y, a.halo_y);
  const int tiles = a.tiles_x * a.tiles_y;
  a.zlen = step_chunk(T, 2 * T + (FINAL ? 1 : 0), FINAL ? 1 : T + 1,
                      static_cast<long>(tiles) * batch, a.nz);
  const int chunks = (a.nz + a.zlen - 1) / a.zlen;
  const dim3 grid(static_cast<unsigned>(tiles * chunks), static_cast<unsigned>(batch));
  const dim3 block(kWaves * 64);
  if (a.dual_plane != whole_quads(a.ny) * a.nx) {
    hipLaunchKernelGGL((k_fgp_steps<T, FIRST, FINAL, Rows::cut, true>), grid, block, 0, s, a);
  } else if (a.ny % kRows != 0) {
    hipLaunchKernelGGL((k_fgp_steps<T, FIRST, FINAL, Rows::filled, true>), grid, block, 0, s, a);
  } else if (exact) {
    hipLaunchKernelGGL((k_fgp_steps<T, FIRST, FINAL, Rows::whole, true>), grid, block, 0, s, a);
  } else {
    hipLaunchKernelGGL((k_fgp_steps<T, FIRST, FINAL, Rows::whole, false>), grid, block, 0, s, a);
  }
}

template <int T>
void launch_steps_of(const StepArgs& a, hipStream_t s, int batch, bool exact) {
  if (a.x) {
    if constexpr (T < kMaxSteps) launch_steps<T, false, true>(a, s, batch, exact);
  } else if (T >= 2 && a.first) {
    // The first of several passes, of 2 to 4 steps: without p_{k-1} at all (256^3: 193 against 200 us
    // for 3 steps, 219 against 240 us for 4; 384^3: 529 against 550 us for 3; a prox of 2 + 2 steps at
    // 128^3 79.5 against 81.5 us).
    launch_steps<T, T >= 2, false>(a, s, batch, exact);
  } else {
    launch_steps<T, false, false>(a, s, batch, exact);
  }
}

// `steps` FGP steps in one pass (up to kMaxSteps); with x set, the prox output after them (up to
// kMaxSteps - 1; 0 steps: of p_k).
void fgp_steps(int steps, const StepArgs& a, hipStream_t s, int batch, bool exact) {
  require(steps + (a.x ? 1 : 0) <= kMaxSteps, "tv: too many steps in a pass");
  switch (steps) {
    case 0: launch_steps<0, true, true>(a, s, batch, exact); break;
    case 1: launch_steps_of<1>(a, s, batch, exact); break;
    case 2: launch_steps_of<2>(a, s, batch, exact); break;
    case 3: launch_steps_of<3>(a, s, batch, exact); break;
    default: launch_steps_of<4>(a, s, batch, exact); break;
  }
  check_launch("fgp_steps");
}

// Floats of one dual buffer (three components per volume of the batch, one volume's after
// another's), rounded up to 256 bytes so that every buffer of a workspace starts 256-byte
// aligned.
std::size_t dual_floats(int nz, long rows, int nx, int batch = 1) {
  const std::size_t three = 3 * static_cast<std::size_t>(nz) * rows * nx * batch;
  return (three + 63) / 64 * 64;
}

}  // namespace

std::size_t TvState::workspace_floats(int nz, int ny, int nx) { return 4 * dual_floats(nz, ny, nx); }

TvState::TvState(int nz, int ny, int nx, int batch)
    : nz_(nz), ny_(ny), nx_(nx), vol_(static_cast<long>(nz) * ny * nx), rows_(whole_quads(ny)),
      cap_(batch), owned_(4 * dual_floats(nz, rows_, nx, std::max(batch, 1))) {
  require(batch >= 1 && batch <= 65535, "tv: the batch must be 1 to 65535");
  const std::size_t stride = dual_floats(nz, rows_, nx, batch);
  for (int i = 0; i < 4; ++i) p_[i] = owned_.get() + i * stride;
}

TvState::TvState(int nz, int ny, int nx, float* workspace, std::size_t floats)
    : nz_(nz), ny_(ny), nx_(nx), vol_(static_cast<long>(nz) * ny * nx), rows_(whole_quads(ny)) {
  require(workspace_floats(nz, ny, nx) <= floats, "tv: the workspace is too small");
  if (4 * dual_floats(nz, rows_, nx) > floats) rows_ = ny;
  const std::size_t stride = dual_floats(nz, rows_, nx);
  for (int i = 0; i < 4; ++i) p_[i] = workspace + i * stride;
}

void TvState::reset(hipStream_t s, int batch) {
  require(batch >= 1 && batch <= cap_, "tv: batch beyond the state's capacity");
  batch_ = batch;
  fill(p_[0], 3 * nz_ * rows_ * nx_ * batch, 0.0f, s);
  cur_ = 0;
}

std::size_t TvState::bytes() const { return owned_.bytes(); }

// tv_prox of the reference (src/cpu/tv.cpp:7-44): r <- p, `inner` FGP steps, out = primal(p).
// The steps go in as few passes as they need, the last of which forms the output where that leaves
// it at most three steps. The dual iterates rotate through four buffers: a pass of T steps reads p_k and p_{k-1} (r is formed
// inside it) and writes p_{k+T-1} and p_{k+T} to buffers nobody reads in that pass; the last pass
// skips p_{k+T-1}, which the next call does not read (its first step uses r = p). The prox leaves
// p in buffer cur_ for the next call.
void TvState::prox(const float* b, float* out, float lambda, int inner, hipStream_t s,
                   bool to_index, float nm2, float inv_k02, Event* t0, Event* t1) {
  if (nx_ > 512) throw InvalidArgument("tv: volume side above 512");
  const float step = 1.0f / (12.0f * lambda);
  // An output that overlaps b is written only by a pass without steps: the stages of the others
  // read b beyond their own points, its last stage at them alone.
  const bool apart = out + vol_ * batch_ <= b || b + vol_ * batch_ <= out;
  // Step counts that are multiples of four: passes of four steps and one of the output alone move
  // the fewest bytes; in small volumes, where a plane's latency bounds a pass, the output counts as
  // a step more and the shares are smaller. A FISTA iteration of 4 / 8 / 20 steps this way and that:
  // 479 / 751 / 1570 against 560 / 807 / 1627 us at 256^3, 216 / 340 / 711 against 251 / 362 / 742
  // at 192^3, 233 / 405 / 919 against 286 / 412 / 896 at 162^3, 114 / 176 / 361 against 121 / 169 /
  // 350 at 128^3, 58 / 88 / 176 against 56 / 82 / 169 at 64^3.
  constexpr long kLarge = 1L << 22;
  const bool whole = inner % kMaxSteps == 0 && vol_ * batch_ >= kLarge;
  const bool joined = fused_ && apart && inner > 0 && !whole;
  const int most = fused_ ? kMaxSteps : 1;
  const int passes = (inner + (joined ? 1 : 0) + most - 1) / most;
  StepArgs a{};
  a.b = b;
  a.vol = vol_;
  a.dual_plane = rows_ * nx_;
  a.dual_vol = nz_ * a.dual_plane;
  a.nz = nz_;
  a.ny = ny_;
  a.nx = nx_;
  a.lambda = lambda;
  a.step = step;
  a.to_index = to_index ? 1 : 0;
  a.nm2 = nm2;
  a.inv_k02 = inv_k02;
  float t = 1.0f;
  float m_prev = 0.0f;
  int cur = cur_;
  int prev = (cur_ + 1) % 4;
  int left = inner;
  launches_ = passes;
  if (t0) t0->record(s);
  for (int k = 0; k < passes; ++k) {
    // Nearly equal shares of what is left, the larger ones first.
    const int steps = (left + passes - k - 1) / (passes - k);
    const bool last = k + 1 == passes;
    left -= steps;
    int f[2] = {0, 0};
    for (int i = 0, n = 0; i < 4; ++i) {
      if (i != cur && i != prev && n < 2) f[n++] = i;
    }
    a.p_k = p_[cur];
    a.p_km1 = p_[prev];
    // A pass of one step leaves p_k as the previous iterate.
    a.p_prev = last || steps == 1 ? nullptr : p_[f[0]];
    a.p_last = p_[f[1]];
    a.x = last && joined ? out : nullptr;
    a.first = k == 0 ? 1 : 0;
    for (int i = 0; i < steps; ++i) {
      a.m[i] = m_prev;
      const float tn = fista_t(t);
      m_prev = (t - 1.0f) / tn;
      t = tn;
    }
    fgp_steps(steps, a, s, batch_, exact_);
    prev = steps == 1 ? cur : f[0];
    cur = f[1];
  }
  if (t1) t1->record(s);
  cur_ = cur;
  if (joined) return;
  a.p_k = p_[cur_];
  a.p_km1 = a.p_prev = a.p_last = nullptr;
  a.x = out;
  a.first = 1;
  fgp_steps(0, a, s, batch_, exact_);
}

}  // namespace qh
