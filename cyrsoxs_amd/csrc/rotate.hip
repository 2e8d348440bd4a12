// E-angle image rotation, rotation mask, angle averaging and detector warp
// (replaces cublasSscal(NaN) + nppiWarpAffine + computeRotationMask +
// cublasSaxpy + averageRotation/cublasSscal + the detector warp:
// src/cudaMain.cu:830-971, include/uniaxial.h:958-992).
//
// Sums over angles are FP64 and run in angle order (deterministic, no atomics).
// Bilinear convention (NPP is closed; the build's own, shared with the oracle):
// destination pixel (X, Y) samples the source at the back-mapped point
// (inverse affine, FP64); it is written iff that point lies in
// [0, Nx-1] x [0, Ny-1]; taps of exactly zero weight are skipped.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <utility>
#include <vector>

#include "geom.hpp"
#include "kernels.hpp"

namespace cyr {

namespace {

struct Inv6 { double c[6]; };

// Pixel of this thread in the rotation kernels: 256-thread blocks cover 16 x 16
// tiles, each wave an 8 x 8 quadrant, so a wave's rotated source footprint is
// compact (a 64-pixel row segment maps to a 64-pixel line of source rows at
// most angles, touching many more cache lines).  Tiles come from `tiles`
// (ty << 16 | tx, sorted by distance from the rotation centre) in XCD order:
// XCD x gets the x-th annulus, and a rotation about the centre maps an annulus
// onto itself, so each XCD's L2 holds only its annulus of the source planes.
__device__ inline bool tile_pixel(const uint32_t *__restrict__ tiles, uint32_t ntiles, uint32_t nx, uint32_t ny,
                                  uint32_t &X, uint32_t &Y) {
  const uint32_t q = xcd_tile(blockIdx.x, gridDim.x);
  if (q >= ntiles) return false;
  const uint32_t tt = tiles[q];
  const uint32_t w = threadIdx.x >> 6, l = threadIdx.x & 63;
  X = (tt & 0xffffu) * 16 + (w & 1) * 8 + (l & 7);
  Y = (tt >> 16) * 16 + (w >> 1) * 8 + (l >> 3);
  return X < nx && Y < ny;
}

// nb angles in turn (the sums stay in angle order): the first batch of a pattern starts
// them, the last one divides and stores the average (128^2, 6 angles: two fills, the sum,
// the average and the copy to the output, 5 launches of 4 to 6 us -> one).
template <typename T>
__global__ void __launch_bounds__(256) rotate_accumulate_kernel(const T *__restrict__ proj, double *__restrict__ acc,
                                                                uint32_t *__restrict__ count, uint32_t nx, uint32_t ny,
                                                                const double *__restrict__ inv_tab, uint32_t nb,
                                                                uint32_t nA, int first, int last, int rot_mask,
                                                                AvgSink<T> avg) {
  const uint64_t P = (uint64_t)nx * ny;
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P) return;
  const uint32_t Y = (uint32_t)(t / nx), X = (uint32_t)(t - (uint64_t)Y * nx);
  double s = first ? 0.0 : acc[t];
  uint32_t c = rot_mask && !first ? count[t] : 0;
#pragma unroll 2
  for (uint32_t b = 0; b < nb; b++) {
    double inv[6];
#pragma unroll
    for (int i = 0; i < 6; i++) inv[i] = inv_tab[6 * (uint64_t)b + i];
    double v;
    if (!bilinear_sample<T>(proj + (uint64_t)b * P, nx, ny, inv, X, Y, &v)) v = __longlong_as_double(0x7ff8000000000000ll);
    if (rot_mask) {
      if (!isnan(v)) {
        s += v;
        c += 1;
      }
    } else {
      s += v;
    }
  }
  if (last) {
    avg.store(0, t, rot_mask ? (c == 0 ? 0.0 : s * (1.0 / (c * 1.0))) : s * (1.0 / (double)nA));
    return;
  }
  acc[t] = s;
  if (rot_mask) count[t] = c;
}

// Material frame: every angle's projection proj[ne][nA][P] rotated, masked and averaged
// (grid z: energies).  A block holds one 8 x 8 quadrant of a tile, its four waves a
// quarter of the angles each; their FP64 sums meet in LDS in angle order.  Each angle has
// a plane of its own, so the split costs no sharing of taps, and small planes get four
// times the waves (128^2, 18 angles: 16 us per energy in a launch of its own -> all of 6
// energies 17 us).
template <typename T>
__global__ void __launch_bounds__(256) rotate_all_kernel(const T *__restrict__ proj, const double *__restrict__ inv_tab,
                                                         uint32_t nA, uint32_t nx, uint32_t ny, int rot_mask,
                                                         AvgSink<T> avg, const uint32_t *__restrict__ tiles,
                                                         uint32_t ntiles) {
  __shared__ double sum[4][64];
  __shared__ uint32_t num[4][64];
  const uint64_t P = (uint64_t)nx * ny;
  const uint32_t b = xcd_tile(blockIdx.x, gridDim.x);
  if (b >= 4 * ntiles) return;  // (the whole block)
  proj += (uint64_t)blockIdx.z * nA * P;
  const uint32_t tt = tiles[b >> 2], w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const uint32_t X = (tt & 0xffffu) * 16 + (b & 1) * 8 + (l & 7);
  const uint32_t Y = (tt >> 16) * 16 + ((b >> 1) & 1) * 8 + (l >> 3);
  const bool in = X < nx && Y < ny;
  const uint64_t t = (uint64_t)Y * nx + X;
  double acc = 0;
  uint32_t cnt = 0;
  const uint32_t a0 = (uint32_t)((uint64_t)nA * w / 4), a1 = in ? (uint32_t)((uint64_t)nA * (w + 1) / 4) : a0;
  // independent gathers per angle; unrolling lets several be in flight (the sum
  // itself stays in angle order)
#pragma unroll 4
  for (uint32_t a = a0; a < a1; a++) {
    double inv[6];
#pragma unroll
    for (int i = 0; i < 6; i++) inv[i] = inv_tab[6 * (uint64_t)a + i];
    double v;
    if (!bilinear_sample<T>(proj + (uint64_t)a * P, nx, ny, inv, X, Y, &v)) v = __longlong_as_double(0x7ff8000000000000ll);
    if (rot_mask) {
      if (!isnan(v)) {
        acc += v;
        cnt++;
      }
    } else {
      acc += v;
    }
  }
  sum[w][l] = acc;
  num[w][l] = cnt;
  __syncthreads();
  if (w != 0 || !in) return;
  for (int i = 1; i < 4; i++) {
    acc += sum[i][l];
    cnt += num[i][l];
  }
  avg.store(blockIdx.z, t, rot_mask ? (cnt == 0 ? 0.0 : acc * (1.0 / (cnt * 1.0))) : acc * (1.0 / (double)nA));
}

// Laboratory frame: every angle's intensity from the per-pixel quadratic form
// q = (q0, q1, q2): I(theta) = c^2 q0 + s^2 q1 + 2 c s q2.  Bilinear sampling is
// linear, so the three components are sampled (same taps, weights and validity
// as bilinear_sample; a tap of zero weight contributes nothing, NaN included)
// and combined once per angle, in the forms' precision.  Each
// angle's back-mapped point, taps and weights serve NE energies.

// Back-mapped point of one (pixel, angle): validity, top-left tap, fractions.
struct QPoint {
  uint32_t x0, y0;
  double sx, sy, fx, fy;
  bool inside;
};

__device__ inline QPoint quad_point(const double *inv, uint32_t X, uint32_t Y, uint32_t nx, uint32_t ny) {
  QPoint p;
  back_map_point(inv, X, Y, p.sx, p.sy);
  const double sx = p.sx, sy = p.sy;
  p.inside = sx >= 0 && sx <= (double)(nx - 1) && sy >= 0 && sy <= (double)(ny - 1);
  const double fx0 = p.inside ? floor(sx) : 0.0, fy0 = p.inside ? floor(sy) : 0.0;
  p.x0 = (uint32_t)fx0;
  p.y0 = (uint32_t)fy0;
  p.fx = p.inside ? sx - fx0 : 0.0;
  p.fy = p.inside ? sy - fy0 : 0.0;
  return p;
}

// One record (q0, q1, q2) of a plane of quadratic forms.
template <typename T> struct Tap3;
template <> struct Tap3<float> { typedef float v __attribute__((ext_vector_type(3))); };
template <> struct Tap3<double> { typedef double v __attribute__((ext_vector_type(3))); };
template <typename T> using Rec = typename Tap3<T>::v;

// The four taps of p (clamped into the image) for NE energy planes.
template <typename T, int NE>
__device__ inline void quad_gather(const T *const (&qp)[NE], const QPoint &p, uint32_t nx, uint32_t ny,
                                   Rec<T> (&tp)[NE][4]) {
  const uint32_t x1 = p.x0 + 1 < nx ? p.x0 + 1 : p.x0, y1 = p.y0 + 1 < ny ? p.y0 + 1 : p.y0;
  const uint32_t off[4] = {quad_index(p.x0, p.y0, nx, ny), quad_index(x1, p.y0, nx, ny), quad_index(p.x0, y1, nx, ny),
                           quad_index(x1, y1, nx, ny)};  // P < 2^32
#pragma unroll
  for (int e = 0; e < NE; e++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const T *r = qp[e] + (uint64_t)off[i] * kQuadRecord;
      tp[e][i] = Rec<T>{r[0], r[1], r[2]};
    }
}

// Bilinear sums (q0, q1, q2) of NE energies at point p from its taps tp.
template <typename T, int NE>
__device__ inline void quad_sums(const QPoint &p, const Rec<T> (&tp)[NE][4], T (&sm)[NE][3]) {
  const double gx = 1 - p.fx, gy = 1 - p.fy;
  const double wd[4] = {gx * gy, p.fx * gy, gx * p.fy, p.fx * p.fy};
  // taps are interpolated in the forms' precision (the weights rounded once per
  // angle); which taps count (weight exactly 0 or not) is decided on the FP64
  // weights, and the sum over angles stays FP64
  T w[4];
  bool z[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    w[i] = (T)wd[i];
    z[i] = wd[i] == 0;
  }
#pragma unroll
  for (int e = 0; e < NE; e++) {
    T s0 = 0, s1 = 0, s2 = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const Rec<T> t = tp[e][i];
      s0 += w[i] * (z[i] ? (T)0 : t.x);
      s1 += w[i] * (z[i] ? (T)0 : t.y);
      s2 += w[i] * (z[i] ? (T)0 : t.z);
    }
    sm[e][0] = s0;
    sm[e][1] = s1;
    sm[e][2] = s2;
  }
}

// Adds one angle's intensity (coefficients c = (c^2, s^2, 2cs)) from the sums sm
// (NaN where the point is outside) to the FP64 sums of NE energies.
template <typename T, int NE>
__device__ inline void quad_combine(bool inside, const T (&sm)[NE][3], const double *c, int rot_mask,
                                    double (&acc)[NE], uint32_t (&cnt)[NE]) {
  const T c0 = (T)c[0], c1 = (T)c[1], c2 = (T)c[2];
#pragma unroll
  for (int e = 0; e < NE; e++) {
    const double v =
        inside ? (double)(c0 * sm[e][0] + c1 * sm[e][1] + c2 * sm[e][2]) : __longlong_as_double(0x7ff8000000000000ll);
    if (rot_mask) {
      const bool ok = !isnan(v);
      acc[e] += ok ? v : 0.0;
      cnt[e] += ok ? 1u : 0u;
    } else {
      acc[e] += v;
    }
  }
}

template <typename T, int NE>
__device__ inline void quad_add(const QPoint &p, const Rec<T> (&tp)[NE][4], const double *c, int rot_mask,
                                double (&acc)[NE], uint32_t (&cnt)[NE]) {
  T sm[NE][3];
  quad_sums<T, NE>(p, tp, sm);
  quad_combine<T, NE>(p.inside, sm, c, rot_mask, acc, cnt);
}

template <typename O, int NE>
__device__ inline void quad_store(const AvgSink<O> &avg, uint64_t t, uint32_t e0, uint32_t ne, uint32_t nA,
                                  int rot_mask, const double (&acc)[NE], const uint32_t (&cnt)[NE]) {
#pragma unroll
  for (int e = 0; e < NE; e++) {
    if (e0 + e >= ne) break;
    avg.store(e0 + e, t,
              rot_mask ? (cnt[e] == 0 ? 0.0 : acc[e] * (1.0 / (cnt[e] * 1.0))) : acc[e] * (1.0 / (double)nA));
  }
}

// Every angle of one pixel, in angle order.
template <typename T, int NE>
__device__ inline void quad_pixel(const T *const (&qp)[NE], const double *__restrict__ inv_tab,
                                  const double *__restrict__ coef, uint32_t nA, uint32_t nx, uint32_t ny, uint32_t X,
                                  uint32_t Y, int rot_mask, double (&acc)[NE], uint32_t (&cnt)[NE]) {
#pragma unroll 2
  for (uint32_t a = 0; a < nA; a++) {
    const QPoint p = quad_point(inv_tab + 6 * (uint64_t)a, X, Y, nx, ny);
    Rec<T> tp[NE][4];
    quad_gather<T, NE>(qp, p, nx, ny, tp);
    quad_add<T, NE>(p, tp, coef + 3 * (uint64_t)a, rot_mask, acc, cnt);
  }
}

// grid y: groups of NE energies (ne in total)
template <typename T, typename O, int NE>
__global__ void __launch_bounds__(256) rotate_quad_kernel(const T *__restrict__ quad, const double *__restrict__ inv_tab,
                                                          const double *__restrict__ coef, uint32_t nA, uint32_t nx,
                                                          uint32_t ny, int rot_mask, AvgSink<O> avg,
                                                          uint32_t ne, const uint32_t *__restrict__ tiles,
                                                          uint32_t ntiles) {
  const uint64_t P = (uint64_t)nx * ny;
  uint32_t X, Y;
  if (!tile_pixel(tiles, ntiles, nx, ny, X, Y)) return;
  const uint32_t e0 = blockIdx.z * NE;
  const T *qp[NE];
#pragma unroll
  for (int e = 0; e < NE; e++) qp[e] = quad + (uint64_t)(e0 + e < ne ? e0 + e : e0) * P * kQuadRecord;
  double acc[NE] = {};
  uint32_t cnt[NE] = {};
  quad_pixel<T, NE>(qp, inv_tab, coef, nA, nx, ny, X, Y, rot_mask, acc, cnt);
  quad_store<O, NE>(avg, (uint64_t)Y * nx + X, e0, ne, nA, rot_mask, acc, cnt);
}

// The same for planes too small to fill the chip: S waves of a block take S runs of the
// angles for one 8 x 8 quadrant of a tile and one energy, and their FP64 sums meet in
// LDS in angle order.  The chain of dependent gathers per wave is S times shorter and
// there are 4 S times as many waves as one tile per block and four energies give:
// 256^2, one energy, 36 angles: 70 us (quarter-turn orbits, 64 blocks) -> 20 us; 64^2,
// 3 energies, 6 angles: 32 -> 6.5 us.
template <typename T, typename O, int S>
__global__ void __launch_bounds__(64 * S) rotate_quad_split_kernel(const T *__restrict__ quad,
                                                                   const double *__restrict__ inv_tab,
                                                                   const double *__restrict__ coef, uint32_t nA,
                                                                   uint32_t nx, uint32_t ny, int rot_mask,
                                                                   AvgSink<O> avg,
                                                                   const uint32_t *__restrict__ tiles,
                                                                   uint32_t ntiles) {
  __shared__ double sum[S][64];
  __shared__ uint32_t num[S][64];
  const uint64_t P = (uint64_t)nx * ny;
  const uint32_t b = xcd_tile(blockIdx.x, gridDim.x);
  if (b >= 4 * ntiles) return;  // (the whole block)
  const uint32_t tt = tiles[b >> 2], w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const uint32_t X = (tt & 0xffffu) * 16 + (b & 1) * 8 + (l & 7);
  const uint32_t Y = (tt >> 16) * 16 + ((b >> 1) & 1) * 8 + (l >> 3);
  const uint32_t e = blockIdx.z;
  const bool in = X < nx && Y < ny;
  double acc[1] = {0};
  uint32_t cnt[1] = {0};
  if (in) {
    const uint32_t a0 = (uint32_t)((uint64_t)nA * w / S), a1 = (uint32_t)((uint64_t)nA * (w + 1) / S);
    const T *qp[1] = {quad + (uint64_t)e * P * kQuadRecord};
    quad_pixel<T, 1>(qp, inv_tab + 6 * (uint64_t)a0, coef + 3 * (uint64_t)a0, a1 - a0, nx, ny, X, Y, rot_mask, acc,
                     cnt);
  }
  sum[w][l] = acc[0];
  num[w][l] = cnt[0];
  __syncthreads();
  if (w != 0 || !in) return;
  for (int i = 1; i < S; i++) {
    acc[0] += sum[i][l];
    cnt[0] += num[i][l];
  }
  quad_store<O, 1>(avg, (uint64_t)Y * nx + X, e, e + 1, nA, rot_mask, acc, cnt);
}

// Tiles of the general order beyond every finite plane value: the averages
// rotate_quad_kernel would form there (NaN, or 0 with the rotation mask), as in
// orbit_fill_kernel.  Same tile and pixel layout as tile_pixel.
template <typename O, int NE>
__global__ void __launch_bounds__(256) quad_fill_kernel(AvgSink<O> avg, uint32_t nx, uint32_t ny,
                                                        uint32_t ne, int rot_mask, const uint32_t *__restrict__ tiles,
                                                        uint32_t first) {
  const uint64_t P = (uint64_t)nx * ny;
  const uint32_t tt = tiles[first + blockIdx.x];
  const uint32_t w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const uint32_t X = (tt & 0xffffu) * 16 + (w & 1) * 8 + (l & 7);
  const uint32_t Y = (tt >> 16) * 16 + (w >> 1) * 8 + (l >> 3);
  if (X >= nx || Y >= ny) return;
  const uint32_t e0 = blockIdx.z * NE;
  const double fill = rot_mask ? 0.0 : __longlong_as_double(0x7ff8000000000000ll);
#pragma unroll
  for (int e = 0; e < NE; e++)
    if (e0 + e < ne) avg.store(e0 + e, (uint64_t)Y * nx + X, fill);
}

// Quarter-turn orbits (square N x N planes whose angle list holds Q quarter turns
// of A4 steps: angle a + q A4 is angle a plus 90q degrees).  The image rotation
// turns about (N/2, N/2), so with s(X, Y) = (N - Y, X) (a 90-degree turn of the
// pixel grid) the point pixel x samples at angle a + q A4 is the point pixel
// s^q(x) samples at angle a.  One lane owns the orbit x, s x, s^2 x, s^3 x of a
// pixel with X - N/2 in [1, N/2 - 1] and Y - N/2 in [0, N/2 - 1] (these orbits tile
// [1, N-1]^2 minus the centre): it back-maps and gathers each (s^i x, a < A4) once
// and serves the Q (pixel, angle) pairs that sample there.
//
// The pairs' own FP64 back-maps (contraction off) differ from the shared point,
// evaluated with fused multiply-adds, by the rounding of the angle tables and
// of the evaluation (~N 1e-15 pixels: at most 4e-12 over every pair of a 4096^2
// plane with 720 angles).  When the shared point lies farther than the margin
// 1e-9 + N 1e-12 from every cell edge and from the image border, all Q pairs have
// its tap cell, validity and nonzero weights, so they reuse its bilinear sums
// (only the weights' last bits can differ from a pair's own).  Such points take
// the lean path: no zero-weight tests, taps through 32-bit buffer offsets (the
// plane is below 2 GiB), the intensity in the forms' precision, and one value
// for the pairs q and q + 2 when their coefficients are equal (`share`).  The
// rest (a point on or near a pixel edge: angles at exact multiples of 90 degrees,
// or special angles such as 60 degrees on the axes) is recorded per angle in a
// 64-bit mask and replayed after each run of 64 angles: there each pair back-maps
// its own point and gathers its own taps, as quad_pixel does.
// Validity and NaN taps are therefore decided exactly as per pair; only the order
// of the FP64 sums over angles differs.  Without the rotation mask a point
// outside the image marks its pairs' pixels NaN (the value the sum would reach).
// Row 0, column 0 and the centre (the tail blocks after the orbit tiles) take
// every angle directly.

// (q0, q1, q2) of the record at byte offset `off` of a plane; offsets past the
// buffer's size read zeros (only taps of points that take the exact path do).
template <typename T> __device__ inline typename Tap3<T>::v tap_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_amdgcn_raw_buffer_load_b96(r, off, 0, 0);
  } else {
    // 24-byte records sit at 8-byte alignment: three 8-byte loads
    typedef int i2 __attribute__((ext_vector_type(2)));
    const i2 a = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
    const i2 b = __builtin_amdgcn_raw_buffer_load_b64(r, off + 8, 0, 0);
    const i2 c = __builtin_amdgcn_raw_buffer_load_b64(r, off + 16, 0, 0);
    typename Tap3<double>::v v;
    v.x = __builtin_bit_cast(double, ((unsigned long long)(unsigned)a.y << 32) | (unsigned)a.x);
    v.y = __builtin_bit_cast(double, ((unsigned long long)(unsigned)b.y << 32) | (unsigned)b.x);
    v.z = __builtin_bit_cast(double, ((unsigned long long)(unsigned)c.y << 32) | (unsigned)c.x);
    return v;
  }
}

// Buffer resource word 3 of a raw (untyped) buffer on gfx9-family devices.
constexpr int kRawBufferFlags = 0x00020000;

// Row 0 (n pixels), column 0 below it (n - 1) and the centre, which are in no orbit: pixel
// j of them by every angle, a quarter of the angles a wave.  Pixels farther than rcut from
// the centre sample nothing finite.
template <typename T, typename O, int NE, bool RM, int R>
__device__ inline void orbit_tail(const T *const (&qp)[NE], const double *__restrict__ inv_tab,
                                  const double *__restrict__ coef, uint32_t nA, uint32_t n, double rcut, uint32_t j,
                                  uint32_t w, uint32_t l, uint32_t e0, uint32_t ne, AvgSink<O> avg,
                                  double (&sum)[4][4][NE][64], uint32_t (&num)[R][R][NE][64]) {
  const uint32_t h = n / 2;
  const bool in = j < 2 * n;
  const uint32_t X = j < n ? j : (j < 2 * n - 1 ? 0 : h);
  const uint32_t Y = j < n ? 0 : (j < 2 * n - 1 ? j - n + 1 : h);
  double acc[NE] = {};
  uint32_t cnt[NE] = {};
  const double dx = (double)X - h, dy = (double)Y - h;
  if (in && dx * dx + dy * dy <= rcut * rcut) {
    const uint32_t a0 = (uint32_t)((uint64_t)nA * w / 4), a1 = (uint32_t)((uint64_t)nA * (w + 1) / 4);
    quad_pixel<T, NE>(qp, inv_tab + 6 * (uint64_t)a0, coef + 3 * (uint64_t)a0, a1 - a0, n, n, X, Y, RM, acc, cnt);
  } else if constexpr (!RM) {
#pragma unroll
    for (int e = 0; e < NE; e++) acc[e] = __longlong_as_double(0x7ff8000000000000ll);
  }
#pragma unroll
  for (int e = 0; e < NE; e++) {
    sum[w][0][e][l] = acc[e];
    if constexpr (RM) num[w][0][e][l] = cnt[e];
  }
  __syncthreads();
  if (w != 0 || !in) return;
#pragma unroll
  for (int e = 0; e < NE; e++)
    for (int i = 1; i < 4; i++) {
      acc[e] += sum[i][0][e][l];
      if constexpr (RM) cnt[e] += num[i][0][e][l];
    }
  quad_store<O, NE>(avg, (uint64_t)Y * n + X, e0, ne, nA, RM, acc, cnt);
}

// A block holds one 8 x 8 quadrant of a tile of orbits; its wave i samples the points of
// orbit pixel i and serves pixel s^-q(i) from them (one pixel per wave, not four in
// turn: four times the waves and a quarter of the chain of gathers for the same work;
// 512^2 FP64 film, 10 energies x 72 angles: 128 us for one energy -> 111 us for all ten;
// 2048^2 film, 10 energies x 180 angles: 1.19 ms, as before).  The waves' sums meet in LDS,
// added in orbit order.
template <typename T, typename O, int NE, int Q, bool RM>
__global__ void __launch_bounds__(256) rotate_orbit_kernel(const T *__restrict__ quad, const double *__restrict__ inv_tab,
                                                           const double *__restrict__ coef,
                                                           const T *__restrict__ coef_t, uint32_t nA, uint32_t A4,
                                                           uint32_t n, AvgSink<O> avg, uint32_t ne,
                                                           const uint32_t *__restrict__ otiles, uint32_t n_otiles,
                                                           double rcut, int share) {
  __shared__ double sum[4][4][NE][64];
  __shared__ uint32_t num[RM ? 4 : 1][RM ? 4 : 1][NE][64];
  const uint64_t P = (uint64_t)n * n;
  const uint32_t h = n / 2;
  const uint32_t qb = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t e0 = blockIdx.z * NE;
  const uint32_t i = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  const T *qp[NE];
#pragma unroll
  for (int e = 0; e < NE; e++) qp[e] = quad + (uint64_t)(e0 + e < ne ? e0 + e : e0) * P * kQuadRecord;
  if (qb >= 4 * n_otiles) {
    orbit_tail<T, O, NE, RM>(qp, inv_tab, coef, nA, n, rcut, (qb - 4 * n_otiles) * 64 + l, i, l, e0, ne, avg, sum, num);
    return;
  }
  const uint32_t tt = otiles[qb >> 2];
  const uint32_t u = (tt & 0xffffu) * 16 + (qb & 1) * 8 + (l & 7) + 1;
  const uint32_t v = (tt >> 16) * 16 + ((qb >> 1) & 1) * 8 + (l >> 3);
  const bool in = u < h && v < h;
  // orbit pixels s^j(x), j = 0..3 (idle lanes: the orbit of (h, h), nothing stored)
  const uint32_t X0 = in ? h + u : h, Y0 = in ? h + v : h;
  auto px = [&](uint32_t j) { return j == 0 ? X0 : j == 1 ? n - Y0 : j == 2 ? n - X0 : Y0; };
  auto py = [&](uint32_t j) { return j == 0 ? Y0 : j == 1 ? X0 : j == 2 ? n - Y0 : n - X0; };
  const uint32_t PXi = px(i), PYi = py(i);
  const double hc = 0.5 * (double)(n - 1);
  const double m = 1e-9 + 1e-12 * (double)n;
  constexpr uint32_t rb = kQuadRecord * (uint32_t)sizeof(T);
  __amdgpu_buffer_rsrc_t rs[NE];
#pragma unroll
  for (int e = 0; e < NE; e++)
    rs[e] = __builtin_amdgcn_make_buffer_rsrc((void *)qp[e], (short)0, (int)(P * rb), kRawBufferFlags);
  // what the points of pixel i give to pixel s^-q(i), q < Q
  double acc[Q][NE] = {};
  uint32_t cnt[Q][NE] = {};
  bool dead = false;
  // angles in chunks of 64: bit (a - a0) of `defer` marks angle a of the chunk
  // whose point takes the exact path
  for (uint32_t a0 = 0; a0 < A4; a0 += 64) {
    const uint32_t a1 = A4 - a0 > 64 ? a0 + 64 : A4;
    uint64_t defer = 0;
    for (uint32_t a = a0; a < a1; a++) {
      const double *inv = inv_tab + 6 * (uint64_t)a;
      const double sx = __builtin_fma(inv[0], (double)PXi, __builtin_fma(inv[1], (double)PYi, inv[2]));
      const double sy = __builtin_fma(inv[3], (double)PXi, __builtin_fma(inv[4], (double)PYi, inv[5]));
      // (half the image's side from its middle: two tests, not four; a point that rounding
      // puts on the wrong side of the border is within the margin of it)
      const double dx = fabs(sx - hc), dy = fabs(sy - hc), far = dx > dy ? dx : dy;
      const bool inside = far <= hc;
      const double fx0 = floor(sx), fy0 = floor(sy);
      const double fx = sx - fx0, fy = sy - fy0;
      const bool safe = inside ? fabs(fx - 0.5) <= 0.5 - m && fabs(fy - 0.5) <= 0.5 - m : far > hc + m;
      const uint32_t x0 = inside ? (uint32_t)fx0 : 0u, y0 = inside ? (uint32_t)fy0 : 0u;
      const uint32_t o00 = quad_index(x0, y0, n, n) * rb, o10 = quad_index(x0 + 1, y0, n, n) * rb;
      const uint32_t o01 = quad_index(x0, y0 + 1, n, n) * rb, o11 = quad_index(x0 + 1, y0 + 1, n, n) * rb;
      typename Tap3<T>::v t[NE][4];
#pragma unroll
      for (int e = 0; e < NE; e++) {
        t[e][0] = tap_load<T>(rs[e], o00);
        t[e][1] = tap_load<T>(rs[e], o10);
        t[e][2] = tap_load<T>(rs[e], o01);
        t[e][3] = tap_load<T>(rs[e], o11);
      }
      if (!safe) {
        defer |= 1ull << (a - a0);
        continue;
      }
      // every pair shares this point's cell, validity and nonzero weights
      const T fxT = (T)fx, fyT = (T)fy, gx = (T)1 - fxT, gy = (T)1 - fyT;
      const T w00 = gx * gy, w10 = fxT * gy, w01 = gx * fyT, w11 = fxT * fyT;
      T sm[NE][3];
#pragma unroll
      for (int e = 0; e < NE; e++) {
        sm[e][0] = w00 * t[e][0].x + w10 * t[e][1].x + w01 * t[e][2].x + w11 * t[e][3].x;
        sm[e][1] = w00 * t[e][0].y + w10 * t[e][1].y + w01 * t[e][2].y + w11 * t[e][3].y;
        sm[e][2] = w00 * t[e][0].z + w10 * t[e][1].z + w01 * t[e][2].z + w11 * t[e][3].z;
      }
      auto add = [&](auto qc, const T(&vq)[NE]) {
        constexpr int q = decltype(qc)::value;
#pragma unroll
        for (int e = 0; e < NE; e++) {
          if constexpr (RM) {
            const double vv = (double)vq[e];
            const bool ok = inside && !isnan(vv);
            acc[q][e] += ok ? vv : 0.0;
            cnt[q][e] += ok ? 1u : 0u;
          } else {
            acc[q][e] += (double)vq[e];
          }
        }
      };
      if constexpr (!RM) dead = dead || !inside;
      auto value = [&](int q, T(&vq)[NE]) {
        const T *c = coef_t + 3 * (uint64_t)(a + q * A4);
#pragma unroll
        for (int e = 0; e < NE; e++) vq[e] = c[0] * sm[e][0] + c[1] * sm[e][1] + c[2] * sm[e][2];
      };
      bool shared = false;
      if constexpr (Q == 4) {
        if (share) {  // pairs q and q + 2 have equal coefficients
          T v0[NE], v1[NE];
          value(0, v0);
          value(1, v1);
          add(std::integral_constant<int, 0>{}, v0);
          add(std::integral_constant<int, 1>{}, v1);
          add(std::integral_constant<int, 2>{}, v0);
          add(std::integral_constant<int, 3>{}, v1);
          shared = true;
        }
      }
      if (!shared) {
        static_for<0, Q>([&](auto qc) {
          T vq[NE];
          value(decltype(qc)::value, vq);
          add(qc, vq);
        });
      }
    }
    // points near a cell edge or the image border: every pair back-maps its own
    // point exactly and gathers its own taps (one pair at a time, so the rare path
    // holds few registers)
    while (defer) {
      const uint32_t a = a0 + (uint32_t)__builtin_ctzll(defer);
      defer &= defer - 1;
#pragma unroll 1
      for (uint32_t q = 0; q < (uint32_t)Q; q++) {
        const uint32_t j = (i - q + 4) & 3;
        const uint32_t aa = a + q * A4;
        const QPoint d = quad_point(inv_tab + 6 * (uint64_t)aa, px(j), py(j), n, n);
        Rec<T> td[NE][4];
        quad_gather<T, NE>(qp, d, n, n, td);
        T sm[NE][3];
        quad_sums<T, NE>(d, td, sm);
        const double *c = coef + 3 * (uint64_t)aa;
        static_for<0, Q>([&](auto qc) {  // constant indices keep the accumulators in registers
          constexpr int qq = decltype(qc)::value;
          if (q == (uint32_t)qq) quad_combine<T, NE>(d.inside, sm, c, RM, acc[qq], cnt[qq]);
        });
      }
    }
  }
#pragma unroll
  for (int q = 0; q < Q; q++)
#pragma unroll
    for (int e = 0; e < NE; e++) {
      sum[i][q][e][l] = dead ? __longlong_as_double(0x7ff8000000000000ll) : acc[q][e];
      if constexpr (RM) num[i][q][e][l] = cnt[q][e];
    }
  __syncthreads();
  if (!in) return;
  // wave i now stores pixel i: the sums of the pixels j whose points serve it, q = j - i
  double a[NE] = {};
  uint32_t c[NE] = {};
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint32_t q = (j - i + 4) & 3;
    if (q >= (uint32_t)Q) continue;  // (uniform)
#pragma unroll
    for (int e = 0; e < NE; e++) {
      a[e] += sum[j][q][e][l];
      if constexpr (RM) c[e] += num[j][q][e][l];
    }
  }
  quad_store<O, NE>(avg, (uint64_t)PYi * n + PXi, e0, ne, nA, RM, a, c);
}

// Full turns (Q = 4): the sum over an angle's four quarter turns first, then the angles.
// With y the point pixel x samples at angle a, x takes Q(s^q y) at angle a + q A4, whose
// coefficients are those of a with c^2 and s^2 exchanged and 2cs negated for odd q.  So
// the four add up to one sample at y of
//   S = q(y) + P q(s y) + q(s^2 y) + P q(s^3 y),   P (q0, q1, q2) = (q1, q0, -q2),
// and as S(s y) = P S(y), pixel s x takes the same sample with P, s^2 x and s^3 x the
// values of x and s x: one gather per orbit and angle a < A4, a quarter of those
// rotate_orbit_kernel makes, from the quadrant u, v in [0, n/2 - 1] about the centre alone
// (every y turns into it; P where by an odd number of quarter turns).  S is summed in FP64
// and kept in the forms' precision, rounded once; its samples, their weights and the angles'
// values are FP64, so in FP32 a pair carries fewer roundings than by orbits (against 64 bits,
// 512^2 films, 72 angles with the mask: 2.17e-7 where orbits leave 2.20e-7 and FP32 sums and
// samples 2.19e-7).  Bound by its gathers through L1 and its FP64 points: 2048^2 film, 10
// energies x 180 angles 1.19 ms by orbits -> 0.43 ms and 25 us for S (FP32 sums and samples:
// 0.40 ms; S kept in FP64, 2.17e-7 too: 0.78 ms; a wave replaying all four pixels of its own
// deferred angles, not one pixel of all, or 1 or 4 energies a pass, not 2: 4 to 11 % slower).

// The quadrant's S of ne planes.  Where a value is not finite the record says what the
// samples that read it come to: q0 and q1 NaN, no pair there has a value (with the mask:
// all four terms NaN; without: any); q0 alone NaN, the exact path decides.  Pixels beyond
// rskip are not read by any sample: neither read nor written here.
template <typename T, bool RM>
__global__ void __launch_bounds__(256) quad_sym_kernel(const T *__restrict__ quad, T *__restrict__ sym, uint32_t n,
                                                       uint32_t tx, double rskip) {
  const uint32_t h = n / 2, w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const uint32_t u = (blockIdx.x % tx) * 16 + (w & 1) * 8 + (l & 7), v = (blockIdx.x / tx) * 16 + (w >> 1) * 8 + (l >> 3);
  if (u >= h || v >= h || (double)u * u + (double)v * v > rskip * rskip) return;
  const T *q = quad + (uint64_t)blockIdx.y * n * n * kQuadRecord;
  T *o = sym + ((uint64_t)blockIdx.y * h * h + quad_index(u, v, h, h)) * kQuadRecord;
  const uint32_t idx[4] = {quad_index(h + u, h + v, n, n), quad_index(h - v, h + u, n, n),
                           quad_index(h - u, h - v, n, n), quad_index(h + v, h - u, n, n)};
  double r[4][3];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int c = 0; c < 3; c++) r[i][c] = (double)q[(uint64_t)idx[i] * kQuadRecord + c];
  const double nan = __longlong_as_double(0x7ff8000000000000ll);
  double s0 = (r[0][0] + r[2][0]) + (r[1][1] + r[3][1]), s1 = (r[0][1] + r[2][1]) + (r[1][0] + r[3][0]);
  const double s2 = (r[0][2] + r[2][2]) - (r[1][2] + r[3][2]);
  if (!(isfinite((T)s0) && isfinite((T)s1) && isfinite((T)s2))) {
    uint32_t bad = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) bad += isnan(r[i][0]) || isnan(r[i][1]) || isnan(r[i][2]) ? 1 : 0;
    s0 = nan;
    s1 = bad >= (RM ? 4u : 1u) ? nan : 0.0;
  }
  o[0] = (T)s0;
  o[1] = (T)s1;
  o[2] = (T)s2;
}

// A block holds one 8 x 8 quadrant of a tile of orbits; its waves take a quarter of the
// angles each.  Points near a cell edge or the image border, and samples of records that
// the exact path decides, are replayed pair by pair from the planes themselves, as in
// rotate_orbit_kernel (the same margins), wave i taking those of orbit pixel i.
template <typename T, typename O, int NE, bool RM>
__global__ void __launch_bounds__(256, sizeof(T) == 4 ? 5 : 4) rotate_sym_kernel(const T *__restrict__ quad, const T *__restrict__ sym,
                                                         const double *__restrict__ inv_tab,
                                                         const double *__restrict__ coef,
                                                         uint32_t nA, uint32_t A4, uint32_t n,
                                                         AvgSink<O> avg, uint32_t ne,
                                                         const uint32_t *__restrict__ otiles, uint32_t n_otiles,
                                                         double rcut) {
  __shared__ double sum[4][4][NE][64];
  __shared__ unsigned long long later[4][64];
  __shared__ uint32_t num[RM ? 4 : 1][RM ? 4 : 1][NE][64];
  const uint64_t P = (uint64_t)n * n;
  const uint32_t h = n / 2;
  const uint32_t qb = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t e0 = blockIdx.z * NE;
  const uint32_t i = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  const T *qp[NE];
#pragma unroll
  for (int e = 0; e < NE; e++) qp[e] = quad + (uint64_t)(e0 + e < ne ? e0 + e : e0) * P * kQuadRecord;
  if (qb >= 4 * n_otiles) {
    if constexpr (!RM)  // (with the mask rotate_orbit_kernel runs too, and takes them)
      orbit_tail<T, O, NE, RM>(qp, inv_tab, coef, nA, n, rcut, (qb - 4 * n_otiles) * 64 + l, i, l, e0, ne, avg, sum, num);
    return;
  }
  const uint32_t tt = otiles[qb >> 2];
  const uint32_t u = (tt & 0xffffu) * 16 + (qb & 1) * 8 + (l & 7) + 1;
  const uint32_t v = (tt >> 16) * 16 + ((qb >> 1) & 1) * 8 + (l >> 3);
  const bool in = u < h && v < h;
  const uint32_t X0 = h + u, Y0 = h + v;  // orbit pixels s^j(x), j = 0..3
  auto px = [&](uint32_t j) { return j == 0 ? X0 : j == 1 ? n - Y0 : j == 2 ? n - X0 : Y0; };
  auto py = [&](uint32_t j) { return j == 0 ? Y0 : j == 1 ? X0 : j == 2 ? n - Y0 : n - X0; };
  const double hh = (double)h, hi = (double)(h - 1);
  const double m = 1e-9 + 1e-12 * (double)n;
  constexpr uint32_t rb = kQuadRecord * (uint32_t)sizeof(T);
  __amdgpu_buffer_rsrc_t rs[NE];
#pragma unroll
  for (int e = 0; e < NE; e++)
    rs[e] = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(sym + (uint64_t)(e0 + e < ne ? e0 + e : e0) * h * h * kQuadRecord), (short)0, (int)((uint64_t)h * h * rb),
        kRawBufferFlags);
  double acc[2][NE] = {};  // pixels x and s^2 x; s x and s^3 x
  uint32_t cnt[NE] = {};
  bool dead = false;
  double ex[NE] = {};  // pixel i's pairs of the exact path
  uint32_t exn[NE] = {};
  const uint32_t chunks = ((A4 + 3) / 4 + 63) / 64, wa1 = in ? A4 * (i + 1) / 4 : 0;
  for (uint32_t ch = 0; ch < chunks; ch++) {  // runs of 64 angles a wave, in step
    const uint32_t a0 = A4 * i / 4 + 64 * ch, a1 = wa1 < a0 + 64 ? wa1 : a0 + 64;
    uint64_t defer = 0;
    for (uint32_t a = a0; a < a1; a++) {
      const double *inv = inv_tab + 6 * (uint64_t)a;
      const double du = __builtin_fma(inv[0], (double)X0, __builtin_fma(inv[1], (double)Y0, inv[2])) - hh;
      const double dv = __builtin_fma(inv[3], (double)X0, __builtin_fma(inv[4], (double)Y0, inv[5])) - hh;
      const bool odd = (du < 0) != (dv < 0);
      const double p = fabs(odd ? dv : du), q = fabs(odd ? du : dv);
      const double far = p > q ? p : q;
      const bool inside = far <= hi;  // (all four turns of the point)
      const double fx0 = floor(p), fy0 = floor(q);
      const double fx = p - fx0, fy = q - fy0;
      const bool safe = inside ? (fabs(fx - 0.5) <= 0.5 - m && fabs(fy - 0.5) <= 0.5 - m)
                               : far > (RM ? hh : hi) + m;  // (with the mask all four outside, else one)
      const uint32_t x0 = inside ? (uint32_t)fx0 : 0u, y0 = inside ? (uint32_t)fy0 : 0u;
      const uint32_t o00 = quad_index(x0, y0, h, h) * rb, o10 = quad_index(x0 + 1, y0, h, h) * rb;
      const uint32_t o01 = quad_index(x0, y0 + 1, h, h) * rb, o11 = quad_index(x0 + 1, y0 + 1, h, h) * rb;
      Rec<T> t[NE][4];
#pragma unroll
      for (int e = 0; e < NE; e++) {
        t[e][0] = tap_load<T>(rs[e], o00);
        t[e][1] = tap_load<T>(rs[e], o10);
        t[e][2] = tap_load<T>(rs[e], o01);
        t[e][3] = tap_load<T>(rs[e], o11);
      }
      const double gx = 1 - fx, gy = 1 - fy;
      const double w00 = gx * gy, w10 = fx * gy, w01 = gx * fy, w11 = fx * fy;
      double sm[NE][3];
      bool exact = !safe;
#pragma unroll
      for (int e = 0; e < NE; e++) {
        sm[e][0] = w00 * (double)t[e][0].x + w10 * (double)t[e][1].x + w01 * (double)t[e][2].x + w11 * (double)t[e][3].x;
        sm[e][1] = w00 * (double)t[e][0].y + w10 * (double)t[e][1].y + w01 * (double)t[e][2].y + w11 * (double)t[e][3].y;
        sm[e][2] = w00 * (double)t[e][0].z + w10 * (double)t[e][1].z + w01 * (double)t[e][2].z + w11 * (double)t[e][3].z;
        exact = exact || (inside && isnan(sm[e][0]) && !isnan(sm[e][1]));
      }
      if (exact) {
        defer |= 1ull << (a - a0);
        continue;
      }
      const double *c = coef + 3 * (uint64_t)a;
      const double c0 = odd ? c[1] : c[0], c1 = odd ? c[0] : c[1], c2 = odd ? -c[2] : c[2];
      if constexpr (!RM) dead = dead || !inside;
#pragma unroll
      for (int e = 0; e < NE; e++) {
        const double v0 = c0 * sm[e][0] + c1 * sm[e][1] + c2 * sm[e][2];
        const double v1 = c1 * sm[e][0] + c0 * sm[e][1] - c2 * sm[e][2];
        if constexpr (RM) {
          const bool ok = inside && !isnan(sm[e][1]);
          acc[0][e] += ok ? v0 : 0.0;
          acc[1][e] += ok ? v1 : 0.0;
          cnt[e] += ok ? 4u : 0u;
        } else {
          acc[0][e] += v0;
          acc[1][e] += v1;
        }
      }
    }
    if (ch) __syncthreads();  // (the masks have been read)
    later[i][l] = defer;
    __syncthreads();
    for (uint32_t w = 0; w < 4; w++)
      for (uint64_t mask = later[w][l]; mask; mask &= mask - 1) {
        const uint32_t a = A4 * w / 4 + 64 * ch + (uint32_t)__builtin_ctzll(mask);
#pragma unroll 2
        for (uint32_t q = 0; q < 4; q++) {
          const uint32_t aa = a + q * A4;
          const QPoint d = quad_point(inv_tab + 6 * (uint64_t)aa, px(i), py(i), n, n);
          Rec<T> td[NE][4];
          quad_gather<T, NE>(qp, d, n, n, td);
          quad_add<T, NE>(d, td, coef + 3 * (uint64_t)aa, RM, ex, exn);
        }
      }
  }
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int e = 0; e < NE; e++) {
      sum[i][j][e][l] = dead ? __longlong_as_double(0x7ff8000000000000ll) : acc[j & 1][e];
      if constexpr (RM) num[i][j][e][l] = cnt[e];
    }
  __syncthreads();
  if (!in) return;
  // wave i stores pixel i
#pragma unroll
  for (int w = 0; w < 4; w++)
#pragma unroll
    for (int e = 0; e < NE; e++) {
      ex[e] += sum[w][i][e][l];
      if constexpr (RM) exn[e] += num[w][i][e][l];
    }
  quad_store<O, NE>(avg, (uint64_t)py(i) * n + px(i), e0, ne, nA, RM, ex, exn);
}

// Orbit tiles beyond every finite plane value (their pixels' taps, within 1.5
// pixels of points as far from the centre as the pixel, are all NaN): the
// averages rotate_orbit_kernel would form there, NaN, or 0 with the rotation
// mask (no valid sample).  Same tile and pixel layout as rotate_orbit_kernel.
template <typename O, int NE, bool RM>
__global__ void __launch_bounds__(256) orbit_fill_kernel(AvgSink<O> avg, uint32_t n, uint32_t ne,
                                                         const uint32_t *__restrict__ otiles, uint32_t first) {
  const uint64_t P = (uint64_t)n * n;
  const uint32_t h = n / 2;
  const uint32_t e0 = blockIdx.z * NE;
  const uint32_t tt = otiles[first + blockIdx.x];
  const uint32_t w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const uint32_t u = (tt & 0xffffu) * 16 + (w & 1) * 8 + (l & 7) + 1;
  const uint32_t v = (tt >> 16) * 16 + (w >> 1) * 8 + (l >> 3);
  if (u >= h || v >= h) return;
  const uint32_t X0 = h + u, Y0 = h + v;
  const uint32_t PX[4] = {X0, n - Y0, n - X0, Y0};
  const uint32_t PY[4] = {Y0, X0, n - Y0, n - X0};
  const double fill = RM ? 0.0 : __longlong_as_double(0x7ff8000000000000ll);
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int e = 0; e < NE; e++)
      if (e0 + e < ne) avg.store(e0 + e, (uint64_t)PY[i] * n + PX[i], fill);
}

// The averaged pattern warped onto the detector (grid y = pattern: avg + y P -> out + y
// out_stride).
template <typename T>
__global__ void __launch_bounds__(256) detector_warp_kernel(const double *__restrict__ avg, T *__restrict__ out,
                                                            uint32_t nx, uint32_t ny, Inv6 inv, int rot_mask,
                                                            uint64_t out_stride) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (uint64_t)nx * ny) return;
  avg += (uint64_t)blockIdx.y * nx * ny;
  out += (uint64_t)blockIdx.y * out_stride;
  const uint32_t Y = (uint32_t)(t / nx), X = (uint32_t)(t - (uint64_t)Y * nx);
  double v;
  if (!bilinear_sample<double>(avg, nx, ny, inv.c, X, Y, &v))
    v = rot_mask ? 0.0 : __longlong_as_double(0x7ff8000000000000ll);
  out[t] = (T)v;
}

template <typename T>
__global__ void __launch_bounds__(256) warp_kernel(const T *__restrict__ src, T *__restrict__ dst, uint32_t nx,
                                                   uint32_t ny, Inv6 inv) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (uint64_t)nx * ny) return;
  const uint32_t Y = (uint32_t)(t / nx), X = (uint32_t)(t - (uint64_t)Y * nx);
  double v;
  if (bilinear_sample<T>(src, nx, ny, inv.c, X, Y, &v)) dst[t] = (T)v;
}

// Waves (8 per CU) below which the rotation splits the angles of a pixel.
constexpr uint64_t kSplitWaves = 2048;

Inv6 mk_inv(const double inv[6]) {
  Inv6 r;
  for (int i = 0; i < 6; i++) r.c[i] = inv[i];
  return r;
}

}  // namespace

uint32_t rotation_tile_count(uint32_t nx, uint32_t ny) { return ceil_div(nx, 16) * ceil_div(ny, 16); }

// Tiles of rotation_tile_order whose centre lies within r pixels of the plane's
// centre: the first ones of that order (same key).
uint32_t rotation_tiles_within(uint32_t nx, uint32_t ny, double r) {
  const uint32_t tx = ceil_div(nx, 16), ty = ceil_div(ny, 16);
  uint32_t c = 0;
  for (uint32_t y = 0; y < ty; y++)
    for (uint32_t x = 0; x < tx; x++) {
      const double dx = (x * 16.0 + 8.0) - nx / 2.0, dy = (y * 16.0 + 8.0) - ny / 2.0;
      c += dx * dx + dy * dy <= r * r ? 1u : 0u;
    }
  return c;
}

void rotation_tile_order(uint32_t nx, uint32_t ny, uint32_t *out) {
  const uint32_t tx = ceil_div(nx, 16), ty = ceil_div(ny, 16);
  std::vector<std::pair<double, uint32_t>> r;
  r.reserve((size_t)tx * ty);
  for (uint32_t y = 0; y < ty; y++)
    for (uint32_t x = 0; x < tx; x++) {
      const double dx = (x * 16.0 + 8.0) - nx / 2.0, dy = (y * 16.0 + 8.0) - ny / 2.0;
      r.emplace_back(dx * dx + dy * dy, (y << 16) | x);
    }
  std::stable_sort(r.begin(), r.end(), [](const auto &a, const auto &b) { return a.first < b.first; });
  for (size_t i = 0; i < r.size(); i++) out[i] = r[i].second;
}

uint32_t rotation_orbit_tile_count(uint32_t n) { return n >= 4 && n % 2 == 0 ? ceil_div(n / 2 - 1, 16) * ceil_div(n / 2, 16) : 0; }

void rotation_orbit_tile_order(uint32_t n, uint32_t *out) {
  // orbit representatives: u = X - n/2 in [1, n/2 - 1] (tile x covers u - 1),
  // v = Y - n/2 in [0, n/2 - 1]; ordered by distance from the centre (0, 0)
  const uint32_t h = n / 2, tx = ceil_div(h - 1, 16), ty = ceil_div(h, 16);
  std::vector<std::pair<double, uint32_t>> r;
  r.reserve((size_t)tx * ty);
  for (uint32_t y = 0; y < ty; y++)
    for (uint32_t x = 0; x < tx; x++) {
      const double du = x * 16.0 + 9.0, dv = y * 16.0 + 8.0;
      r.emplace_back(du * du + dv * dv, (y << 16) | x);
    }
  std::stable_sort(r.begin(), r.end(), [](const auto &a, const auto &b) { return a.first < b.first; });
  for (size_t i = 0; i < r.size(); i++) out[i] = r[i].second;
}

// Orbit tiles whose centre (du, dv of rotation_orbit_tile_order) lies within r
// pixels of the plane's centre: the first ones of that order.
uint32_t rotation_orbit_tiles_within(uint32_t n, double r) {
  const uint32_t h = n / 2, tx = ceil_div(h - 1, 16), ty = ceil_div(h, 16);
  uint32_t c = 0;
  for (uint32_t y = 0; y < ty; y++)
    for (uint32_t x = 0; x < tx; x++) {
      const double du = x * 16.0 + 9.0, dv = y * 16.0 + 8.0;
      c += du * du + dv * dv <= r * r ? 1u : 0u;
    }
  return c;
}

uint32_t rotation_quarter_turns(uint32_t nx, uint32_t ny, uint32_t nA, uint32_t quarter) {
  if (quarter == 0 || nx != ny || nx < 4 || nx % 2 != 0 || nA % quarter != 0) return 0;
  const uint32_t q = nA / quarter;
  return q >= 2 && q <= 4 ? q : 0;
}

template <typename T>
cyr_status launch_rotate_accumulate(const T *proj, double *acc, uint32_t *count, uint32_t nx, uint32_t ny,
                                    const double *inv, uint32_t nb, uint32_t nA, bool first, bool last, int rot_mask,
                                    const AvgSink<T> &avg, hipStream_t st) {
  const uint64_t P = (uint64_t)nx * ny;
  hipLaunchKernelGGL((rotate_accumulate_kernel<T>), dim3(ceil_div(P, 256)), dim3(256), 0, st, proj, acc, count, nx,
                     ny, inv, nb, nA, first ? 1 : 0, last ? 1 : 0, rot_mask, avg);
  CYR_LAUNCHED();
  return CYR_OK;
}

template <typename T>
cyr_status launch_rotate_all(const T *proj, const double *inv_tab, uint32_t nA, uint32_t nx, uint32_t ny, int rot_mask,
                             const AvgSink<T> &avg, uint32_t ne, const uint32_t *tiles, double rfin, hipStream_t st) {
  const uint32_t ntiles = rotation_tile_count(nx, ny);
  if (!tiles) return fail(CYR_E_INVALID, "rotation: tile order missing");
  // the finite-radius cut of launch_rotate_quad (the projections are NaN where the
  // forms are)
  const uint32_t n_act = rfin >= 0 ? std::min(ntiles, rotation_tiles_within(nx, ny, rfin + 14.0)) : ntiles;
  hipLaunchKernelGGL((rotate_all_kernel<T>), dim3(xcd_grid(4ull * n_act), 1, ne), dim3(256), 0, st, proj, inv_tab, nA, nx, ny,
                     rot_mask, avg, tiles, n_act);
  CYR_LAUNCHED();
  if (n_act < ntiles) {
    hipLaunchKernelGGL((quad_fill_kernel<T, 1>), dim3(ntiles - n_act, 1, ne), dim3(256), 0, st, avg, nx, ny, ne, rot_mask,
                       tiles, n_act);
    CYR_LAUNCHED();
  }
  return CYR_OK;
}

template <typename T, typename O, int NE, bool RM>
hipError_t launch_orbit_rm(uint32_t Q, dim3 grid, hipStream_t st, const T *quad, const double *inv_tab,
                           const double *coef, const T *coef_t, uint32_t nA, uint32_t A4, uint32_t n, const AvgSink<O> &avg,
                           uint32_t ne, const uint32_t *otiles, uint32_t n_otiles, double rcut, int share) {
  switch (Q) {
    case 2:
      hipLaunchKernelGGL((rotate_orbit_kernel<T, O, NE, 2, RM>), grid, dim3(256), 0, st, quad, inv_tab, coef, coef_t, nA,
                         A4, n, avg, ne, otiles, n_otiles, rcut, share);
      break;
    case 3:
      hipLaunchKernelGGL((rotate_orbit_kernel<T, O, NE, 3, RM>), grid, dim3(256), 0, st, quad, inv_tab, coef, coef_t, nA,
                         A4, n, avg, ne, otiles, n_otiles, rcut, share);
      break;
    default:
      hipLaunchKernelGGL((rotate_orbit_kernel<T, O, NE, 4, RM>), grid, dim3(256), 0, st, quad, inv_tab, coef, coef_t, nA,
                         A4, n, avg, ne, otiles, n_otiles, rcut, share);
      break;
  }
  return hipGetLastError();
}

template <typename T, typename O>
cyr_status launch_rotate_quad(const T *quad, const double *inv_tab, const double *coef, const T *coef_t, uint32_t nA,
                              uint32_t nx, uint32_t ny, int rot_mask, const AvgSink<O> &avg, uint32_t ne,
                              const uint32_t *tiles,
                              uint32_t quarter, const uint32_t *otiles, QuadTurns turns, double rfin, void *scratch,
                              size_t scratch_bytes, hipStream_t st) {
  if (ne == 0) return CYR_OK;
  if ((uint64_t)nx * ny > 0xffffffffull) return fail(CYR_E_UNSUPPORTED, "rotation: more than 2^32 pixels");
  if (!tiles) return fail(CYR_E_INVALID, "rotation: tile order missing");
  const uint32_t ntiles = rotation_tile_count(nx, ny);
  // tiles (in order of distance from the centre (Nx/2, Ny/2), about which the
  // image turns) whose pixels all lie more than rfin + 2 pixels out are filled:
  // a 16 x 16 tile's pixels are within 8 sqrt(2) of its centre
  const uint32_t n_act = rfin >= 0 ? std::min(ntiles, rotation_tiles_within(nx, ny, rfin + 14.0)) : ntiles;
  // planes whose sampled tiles, four waves each, give fewer waves than kSplitWaves over
  // all energies: angles split over the waves of a block
  if ((uint64_t)n_act * 4 * ne < kSplitWaves) {
    const dim3 grid(xcd_grid(4ull * n_act), 1, ne);
    if ((uint64_t)n_act * 16 * ne < kSplitWaves && nA >= 8)
      hipLaunchKernelGGL((rotate_quad_split_kernel<T, O, 16>), grid, dim3(1024), 0, st, quad, inv_tab, coef, nA, nx, ny,
                         rot_mask, avg, tiles, n_act);
    else
      hipLaunchKernelGGL((rotate_quad_split_kernel<T, O, 4>), grid, dim3(256), 0, st, quad, inv_tab, coef, nA, nx, ny,
                         rot_mask, avg, tiles, n_act);
    CYR_LAUNCHED();
    if (n_act < ntiles) {
      hipLaunchKernelGGL((quad_fill_kernel<O, 1>), dim3(ntiles - n_act, 1, ne), dim3(256), 0, st, avg, nx, ny, ne,
                         rot_mask, tiles, n_act);
      CYR_LAUNCHED();
    }
    return CYR_OK;
  }
  // the orbit kernel addresses a plane through 32-bit buffer offsets
  const bool small_plane = (uint64_t)nx * ny * kQuadRecord * sizeof(T) < (1ull << 31);
  const uint32_t Q = otiles && small_plane ? rotation_quarter_turns(nx, ny, nA, quarter) : 0;
  if (Q) {
    // quarter-turn orbits: each gathered tap cell serves Q (pixel, angle) pairs
    const uint32_t n_otiles = rotation_orbit_tile_count(nx);
    // tiles (in order of distance from the centre) whose pixels all lie more than
    // rfin + 2 pixels out are filled, not sampled: a tile's pixels are within
    // 8 sqrt(2) < 11.4 pixels of its centre, hence the cut at rfin + 14
    const uint32_t o_act = rfin >= 0 ? std::min(n_otiles, rotation_orbit_tiles_within(nx, rfin + 14.0)) : n_otiles;
    // 2 energies per pass (measured against 1 and 4: 512^2 x 20 energies 415 / 384 us
    // for 4 / 2; 2048^2 film 7.30 / 6.75 / 8.92 ms per 10 energies for 1 / 2 / 4)
    const uint64_t blocks = 4ull * o_act + ceil_div(2ull * nx, 64);
    const double rcut = rfin >= 0 ? rfin + 2.0 : 4.0 * nx;
    hipError_t e;
    // Full turns: summed over the quarter turns first, as many energies at a time as the
    // scratch buffer has quadrants for.  With the mask only the tiles that sample finite
    // values alone (turns.rin): near the disc's edge, which is not quite its own quarter
    // turn, every angle of a pixel would take the exact path (512^2 FP64 film, 72 angles:
    // 229 us for all tiles, 107 us so, 111 us by orbits alone).
    const uint32_t h = nx / 2;
    const uint64_t plane = (uint64_t)h * h * kQuadRecord, fit = scratch ? scratch_bytes / (plane * sizeof(T)) : 0;
    uint32_t o_sym = 0;
    if (Q == 4 && turns.turn && fit)
      o_sym = rot_mask ? std::min(o_act, rotation_orbit_tiles_within(nx, std::max(0.0, turns.rin - 14.0))) : o_act;
    if (o_sym) {
      T *sym = reinterpret_cast<T *>(scratch);
      const double rskip = rfin >= 0 ? rfin + kQuadMargin : 4.0 * nx;
      const uint32_t tx = ceil_div(rfin >= 0 ? std::min(h, (uint32_t)rskip + 1) : h, 16);
      const uint32_t passes = ceil_div(ne, fit), per = ceil_div(ne, passes);  // (alike)
      for (uint32_t b0 = 0; b0 < ne;) {
        const uint32_t nb = std::min(per, ne - b0);
        const T *qb = quad + (uint64_t)b0 * nx * nx * kQuadRecord;
        const AvgSink<O> ab = avg.from(b0);
        const dim3 gs(tx * tx, nb);
        const dim3 gr(xcd_grid(rot_mask ? 4ull * o_sym : blocks), 1, ceil_div(nb, 2));
        auto run = [&](auto rm) {
          constexpr bool RM = decltype(rm)::value;
          hipLaunchKernelGGL((quad_sym_kernel<T, RM>), gs, dim3(256), 0, st, qb, sym, nx, tx, rskip);
          if (nb == 1)  // (one plane, not gathered twice)
            hipLaunchKernelGGL((rotate_sym_kernel<T, O, 1, RM>), gr, dim3(256), 0, st, qb, sym, inv_tab, coef, nA,
                               quarter, nx, ab, nb, otiles, o_sym, rcut);
          else
            hipLaunchKernelGGL((rotate_sym_kernel<T, O, 2, RM>), gr, dim3(256), 0, st, qb, sym, inv_tab, coef, nA,
                               quarter, nx, ab, nb, otiles, o_sym, rcut);
        };
        if (rot_mask) run(std::true_type{});
        else run(std::false_type{});
        e = hipGetLastError();
        if (e != hipSuccess) return hip_fail(e, "rotate_sym_kernel", __FILE__, __LINE__);
        b0 += nb;
      }
    }
    if (!o_sym || rot_mask) {
      const uint32_t o_n = o_act - o_sym;
      const dim3 grid(xcd_grid(4ull * o_n + ceil_div(2ull * nx, 64)), 1, ceil_div(ne, 2));
      auto run = [&](auto energies, auto rm) {
        return launch_orbit_rm<T, O, decltype(energies)::value, decltype(rm)::value>(
            Q, grid, st, quad, inv_tab, coef, coef_t, nA, quarter, nx, avg, ne, rot_mask ? otiles + o_sym : otiles, o_n,
            rcut, turns.share ? 1 : 0);
      };
      using One = std::integral_constant<int, 1>;
      using Two = std::integral_constant<int, 2>;
      e = rot_mask ? (ne == 1 ? run(One{}, std::true_type{}) : run(Two{}, std::true_type{}))
                   : (ne == 1 ? run(One{}, std::false_type{}) : run(Two{}, std::false_type{}));
      if (e != hipSuccess) return hip_fail(e, "rotate_orbit_kernel", __FILE__, __LINE__);
    }
    if (o_act < n_otiles) {
      const dim3 gf(n_otiles - o_act, 1, ceil_div(ne, 2));
      if (rot_mask) hipLaunchKernelGGL((orbit_fill_kernel<O, 2, true>), gf, dim3(256), 0, st, avg, nx, ne, otiles, o_act);
      else hipLaunchKernelGGL((orbit_fill_kernel<O, 2, false>), gf, dim3(256), 0, st, avg, nx, ne, otiles, o_act);
      e = hipGetLastError();
      if (e != hipSuccess) return hip_fail(e, "orbit_fill_kernel", __FILE__, __LINE__);
    }
    return CYR_OK;
  }
  // Energies per pass: 4 share each angle's taps; once a plane of quadratic forms
  // exceeds 16 MB (2048^2: 64 MB), one energy per pass keeps the gathers' working
  // set in cache (measured 19% faster there, equal at 512^2).
  const bool one = (uint64_t)nx * ny * kQuadRecord * sizeof(T) > (16ull << 20);
  if (one)
    hipLaunchKernelGGL((rotate_quad_kernel<T, O, 1>), dim3(xcd_grid(n_act), 1, ne), dim3(256), 0, st, quad, inv_tab,
                       coef, nA, nx, ny, rot_mask, avg, ne, tiles, n_act);
  else
    hipLaunchKernelGGL((rotate_quad_kernel<T, O, 4>), dim3(xcd_grid(n_act), 1, ceil_div(ne, 4)), dim3(256), 0, st, quad,
                       inv_tab, coef, nA, nx, ny, rot_mask, avg, ne, tiles, n_act);
  CYR_LAUNCHED();
  if (n_act < ntiles) {
    if (one)
      hipLaunchKernelGGL((quad_fill_kernel<O, 1>), dim3(ntiles - n_act, 1, ne), dim3(256), 0, st, avg, nx, ny, ne, rot_mask,
                         tiles, n_act);
    else
      hipLaunchKernelGGL((quad_fill_kernel<O, 4>), dim3(ntiles - n_act, 1, ceil_div(ne, 4)), dim3(256), 0, st, avg, nx, ny,
                         ne, rot_mask, tiles, n_act);
    CYR_LAUNCHED();
  }
  return CYR_OK;
}

template <typename T>
cyr_status launch_detector_warp(const double *avg, T *out, uint64_t out_stride, uint32_t ne, uint32_t nx, uint32_t ny,
                                const double inv[6], int rot_mask, hipStream_t st) {
  if (ne == 0 || identity_warp(inv)) return CYR_OK;
  hipLaunchKernelGGL((detector_warp_kernel<T>), dim3(ceil_div((uint64_t)nx * ny, 256), ne), dim3(256), 0, st, avg, out,
                     nx, ny, mk_inv(inv), rot_mask, out_stride);
  CYR_LAUNCHED();
  return CYR_OK;
}

template <typename T>
cyr_status launch_warp(const T *src, T *dst, uint32_t nx, uint32_t ny, const double inv[6], hipStream_t st) {
  const uint64_t P = (uint64_t)nx * ny;
  hipLaunchKernelGGL((warp_kernel<T>), dim3(ceil_div(P, 256)), dim3(256), 0, st, src, dst, nx, ny, mk_inv(inv));
  CYR_LAUNCHED();
  return CYR_OK;
}

#define CYR_INST(T)                                                                                                \
  template cyr_status launch_rotate_accumulate<T>(const T *, double *, uint32_t *, uint32_t, uint32_t,             \
                                                  const double *, uint32_t, uint32_t, bool, bool, int,             \
                                                  const AvgSink<T> &, hipStream_t);                                \
  template cyr_status launch_rotate_all<T>(const T *, const double *, uint32_t, uint32_t, uint32_t, int,           \
                                           const AvgSink<T> &, uint32_t, const uint32_t *, double, hipStream_t);   \
  template cyr_status launch_detector_warp<T>(const double *, T *, uint64_t, uint32_t, uint32_t, uint32_t,         \
                                              const double *, int, hipStream_t);                                   \
  template cyr_status launch_warp<T>(const T *, T *, uint32_t, uint32_t, const double *, hipStream_t);
CYR_INST(float)
CYR_INST(double)
#undef CYR_INST

#define CYR_INST(T, O)                                                                                            \
  template cyr_status launch_rotate_quad<T, O>(const T *, const double *, const double *, const T *, uint32_t,    \
                                               uint32_t, uint32_t, int, const AvgSink<O> &, uint32_t,             \
                                               const uint32_t *, uint32_t, const uint32_t *, QuadTurns, double,   \
                                               void *, size_t, hipStream_t);
CYR_INST(float, float)
CYR_INST(double, float)
CYR_INST(double, double)
#undef CYR_INST

}  // namespace cyr
