// Per-voxel fields + X FFT: the first kernel of both fused executors.
//
// A block holds pp rows of tpp threads (F::kE elements each); the compile-time
// plans' WG = 64 makes every row exchange wave-local (the barriers compile to LDS
// waits).  LDS: the
// pp x row tile, plus the X twiddle table: the 4-7 FFTs per row read their
// twiddles from LDS (the pair kernel's vector-memory instructions drop from 124 to
// 34 per wave: 731 -> 621 us at 512^2 x 128; the tensor kernel 780 -> 742 us).
// Looping a block over several rows spills registers.
//
// What a voxel contributes is selected by MODE:
//   kXTensor  the five E-basis tensor fields N'00, N'01, N'02, N'11, N'12 of one
//             energy (complex, summed over all materials);
//   kXPair    the seven energy-independent real basis fields of two materials
//             m0, m0+1, packed as (basis of m0) + i (basis of m0+1);
//   kXSingle  the seven basis fields of material m0 packed into four volumes
//             (alpha + i beta, q00 + i q11, q01 + i q02, q12).
// Basis fields of a material (all windowed and scaled by 1/4pi; s' = Q^T s):
//   alpha = phi_a (Euler) | |s|^2 (vector),  beta = phi_u (Euler) | phi (vector),
//   q00 = phi_a s'0^2, q11 = phi_a s'1^2, q01 = phi_a s'0 s'1, q02 = phi_a s'0 s'2,
//   q12 = phi_a s'1 s'2   (phi_a = 1 for vector morphologies),
// so that the tensor fields of an energy are, per material,
//   N'00 += b alpha + c beta + d q00,  N'11 += b alpha + c beta + d q11,
//   N'01 += d q01,  N'02 += d q02,  N'12 += d q12
// with b = nperp^2 - 1, c = niso^2 - 1, d = npara^2 - nperp^2 (include/uniaxial.h:106-150, 215-240).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "fft.hpp"
#include "fftpolicy.hpp"
#include "kernels.hpp"
#include "stockham.hpp"
#include "tensor.hpp"

namespace cyr {

template <int MODE> constexpr int x_outputs() { return MODE == kXTensor ? kEbFields : (MODE == kXPair ? 7 : 4); }

// ---- the five tensor fields of one voxel -------------------------------------
template <typename T, typename S, int MORPH>
__device__ inline void tensor_fields(const S *__restrict__ vox, const MatConst<T> *__restrict__ mats, uint32_t M,
                                     uint64_t V, uint64_t idx, const Mat3<T> &Q, bool rot, T fr[kEbFields],
                                     T fi[kEbFields]) {
#pragma unroll
  for (int j = 0; j < kEbFields; j++) fr[j] = fi[j] = 0;
  for (uint32_t m = 0; m < M; m++) {
    const MatConst<T> mc = mats[m];
    T v[4];
    VoxLoad<T, S>::get(vox, (uint64_t)m * V + idx, v);
    T sx, sy, sz, pa, isor, isoi;
    if (MORPH == 1) {
      sx = v[0];
      sy = v[1];
      sz = v[2];
      pa = (T)1;
      const T ss = sx * sx + sy * sy + sz * sz;
      isor = mc.br * ss + mc.cr * v[3];
      isoi = mc.bi * ss + mc.ci * v[3];
    } else {
      T st, ct, sp, cp;
      sincos_t(v[1], &st, &ct);
      sincos_t(v[2], &sp, &cp);
      sx = cp * st;
      sy = sp * st;
      sz = ct;
      pa = v[3] * v[0];
      const T pu = v[3] - pa;
      isor = mc.br * pa + mc.cr * pu;
      isoi = mc.bi * pa + mc.ci * pu;
    }
    if (rot) {  // s' = Q^T s
      const T a = Q.m[0] * sx + Q.m[3] * sy + Q.m[6] * sz;
      const T b = Q.m[1] * sx + Q.m[4] * sy + Q.m[7] * sz;
      const T c = Q.m[2] * sx + Q.m[5] * sy + Q.m[8] * sz;
      sx = a;
      sy = b;
      sz = c;
    }
    const T tx = pa * sx, ty = pa * sy;
    const T q00 = tx * sx, q01 = tx * sy, q02 = tx * sz, q11 = ty * sy, q12 = ty * sz;
    fr[0] += isor + mc.dr * q00;
    fi[0] += isoi + mc.di * q00;
    fr[1] += mc.dr * q01;
    fi[1] += mc.di * q01;
    fr[2] += mc.dr * q02;
    fi[2] += mc.di * q02;
    fr[3] += isor + mc.dr * q11;
    fi[3] += isoi + mc.di * q11;
    fr[4] += mc.dr * q12;
    fi[4] += mc.di * q12;
  }
}

// ---- the seven real basis fields of one material at one voxel ------------------
// b = (alpha, beta, q00, q11, q01, q02, q12)
template <typename T, typename S, int MORPH>
__device__ inline void basis_fields(const S *__restrict__ vox, uint64_t V, uint32_t m, uint64_t idx, const Mat3<T> &Q,
                                    bool rot, T b[7]) {
  T v[4];
  VoxLoad<T, S>::get(vox, (uint64_t)m * V + idx, v);
  T sx, sy, sz, pa;
  if (MORPH == 1) {
    sx = v[0];
    sy = v[1];
    sz = v[2];
    pa = (T)1;
    b[0] = sx * sx + sy * sy + sz * sz;
    b[1] = v[3];
  } else {
    T st, ct, sp, cp;
    sincos_t(v[1], &st, &ct);
    sincos_t(v[2], &sp, &cp);
    sx = cp * st;
    sy = sp * st;
    sz = ct;
    pa = v[3] * v[0];
    b[0] = pa;
    b[1] = v[3] - pa;
  }
  if (rot) {
    const T a = Q.m[0] * sx + Q.m[3] * sy + Q.m[6] * sz;
    const T c = Q.m[1] * sx + Q.m[4] * sy + Q.m[7] * sz;
    const T d = Q.m[2] * sx + Q.m[5] * sy + Q.m[8] * sz;
    sx = a;
    sy = c;
    sz = d;
  }
  const T tx = pa * sx, ty = pa * sy;
  b[2] = tx * sx;
  b[3] = ty * sy;
  b[4] = tx * sy;
  b[5] = tx * sz;
  b[6] = ty * sz;
}

template <typename T, typename S, int MORPH, int MODE>
__device__ inline void voxel_fields(const S *__restrict__ vox, const PolxArgs<T> &a, uint64_t idx, bool rot,
                                    T fr[x_outputs<MODE>()], T fi[x_outputs<MODE>()]) {
  if constexpr (MODE == kXTensor) {
    tensor_fields<T, S, MORPH>(vox, a.mats, a.M, a.V, idx, a.Q, rot, fr, fi);
  } else if constexpr (MODE == kXPair) {
    T b0[7], b1[7];
    basis_fields<T, S, MORPH>(vox, a.V, a.m0, idx, a.Q, rot, b0);
    basis_fields<T, S, MORPH>(vox, a.V, a.m0 + 1, idx, a.Q, rot, b1);
#pragma unroll
    for (int r = 0; r < 7; r++) {
      fr[r] = b0[r];
      fi[r] = b1[r];
    }
  } else {
    T b[7];
    basis_fields<T, S, MORPH>(vox, a.V, a.m0, idx, a.Q, rot, b);
    fr[0] = b[0];
    fi[0] = b[1];
    fr[1] = b[2];
    fi[1] = b[3];
    fr[2] = b[4];
    fi[2] = b[5];
    fr[3] = b[6];
    fi[3] = 0;
  }
}

// Waves per SIMD the registers are held to: the any-length kernels wait on LDS and
// barriers and want all that fit without spilling.
template <typename T, class F, int MODE> constexpr int x_min_waves() {
  if constexpr (F::kCt) return MODE == kXTensor && F::kE <= 8 ? 4 : 2;
  else return sizeof(T) == 8 ? (F::kE <= 2 ? 3 : 2) : F::kNarrow && F::kE <= 4 && sizeof(typename F::Comp) == 4 ? 4 : 2;
}

// ---- fields + X FFT --------------------------------------------------------------
template <typename T, typename S, class F, int WG, int MODE>
__global__ void __launch_bounds__(WG, (x_min_waves<T, F, MODE>()))
    xfields_kernel(typename F::Plan plan, PolxArgs<T> a, const S *__restrict__ vox, int morph, int hann) {
  constexpr int E = F::kE, NO = x_outputs<MODE>();
  extern __shared__ unsigned char smem_raw[];
  auto *lds = reinterpret_cast<cx<typename F::Comp> *>(smem_raw);
  const F fft(plan);
  const uint32_t tpp = a.tpp;
  const uint32_t t = threadIdx.x % tpp, p = threadIdx.x / tpp;
  const uint32_t row = blockIdx.x * a.pp + p;  // row = y + ny z
  const bool active = row < a.rows;
  const uint32_t y = active ? row % a.ny : 0, z = active ? row / a.ny : 0;
  const T k4 = (T)(1.0 / (4.0 * M_PI));
  const T wyz = hann ? a.hy[y] * a.hz[z] * k4 : k4;
  const bool rot = a.rot != 0;
  // twiddles staged in LDS.  The X transform (the first of the three) keeps
  // plain products: this kernel is register- and latency-bound, compensated
  // products here cost 12% of its time (512^2 x 128, material pair) and left the
  // FP32 pattern error unchanged to three digits; the later Y and Z passes
  // apply them.
  if constexpr (F::kCt) fft.stage(lds, a.pp, a.twx);
  else fft.stage(lds, a.pp);
  lds_sync();  // (single-wave blocks: an LDS wait only)
  // fill(c, v) forms output c, which is transformed and written.  Compile-time plans
  // unroll the outputs; the any-length transform is too large to copy per output.
  // (touch() marks what fill reads as changed: the products of every output would
  // otherwise be hoisted out of the loop and held in registers)
  auto each_output = [&](auto touch, auto fill) {
    auto emit = [&](cx<T>(&v)[E], cx<T> *vol) {
      // (transform() ends with a barrier after its last LDS reads, so the next
      // output's first LDS store cannot overtake them)
      if constexpr (F::kCt) {
        cx<T> *o = vol + (uint64_t)(active ? row : 0) * a.nx;
        fft.transform(v, t, p, a.pp, lds, [&](uint32_t, uint32_t k, cx<T> x) {
          if (active) o[k] = x;
        });
      } else {
        const uint32_t r0 = blockIdx.x * a.pp;
        cx<T> *o = vol + (uint64_t)r0 * a.nx;
        fft.transform(v, t, p, a.pp, lds, [&](uint32_t r, uint32_t k, cx<T> x) {
          if (r0 + r < a.rows) o[(uint64_t)r * a.nx + k] = x;
        });
      }
    };
    if constexpr (F::kCt) {
      static_for<0, NO>([&](auto cc) {
        cx<T> v[E];
        fill(cc, v);
        emit(v, a.out[decltype(cc)::value]);
      });
    } else {
#pragma unroll 1
      for (uint32_t c = blockIdx.y; c < (uint32_t)NO; c += gridDim.y) {
        cx<T> v[E];
        cx<T> *vol = nullptr;
        touch();
        static_for<0, NO>([&](auto cc) {  // (uniform)
          if (c == (uint32_t)decltype(cc)::value) {
            fill(cc, v);
            vol = a.out[decltype(cc)::value];
          }
        });
        emit(v, vol);
      }
    }
  };
  if constexpr (MODE == kXPair) {
    // Material pair: a compact per-material state per element (window-weighted
    // phi_a, the second scalar field, the director s'; 5-6 values instead of the
    // 7 fields) and each output's fields formed just before its FFT, so the
    // loads are consumed early and the field products interleave with the FFTs
    // (512-point rows, 2 materials: 577 us against 625 us with all 7 x 2 fields
    // formed up front).
    auto pair_rows = [&](auto mtag) {
      constexpr int MORPH = decltype(mtag)::value;
      T wal[MORPH == 1 ? 2 : 1][E], wpa[2][E], wbe[2][E], sxa[2][E], sya[2][E], sza[2][E];
#pragma unroll
      for (int i = 0; i < E; i++) {
        const uint32_t x = fft.in_pos(t, i);
        const bool in = active && fft.holds(t, i);
        const T w = in ? (hann ? a.hx[x] * wyz : wyz) : (T)0;
#pragma unroll
        for (int m = 0; m < 2; m++) {
          T vv[4] = {0, 0, 0, 0};
          if (in) VoxLoad<T, S>::get(vox, (uint64_t)(a.m0 + m) * a.V + (uint64_t)row * a.nx + x, vv);
          T sx, sy, sz;
          if constexpr (MORPH == 1) {  // alpha = |s|^2, beta = phi_u, phi_a = 1
            sx = vv[0];
            sy = vv[1];
            sz = vv[2];
            wal[m][i] = w * (sx * sx + sy * sy + sz * sz);
            wpa[m][i] = w;
            wbe[m][i] = w * vv[3];
          } else {  // alpha = phi_a = Vfrac S, beta = Vfrac - phi_a
            T st, ct, sp, cp;
            sincos_t(vv[1], &st, &ct);
            sincos_t(vv[2], &sp, &cp);
            sx = cp * st;
            sy = sp * st;
            sz = ct;
            const T pa = vv[3] * vv[0];
            wpa[m][i] = w * pa;
            wbe[m][i] = w * (vv[3] - pa);
          }
          if (rot) {  // s' = Q^T s
            const T q0 = a.Q.m[0] * sx + a.Q.m[3] * sy + a.Q.m[6] * sz;
            const T q1 = a.Q.m[1] * sx + a.Q.m[4] * sy + a.Q.m[7] * sz;
            const T q2 = a.Q.m[2] * sx + a.Q.m[5] * sy + a.Q.m[8] * sz;
            sx = q0;
            sy = q1;
            sz = q2;
          }
          sxa[m][i] = sx;
          sya[m][i] = sy;
          sza[m][i] = sz;
        }
      }
      // outputs c = 0..6: (alpha, beta, q00, q11, q01, q02, q12) of material m0
      // (real part) and m0 + 1 (imaginary part), q_ij = phi_a s'_i s'_j
      auto touch = [&] {
#pragma unroll
        for (int i = 0; i < E; i++)
#pragma unroll
          for (int m = 0; m < 2; m++) {
            asm volatile("" : "+v"(wpa[m][i]), "+v"(wbe[m][i]), "+v"(sxa[m][i]), "+v"(sya[m][i]), "+v"(sza[m][i]));
            if constexpr (MORPH == 1) asm volatile("" : "+v"(wal[m][i]));
          }
      };
      each_output(touch, [&](auto cc, cx<T>(&v)[E]) {
        constexpr int c = decltype(cc)::value;
#pragma unroll
        for (int i = 0; i < E; i++) {
          T f[2];
#pragma unroll
          for (int m = 0; m < 2; m++) {
            if constexpr (c == 0) f[m] = MORPH == 1 ? wal[MORPH == 1 ? m : 0][i] : wpa[m][i];
            else if constexpr (c == 1) f[m] = wbe[m][i];
            else if constexpr (c == 2) f[m] = wpa[m][i] * sxa[m][i] * sxa[m][i];
            else if constexpr (c == 3) f[m] = wpa[m][i] * sya[m][i] * sya[m][i];
            else if constexpr (c == 4) f[m] = wpa[m][i] * sxa[m][i] * sya[m][i];
            else if constexpr (c == 5) f[m] = wpa[m][i] * sxa[m][i] * sza[m][i];
            else f[m] = wpa[m][i] * sya[m][i] * sza[m][i];
          }
          v[i] = mk<T>(f[0], f[1]);
        }
      });
    };
    if (morph == 1) pair_rows(std::integral_constant<int, 1>{});
    else pair_rows(std::integral_constant<int, 0>{});
    return;
  }
  T fre[NO][E], fim[NO][E];
#pragma unroll
  for (int i = 0; i < E; i++) {
    const uint32_t x = fft.in_pos(t, i);
    T fr[NO], fi[NO];
    if (active && fft.holds(t, i)) {
      const uint64_t idx = (uint64_t)row * a.nx + x;
      if (morph == 1) voxel_fields<T, S, 1, MODE>(vox, a, idx, rot, fr, fi);
      else voxel_fields<T, S, 0, MODE>(vox, a, idx, rot, fr, fi);
      const T w = hann ? a.hx[x] * wyz : wyz;
#pragma unroll
      for (int c = 0; c < NO; c++) {
        fr[c] *= w;
        fi[c] *= w;
      }
    } else {
#pragma unroll
      for (int c = 0; c < NO; c++) fr[c] = fi[c] = 0;
    }
#pragma unroll
    for (int c = 0; c < NO; c++) {
      fre[c][i] = fr[c];
      fim[c][i] = fi[c];
    }
  }
  each_output([] {}, [&](auto cc, cx<T>(&v)[E]) {
    constexpr int c = decltype(cc)::value;
#pragma unroll
    for (int i = 0; i < E; i++) v[i] = mk<T>(fre[c][i], fim[c][i]);
  });
}

// ---- plan helpers shared by the fused executors ------------------------------
// Launch shape of the compile-time X plans: rows of <= 64 threads share a wave.
constexpr int ct_polx_wg(int N, int E) { return N / E <= 64 ? 64 : N / E; }

// Plan, shape and elements per thread of the any-length X transforms: FP32 4, FP64 2, and
// for rows that would need more than kLfRowThreads threads twice that, in FP32 up to four
// times (rows of 4097 to 8192 points).  Narrow plans: the
// per-element state and butterflies of up to 8 then fit 128 registers in FP32, 4 waves per
// SIMD, where radices up to 13 took 182 (200 x 240 x 50, 3 materials: 109 -> 84 us per
// volume; 101 x 94 x 21: 58 -> 37 us).  Lengths with factors 11 and 13 would be
// Bluestein's in a narrow plan, so those keep the wide one in FP32 (156 x 156 x 64, 4
// materials: 183 us per volume by Bluestein, 98 so).  Short convolutions: narrow FP64 plans.
constexpr uint64_t kXSplitThreads = 256 * 384;  // one and a half waves per SIMD
inline bool lf_x_shape(uint32_t n, int precision, LfPlan &P, LfShape &s, uint32_t &e) {
  e = precision == CYR_FP64 ? 2 : 4;
  if (lf_precision(n, precision) != precision)
    return lf_plan(n, CYR_FP64, true, P) && lf_rows_shape(P, CYR_FP64, e, true, s);
  const bool fits = lf_plan(n, precision, true, P);
  if (precision == CYR_FP32 && fits && P.blue) {
    LfPlan W;
    if (lf_plan(n, precision, false, W) && !W.blue && lf_rows_shape(W, precision, e, true, s)) {
      P = W;
      return true;
    }
  }
  if (!fits) return false;
  for (const uint32_t last = precision == CYR_FP64 ? 4 : 16; e <= last; e *= 2)
    if (lf_rows_shape(P, precision, e, true, s)) return true;
  return false;
}

// The compile-time plan applies (its elements per thread are compiled for T).
inline bool ct_usable(uint32_t n, int precision) {
  return ct_length(n) && (precision != CYR_FP64 || ct_elements(n) <= 8);
}

// Blocks over which the any-length outputs are split (each evaluates the voxels again,
// from L2): all of them when the rows alone leave the chip short of waves, so that the
// chain of transforms that a block runs one after another is one transform long.  A pair of
// materials, split / not (us), by threads of the rows alone: FP32 32 x 32 x 16 (4k) 8.4 /
// 21.2, 101 x 94 x 21 (51k) 44.8 / 75.2, 147 x 147 x 16 (87k) 29.7 / 38.7, 200 x 240 x 8
// (96k) 29.9 / 34.7, 96 x 96 x 48 (111k) 37.1 / 34.7, 1000 x 500 (125k) 47 / 42; FP64, whose
// sines weigh more, 250 x 250 (31k) 22.5 / 36.3, 50 x 60 x 20 (30k) 20.9 / 29.2, 300 x 271
// (41k) 27.6 / 38.6, 500 x 500 (125k) 56 / 42, 200 x 240 x 8 (192k) 87 / 61.  Not for the
// compile-time plans, whose transforms are short (64^3: 13.7 against 15.2 us).
template <typename T, int MODE> uint32_t x_split(uint64_t blocks, uint32_t threads) {
  return blocks * threads < kXSplitThreads ? (uint32_t)x_outputs<MODE>() : 1;
}

template <typename T, typename S, int E, bool NARROW, int MODE, typename C>
hipError_t launch_xfields_lf(const LfTab<C> &tb, const LfShape &sh, hipStream_t st, const PolxArgs<T> &a,
                             const void *vox, int morph, int hann) {
  using F = LfRowFft<T, E, NARROW, C>;
  const typename F::Plan plan{tb, sh.tpp, sh.pitch, sh.pad};
  hipLaunchKernelGGL((xfields_kernel<T, S, F, kLfRowThreads, MODE>),
                     dim3(ceil_div(a.rows, sh.pp), x_split<T, MODE>(ceil_div(a.rows, sh.pp), sh.pp * sh.tpp)),
                     dim3(sh.pp * sh.tpp), sh.lds, st, plan, a, (const S *)vox, morph, hann);
  return hipGetLastError();
}

template <typename T, typename S, int N, int MODE>
hipError_t launch_xfields_ct(dim3 grid, size_t lds, hipStream_t st, const PolxArgs<T> &a, const void *vox, int morph,
                             int hann) {
  using F = typename CtPlan<T, N, true, 1>::type;
  constexpr int WG = ct_polx_wg(N, F::kE);
  hipLaunchKernelGGL((xfields_kernel<T, S, F, WG, MODE>), grid, dim3(WG), lds, st, typename F::Plan{}, a,
                     (const S *)vox, morph, hann);
  return hipGetLastError();
}

template <typename T, typename S, int MODE>
hipError_t launch_xfields_ct_n(uint32_t n, dim3 grid, size_t lds, hipStream_t st, const PolxArgs<T> &a,
                               const void *vox, int morph, int hann, bool *found) {
  *found = true;
  switch (n) {
    case 64: return launch_xfields_ct<T, S, 64, MODE>(grid, lds, st, a, vox, morph, hann);
    case 128: return launch_xfields_ct<T, S, 128, MODE>(grid, lds, st, a, vox, morph, hann);
    case 256: return launch_xfields_ct<T, S, 256, MODE>(grid, lds, st, a, vox, morph, hann);
    case 384:
      if constexpr (sizeof(T) == 4) return launch_xfields_ct<T, S, 384, MODE>(grid, lds, st, a, vox, morph, hann);
      break;
    case 512: return launch_xfields_ct<T, S, 512, MODE>(grid, lds, st, a, vox, morph, hann);
    case 1024: return launch_xfields_ct<T, S, 1024, MODE>(grid, lds, st, a, vox, morph, hann);
    case 2048: return launch_xfields_ct<T, S, 2048, MODE>(grid, lds, st, a, vox, morph, hann);
    default: break;
  }
  *found = false;
  return hipSuccess;
}

// Plans and launches the fields + X FFT kernel of one MODE (instantiated per precision
// and mode in a file of its own: xfields_*.hip).
template <typename T, int MODE>
cyr_status launch_xfields(PolxArgs<T> a, const void *vox, int storage, int morph, bool hann, hipStream_t st) {
  const int prec = sizeof(T) == 8 ? CYR_FP64 : CYR_FP32;
  const bool ct = ct_usable(a.nx, prec);
  LfTab<T> tb{};
  LfTab<double> tb64{};
  LfShape sh;
  uint32_t e_lf = 0;
  bool narrow = true;
  const bool conv64 = !ct && lf_precision(a.nx, prec) != prec;
  size_t lds = 0;
  if (ct) {
    // rows of <= 64 threads share one wave
    a.tpp = a.nx / ct_elements(a.nx);
    a.pp = a.tpp <= 64 ? 64 / a.tpp : 1;
    lds = ((size_t)a.pp * ct_row_pitch(a.nx) + a.nx) * sizeof(cx<T>);
    if (lds > device_max_lds()) return fail(CYR_E_UNSUPPORTED, "fused X kernel: row does not fit in LDS");
    cyr_status s;
    a.twx = twiddles<T>(a.nx, &s);
    if (!a.twx) return s;
  } else {
    LfPlan P;
    if (!lf_x_shape(a.nx, prec, P, sh, e_lf))
      return fail(CYR_E_UNSUPPORTED, "fused X kernel: row does not fit its block");
    narrow = P.narrow;
    if (conv64) CYR_TRY(lf_tables<double>(P, tb64));
    else CYR_TRY(lf_tables<T>(P, tb));
    a.tpp = sh.tpp;
    a.pp = sh.pp;
  }
  const dim3 grid(ceil_div(a.rows, a.pp));
  bool found = true;
  hipError_t e = hipSuccess;
  constexpr int E0 = sizeof(T) == 4 ? 4 : 2;
  auto go = [&](auto tag) {
    using S = decltype(tag);
    if (ct) e = launch_xfields_ct_n<T, S, MODE>(a.nx, grid, lds, st, a, vox, morph, hann ? 1 : 0, &found);
    else if (conv64) {
      if constexpr (sizeof(T) == 4) e = launch_xfields_lf<T, S, E0, true, MODE>(tb64, sh, st, a, vox, morph, hann ? 1 : 0);
    } else if (!narrow) {
      if constexpr (sizeof(T) == 4) e = launch_xfields_lf<T, S, E0, false, MODE>(tb, sh, st, a, vox, morph, hann ? 1 : 0);
    } else if (e_lf == E0) e = launch_xfields_lf<T, S, E0, true, MODE>(tb, sh, st, a, vox, morph, hann ? 1 : 0);
    else if (e_lf == 2 * E0) e = launch_xfields_lf<T, S, 2 * E0, true, MODE>(tb, sh, st, a, vox, morph, hann ? 1 : 0);
    else if constexpr (sizeof(T) == 4) e = launch_xfields_lf<T, S, 4 * E0, true, MODE>(tb, sh, st, a, vox, morph, hann ? 1 : 0);
  };
  if constexpr (sizeof(T) == 4) {
    if (storage == CYR_STORE_FP16) go(half4{});
    else if (storage == CYR_STORE_BF16) go(bf164{});
    else go(float4{});
  } else {
    if (storage != CYR_STORE_NATIVE) return fail(CYR_E_UNSUPPORTED, "fused X kernel FP64: native morphology storage only");
    go(double4{});
  }
  if (e != hipSuccess) return hip_fail(e, "xfields_kernel", __FILE__, __LINE__);
  if (!found) return fail(CYR_E_UNSUPPORTED, "fused X kernel: no kernel for this length");
  return CYR_OK;
}

}  // namespace cyr
