// Transforms of any length inside one work group: the lengths without a
// compile-time codelet (fftpolicy.hpp).
//
// A pencil lives in LDS for the whole transform.  Every stage is an in-place
// decimation-in-frequency butterfly: butterfly b = blk q + j (j < q = L / R) of a
// stage with block length L and radix R reads the elements blk L + j + r q,
// transforms them, multiplies output r by W_L^(r j) and writes them back where
// they were.  One copy of the pencil (not two, as an autosort exchange needs when
// a thread's butterflies do not divide the pencil evenly) and one barrier per
// stage; radices may be any mix, so threads simply loop over the butterflies of a
// stage.  The first stage takes its inputs from a functor (HBM) and the last hands
// its outputs to one, in natural order: output kk + r n / R comes from the butterfly
// at slot pos[kk], the digit reversal, so nothing is reordered.
//
// Lengths with a prime factor above 13 (FP64: above 7) run Bluestein's algorithm in
// the same tile (short ones in FP64 arithmetic, lf_precision): with c_n = exp(-i pi n^2 / N), X_k = c_k sum_n (x_n c_n) conj(c_(k-n)),
// a circular convolution of length M >= 2N - 1 (M = 2^a 3^b 5^c 7^d).  The forward
// transform leaves digit-reversed order, the spectrum of the chirp is stored in
// that order, and the stages run backwards (decimation in time, digit-reversed in,
// natural out) give the inverse; the last forward butterfly, the product and the first
// inverse butterfly act on the same slots and stay in registers.  The direct O(N) sum
// per output that it replaces took 255 us for three 101 x 94 x 21 volumes.
//
// What bounds it: vector arithmetic and latency (about 20 instructions per element and
// stage, a third of them addresses and twiddles that a compile-time plan folds into
// immediates), not LDS (2 x (stages - 1) x 8 B per element plus twiddles).
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "stockham.hpp"

namespace cyr {

constexpr int kLfStages = 12;
constexpr uint32_t kLfMaxLength = 20480;       // one FP32 pencil in 160 KB of LDS
constexpr uint32_t kLfMaxConvolution = 16384;  // Bluestein's

struct LfStage {
  uint32_t radix;
  uint32_t L;   // block length
  uint32_t q;   // L / radix
  uint32_t mg;  // ceil(2^32 / q): b / q = mulhi(b, mg) for b q < 2^32 (q > 1)
  uint32_t nb;  // butterflies, m / radix
  uint32_t mb;  // ceil(2^32 / nb): i / nb = mulhi(i, mb) for i nb < 2^32 (nb > 1)
  uint32_t ts;  // twiddle step, m / L
};

struct LfPlan {
  uint32_t n;     // pencil length
  uint32_t m;     // transform length (n, or the convolution's)
  uint32_t blue;  // 1: Bluestein
  uint32_t nst;
  uint32_t narrow;
  LfStage st[kLfStages];
};

// Device tables of one length: W_m^k (k < m); pos[k], the slot of output k (uint16);
// Bluestein: chirp c_n (n < N) and the chirp's spectrum / m by slot.  In FP32 the twiddles
// are followed by their rounding residuals.
template <typename T> struct LfTab {
  uint32_t n, m, blue, nst;  // of the plan
  uint32_t nlast;            // butterflies of the last stage: pos[k] below it are used
  const LfStage *st;         // (device memory: stage numbers are run-time, and a kernel
                             // argument indexed by them would be copied to scratch)
  const cx<T> *tw;
  const cx<T> *chirp;
  const cx<T> *spec;
  const uint16_t *pos;
};

// The precision of the arithmetic of a length: FP64 for FP32 pencils of fewer than 208 points
// that need a convolution.  There the direct sum of compensated products is as close as an
// FP32 convolution or closer, whose intermediate values carry the pencil's mean through every
// slot: values about an offset, errors 2.0 (23 points), 1.6 (47), 1.2 (101) and 1.06 (202)
// times the sum's; from 211 on (0.86) it is the sum that is further off (499: 0.63), with
// compensated products in the convolution hardly more (0.82, 0.61).  In FP64 the error is
// the result's own rounding (101 x 94 x 21, 4 energies: 131 -> 153 us).
constexpr uint32_t kLfShortConvolution = 208;
int lf_precision(uint32_t n, int precision);

// Plan of a length (false: longer than the tile limit).  lf_tables builds its
// tables once per device (or in the caller's scratch arena).
// narrow: radices up to 8 only, for kernels that hold state of their own in registers.
bool lf_plan(uint32_t n, int precision, bool narrow, LfPlan &P);
template <typename T> cyr_status lf_tables(const LfPlan &P, LfTab<T> &t);

// Launch shape of a tile: pencils, threads per pencil and block, row pitch and padding, the
// dynamic LDS and whether it includes the tables (returns false when the pencil does
// not fit the tile).  Columns: at most max_cols (a power of two <= 32).  Rows: e > 0 for
// kernels that hold e elements of a row per thread (tpp threads of a row, at most
// kLfRowThreads).
constexpr uint32_t kLfRowThreads = 512;
struct LfShape {
  uint32_t pp = 0, lpp = 0, tpp = 0, threads = 0, pitch = 0, pad = 0;
  bool tables = false;
  size_t lds = 0;
};
// The longest columns go without tables, and rows do without `need_tables`.
bool lf_cols_shape(const LfPlan &P, int precision, uint32_t max_cols, LfShape &s);
bool lf_rows_shape(const LfPlan &P, int precision, uint32_t e, bool need_tables, LfShape &s);

// ---- butterflies beyond stockham.hpp's 2, 3, 4, 5, 8 (forward) -------------------
// cos and sin of 2 pi k / P, k = 1 .. (P - 1) / 2
template <int P> struct PrimeRoots;
template <> struct PrimeRoots<7> {
  static constexpr double c[3] = {0.62348980185873353052500488400424, -0.22252093395631440428890256449679,
                                  -0.90096886790241912623610231950745};
  static constexpr double s[3] = {0.78183148246802980870844452667406, 0.97492791218182360701813168299393,
                                  0.43388373911755812047576833284836};
};
template <> struct PrimeRoots<11> {
  static constexpr double c[5] = {0.84125353283118116886181164892437, 0.41541501300188642552927414923037,
                                  -0.14231483827328514044379266861756, -0.65486073394528506405692507247390,
                                  -0.95949297361449738989036805707332};
  static constexpr double s[5] = {0.54064081745559758210763595432092, 0.90963199535451837141171538309067,
                                  0.98982144188093273237609203778009, 0.75574957435425828377403584396855,
                                  0.28173255684142969771141791535280};
};
template <> struct PrimeRoots<13> {
  static constexpr double c[6] = {0.88545602565320989589719492060770, 0.56806474673115580251180755912752,
                                  0.12053668025532305334906768745255, -0.35460488704253562596963789260002,
                                  -0.74851074817110109863463059970135, -0.97094181742605202715698227629379};
  static constexpr double s[6] = {0.46472317204376854565588859600131, 0.82298386589365639457961060209735,
                                  0.99270887409805399280075164949252, 0.93501624268541482343978459979690,
                                  0.66312265824079520237678549266050, 0.23931566428755776715017104454620};
};

// X_j, X_(P-j) = a_0 + sum_k cos(2 pi j k / P) (a_k + a_(P-k)) -/+ i sum_k sin(...) (a_k - a_(P-k))
// (FP32, 13: constants with their rounding residuals, without which 13 points were 1.18 times
// as far off as the direct sum; 7 and 11 are no further than that either way)
template <typename T, int P> __device__ inline void bfly_prime(cx<T> *a) {
  constexpr int H = (P - 1) / 2;
  cx<T> t[H], d[H];
  cx<T> s0 = a[0];
#pragma unroll
  for (int k = 0; k < H; k++) {
    t[k] = cadd<T>(a[k + 1], a[P - 1 - k]);
    d[k] = csub<T>(a[k + 1], a[P - 1 - k]);
    s0 = cadd<T>(s0, t[k]);
  }
  const cx<T> a0 = a[0];
  a[0] = s0;
  static_for<1, H + 1>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    cx<T> m = a0, n = mk<T>(0, 0);
    static_for<1, H + 1>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      constexpr int e = (j * k) % P;
      constexpr T c = (T)PrimeRoots<P>::c[(e <= H ? e : P - e) - 1];
      constexpr double sd = e <= H ? PrimeRoots<P>::s[e - 1] : -PrimeRoots<P>::s[P - e - 1];
      constexpr T s = (T)sd;
      if constexpr (sizeof(T) == 4 && P == 13) {
        constexpr T cl = (T)(PrimeRoots<P>::c[(e <= H ? e : P - e) - 1] - (double)c), sl = (T)(sd - (double)s);
        m.x += cl * t[k - 1].x;
        m.y += cl * t[k - 1].y;
        n.x += sl * d[k - 1].x;
        n.y += sl * d[k - 1].y;
      }
      m.x += c * t[k - 1].x;
      m.y += c * t[k - 1].y;
      n.x += s * d[k - 1].x;
      n.y += s * d[k - 1].y;
    });
    a[j] = mk<T>(m.x + n.y, m.y - n.x);
    a[P - j] = mk<T>(m.x - n.y, m.y + n.x);
  });
}

// v (c + i s) with both constants' rounding residuals (FP32), as the table's finest products
template <typename T> __device__ inline cx<T> cmul_const(cx<T> v, double c, double s) {
  const cx<T> hi = mk<T>((T)c, (T)s);
  return cmul_comp<T>(v, hi, mk<T>((T)(c - (double)hi.x), (T)(s - (double)hi.y)));
}

template <typename T> __device__ inline void bfly6(cx<T> *a) {
  constexpr double r = 0.86602540378443864676372317075293618347;
  cx<T> e[3] = {a[0], a[2], a[4]}, o[3] = {a[1], a[3], a[5]};
  bfly3<T>(e);
  bfly3<T>(o);
  o[1] = cmul_const<T>(o[1], 0.5, -r);
  o[2] = cmul_const<T>(o[2], -0.5, -r);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    a[k] = cadd<T>(e[k], o[k]);
    a[k + 3] = csub<T>(e[k], o[k]);
  }
}

template <typename T> __device__ inline void bfly9(cx<T> *a) {
  // W_9^1, W_9^2, W_9^4
  constexpr double c1 = 0.76604444311897803520239265055542, s1 = -0.64278760968653932632264340990726;
  constexpr double c2 = 0.17364817766693034885171662676931, s2 = -0.98480775301220805936674302458952;
  constexpr double c4 = -0.93969262078590838405410927732473, s4 = -0.34202014332566873304409961468226;
  cx<T> c[3][3];
#pragma unroll
  for (int n = 0; n < 3; n++) {
    c[n][0] = a[n];
    c[n][1] = a[n + 3];
    c[n][2] = a[n + 6];
    bfly3<T>(c[n]);
  }
  c[1][1] = cmul_const<T>(c[1][1], c1, s1);
  c[1][2] = cmul_const<T>(c[1][2], c2, s2);
  c[2][1] = cmul_const<T>(c[2][1], c2, s2);
  c[2][2] = cmul_const<T>(c[2][2], c4, s4);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    cx<T> v[3] = {c[0][k], c[1][k], c[2][k]};
    bfly3<T>(v);
    a[k] = v[0];
    a[k + 3] = v[1];
    a[k + 6] = v[2];
  }
}

template <typename T> __device__ inline void bfly10(cx<T> *a) {
  // W_10^k = (cos 36k, -sin 36k)
  constexpr double c1 = 0.80901699437494742410229341718282, s1 = 0.58778525229247312916870595463907;
  constexpr double c2 = 0.30901699437494742410229341718282, s2 = 0.95105651629515357211643933337938;
  cx<T> e[5] = {a[0], a[2], a[4], a[6], a[8]}, o[5] = {a[1], a[3], a[5], a[7], a[9]};
  bfly5<T>(e);
  bfly5<T>(o);
  o[1] = cmul_const<T>(o[1], c1, -s1);
  o[2] = cmul_const<T>(o[2], c2, -s2);
  o[3] = cmul_const<T>(o[3], -c2, -s2);
  o[4] = cmul_const<T>(o[4], -c1, -s1);
#pragma unroll
  for (int k = 0; k < 5; k++) {
    a[k] = cadd<T>(e[k], o[k]);
    a[k + 5] = csub<T>(e[k], o[k]);
  }
}

template <typename T, int R> __device__ inline void bfly_any(cx<T> *a) {
  if constexpr (R == 6) bfly6<T>(a);
  else if constexpr (R == 9) bfly9<T>(a);
  else if constexpr (R == 10) bfly10<T>(a);
  else if constexpr (R == 7 || R == 11 || R == 13) bfly_prime<T, R>(a);
  else bfly<T, R>(a);
}

// ---- who does which butterfly ------------------------------------------------------
// Column tiles: the lanes run over the columns, thread t of column p takes butterflies
// t, t + nt, ...; element e at (e << lpp) + p.
struct LfCols {
  uint32_t lpp, p, t, nt;
  __device__ inline uint32_t first() const { return t; }
  __device__ inline uint32_t step() const { return nt; }
  __device__ inline uint32_t count(const LfStage &S) const { return S.nb; }
  __device__ inline void split(uint32_t i, const LfStage &, uint32_t &pencil, uint32_t &b) const {
    pencil = p;
    b = i;
  }
  // slot of element e0 + r q of the pencil, a0 that of e0
  __device__ inline uint32_t at(uint32_t, uint32_t e) const { return (e << lpp) + p; }
  __device__ inline uint32_t at(uint32_t, uint32_t a0, uint32_t, uint32_t r, uint32_t q) const {
    return a0 + r * (q << lpp);
  }
};
// Row tiles: the block's threads run over all butterflies of all its rows (a row's own
// threads would leave half a wave idle in every stage with fewer butterflies); element e
// of row p at p pitch + e + (e >> pad), one slot of padding per 8 elements (the late
// stages' stride-R accesses then spread over the banks; rows that only fit without it go
// unpadded).
struct LfRows {
  uint32_t pitch, pad, rows;
  __device__ inline uint32_t first() const { return threadIdx.x; }
  __device__ inline uint32_t step() const { return blockDim.x; }
  __device__ inline uint32_t count(const LfStage &S) const { return rows * S.nb; }
  __device__ inline void split(uint32_t i, const LfStage &S, uint32_t &pencil, uint32_t &b) const {
    pencil = S.nb == 1 ? i : __umulhi(i, S.mb);
    b = i - pencil * S.nb;
  }
  __device__ inline uint32_t at(uint32_t p, uint32_t e) const { return p * pitch + e + (e >> pad); }
  __device__ inline uint32_t at(uint32_t p, uint32_t, uint32_t e0, uint32_t r, uint32_t q) const {
    return at(p, e0 + r * q);
  }
};
constexpr uint32_t kLfPad = 3, kLfNoPad = 31;
inline uint32_t lf_row_pitch(uint32_t m, uint32_t pad) { return m + (m >> pad) + (pad == kLfNoPad ? 0 : 1); }

// The tables a block keeps in LDS behind its tile (twiddles and digit reversal; a
// pointer that could be either LDS or memory would make every twiddle load a flat
// one).
template <typename T> struct LfLds {
  const cx<T> *tw, *lo;  // (lo: FP32 residuals)
  const uint16_t *pos;
};
// Twiddle entries a block keeps: with comp (not in convolutions), FP32 residuals too.
template <typename T> __host__ __device__ constexpr uint32_t lf_lds_twiddles(uint32_t m, bool comp) {
  return comp ? (uint32_t)tw_len<T>(m) : m;
}
// LDS bytes of the tables.
template <typename T> __host__ __device__ constexpr size_t lf_lds_tables(uint32_t m, uint32_t nlast, bool comp) {
  return sizeof(cx<T>) * lf_lds_twiddles<T>(m, comp) + ((sizeof(uint16_t) * nlast + 15) & ~(size_t)15);
}
// Copies them to `at` (a barrier must follow).
template <typename T, bool COMP> __device__ inline LfLds<T> lf_stage_tables(const LfTab<T> &P, cx<T> *at) {
  const uint32_t n = lf_lds_twiddles<T>(P.m, COMP && !P.blue);
  uint16_t *pos = reinterpret_cast<uint16_t *>(at + n);
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) at[i] = P.tw[i];
  for (uint32_t i = threadIdx.x; i < P.nlast; i += blockDim.x) pos[i] = P.pos[i];
  return LfLds<T>{at, at + P.m, pos};
}

// ---- stages -------------------------------------------------------------------------
// What a stage does besides the butterflies (uniform over the grid):
enum LfRole : uint32_t {
  kLfIn = 1,   // inputs from the functor (times the chirp, zeros from n on: Bluestein)
  kLfOut = 2,  // outputs to the functor
  kLfInv = 4,  // run backwards: twiddles before the butterfly
  kLfMid = 8   // Bluestein's turn: last forward butterfly, spectrum, first inverse one
};

// Stage S of the block's pencils.
// COMP, FP32: the finest twiddles, those of the first stage, are compensated products, as the
// finest of the codelets' passes are (not in convolutions).  Their residuals lie in LDS
// beside them (200 x 240 x 50, 12 energies: 491 us with plain products, 522 with residuals
// read from L2 ahead of the butterfly, 511 from LDS).
template <typename T, int R, bool COMP, class AD, class IN, class OUT>
__device__ inline void lf_stage(const LfTab<T> &P, const LfStage &S, uint32_t role, const LfLds<T> &tab, cx<T> *buf,
                                const AD &ad, IN &in, OUT &out) {
  const uint32_t q = S.q, count = ad.count(S);
#pragma unroll 1
  for (uint32_t i = ad.first(); i < count; i += ad.step()) {
    uint32_t p, b;
    ad.split(i, S, p, b);
    // (the last forward stage, q = 1, goes by output: block pos[b] / R)
    const bool last = q == 1;
    const uint32_t blk = last ? b : __umulhi(b, S.mg);
    const uint32_t j = last ? 0 : b - blk * q;
    const uint32_t e0 = (role & (kLfOut | kLfInv)) == kLfOut ? tab.pos[b] : blk * S.L + j;
    const uint32_t a0 = ad.at(p, e0);
    cx<T> v[R];
    if (role & kLfIn) {
      if (!P.blue) {
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = in.load(p, e0, r, q);
      } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
          const uint32_t e = e0 + r * q, ec = e < P.n ? e : 0;
          v[r] = in.load(p, ec, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
          const uint32_t e = e0 + r * q;
          const cx<T> c = cmul<T>(v[r], P.chirp[e < P.n ? e : 0]);
          v[r] = e < P.n ? c : mk<T>(0, 0);
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; r++) v[r] = buf[ad.at(p, a0, e0, r, q)];
    }
    const uint32_t w = j * S.ts;
    auto twiddle = [&] {
      if constexpr (COMP && sizeof(T) == 4) {
        if (S.ts == 1 && !P.blue) {  // (uniform)
#pragma unroll
          for (int r = 1; r < R; r++) v[r] = cmul_comp<T>(v[r], tab.tw[r * w], tab.lo[r * w]);
          return;
        }
      }
#pragma unroll
      for (int r = 1; r < R; r++) v[r] = cmul<T>(v[r], tab.tw[r * w]);
    };
    if ((role & kLfInv) && !last) twiddle();
    bfly_any<T, R>(v);
    if constexpr (R <= 10) {
      if (role & kLfMid) {
        // times the chirp's spectrum; real and imaginary parts swapped, so that
        // forward butterflies give the inverse transform (swapped back at the end)
#pragma unroll
        for (int r = 0; r < R; r++) {
          const cx<T> u = cmul<T>(v[r], P.spec[e0 + r]);
          v[r] = mk<T>(u.y, u.x);
        }
        bfly_any<T, R>(v);
      }
    }
    if (!(role & kLfInv) && !last) twiddle();
    if (role & kLfOut) {
      if (role & kLfInv) {
#pragma unroll
        for (int r = 0; r < R; r++) {
          const uint32_t k = e0 + r * q;
          if (k < P.n) out(p, k, 0, 0, cmul<T>(mk<T>(v[r].y, v[r].x), P.chirp[k]));
        }
      } else {
#pragma unroll
        for (int r = 0; r < R; r++) out(p, b, r, S.nb, v[r]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; r++) buf[ad.at(p, a0, e0, r, q)] = v[r];
    }
  }
}

template <bool NARROW, bool COMP, typename T, class AD, class IN, class OUT>
__device__ inline void lf_stage_any(const LfTab<T> &P, uint32_t s, uint32_t role, const LfLds<T> &tab, cx<T> *buf,
                                    const AD &ad, IN &in, OUT &out) {
  const LfStage S = P.st[s];
  // (uniform over the grid; FP64 butterflies of 11 and 13 would spill: those lengths run
  // Bluestein)
  switch (S.radix) {
    case 2: lf_stage<T, 2, COMP>(P, S, role, tab, buf, ad, in, out); break;
    case 3: lf_stage<T, 3, COMP>(P, S, role, tab, buf, ad, in, out); break;
    case 4: lf_stage<T, 4, COMP>(P, S, role, tab, buf, ad, in, out); break;
    case 5: lf_stage<T, 5, COMP>(P, S, role, tab, buf, ad, in, out); break;
    case 6: lf_stage<T, 6, COMP>(P, S, role, tab, buf, ad, in, out); break;
    case 7: lf_stage<T, 7, COMP>(P, S, role, tab, buf, ad, in, out); break;
    case 8: lf_stage<T, 8, COMP>(P, S, role, tab, buf, ad, in, out); break;
    case 9: if constexpr (!NARROW) lf_stage<T, 9, COMP>(P, S, role, tab, buf, ad, in, out); break;
    case 10: if constexpr (!NARROW) lf_stage<T, 10, COMP>(P, S, role, tab, buf, ad, in, out); break;
    case 11: if constexpr (!NARROW && sizeof(T) == 4) lf_stage<T, 11, COMP>(P, S, role, tab, buf, ad, in, out); break;
    default: if constexpr (!NARROW && sizeof(T) == 4) lf_stage<T, 13, COMP>(P, S, role, tab, buf, ad, in, out); break;
  }
}

// Inputs already in LDS.
template <typename T> struct LfNoInput {
  __device__ inline cx<T> load(uint32_t, uint32_t, uint32_t, uint32_t) const { return mk<T>(0, 0); }
};

// Transforms the block's pencils: in.load(p, e0, r, q) gives input e0 + r q < n of pencil
// p, out(p, k0, r, dk, v) takes its output k0 + r dk (q and dk uniform: addresses step by
// scalars).  FROM_LDS: the inputs are already stored in LDS, behind a barrier (Bluestein:
// times the chirp, zeros from n on).  NARROW: a narrow plan.  COMP: see lf_stage.  Every thread of the block
// calls it; barriers separate the stages, none follows the last.
template <bool FROM_LDS, bool NARROW, bool COMP, typename T, class AD, class IN, class OUT>
__device__ inline void lf_run(const LfTab<T> &P, const LfLds<T> &tab, cx<T> *buf, const AD &ad, IN &in, OUT &out) {
  const uint32_t steps = P.blue ? 2 * P.nst - 1 : P.nst;
#pragma unroll 1
  for (uint32_t i = 0; i < steps; i++) {
    uint32_t role = (!FROM_LDS && i == 0 ? kLfIn : 0) | (i + 1 == steps ? kLfOut : 0);
    if (P.blue) role |= i + 1 == P.nst ? kLfMid : i >= P.nst ? kLfInv : 0;
    lf_stage_any<NARROW, COMP, T>(P, i < P.nst ? i : steps - 1 - i, role, tab, buf, ad, in, out);
    if (i + 1 < steps) lds_sync();
  }
}

}  // namespace cyr
