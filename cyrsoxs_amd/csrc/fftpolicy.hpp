// Register/LDS FFT policies shared by the FFT passes and the fused kernels.
//
// A policy transforms one pencil held by tpp threads, E elements each:
//   in_pos(t, i)   pencil index loaded into register slot i
//   holds(t, i)    whether slot i is an element of the pencil at all
//   stage(lds, pp, ...)  copies its tables behind the tile of pp pencils
//   transform(v, t, p, pp, lds, out)  the transform, exchanging through LDS;
//                  out(row, k, v) takes output k of a row
// Layouts: CONTIG pencils are rows of the LDS tile; otherwise pencils are
// columns (element e of pencil p at e pp + p), which keeps a wave's accesses to
// consecutive pencils in consecutive LDS words.
//
// CtFft: Stockham autosort with the radix sequence, the pencil length and the LDS
// pitch fixed at compile time, so every LDS offset and most index arithmetic fold
// into immediates.  Butterfly j (0 <= j < n/R) of a stage with sub-transform length
// Ls reads x[j + r n/R], multiplies by W_{Ls R}^{r (j mod Ls)}, does an R-point DFT
// and writes y[(j / Ls) Ls R + (j mod Ls) + r Ls]; a thread holds E elements (E/R
// butterflies, j = t + b tpp).  LfFft: any length (lfft.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include "lfft.hpp"
#include "stockham.hpp"

namespace cyr {

template <int A, int... B> struct FirstOf { static constexpr int value = A; };
template <int A, int... B> struct LastOf { static constexpr int value = LastOf<B...>::value; };
template <int A> struct LastOf<A> { static constexpr int value = A; };

// LDS addressing of the compile-time stages.  Column tiles (pencils are
// columns, PE = pencils per tile) place element e at e * PE; row tiles (PE = 1)
// pad one slot per 8 elements, e -> e + e / 8, so the radix-R scatter of a
// Stockham stage (lane stride R elements) spreads over the LDS banks.
__host__ __device__ constexpr uint32_t pad8(uint32_t e) { return e + (e >> 3); }

// Largest (A mod 8) over the stage's runtime store bases A = (t / LS) LS R + t mod LS.
template <int LS, int R> constexpr uint32_t max_base_mod8() {
  uint32_t m = 0;
  for (uint32_t t = 0; t < 8u * LS; t++) {
    const uint32_t a = ((t / LS) * (LS * R) + (t % LS)) % 8;
    m = a > m ? a : m;
  }
  return m;
}

// LDS slot of element A + B (A runtime, B compile-time).  For row tiles the
// padding splits when the low bits of A and B cannot carry into bit 3.
template <int PE, int LS, int R, uint32_t B> __device__ inline uint32_t lds_slot(uint32_t A) {
  if constexpr (PE != 1) {
    return (A + B) * PE;
  } else if constexpr (max_base_mod8<LS, R>() + (B % 8) <= 7) {
    return pad8(A) + (B / 8) * 9 + (B % 8);
  } else {
    return pad8(A + B);
  }
}

// Register slot i = b R + r -> LDS element o0 + (b TPP / LS) LS R + r LS (stage outputs).
template <typename T, int E, int PE, int LS, int R, int TPP, int I>
__device__ inline void ct_store(const cx<T> (&v)[E], uint32_t o0, cx<T> *lb) {
  if constexpr (I < E) {
    constexpr int b = I / R, r = I % R;
    constexpr uint32_t B = (uint32_t)((b * TPP / LS) * (LS * R) + r * LS);
    lb[lds_slot<PE, LS, R, B>(o0)] = v[I];
    ct_store<T, E, PE, LS, R, TPP, I + 1>(v, o0, lb);
  }
}

// Register slot i = b R2 + r <- LDS element t + b TPP + r M2 (next stage's inputs).
template <typename T, int E, int PE, int TPP, int M2, int R2, int I>
__device__ inline void ct_load(cx<T> (&v)[E], uint32_t t, const cx<T> *lb) {
  if constexpr (I < E) {
    constexpr int b = I / R2, r = I % R2;
    constexpr uint32_t B = (uint32_t)(b * TPP + r * M2);
    static_assert(PE != 1 || B % 8 == 0, "row-tile loads need 8-aligned offsets");
    if constexpr (PE != 1) v[I] = lb[(t + B) * PE];
    else v[I] = lb[pad8(t) + (B / 8) * 9];
    ct_load<T, E, PE, TPP, M2, R2, I + 1>(v, t, lb);
  }
}

// Stage with sub-transform length LS and radix R on registers, then (unless it
// is the last) the LDS exchange into the next stage's input order.  lb is the
// pencil's LDS base, PE the LDS stride between consecutive pencil elements
// (PE = 1: padded row, see lds_slot).
template <typename T, int N, int E, int PE, bool CP, int LS, int R, int... Rest>
__device__ inline void ct_stages(cx<T> (&v)[E], uint32_t t, cx<T> *lb, const cx<T> *__restrict__ tw,
                                 const cx<T> *__restrict__ twlo) {
  constexpr int TPP = N / E, NB = E / R, TSTEP = N / (LS * R);
  // with CP the last stage applies the finest twiddles as compensated products (FP32 hi + lo)
  constexpr bool COMP = CP && sizeof...(Rest) == 0 && tw_blocks<T>() == 2;
  static_assert(E % R == 0, "elements per thread must be a multiple of every radix");
  if constexpr (LS > 1) {
    if constexpr (TPP % LS == 0) {
      // every butterfly of this thread has the same twiddle exponent k = t mod LS
      const uint32_t k = t % LS;
      if (k != 0) {
        cx<T> w[R], wl[R];
#pragma unroll
        for (int r = 1; r < R; r++) {
          w[r] = tw[r * k * TSTEP];
          if constexpr (COMP) wl[r] = twlo[r * k * TSTEP];
        }
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int r = 1; r < R; r++) {
            if constexpr (COMP) v[b * R + r] = cmul_comp<T>(v[b * R + r], w[r], wl[r]);
            else v[b * R + r] = cmul<T>(v[b * R + r], w[r]);
          }
      }
    } else {
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const uint32_t k = (t + b * TPP) % LS;
        if (k != 0) {
#pragma unroll
          for (int r = 1; r < R; r++) {
            if constexpr (COMP) v[b * R + r] = cmul_comp<T>(v[b * R + r], tw[r * k * TSTEP], twlo[r * k * TSTEP]);
            else v[b * R + r] = cmul<T>(v[b * R + r], tw[r * k * TSTEP]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int b = 0; b < NB; b++) bfly<T, R>(&v[b * R]);
  if constexpr (sizeof...(Rest) > 0) {
    if constexpr (TPP % LS == 0) {
      const uint32_t o0 = (t / LS) * (LS * R) + (t % LS);
      ct_store<T, E, PE, LS, R, TPP, 0>(v, o0, lb);
    } else {
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const uint32_t j = t + b * TPP;
        const uint32_t o0 = (j / LS) * (LS * R) + (j % LS);
#pragma unroll
        for (int r = 0; r < R; r++) lb[PE == 1 ? pad8(o0 + r * LS) : (o0 + r * LS) * PE] = v[b * R + r];
      }
    }
    lds_sync();
    constexpr int R2 = FirstOf<Rest...>::value;
    static_assert(E % R2 == 0, "elements per thread must be a multiple of every radix");
    ct_load<T, E, PE, TPP, N / R2, R2, 0>(v, t, lb);
    lds_sync();
    ct_stages<T, N, E, PE, CP, LS * R, Rest...>(v, t, lb, tw, twlo);
  }
}

// CONTIG: pencil p at lds + p * pitch(N) as a padded row; otherwise lds + p with
// element stride PP.
template <typename T, int N, int E, bool CONTIG, int PP, int... R> struct CtFft {
  static constexpr uint32_t kPitch = N + N / 8;  // padded row length (CONTIG)
  static constexpr int kE = E, TPP = N / E;
  static constexpr int R0 = FirstOf<R...>::value, RL = LastOf<R...>::value;
  static constexpr int PE = CONTIG ? 1 : PP;
  static constexpr bool kCt = true;
  using Comp = T;  // precision of the arithmetic
  struct Plan {};
  __device__ explicit CtFft(const Plan &) {}
  __device__ static constexpr bool holds(uint32_t, int) { return true; }
  // rows: twiddles staged behind them (a barrier must follow), plain twiddle products
  __device__ static void stage(cx<T> *lds, uint32_t pp, const cx<T> *__restrict__ tw) {
    for (uint32_t i = threadIdx.x; i < (uint32_t)N; i += blockDim.x) lds[pp * kPitch + i] = tw[i];
  }
  template <class OUT>
  __device__ static void transform(cx<T> (&v)[E], uint32_t t, uint32_t p, uint32_t pp, cx<T> *lds, OUT out) {
    run<false>(v, t, p, lds, lds + pp * kPitch, nullptr);
#pragma unroll
    for (int i = 0; i < E; i++) out(p, out_pos(t, i), v[i]);
  }
  __device__ static uint32_t in_pos(uint32_t t, int i) { return t + (i / R0) * TPP + (i % R0) * (N / R0); }
  __device__ static uint32_t out_pos(uint32_t t, int i) { return t + (i / RL) * TPP + (i % RL) * (N / RL); }
  __device__ static constexpr uint32_t in_delta(int i) { return (i / R0) * TPP + (i % R0) * (N / R0); }
  template <bool COMP = true>
  __device__ static void run(cx<T> (&v)[E], uint32_t t, uint32_t p, cx<T> *lds, const cx<T> *__restrict__ tw,
                             const cx<T> *__restrict__ twlo) {
    cx<T> *lb = CONTIG ? lds + (size_t)p * kPitch : lds + p;
    ct_stages<T, N, E, PE, COMP, 1, R...>(v, t, lb, tw, twlo);
  }
};

// Any length (lfft.hpp), rows: slot i of thread t is element t + i tpp (E tpp >= n;
// the last slots may be empty).  Plain twiddle products.  C: precision of the arithmetic
// (lf_precision).
template <typename T, int E, bool NARROW, typename C = T> struct LfRowFft {
  static constexpr int kE = E;
  static constexpr bool kCt = false, kNarrow = NARROW;
  using Comp = C;
  struct Plan {
    LfTab<C> tb;
    uint32_t tpp;    // threads per row
    uint32_t pitch;  // LDS elements per row
    uint32_t pad;    // one slot of padding per 2^pad elements
  };
  const Plan P;
  __device__ explicit LfRowFft(const Plan &plan) : P(plan) {}
  __device__ uint32_t in_pos(uint32_t t, int i) const { return t + (uint32_t)i * P.tpp; }
  __device__ bool holds(uint32_t t, int i) const { return t + (uint32_t)i * P.tpp < P.tb.n; }
  // (the tables lie behind the rows: stage() copies them, a barrier must follow)
  __device__ void stage(cx<C> *lds, uint32_t pp) const { lf_stage_tables<C, false>(P.tb, lds + pp * P.pitch); }
  template <class OUT>
  __device__ void transform(cx<T> (&v)[E], uint32_t t, uint32_t p, uint32_t pp, cx<C> *lds, OUT out) const {
    const cx<C> *tw = lds + pp * P.pitch;
    const LfLds<C> tab{tw, nullptr, reinterpret_cast<const uint16_t *>(tw + P.tb.m)};
    const LfRows ad{P.pitch, P.pad, pp};
#pragma unroll
    for (int i = 0; i < E; i++)
      if (holds(t, i)) {
        const uint32_t e = in_pos(t, i);
        const cx<C> x = cx_as<C, T>(v[i]);
        lds[ad.at(p, e)] = P.tb.blue ? cmul<C>(x, P.tb.chirp[e]) : x;
      }
    if (P.tb.blue)
      for (uint32_t e = P.tb.n + t; e < P.tb.m; e += P.tpp) lds[ad.at(p, e)] = mk<C>(0, 0);
    lds_sync();
    LfNoInput<C> in;
    auto emit = [&](uint32_t row, uint32_t k, uint32_t r, uint32_t dk, cx<C> x) { out(row, k + r * dk, cx_as<T, C>(x)); };
    lf_run<true, NARROW, false, C>(P.tb, tab, lds, ad, in, emit);
    lds_sync();  // the rows may be refilled
  }
};

// Compile-time plans of the lengths the workloads use: elements per thread and
// radix sequence (radix-8 first; E = lcm of the radices).
template <typename T, int N, bool CONTIG, int PP> struct CtPlan;
template <typename T, bool C, int PP> struct CtPlan<T, 64, C, PP> { using type = CtFft<T, 64, 8, C, PP, 8, 8>; };
template <typename T, bool C, int PP> struct CtPlan<T, 128, C, PP> { using type = CtFft<T, 128, 8, C, PP, 8, 8, 2>; };
template <typename T, bool C, int PP> struct CtPlan<T, 256, C, PP> { using type = CtFft<T, 256, 8, C, PP, 8, 8, 4>; };
template <typename T, bool C, int PP> struct CtPlan<T, 384, C, PP> {
  using type = CtFft<T, 384, 12, C, PP, 4, 4, 4, 2, 3>;
};
template <typename T, bool C, int PP> struct CtPlan<T, 512, C, PP> { using type = CtFft<T, 512, 8, C, PP, 8, 8, 8>; };
template <typename T, bool C, int PP> struct CtPlan<T, 1024, C, PP> {
  using type = CtFft<T, 1024, 8, C, PP, 8, 8, 8, 2>;
};
template <typename T, bool C, int PP> struct CtPlan<T, 2048, C, PP> {
  using type = CtFft<T, 2048, 8, C, PP, 8, 8, 8, 4>;
};

// Lengths with a compile-time plan, its elements per thread, and the LDS
// elements one padded row of it takes.
inline bool ct_length(uint32_t n) {
  return n == 64 || n == 128 || n == 256 || n == 384 || n == 512 || n == 1024 || n == 2048;
}
inline uint32_t ct_elements(uint32_t n) { return n == 384 ? 12u : 8u; }
inline uint32_t ct_row_pitch(uint32_t n) { return n + n / 8; }

}  // namespace cyr
