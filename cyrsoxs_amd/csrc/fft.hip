// Forward complex-to-complex FFT pencils for gfx950 (replaces the reference's
// cufftExecC2C/Z2Z calls, include/cudaMain.h:184-190, src/cudaMain.cu:668-670).
//
// Contract: F[k] = sum_n x[n] exp(-2 pi i n k / N) along one axis, unnormalised,
// in place.  A 3D transform is three axis passes (X, Y, Z).
//
// Design (wave64 / LDS):
//   * A block owns `pp` whole pencils.  For the contiguous X axis the threads of a
//     pencil are consecutive lanes (row loads are unit-stride); for the strided
//     Y/Z axes the lanes run across `pp` adjacent pencils (each element load is a
//     pp*sizeof(complex) contiguous segment).
//   * The first stage's butterflies load from HBM, the stages exchange through LDS, and
//     the last stage's butterflies store to HBM: each element is read once and written
//     once per pass.  Lengths 64-2048 with a compile-time codelet run it (fftpolicy.hpp);
//     every other length runs the any-length transform (lfft.hpp).
//   * Twiddles come from a per-length table generated in FP64 on the host.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "fft.hpp"
#include "fftpolicy.hpp"
#include "stockham.hpp"

namespace cyr {

namespace {

constexpr uint32_t kPassVols = 24;  // volumes of one launch
struct PassArgs {
  void *vol[kPassVols];
  uint32_t nvol;  // volumes of this launch (1D XCD-ordered grids)
  uint64_t elem_stride;
  uint64_t inner_stride;
  uint64_t outer_stride;
  uint32_t inner_count;
  uint32_t outer_count;
  uint32_t groups;  // launched, of ceil(inner_count / pp)
  uint32_t pp;
  uint32_t glo = 0xffffffffu, gskip = 0;  // groups from glo on lie gskip further (column_groups)
  double2 *dcz;        // non-null: the Y pass adds the DC-neighbour partial sums (FftDc)
  const void *dc_twy;  // Y and Z twiddles of those sums (twz null in 2D)
  const void *dc_twz;
  uint32_t dc_nz;
  const uint32_t *span;  // Y pass: per output row, the shifted x range it writes (null: all)
  uint32_t reach = 0xffffffffu;  // Y pass: columns from bin 0, either way round, that are read later
};

// The column groups of a strided pass: all, or those within reach of bin 0 (the others are
// neither read nor written; 2048^2 film at 1 nm, 7 and 4 volumes: 307 -> 175 us).
inline void column_groups(PassArgs &A) {
  const uint32_t n = A.inner_count, total = (n + A.pp - 1) / A.pp;
  A.groups = total;
  A.glo = 0xffffffffu;
  A.gskip = 0;
  if (A.reach >= n / 2) return;
  const uint32_t lo = A.reach / A.pp + 1, hi = (n - A.reach) / A.pp;
  if (hi <= lo) return;
  A.glo = lo;
  A.gskip = hi - lo;
  A.groups = total - A.gskip;
}

// Compile-time codelet pass (lengths with a CtPlan): pencils held in registers,
// stages exchanged through LDS with immediate offsets.  Contiguous pencils (X)
// are padded LDS rows, several per wave when short, twiddles read from the
// global table; strided pencils (Y, Z) are PP-column tiles whose twiddles are
// staged in LDS next to the tile once per block.
// Load of one complex element marked non-temporal (streamed: each element of a
// strided pass is read once).  For the 512-point Y pass over 7 volumes of
// 512^2 x 128 it cuts the pass from 717 to 637 us; non-temporal stores add nothing.
template <typename T> __device__ inline cx<T> stream_load(const cx<T> *p) {
  if constexpr (sizeof(T) == 4) {
    const unsigned long long v = __builtin_nontemporal_load(reinterpret_cast<const unsigned long long *>(p));
    return mk<T>(__uint_as_float((unsigned)v), __uint_as_float((unsigned)(v >> 32)));
  } else {
    const double *d = reinterpret_cast<const double *>(p);
    return mk<T>(__builtin_nontemporal_load(d), __builtin_nontemporal_load(d + 1));
  }
}

template <typename T, class F, bool CONTIG, int WG>
__global__ void __launch_bounds__(WG) fft_ct_kernel(PassArgs A, const cx<T> *__restrict__ tw) {
  constexpr int E = F::kE, TPP = F::TPP, N = TPP * E;
  constexpr bool LO = !CONTIG && tw_lo_in_lds<T>((size_t)F::PE * N, N, WG);
  extern __shared__ unsigned char smem_raw[];
  cx<T> *lds = reinterpret_cast<cx<T> *>(smem_raw);
  const cx<T> *twp = tw;
  uint32_t t, p;
  if constexpr (CONTIG) {
    t = threadIdx.x % TPP;
    p = threadIdx.x / TPP;
  } else {
    if (xcd_tile(blockIdx.x, gridDim.x) >= A.groups * A.outer_count * A.nvol)
      return;  // grid padding: the whole block leaves before any barrier
    p = threadIdx.x % A.pp;
    t = threadIdx.x / A.pp;
  }
  uint32_t tile = blockIdx.x, vol = blockIdx.y;
  if constexpr (!CONTIG) {
    // 1D grid in XCD order: neighbouring column groups (sharing HBM sectors) on one XCD
    const uint32_t q = xcd_tile(blockIdx.x, gridDim.x);
    const uint32_t per_vol = A.groups * A.outer_count;
    vol = q / per_vol;
    tile = q % per_vol;
  }
  uint32_t g = tile % A.groups;
  const uint32_t o = tile / A.groups;
  if (g >= A.glo) g += A.gskip;
  const uint32_t pencil = g * A.pp + p;
  const bool active = pencil < A.inner_count;
  cx<T> *gbase = reinterpret_cast<cx<T> *>(A.vol[vol]) + (uint64_t)(active ? pencil : 0) * A.inner_stride +
                 (uint64_t)o * A.outer_stride;
  cx<T> v[E];
#pragma unroll
  for (int i = 0; i < E; i++) {
    if constexpr (CONTIG) v[i] = active ? gbase[(uint64_t)F::in_pos(t, i) * A.elem_stride] : mk<T>(0, 0);
    else v[i] = active ? stream_load<T>(gbase + (uint64_t)F::in_pos(t, i) * A.elem_stride) : mk<T>(0, 0);
  }
  if constexpr (!CONTIG) {
    // DC-neighbour sums (Y pass of X-transformed volumes, Nx >= 3): columns 0, 1
    // and Nx - 1 of slice z = o add sum_y w G(x, y, z), w = 2 cos(2 pi y / Ny)
    // + 2 cos(2 pi z / Nz) (3D) at x = 0 and 1 otherwise; one FP64 partial per
    // (volume, z, column, wave), the lanes of a wave that hold one column (lane
    // stride pp) combined in a fixed order
    if (A.dcz && (g == 0 || g == A.groups + A.gskip - 1)) {  // the same for the whole block
      const bool mine = active && (pencil <= 1 || pencil == A.inner_count - 1);
      const uint32_t which = pencil <= 1 ? pencil : 2;
      double sr = 0, si = 0;
      if (mine) {
        const double cz =
            A.dc_nz > 1 ? 2.0 * tw_cos<T>(reinterpret_cast<const cx<T> *>(A.dc_twz), A.dc_nz, o) : 0.0;
#pragma unroll
        for (int i = 0; i < E; i++) {
          const double w = which == 0 ? 2.0 * tw_cos<T>(reinterpret_cast<const cx<T> *>(A.dc_twy), N, F::in_pos(t, i)) + cz : 1.0;
          sr += w * (double)v[i].x;
          si += w * (double)v[i].y;
        }
      }
      for (uint32_t off = A.pp; off < 64; off <<= 1) {
        sr += __shfl_xor(sr, (int)off);
        si += __shfl_xor(si, (int)off);
      }
      if (mine && (threadIdx.x & 63) < A.pp)
        A.dcz[(((uint64_t)vol * A.dc_nz + o) * 3 + which) * (WG / 64) + threadIdx.x / 64] = make_double2(sr, si);
    }
  }
  if constexpr (!CONTIG) {
    // twiddles staged while the pencil loads are in flight, with the last
    // stage's FP32 residuals when they fit without costing occupancy (else they
    // are read from the global table, L2 resident)
    cx<T> *ltw = lds + (size_t)A.pp * N;
    for (uint32_t i = threadIdx.x; i < (uint32_t)(LO ? 2 * N : N); i += WG) ltw[i] = tw[i];
    if (A.span) {  // row spans beside the twiddles
      uint32_t *ls = reinterpret_cast<uint32_t *>(ltw + (LO ? 2 * N : N));
      for (uint32_t i = threadIdx.x; i < (uint32_t)N; i += WG) ls[i] = A.span[i];
    }
    lds_sync();
    twp = ltw;
  }
  // Row spans: output row y is written only where some Ewald band reads it, in
  // whole lines of the block's pp columns (a line is kept when any of its
  // columns' shifted x coordinates, m - x for bins x <= m = n/2 and n + m - x
  // above, lies in the row's lo..hi).  Skipping single columns leaves partial
  // lines, which made the pass slower than writing everything.
  uint32_t keep = (1u << E) - 1;
  if (!CONTIG && A.span) {
    const uint32_t *ls = reinterpret_cast<const uint32_t *>(lds + (size_t)A.pp * N + (LO ? 2 * N : N));
    const uint32_t n = A.inner_count, m = n / 2;
    const uint32_t x0 = g * A.pp, x1 = (x0 + A.pp < n ? x0 + A.pp : n) - 1;
    const bool lo_part = x0 <= m, hi_part = x1 > m;  // the line's bins <= m and > m
    const uint32_t a0 = m - (x1 < m ? x1 : m), a1 = m - x0;
    const uint32_t b0 = n + m - x1, b1 = n + m - (x0 > m + 1 ? x0 : m + 1);
    keep = 0;
#pragma unroll
    for (int i = 0; i < E; i++) {
      const uint32_t sp = ls[F::out_pos(t, i)], lo = sp & 0xffffu, hi = sp >> 16;
      const bool meet = lo <= hi && ((lo_part && a0 <= hi && a1 >= lo) || (hi_part && b0 <= hi && b1 >= lo));
      keep |= meet ? 1u << i : 0u;
    }
  }
  F::run(v, t, p, lds, twp, LO ? twp + N : tw + N);
  if (active) {
#pragma unroll
    for (int i = 0; i < E; i++)
      if (keep & (1u << i)) gbase[(uint64_t)F::out_pos(t, i) * A.elem_stride] = v[i];
  }
}

template <typename T, int N>
hipError_t launch_ct_n(bool contig, uint32_t nc, PassArgs &A, hipStream_t stream, const cx<T> *tw) {
  constexpr int E = N == 384 ? 12 : 8, TPP = N / E;
  if (contig) {
    using F = typename CtPlan<T, N, true, 1>::type;
    constexpr int WG = TPP <= 64 ? 64 : TPP;
    A.pp = WG / TPP;
    A.groups = (A.inner_count + A.pp - 1) / A.pp;
    const uint64_t blocks = (uint64_t)A.groups * A.outer_count;
    if (blocks > 0x7fffffffull) return hipErrorInvalidConfiguration;
    const size_t lds = (size_t)A.pp * F::kPitch * sizeof(cx<T>);
    hipLaunchKernelGGL((fft_ct_kernel<T, F, true, WG>), dim3((unsigned)blocks, nc), dim3(WG), lds, stream, A, tw);
  } else {
    constexpr int PP = N <= 512 ? 16 : (N == 1024 ? 8 : 4);
    using F = typename CtPlan<T, N, false, PP>::type;
    constexpr int WG = PP * TPP;
    A.pp = PP;
    column_groups(A);
    A.nvol = nc;
    const uint64_t tiles = (uint64_t)A.groups * A.outer_count * nc;
    if (tiles > 0x7ffffff0ull) return hipErrorInvalidConfiguration;
    constexpr bool LO = tw_lo_in_lds<T>((size_t)PP * N, N, WG);
    const size_t lds = ((size_t)PP * N + (LO ? 2 * N : N)) * sizeof(cx<T>) + (A.span ? 4 * (size_t)N : 0);
    hipLaunchKernelGGL((fft_ct_kernel<T, F, false, WG>), dim3(xcd_grid(tiles)), dim3(WG), lds, stream, A, tw);
  }
  return hipGetLastError();
}

template <typename T>
hipError_t launch_ct(uint32_t n, bool contig, uint32_t nc, PassArgs &A, hipStream_t stream, const cx<T> *tw,
                     bool *found) {
  *found = true;
  switch (n) {
    case 64: return launch_ct_n<T, 64>(contig, nc, A, stream, tw);
    case 128: return launch_ct_n<T, 128>(contig, nc, A, stream, tw);
    case 256: return launch_ct_n<T, 256>(contig, nc, A, stream, tw);
    case 384:
      if constexpr (sizeof(T) == 4) return launch_ct_n<T, 384>(contig, nc, A, stream, tw);
      break;
    case 512: return launch_ct_n<T, 512>(contig, nc, A, stream, tw);
    case 1024: return launch_ct_n<T, 1024>(contig, nc, A, stream, tw);
    case 2048: return launch_ct_n<T, 2048>(contig, nc, A, stream, tw);
    default: break;
  }
  *found = false;
  return hipSuccess;
}

// Any-length pass (lfft.hpp): rows (CONTIG) or tiles of pp columns, tpp threads per
// pencil.  In place: a block owns whole pencils, and its first stage has read every
// element before its last stage writes (a barrier lies between them; a one-stage
// transform's butterfly is the whole pencil).  DC sums and row spans as in
// fft_ct_kernel.
struct AnyShape {
  uint32_t tpp, lpp, pitch, pad;  // (tpp, lpp: columns; pitch, pad: rows)
};

// Inputs: of one column, or of the block's rows (rows past the last read the last).
template <typename T, typename C, bool CONTIG> struct AnyIn {
  const cx<T> *gp;
  uint64_t es;     // columns: element stride; rows: row stride
  uint32_t rows;   // rows of this block
  __device__ inline cx<C> load(uint32_t p, uint32_t e, uint32_t r, uint32_t q) const {
    if constexpr (CONTIG) return cx_as<C, T>(gp[(uint64_t)(p < rows ? p : rows - 1) * es + e + r * q]);
    else return cx_as<C, T>(stream_load<T>(gp + e * es + r * (q * es)));
  }
};

// TAB: the tables are in LDS (false: the longest pencils, read from memory).  C: the
// precision of the arithmetic (lf_precision).
template <typename T, typename C, bool CONTIG, bool TAB>
__global__ void __launch_bounds__(1024) fft_any_kernel(LfTab<C> tb, AnyShape sh, PassArgs A) {
  extern __shared__ unsigned char smem_raw[];
  cx<C> *lds = reinterpret_cast<cx<C> *>(smem_raw);
  uint32_t t = 0, p = 0, tile = blockIdx.x, vol = blockIdx.y;
  if constexpr (!CONTIG) {
    const uint32_t q = xcd_tile(blockIdx.x, gridDim.x);
    const uint32_t per_vol = A.groups * A.outer_count;
    if (q >= per_vol * A.nvol) return;  // grid padding: the whole block leaves before any barrier
    p = threadIdx.x & (A.pp - 1);
    t = threadIdx.x >> sh.lpp;
    vol = q / per_vol;
    tile = q % per_vol;
  }
  uint32_t g = tile % A.groups;
  const uint32_t o = tile / A.groups;
  if (g >= A.glo) g += A.gskip;
  const uint32_t pencil = g * A.pp + p;
  const bool active = pencil < A.inner_count;
  // (idle pencils read pencil 0 and write nothing)
  cx<T> *gp = reinterpret_cast<cx<T> *>(A.vol[vol]) + (uint64_t)o * A.outer_stride +
              (uint64_t)(active ? pencil : 0) * A.inner_stride;
  LfLds<C> tab{tb.tw, tb.tw + tb.m, tb.pos};
  cx<C> *after = lds + (CONTIG ? A.pp * sh.pitch : tb.m << sh.lpp);
  const uint32_t *span = A.span;
  if constexpr (TAB) {
    tab = lf_stage_tables<C, true>(tb, after);
    if (!CONTIG && A.span) {
      uint32_t *ls = reinterpret_cast<uint32_t *>(reinterpret_cast<unsigned char *>(after) +
                                                  lf_lds_tables<C>(tb.m, tb.nlast, !tb.blue));
      for (uint32_t i = threadIdx.x; i < tb.n; i += blockDim.x) ls[i] = A.span[i];
      span = ls;
    }
    lds_sync();
  }
  if constexpr (!CONTIG) {
    // DC-neighbour sums (fft_ct_kernel has the formula) of columns 0, 1 and Nx - 1, in the
    // blocks that hold them (of one-column tiles, column 1 is group 1): one more read of
    // those lines, ahead of the transform's own
    if (A.dcz && (g * A.pp <= 1 || g == A.groups + A.gskip - 1)) {
      const bool mine = active && (pencil <= 1 || pencil == A.inner_count - 1);
      const uint32_t which = pencil <= 1 ? pencil : 2;
      double sr = 0, si = 0;
      if (mine) {
        const double cz =
            A.dc_nz > 1 ? 2.0 * tw_cos<T>(reinterpret_cast<const cx<T> *>(A.dc_twz), A.dc_nz, o) : 0.0;
        for (uint32_t e = t; e < tb.n; e += sh.tpp) {
          const cx<T> v = gp[e * A.elem_stride];
          const double w =
              which == 0 ? 2.0 * tw_cos<T>(reinterpret_cast<const cx<T> *>(A.dc_twy), tb.n, e) + cz : 1.0;
          sr += w * (double)v.x;
          si += w * (double)v.y;
        }
      }
      for (uint32_t off = A.pp; off < 64; off <<= 1) {
        sr += __shfl_xor(sr, (int)off);
        si += __shfl_xor(si, (int)off);
      }
      if (mine && (threadIdx.x & 63) < A.pp)
        A.dcz[(((uint64_t)vol * A.dc_nz + o) * 3 + which) * (blockDim.x / 64) + threadIdx.x / 64] =
            make_double2(sr, si);
    }
  }
  const uint32_t rows = CONTIG ? (A.inner_count - g * A.pp < A.pp ? A.inner_count - g * A.pp : A.pp) : 1;
  AnyIn<T, C, CONTIG> in{gp, CONTIG ? A.inner_stride : A.elem_stride, rows};
  // the line's shifted x range (see fft_ct_kernel)
  const uint32_t n = A.inner_count, m = n / 2;
  const uint32_t x0 = g * A.pp, x1 = (x0 + A.pp < n ? x0 + A.pp : n) - 1;
  const bool lo_part = x0 <= m, hi_part = x1 > m;
  const uint32_t a0 = m - (x1 < m ? x1 : m), a1 = m - x0;
  const uint32_t b0 = n + m - x1, b1 = n + m - (x0 > m + 1 ? x0 : m + 1);
  auto out = [&](uint32_t row, uint32_t k0, uint32_t r, uint32_t dk, cx<C> v) {
    const uint32_t k = k0 + r * dk;
    bool keep = CONTIG ? row < rows : active;
    if constexpr (!CONTIG) {
      if (A.span) {
        const uint32_t sp = span[k], lo = sp & 0xffffu, hi = sp >> 16;
        keep = keep && lo <= hi && ((lo_part && a0 <= hi && a1 >= lo) || (hi_part && b0 <= hi && b1 >= lo));
      }
    }
    if (keep) {
      if constexpr (CONTIG) gp[row * in.es + k] = cx_as<T, C>(v);
      else gp[k0 * in.es + r * (dk * in.es)] = cx_as<T, C>(v);
    }
  };
  if constexpr (CONTIG) lf_run<false, false, true, C>(tb, tab, lds, LfRows{sh.pitch, sh.pad, A.pp}, in, out);
  else lf_run<false, false, true, C>(tb, tab, lds, LfCols{sh.lpp, p, t, sh.tpp}, in, out);
}

// Direct O(n^2) DFT of each pencil for lengths beyond the any-length tile (e.g. a
// large prime whose convolution does not fit in LDS): the pencil is staged in LDS,
// then every thread produces outputs.
template <typename T>
__global__ void __launch_bounds__(256) dft_pencil_kernel(uint32_t n, PassArgs A, const cx<T> *__restrict__ tw) {
  extern __shared__ unsigned char smem_raw[];
  cx<T> *x = reinterpret_cast<cx<T> *>(smem_raw);
  const uint32_t g = blockIdx.x % A.inner_count;
  const uint32_t o = blockIdx.x / A.inner_count;
  cx<T> *base = reinterpret_cast<cx<T> *>(A.vol[blockIdx.y]) + (uint64_t)g * A.inner_stride +
                (uint64_t)o * A.outer_stride;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) x[i] = base[(uint64_t)i * A.elem_stride];
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) {
    T re = 0, im = 0;
    uint32_t e = 0;
    for (uint32_t i = 0; i < n; i++) {
      const cx<T> u = cmul_tw<T>(x[i], tw, n, e);
      re += u.x;
      im += u.y;
      e += k;
      if (e >= n) e -= n;
    }
    base[(uint64_t)k * A.elem_stride] = mk<T>(re, im);
  }
}

// ---- host-side planning ------------------------------------------------------

std::mutex g_mu;
std::map<std::tuple<int, uint32_t, int>, DeviceBuffer> g_tw;  // (device, n, precision)
std::map<std::tuple<int, uint32_t, int>, DeviceBuffer> g_lf;  // (device, n, precision + 2 narrow): lfft.hpp tables

template <typename T> constexpr int prec_of() { return sizeof(T) == 8 ? CYR_FP64 : CYR_FP32; }

size_t max_lds_bytes() {
  static size_t v = 0;
  if (!v) {
    int dev = 0;
    hipGetDevice(&dev);
    int b = 0;
    if (hipDeviceGetAttribute(&b, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || b <= 0)
      b = 160 * 1024;  // gfx950 (the only target this library is built for)
    v = (size_t)b;
  }
  return v;
}

}  // namespace

size_t device_max_lds() { return max_lds_bytes(); }

// Host image of the length-n table (tw_len<T>(n) entries).
template <typename T> void twiddle_host(uint32_t n, cx<T> *h) {
  for (uint32_t m = 0; m < n; m++) {
    // exact-angle FP64 twiddle, rounded once to the compute precision; FP32
    // tables also keep the rounding residual (block 2)
    const double a = 2.0 * M_PI * (double)m / (double)n;
    const double c = std::cos(a), sn = -std::sin(a);
    h[m].x = (T)c;
    h[m].y = (T)sn;
    if (tw_blocks<T>() == 2) {
      h[n + m].x = (T)(c - (double)h[m].x);
      h[n + m].y = (T)(sn - (double)h[m].y);
    }
  }
}

// Under an installed scratch arena the table is built into the arena for this
// call (queued on the arena's stream), never into the process-wide cache.
template <typename T> const cx<T> *arena_twiddles(ScratchArena &a, uint32_t n, cyr_status *st) {
  const auto key = std::make_pair(n, prec_of<T>());
  auto it = a.tw.find(key);
  if (it != a.tw.end()) {
    *st = CYR_OK;
    return reinterpret_cast<const cx<T> *>(it->second);
  }
  const size_t bytes = sizeof(cx<T>) * tw_len<T>(n);
  void *d = a.carve(bytes);
  if (!d) {
    *st = fail(CYR_E_NOMEM, "allocation-free call: twiddle tables exceed the scratch array");
    return nullptr;
  }
  a.keep.emplace_back(bytes);
  twiddle_host<T>(n, reinterpret_cast<cx<T> *>(a.keep.back().data()));
  if (hipMemcpyAsync(d, a.keep.back().data(), bytes, hipMemcpyHostToDevice, a.stream) != hipSuccess) {
    (void)hipGetLastError();
    *st = fail(CYR_E_DEVICE, "twiddle upload failed");
    return nullptr;
  }
  a.tw[key] = d;
  *st = CYR_OK;
  return reinterpret_cast<const cx<T> *>(d);
}

template <typename T> const cx<T> *twiddles(uint32_t n, cyr_status *st) {
  if (ScratchArena *a = scratch_arena()) return arena_twiddles<T>(*a, n, st);
  int dev = 0;
  hipGetDevice(&dev);
  std::lock_guard<std::mutex> lk(g_mu);
  auto key = std::make_tuple(dev, n, prec_of<T>());
  auto it = g_tw.find(key);
  if (it != g_tw.end()) {
    *st = CYR_OK;
    return reinterpret_cast<const cx<T> *>(it->second.ptr);
  }
  const size_t len = tw_len<T>(n);
  std::vector<cx<T>> h(len);
  twiddle_host<T>(n, h.data());
  DeviceBuffer b;
  cyr_status s = ensure_buffer(b, sizeof(cx<T>) * len);
  if (s != CYR_OK) {
    *st = s;
    return nullptr;
  }
  if (hipMemcpy(b.ptr, h.data(), sizeof(cx<T>) * len, hipMemcpyHostToDevice) != hipSuccess) {
    free_buffer(b);
    *st = fail(CYR_E_DEVICE, "twiddle upload failed");
    return nullptr;
  }
  g_tw[key] = b;
  *st = CYR_OK;
  return reinterpret_cast<const cx<T> *>(b.ptr);
}

void fft_release() {
  std::lock_guard<std::mutex> lk(g_mu);
  for (auto &kv : g_tw) free_buffer(kv.second);
  g_tw.clear();
  for (auto &kv : g_lf) free_buffer(kv.second);
  g_lf.clear();
}

// ---- any-length plans and tables (lfft.hpp) -------------------------------------
namespace {

// Radices in the order of their stages' preference (odd ones last: the late stages
// step through LDS rows by the radix) and the relative cost of a stage: the LDS round
// trip and barrier every radix pays, plus its arithmetic and registers.
struct RadixCost {
  uint32_t r;
  double c;
};
constexpr RadixCost kRadices[] = {{10, 1.5}, {8, 1.25}, {6, 1.2}, {4, 1.05}, {2, 1.0}, {13, 2.4},
                                  {11, 2.1}, {9, 1.45}, {7, 1.4}, {5, 1.15}, {3, 1.02}};

// Cheapest sequence of radices (at most `cap`) with product n.
void radix_search(uint32_t n, uint32_t cap, size_t from, double cost, std::vector<uint32_t> &cur, double &best,
                  std::vector<uint32_t> &out) {
  if (n == 1) {
    if (cost < best && cur.size() <= (size_t)kLfStages) {
      best = cost;
      out = cur;
    }
    return;
  }
  for (size_t i = from; i < sizeof(kRadices) / sizeof(kRadices[0]); i++) {
    const uint32_t r = kRadices[i].r;
    if (r > cap || n % r != 0 || cost + kRadices[i].c >= best) continue;
    cur.push_back(r);
    radix_search(n / r, cap, i, cost + kRadices[i].c, cur, best, out);
    cur.pop_back();
  }
}

bool radix_sequence(uint32_t n, uint32_t cap, std::vector<uint32_t> &out, double &cost) {
  uint32_t r = n;
  for (uint32_t p : {2u, 3u, 5u, 7u, 11u, 13u})
    while (p <= cap && r % p == 0) r /= p;
  if (r != 1) return false;
  std::vector<uint32_t> cur;
  cost = 1e9;
  out.clear();
  radix_search(n, cap, 0, 0.0, cur, cost, out);
  return !out.empty();
}

// The tables are formed in extended precision and rounded once (their entries' errors
// would add to those of the arithmetic).
using xcomplex = std::complex<long double>;
constexpr long double kPiL = 3.14159265358979323846264338327950288L;

// exp(-2 pi i k / n)
xcomplex root_of(uint64_t k, uint64_t n) {
  const long double a = -2 * kPiL * (long double)(k % n) / (long double)n;
  return {std::cos(a), std::sin(a)};
}

// Forward FFT of a host vector whose length is a product of small primes (roots: those of
// the whole transform, `step` apart for this length).
void host_fft(std::vector<xcomplex> &x, const std::vector<xcomplex> &roots, size_t step) {
  const size_t n = x.size();
  if (n == 1) return;
  size_t p = 2;
  while (n % p != 0) p++;
  const size_t m = n / p;
  std::vector<std::vector<xcomplex>> sub(p, std::vector<xcomplex>(m));
  for (size_t i = 0; i < n; i++) sub[i % p][i / p] = x[i];
  for (auto &v : sub) host_fft(v, roots, step * p);
  for (size_t k = 0; k < n; k++) {
    xcomplex acc = 0;
    for (size_t r = 0; r < p; r++) acc += sub[r][k % m] * roots[(r * k) % n * step];
    x[k] = acc;
  }
}

size_t al64(size_t x) { return (x + 63) & ~(size_t)63; }

template <typename T> struct LfOffsets {
  size_t tw, chirp, spec, pos, total;  // (the stages come first)
  explicit LfOffsets(const LfPlan &P) {
    const size_t cs = sizeof(cx<T>);
    tw = al64(sizeof(P.st));
    chirp = tw + al64(cs * tw_len<T>(P.m));
    spec = chirp + (P.blue ? al64(cs * P.n) : 0);
    pos = spec + (P.blue ? al64(cs * P.m) : 0);
    total = pos + al64(sizeof(uint16_t) * P.m);
  }
};

// Host image of the tables of P.
template <typename T> std::vector<unsigned char> lf_host(const LfPlan &P) {
  const LfOffsets<T> o(P);
  std::vector<unsigned char> h(o.total, 0);
  std::memcpy(h.data(), P.st, sizeof(P.st));
  auto round = [](const xcomplex &c) { return mk<T>((T)c.real(), (T)c.imag()); };
  cx<T> *tw = reinterpret_cast<cx<T> *>(h.data() + o.tw);
  for (uint32_t k = 0; k < P.m; k++) {
    const xcomplex c = root_of(k, P.m);
    tw[k] = round(c);
    if (tw_blocks<T>() == 2) tw[P.m + k] = round(c - xcomplex(tw[k].x, tw[k].y));
  }
  uint16_t *pos = reinterpret_cast<uint16_t *>(h.data() + o.pos);
  for (uint32_t k = 0; k < P.m; k++) {
    uint32_t x = k, at = 0;
    for (uint32_t s = 0; s < P.nst; s++) {
      at += (x % P.st[s].radix) * P.st[s].q;
      x /= P.st[s].radix;
    }
    pos[k] = (uint16_t)at;
  }
  if (P.blue) {
    cx<T> *ch = reinterpret_cast<cx<T> *>(h.data() + o.chirp), *sp = reinterpret_cast<cx<T> *>(h.data() + o.spec);
    std::vector<xcomplex> b(P.m, 0.0L), roots(P.m);
    for (uint32_t k = 0; k < P.m; k++) roots[k] = root_of(k, P.m);
    for (uint32_t k = 0; k < P.n; k++) {
      const xcomplex c = root_of((uint64_t)k * k, 2ull * P.n);  // exp(-i pi k^2 / n)
      ch[k] = round(c);
      b[k] = std::conj(c);
      if (k) b[P.m - k] = std::conj(c);
    }
    host_fft(b, roots, 1);
    for (uint32_t k = 0; k < P.m; k++) sp[pos[k]] = round(b[k] / (long double)P.m);
  }
  return h;
}

}  // namespace

namespace {

// (cached by lf_plan: the search for a convolution length tries hundreds)
bool lf_search(uint32_t n, int precision, bool narrow, LfPlan &P) {
  std::vector<uint32_t> seq;
  double c;
  P = LfPlan{};
  P.n = P.m = n;
  P.narrow = narrow ? 1 : 0;
  if (!radix_sequence(n, narrow ? 8 : precision == CYR_FP64 ? 10 : 13, seq, c)) {
    // Bluestein: the cheapest convolution length (radices <= 10: the stages also
    // run backwards)
    double best = 1e18;
    std::vector<uint32_t> s2;
    for (uint32_t m = 2 * n - 1; m <= std::min(kLfMaxConvolution, 3 * n); m++) {
      if (!radix_sequence(m, narrow ? 8 : 10, s2, c)) continue;
      if (m * (2 * c + 2) < best) {
        best = m * (2 * c + 2);
        P.m = m;
        seq = s2;
      }
    }
    if (best > 1e17) return false;
    P.blue = 1;
  }
  P.nst = (uint32_t)seq.size();
  uint32_t L = P.m;
  for (uint32_t s = 0; s < P.nst; s++) {
    const uint32_t q = L / seq[s];
    P.st[s] = LfStage{seq[s], L, q, q > 1 ? (uint32_t)(((1ull << 32) + q - 1) / q) : 0, P.m / seq[s], 0, P.m / L};
    P.st[s].mb = P.st[s].nb > 1 ? (uint32_t)(((1ull << 32) + P.st[s].nb - 1) / P.st[s].nb) : 0;
    L = q;
  }
  return true;
}

}  // namespace

bool lf_plan(uint32_t n, int precision, bool narrow, LfPlan &P) {
  if (n < 2 || n > kLfMaxLength) return false;
  // by length, precision and width (at most 4 x kLfMaxLength small entries); n = 0: no
  // plan
  static std::mutex mu;
  static std::map<std::tuple<uint32_t, int, bool>, LfPlan> plans;
  std::lock_guard<std::mutex> lk(mu);
  const auto key = std::make_tuple(n, precision, narrow);
  auto it = plans.find(key);
  if (it == plans.end()) {
    LfPlan p;
    if (!lf_search(n, precision, narrow, p)) p.n = 0;
    it = plans.emplace(key, p).first;
  }
  P = it->second;
  return P.n != 0;
}

int lf_precision(uint32_t n, int precision) {
  LfPlan P;
  return precision == CYR_FP32 && n < kLfShortConvolution && lf_plan(n, CYR_FP32, false, P) && P.blue ? CYR_FP64
                                                                                                      : precision;
}

template <typename T> cyr_status lf_tables(const LfPlan &P, LfTab<T> &t) {
  const LfOffsets<T> o(P);
  const unsigned char *base = nullptr;
  if (ScratchArena *a = scratch_arena()) {
    // built into the arena for this call, never into the process-wide cache
    const auto key = std::make_pair(P.n, prec_of<T>() + 2 * (int)P.narrow);
    auto it = a->lf.find(key);
    if (it == a->lf.end()) {
      void *d = a->carve(o.total);
      if (!d) return fail(CYR_E_NOMEM, "allocation-free call: transform tables exceed the scratch array");
      a->keep.push_back(lf_host<T>(P));
      CYR_HIP(hipMemcpyAsync(d, a->keep.back().data(), o.total, hipMemcpyHostToDevice, a->stream));
      it = a->lf.emplace(key, d).first;
    }
    base = reinterpret_cast<const unsigned char *>(it->second);
  } else {
    int dev = 0;
    CYR_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_mu);
    const auto key = std::make_tuple(dev, P.n, prec_of<T>() + 2 * (int)P.narrow);
    auto it = g_lf.find(key);
    if (it == g_lf.end()) {
      const std::vector<unsigned char> h = lf_host<T>(P);
      DeviceBuffer b;
      CYR_TRY(ensure_buffer(b, h.size()));
      if (hipMemcpy(b.ptr, h.data(), h.size(), hipMemcpyHostToDevice) != hipSuccess) {
        free_buffer(b);
        return fail(CYR_E_DEVICE, "transform table upload failed");
      }
      it = g_lf.emplace(key, b).first;
    }
    base = reinterpret_cast<const unsigned char *>(it->second.ptr);
  }
  t.n = P.n;
  t.m = P.m;
  t.blue = P.blue;
  t.nst = P.nst;
  t.nlast = P.st[P.nst - 1].nb;
  t.st = reinterpret_cast<const LfStage *>(base);
  t.tw = reinterpret_cast<const cx<T> *>(base + o.tw);
  t.chirp = reinterpret_cast<const cx<T> *>(base + o.chirp);
  t.spec = reinterpret_cast<const cx<T> *>(base + o.spec);
  t.pos = reinterpret_cast<const uint16_t *>(base + o.pos);
  return CYR_OK;
}

// Threads per pencil, a multiple of `unit`: blocks of about 256 threads (more, smaller
// blocks per CU overlap one block's loads with another's stages), the count whose
// stages, in whole rounds of butterflies, keep the fewest threads idle.
uint32_t lf_threads(const LfPlan &P, uint32_t unit, uint32_t pencils) {
  uint32_t pick = 0;
  double best = 1e30;
  for (uint32_t t = unit; t * pencils <= 1024 && t < P.m / 2 + unit; t += unit) {
    double c = 0;
    for (uint32_t s = 0; s < P.nst; s++)
      for (const RadixCost &k : kRadices)
        if (k.r == P.st[s].radix) {
          const uint32_t rounds = (P.st[s].nb + t - 1) / t;
          c += (double)t * rounds * k.r * k.c + 0.1 * P.m * rounds;
        }
    const uint32_t wg = t * pencils;
    if (wg < 256) c *= 1.0 + 0.1 * (256 - wg) / 64.0;
    if (wg > 320) c *= 1.0 + 0.1 * (wg - 320) / 64.0;
    if (c < best) {
      best = c;
      pick = t;
    }
  }
  return pick;
}

// (comp: with the FP32 residuals of compensated products)
size_t lf_tables_lds(const LfPlan &P, int precision, bool comp) {
  const uint32_t nlast = P.st[P.nst - 1].nb;
  comp = comp && !P.blue;
  return precision == CYR_FP64 ? lf_lds_tables<double>(P.m, nlast, comp) : lf_lds_tables<float>(P.m, nlast, comp);
}

// Column tiles: max_cols adjacent pencils where three blocks of them (with room for a
// row-span table) fit in a CU's LDS, else fewer; whole waves.  One column that fits without
// its tables reads them from memory.
bool lf_cols_shape(const LfPlan &P, int precision, uint32_t max_cols, LfShape &s) {
  const size_t cs = precision == CYR_FP64 ? 16 : 8, cap = max_lds_bytes();
  s = LfShape{};
  for (uint32_t lpp = 6; lpp-- > 0;) {
    if (1u << lpp > max_cols) continue;
    const uint32_t pp = 1u << lpp;
    const size_t tile = cs * ((size_t)P.m << lpp), with = tile + lf_tables_lds(P, precision, true) + 4 * (size_t)P.n;
    if (lpp > 2 && with > cap / 3) continue;
    if (lpp > 0 && with > cap) continue;
    const bool tables = with <= cap;
    if (tile > cap) continue;
    const uint32_t tpp = lf_threads(P, 64 / pp, pp);
    if (!tpp) continue;
    s.pp = pp;
    s.lpp = lpp;
    s.tpp = tpp;
    s.threads = pp * tpp;
    s.tables = tables;
    s.lds = tables ? with : tile;
    return true;
  }
  return false;
}

// Rows: 2048 points of transforms for 256 threads, or, with e elements of a row per
// thread, as many rows as 256 threads hold (plain twiddle products).
bool lf_rows_shape(const LfPlan &P, int precision, uint32_t e, bool need_tables, LfShape &s) {
  const size_t cs = precision == CYR_FP64 ? 16 : 8, cap = max_lds_bytes();
  const size_t tab = lf_tables_lds(P, precision, e == 0);
  s = LfShape{};
  s.tpp = e ? (P.n + e - 1) / e : 0;
  if (s.tpp > kLfRowThreads) return false;
  uint32_t rows = e ? std::max(1u, 256 / s.tpp) : std::max(1u, 2048 / P.m);
  s.pad = kLfPad;
  auto tile = [&] { return cs * (size_t)rows * lf_row_pitch(P.m, s.pad); };
  while (rows > 1 && tile() + tab > cap / 3) rows /= 2;
  s.tables = tile() + tab <= cap;
  if (tile() > cap) s.pad = kLfNoPad;
  if (tile() > cap || (need_tables && !s.tables)) return false;
  s.pp = rows;
  s.threads = e ? rows * s.tpp : P.m > 4096 ? 512 : 256;
  s.pitch = lf_row_pitch(P.m, s.pad);
  s.lds = tile() + (s.tables ? tab : 0);
  return true;
}

namespace {

// One pass by the any-length transform (*done = false: the length is beyond it).
template <typename T>
cyr_status launch_any(uint32_t n, bool contig, uint32_t nc, PassArgs &A, hipStream_t st, bool *done) {
  LfPlan P;
  LfShape s;
  *done = false;
  const int prec = lf_precision(n, prec_of<T>());
  if (!lf_plan(n, prec, false, P)) return CYR_OK;
  if (!(contig ? lf_rows_shape(P, prec, 0, false, s) : lf_cols_shape(P, prec, 16, s))) return CYR_OK;
  A.pp = s.pp;
  column_groups(A);
  A.nvol = nc;
  const uint64_t tiles = (uint64_t)A.groups * A.outer_count;
  if (tiles * (contig ? 1 : nc) > 0x7ffffff0ull)
    return fail(CYR_E_UNSUPPORTED, "FFT grid too large");
  const AnyShape sh{s.tpp, s.lpp, s.pitch, s.pad};
  const dim3 block(s.threads), grid = contig ? dim3((unsigned)tiles, nc) : dim3(xcd_grid(tiles * nc));
#define CYR_ANY(C, CT, TB) hipLaunchKernelGGL((fft_any_kernel<T, C, CT, TB>), grid, block, s.lds, st, tb, sh, A)
  if (prec != prec_of<T>()) {  // (short: the tables are in LDS)
    LfTab<double> tb;
    CYR_TRY(lf_tables<double>(P, tb));
    if (contig) CYR_ANY(double, true, true);
    else CYR_ANY(double, false, true);
  } else {
    LfTab<T> tb;
    CYR_TRY(lf_tables<T>(P, tb));
    if (contig && s.tables) CYR_ANY(T, true, true);
    else if (contig) CYR_ANY(T, true, false);
    else if (s.tables) CYR_ANY(T, false, true);
    else CYR_ANY(T, false, false);
  }
#undef CYR_ANY
  CYR_LAUNCHED();
  *done = true;
  return CYR_OK;
}

}  // namespace

// Whether a strided pass of length n runs the compile-time codelets.
template <typename T> bool strided_ct(uint32_t n) {
  if (!ct_length(n) || (sizeof(T) == 8 && ct_elements(n) > 8)) return false;
  const uint32_t pp = n <= 512 ? 16 : (n == 1024 ? 8 : 4);
  return ((size_t)pp * n + n) * sizeof(cx<T>) <= max_lds_bytes();
}

// The compile-time block of length n also holds the row-span table (4 bytes per
// row) when that costs no occupancy; the any-length pass keeps it with its tables.
template <typename T> bool fft_span_fits(uint32_t n) {
  if (!strided_ct<T>(n)) {
    LfPlan P;
    LfShape s;
    const int prec = lf_precision(n, prec_of<T>());
    return lf_plan(n, prec, false, P) && lf_cols_shape(P, prec, 16, s);
  }
  const uint32_t pp = n <= 512 ? 16 : (n == 1024 ? 8 : 4), wg = pp * (n / ct_elements(n));
  const bool lo = tw_lo_in_lds<T>((size_t)pp * n, n, wg);
  const size_t lds = ((size_t)pp * n + (lo ? 2 * n : n)) * sizeof(cx<T>), with = lds + 4 * (size_t)n;
  return with <= max_lds_bytes() && cu_blocks(with, wg) >= cu_blocks(lds, wg);
}

// (partials per wave of the pass's block: pp pencils x threads per pencil)
template <typename T> uint32_t fft_dc_slots(uint32_t nx, uint32_t ny) {
  if (nx < 3 || ny < 2) return 0;
  if (strided_ct<T>(ny)) {
    const uint32_t pp = ny <= 512 ? 16 : (ny == 1024 ? 8 : 4);
    return 3 * (pp * (ny / ct_elements(ny)) / 64);
  }
  LfPlan P;
  LfShape s;
  const int prec = lf_precision(ny, prec_of<T>());
  return lf_plan(ny, prec, false, P) && lf_cols_shape(P, prec, 16, s) ? 3 * (s.pp * s.tpp / 64) : 0;
}

template <typename T>
cyr_status fft_axis(void *const *vols, uint32_t count, uint32_t nx, uint32_t ny, uint32_t nz, int axis,
                    hipStream_t stream, const FftDc *dc) {
  const uint32_t n = axis == 0 ? nx : axis == 1 ? ny : nz;
  if (n <= 1 || count == 0) return CYR_OK;
  cyr_status st;
  const cx<T> *tw = twiddles<T>(n, &st);
  if (!tw) return st;
  PassArgs A{};
  const bool contig = axis == 0;
  if (axis == 0) {
    A.elem_stride = 1;
    A.inner_stride = nx;
    A.inner_count = ny;
    A.outer_stride = (uint64_t)nx * ny;
    A.outer_count = nz;
  } else if (axis == 1) {
    A.elem_stride = nx;
    A.inner_stride = 1;
    A.inner_count = nx;
    A.outer_stride = (uint64_t)nx * ny;
    A.outer_count = nz;
  } else {
    A.elem_stride = (uint64_t)nx * ny;
    A.inner_stride = 1;
    A.inner_count = nx;
    A.outer_stride = nx;
    A.outer_count = ny;
  }
  const size_t lds_max = max_lds_bytes();
  bool use_ct;
  if (contig) {
    use_ct = ct_length(n) && (sizeof(T) == 4 || ct_elements(n) <= 8);
    if (use_ct) {
      const size_t need = (size_t)(64 / (n / ct_elements(n)) > 1 ? 64 / (n / ct_elements(n)) : 1) *
                          ct_row_pitch(n) * sizeof(cx<T>);
      if (need > lds_max) use_ct = false;
    }
  } else {
    use_ct = strided_ct<T>(n);
  }
  const uint64_t dc_per_vol = dc ? (uint64_t)nz * fft_dc_slots<T>(nx, ny) : 0;
  if (dc && (axis != 1 || dc_per_vol == 0)) return fail(CYR_E_INVALID, "FFT: DC sums need a Y pass and Nx >= 3");
  for (uint32_t c0 = 0; c0 < count; c0 += kPassVols) {
    const uint32_t nc = count - c0 < kPassVols ? count - c0 : kPassVols;
    for (uint32_t i = 0; i < nc; i++) A.vol[i] = vols[c0 + i];
    A.dcz = dc ? dc->dcz + c0 * dc_per_vol : nullptr;
    A.dc_twy = tw;
    A.dc_twz = dc ? dc->twz : nullptr;
    A.dc_nz = nz;
    A.reach = dc && dc->reach > 1 ? dc->reach : dc ? 1 : 0xffffffffu;
    A.span = dc && dc->span && fft_span_fits<T>(ny) ? dc->span : nullptr;
    bool done = false;
    if (use_ct) {
      bool found = false;
      const hipError_t e = launch_ct<T>(n, contig, nc, A, stream, tw, &found);
      if (e != hipSuccess) return hip_fail(e, "fft_ct_kernel", __FILE__, __LINE__);
      done = found;
    }
    if (!done) CYR_TRY(launch_any<T>(n, contig, nc, A, stream, &done));
    if (!done) {
      if (dc) return fail(CYR_E_INVALID, "FFT: DC sums need a tiled Y pass");
      if ((size_t)n * sizeof(cx<T>) > lds_max) return fail(CYR_E_UNSUPPORTED, "FFT length not supported");
      const uint64_t blocks = (uint64_t)A.inner_count * A.outer_count;
      if (blocks > 0x7fffffffull) return fail(CYR_E_UNSUPPORTED, "FFT grid too large");
      dim3 grid((unsigned)blocks, nc), block(256);
      hipLaunchKernelGGL((dft_pencil_kernel<T>), grid, block, (size_t)n * sizeof(cx<T>), stream, n, A, tw);
      CYR_LAUNCHED();
    }
  }
  return CYR_OK;
}

template <typename T>
cyr_status fft3d(void *const *vols, uint32_t count, uint32_t nx, uint32_t ny, uint32_t nz, hipStream_t stream) {
  CYR_TRY(fft_axis<T>(vols, count, nx, ny, nz, 0, stream));
  CYR_TRY(fft_axis<T>(vols, count, nx, ny, nz, 1, stream));
  CYR_TRY(fft_axis<T>(vols, count, nx, ny, nz, 2, stream));
  return CYR_OK;
}

template cyr_status lf_tables<float>(const LfPlan &, LfTab<float> &);
template cyr_status lf_tables<double>(const LfPlan &, LfTab<double> &);
template const cx<float> *twiddles<float>(uint32_t, cyr_status *);
template const cx<double> *twiddles<double>(uint32_t, cyr_status *);
template cyr_status fft_axis<float>(void *const *, uint32_t, uint32_t, uint32_t, uint32_t, int, hipStream_t,
                                    const FftDc *);
template cyr_status fft_axis<double>(void *const *, uint32_t, uint32_t, uint32_t, uint32_t, int, hipStream_t,
                                     const FftDc *);
template uint32_t fft_dc_slots<float>(uint32_t, uint32_t);
template uint32_t fft_dc_slots<double>(uint32_t, uint32_t);
template bool fft_span_fits<float>(uint32_t);
template bool fft_span_fits<double>(uint32_t);
template cyr_status fft3d<float>(void *const *, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t);
template cyr_status fft3d<double>(void *const *, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t);

}  // namespace cyr
