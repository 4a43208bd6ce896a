// Longitude transform of lengths up to 513 with a prime factor above 7 (67,
// 268, 341, 511, ...: grids of 2M + 1 or 3M + 1 longitudes), and of all lengths from 8
// to 63 but powers of two, as a folded real DFT on the matrix cores.
//
// With e_n = x_n + x_{N-n} and o_n = x_n - x_{N-n} (0 < n < N / 2) the rows are
//   cos row m = s_m (x_0 + (-1)^m x_{N/2}) + sum_n s_m cos(2 pi m n / N) e_n,
//   sin row m = sum_n s_m sin(2 pi m n / N) o_n
// (the x_{N/2} term for even N only), half the products of the unfolded sum,
// and in the other direction E_n = row 0 + sum_m cos .. g_cos, O_n = sum_m
// sin .. g_sin give x_n = E + O, x_{N-n} = E - O.  A wave owns 16 columns of
// one field: it holds the folded column (or its Fourier rows) in registers as
// MFMA B operands and sweeps tiles of 16 output rows, whose cos and sin
// coefficients come from a plan table in fragment order, staged through a
// double-buffered LDS tile that the waves of the block share.  Prime lengths cost the
// same as composite ones.
//
// The bound: I (2M - 1) flops a column on the FP32 / FP64 matrix cores (150 /
// 72 TFLOP/s) against 4 / 8 (I + 2M - 1) bytes at 4.7 TB/s.  I = 268, J = 134,
// B = 64, FP32: 22 / 18 us forward / inverse (0.36 GFLOP folded, 15 MB) against 206 / 141
// with the direct kernel, whose every product read LDS; I = 511, J = 256,
// B = 100: 75 / 66 us against 847 / 886.
#include <algorithm>

#include "dino_common.h"

namespace dino {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Frag;
template <>
struct Frag<float> {
  using V4 = f4;
  __device__ static V4 mma(float a, float b, V4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // output row of accumulator register i in lane group g
  __device__ static int row(int g, int i) { return 4 * g + i; }
};
template <>
struct Frag<double> {
  using V4 = d4;
  __device__ static V4 mma(double a, double b, V4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static int row(int g, int i) { return 4 * i + g; }
};

constexpr int kMaxGroups = 16;  // 16-term groups of the reduction: 256 folded terms

struct GemmArgs {
  int N, J, R, M;
  int terms;           // folded terms of the reduction: (N - 1) / 2 or M - 1
  int kg, tiles, gpf;  // term groups, output tiles, 16-column groups per field
  int weighted;
  int64_t groups;      // B * gpf
};

// KG: term groups the registers hold (kg <= KG of them in use).
template <typename T, int KG, int NW, bool INV>
__global__ __launch_bounds__(64 * NW) void dft_gemm_kernel(
    const T* __restrict__ in, T* __restrict__ out, const T* __restrict__ tab,
    const T* __restrict__ qw, GemmArgs a) {
  using V4 = typename Frag<T>::V4;
  constexpr int NTH = 64 * NW;
  constexpr int PER = (2 * KG * 64 + NTH - 1) / NTH;  // fragments a thread stages
  extern __shared__ __align__(32) unsigned char smem_raw[];
  V4* const lds = reinterpret_cast<V4*>(smem_raw);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c16 = lane & 15;
  const int N = a.N, J = a.J, M = a.M, kg = a.kg;
  const int tf = 2 * kg * 64;  // fragments of an output tile
  const V4* const tb = reinterpret_cast<const V4*>(tab);
  V4 st[PER];
  auto load_table = [&](int i) {
    const V4* src = tb + (int64_t)i * tf;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int idx = tid + NTH * q;
      st[q] = src[idx < tf ? idx : 0];
    }
  };
  load_table(0);

  // this wave's columns; waves past the last group and lanes past the last
  // column compute on a valid one and store nothing
  const int64_t grp = (int64_t)blockIdx.x * NW + wave;
  const int64_t gid = grp < a.groups ? grp : a.groups - 1;
  const int64_t b = gid / a.gpf;
  const int j = (int)(gid - b * a.gpf) * 16 + c16;
  const bool ok = grp < a.groups && j < J;
  const int jc = j < J ? j : J - 1;
  const T w = a.weighted ? qw[jc] : (T)1;
  const T* const src = in + b * (int64_t)(INV ? a.R : N) * J + jc;
  T* const dst = out + b * (int64_t)(INV ? N : a.R) * J + jc;

  // x0 / x1: cos and sin operands of the terms 1 + 16 t + 4 g + u
  T x0[KG][4], x1[KG][4];
#pragma unroll
  for (int t = 0; t < KG; ++t) {
    if (t >= kg) continue;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = 1 + 16 * t + 4 * g + u;
      const int kc = k <= a.terms ? k : 1;
      const T p = src[(int64_t)(INV ? 2 * kc - 1 : kc) * J];
      const T q = src[(int64_t)(INV ? 2 * kc : N - kc) * J];
      x0[t][u] = INV ? p : (p + q) * w;
      x1[t][u] = INV ? q : (p - q) * w;
      if (k > a.terms) x0[t][u] = x1[t][u] = (T)0;
    }
  }
  const T inv_sqrt_2pi = (T)0.39894228040143267794;
  const T inv_sqrt_pi = (T)0.56418958354775628695;
  T first, half = (T)0;  // x_0 and x_{N/2}, or the constant row
  first = src[0];
  if (INV) {
    first *= inv_sqrt_2pi;
  } else {
    first *= w;
    if ((N & 1) == 0) half = src[(int64_t)(N / 2) * J] * w;
  }

  for (int i = 0; i < a.tiles; ++i) {
    V4* const buf = lds + (i & 1) * tf;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int idx = tid + NTH * q;
      if (idx < tf) buf[idx] = st[q];
    }
    __syncthreads();
    // the last iteration reloads its own tile, which is never stored
    load_table(i + 1 < a.tiles ? i + 1 : i);
    __builtin_amdgcn_sched_barrier(0);
    V4 c, s = {0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * i + Frag<T>::row(g, r);
      c[r] = INV ? first
                 : (first + ((m & 1) ? -half : half)) * (m == 0 ? inv_sqrt_2pi : inv_sqrt_pi);
    }
#pragma unroll
    for (int t = 0; t < KG; ++t) {
      if (t >= kg) continue;
      const V4 pc = buf[t * 64 + lane];
      const V4 ps = buf[(kg + t) * 64 + lane];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        c = Frag<T>::mma(pc[u], x0[t][u], c);
        s = Frag<T>::mma(ps[u], x1[t][u], s);
      }
    }
    if (ok) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 16 * i + Frag<T>::row(g, r);
        if (INV) {
          if (2 * k <= N) dst[(int64_t)k * J] = (c[r] + s[r]) * w;
          if (k > 0 && 2 * k < N) dst[(int64_t)(N - k) * J] = (c[r] - s[r]) * w;
        } else {
          if (k < M) dst[(int64_t)(k == 0 ? 0 : 2 * k - 1) * J] = c[r];
          if (k > 0 && k < M) dst[(int64_t)(2 * k) * J] = s[r];
        }
      }
    }
  }
}

// Coefficients in fragment order: [tile][cos, sin][group][lane][u], the lane's
// output row 16 tile + lane % 16 and the term 1 + 16 group + 4 (lane / 16) + u.
template <typename T>
__global__ void dft_gemm_table_kernel(T* tab, int N, int M, int terms, int kg, int inverse,
                                      int64_t n) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  const int u = (int)(idx % 4), lane = (int)(idx / 4 % 64);
  const int64_t f = idx / 256;
  const int t = (int)(f % kg), part = (int)(f / kg % 2), i = (int)(f / (2 * kg));
  const int row = 16 * i + lane % 16, k = 1 + 16 * t + 4 * (lane / 16) + u;
  double v = 0;
  if (k <= terms && (inverse ? 2 * row <= N : row < M)) {
    double sn, cs;
    sincospi(2.0 * ((int64_t)row * k % N) / N, &sn, &cs);
    const double scale = !inverse && row == 0 ? 0.39894228040143267794 : 0.56418958354775628695;
    v = scale * (part ? sn : cs);
  }
  tab[idx] = (T)v;
}

inline int gemm_terms(const dino_plan* pl, bool inverse) {
  return inverse ? pl->M - 1 : (pl->I - 1) / 2;
}
inline int gemm_groups(const dino_plan* pl, bool inverse) {
  return std::max((gemm_terms(pl, inverse) + 15) / 16, 1);
}
inline int gemm_tiles(const dino_plan* pl, bool inverse) {
  return inverse ? pl->I / 32 + 1 : (pl->M + 15) / 16;
}

template <typename T, int KG, int NW, bool INV>
int launch_gemm(const T* in, T* out, const T* tab, const T* qw, const GemmArgs& a,
                hipStream_t s) {
  const size_t lds = sizeof(T) * 4 * 64 * 2 * 2 * (size_t)a.kg;
  const void* k = (const void*)dft_gemm_kernel<T, KG, NW, INV>;
  if (lds > 65536)
    DINO_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const unsigned grid = (unsigned)((a.groups + NW - 1) / NW);
  dft_gemm_kernel<T, KG, NW, INV><<<grid, 64 * NW, lds, s>>>(in, out, tab, qw, a);
  DINO_LAUNCH_CHECK("dft gemm kernel");
  return DINO_OK;
}

template <typename T, bool INV>
int gemm_by_groups(const T* in, T* out, const T* tab, const T* qw, const GemmArgs& a,
                   hipStream_t s) {
  // FP32: 4 waves a block spread a small batch over more CUs (I = 268, J = 134,
  // B = 64: 22 / 18 us against 26 / 23 with 8) and cost nothing on a large one.  FP64: 8, so that the
  // tables, twice as large, are fetched half as often (I = 320, B = 600: 174 us
  // against 206).
  constexpr int NW = sizeof(T) == 8 ? 8 : 4;
  if (a.kg <= 4) return launch_gemm<T, 4, NW, INV>(in, out, tab, qw, a, s);
  if (a.kg <= 8) return launch_gemm<T, 8, NW, INV>(in, out, tab, qw, a, s);
  if (a.kg <= 12) return launch_gemm<T, 12, NW, INV>(in, out, tab, qw, a, s);
  // FP64: 256 registers of operands leave one wave per SIMD
  return launch_gemm<T, 16, 4, INV>(in, out, tab, qw, a, s);
}

}  // namespace

bool dft_gemm_available(int I, int M) {
  return M >= 2 && I >= 8 && I <= 2 * 16 * kMaxGroups + 1 && M - 1 <= 16 * kMaxGroups;
}

// Lengths of factors 2, 3, 5, 7 that take this kernel rather than the mixed-radix FFT
// (dft_mixed.hip), whose passes are a chain of barriers however short the column is.
// Below 64 it is the faster one in both types at every batch; beyond, not for few
// fields in FP64.  Forward, FFT / here, us: I = 30, FP32, 12 fields 15.7 / 3.8, 1000 10.1 /
// 4.1; I = 45 13.6 / 4.7, 9.9 / 5.8, FP64 11.4 / 6.4, 10.9 / 7.9; I = 63 17.8 / 4.7, 12.6 / 6.6,
// 19.7 / 6.7, 15.8 / 9.8; I = 72 6.7 / 6.0, 12.7 / 11.0, 8.3 / 9.8, 20.5 / 19.7.  (The direct
// kernel: I = 30 7.5 and 11.0, I = 45 12.2 and 19.7.)
bool dft_gemm_short(int I) { return I < 64; }

int64_t dft_gemm_table_elems(const dino_plan* pl, bool inverse) {
  return (int64_t)gemm_tiles(pl, inverse) * 2 * gemm_groups(pl, inverse) * 256;
}

void dft_gemm_table_fill(const dino_plan* pl, hipStream_t s) {
  for (int inv = 0; inv < 2; ++inv) {
    const int64_t n = dft_gemm_table_elems(pl, inv);
    const unsigned grid = (unsigned)((n + 255) / 256);
    const int terms = gemm_terms(pl, inv), kg = gemm_groups(pl, inv);
    dft_gemm_table_kernel<float><<<grid, 256, 0, s>>>(pl->dftg32[inv], pl->I, pl->M, terms, kg,
                                                      inv, n);
    dft_gemm_table_kernel<double><<<grid, 256, 0, s>>>(pl->dftg64[inv], pl->I, pl->M, terms, kg,
                                                       inv, n);
  }
}

template <typename T>
int dft_gemm(bool forward, const dino_plan* pl, const T* in, T* out, const T* qw, int64_t B,
             int weighted, hipStream_t s) {
  GemmArgs a = {};
  a.N = pl->I;
  a.J = pl->J;
  a.R = pl->R;
  a.M = pl->M;
  a.terms = gemm_terms(pl, !forward);
  a.kg = gemm_groups(pl, !forward);
  a.tiles = gemm_tiles(pl, !forward);
  a.gpf = (pl->J + 15) / 16;
  a.groups = B * a.gpf;
  a.weighted = weighted;
  const T* tab;
  if constexpr (sizeof(T) == 8) tab = pl->dftg64[forward ? 0 : 1];
  else tab = pl->dftg32[forward ? 0 : 1];
  return forward ? gemm_by_groups<T, false>(in, out, tab, qw, a, s)
                 : gemm_by_groups<T, true>(in, out, tab, qw, a, s);
}

template int dft_gemm<float>(bool, const dino_plan*, const float*, float*, const float*, int64_t,
                             int, hipStream_t);
template int dft_gemm<double>(bool, const dino_plan*, const double*, double*, const double*,
                              int64_t, int, hipStream_t);

}  // namespace dino
