// Longitude transform for smooth I from 64 on that is no power of two (96, 192, 320,
// 360, 640, 1280, ... : every factor 2, 3, 5 or 7): mixed-radix Stockham FFT
// in LDS, same packing and unpacking as dft.hip (two real latitude columns
// form one complex column).
//
// The transform moves 4 (I + 2M - 1) bytes a column and should run at the
// copy rate; the direct DFT that served these I before took O(I M) operations
// and LDS reads a column.  FP32, forward / inverse: I = 1280, J = 640, B = 37: 7.2 /
// 5.1 ms direct, 0.110 / 0.100 now (2.2 / 2.4 TB/s); I = 320, J = 160, B = 600,
// 0.061 / 0.061 (3.4 TB/s).  What bounds it now is the passes' index and
// butterfly arithmetic, overlapped with the loads and stores of the other
// workgroups on the CU.
//
// Persistent workgroups walk tiles of one field and 2P latitude columns: one
// coalesced read of the tile (2P * sizeof(T) bytes of each row), prefetched
// while the previous tile is transformed, passes of radix up to 10 in place
// (all butterflies of a pass in registers, at most kElems complex values a
// thread), one write.  The length, the pass radices and the
// divisions by the running transform length are launch arguments, so one
// kernel per (type, P) serves every length.
#include <algorithm>

#include "dft_common.h"

namespace dino {

int device_cus();  // dft.hip

namespace {

constexpr int kMaxPasses = 12;
constexpr int kElems = 8;       // complex elements of the tile per thread, at most
constexpr int kThreads = 1024;  // per workgroup, at most

struct MixedArgs {
  int N, J, R, M;  // longitudes, latitudes, Fourier rows, wavenumbers
  int npass, tpf, weighted, vec;  // tiles per field; vec: 16-byte rows and buffers
  int64_t ntiles;
  int radix[kMaxPasses];
  unsigned magic[kMaxPasses];  // ceil(2^32 / Ns), Ns = product of the previous radices
};

// Thread index that the compiler takes as new at each call, so that index
// arithmetic is not hoisted out of the pass and tile loops (every radix's at
// once: 150 / 190 registers in the forward / inverse kernel instead of 78 / 77).
__device__ __forceinline__ int opaque_tid() {
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  return tid;
}

template <typename T, int P, int R, bool INV>
__device__ __forceinline__ void mixed_pass(cplx<T>* buf, const cplx<T>* tws, int N, int Ns,
                                           unsigned magic) {
  constexpr int BPT = (kElems + R - 1) / R;
  const int NB = N / R, tot = NB * P;
  const int step = NB / Ns;  // N / (Ns R)
  const int NT = blockDim.x;
  const int tid = opaque_tid();
  cplx<T> v[BPT][R];
#pragma unroll
  for (int q = 0; q < BPT; ++q) {
    const int t = tid + q * NT;
    if (t < tot) {
      const int p = t % P, j = t / P;
#pragma unroll
      for (int r = 0; r < R; ++r) v[q][r] = buf[(j + r * NB) * P + p];
      if (Ns > 1) {
        const int k = j - (int)__umulhi((unsigned)j, magic) * Ns;
#pragma unroll
        for (int r = 1; r < R; ++r) {
          cplx<T> w = tws[r * k * step];
          if (INV) w.y = -w.y;
          v[q][r] = cmul(v[q][r], w);
        }
      }
      dft_r<T, R, INV>(v[q]);
    }

  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < BPT; ++q) {
    const int t = tid + q * NT;
    if (t < tot) {
      const int p = t % P, j = t / P;
      const int g = Ns > 1 ? (int)__umulhi((unsigned)j, magic) : j;
      const int d = g * Ns * (R - 1) + j;  // g Ns R + (j - g Ns)
#pragma unroll
      for (int r = 0; r < R; ++r) buf[(d + r * Ns) * P + p] = v[q][r];
    }
  }
  __syncthreads();
}

template <typename T, int P, bool INV>
__device__ __forceinline__ void mixed_fft(cplx<T>* buf, const cplx<T>* tws, const MixedArgs& a) {
  int Ns = 1;
  for (int i = 0; i < a.npass; ++i) {
    const int r = a.radix[i];
    const unsigned mg = a.magic[i];
    switch (r) {
      case 2: mixed_pass<T, P, 2, INV>(buf, tws, a.N, Ns, mg); break;
      case 3: mixed_pass<T, P, 3, INV>(buf, tws, a.N, Ns, mg); break;
      case 4: mixed_pass<T, P, 4, INV>(buf, tws, a.N, Ns, mg); break;
      case 5: mixed_pass<T, P, 5, INV>(buf, tws, a.N, Ns, mg); break;
      case 6: mixed_pass<T, P, 6, INV>(buf, tws, a.N, Ns, mg); break;
      case 7: mixed_pass<T, P, 7, INV>(buf, tws, a.N, Ns, mg); break;
      case 8: mixed_pass<T, P, 8, INV>(buf, tws, a.N, Ns, mg); break;
      case 9: mixed_pass<T, P, 9, INV>(buf, tws, a.N, Ns, mg); break;
      default: mixed_pass<T, P, 10, INV>(buf, tws, a.N, Ns, mg); break;
    }
    Ns *= r;
  }
}

// 16-byte vector of the data type
template <typename T>
struct vec16;
template <>
struct vec16<float> {
  typedef float type __attribute__((ext_vector_type(4)));
};
template <>
struct vec16<double> {
  typedef double type __attribute__((ext_vector_type(2)));
};

// Tiles of a persistent workgroup: each XCD takes a contiguous eighth of the
// tiles and its workgroups walk it side by side, so the column tiles of one
// field, which share 128-byte lines when 2P columns are less than a line or
// J is not a multiple of it, share an L2.
struct TileWalk {
  int64_t next, end;
  int stride;
  __device__ explicit TileWalk(int64_t n) {
    const int x = gridDim.x < 8 ? (int)gridDim.x : 8;
    const int k = (int)blockIdx.x % x;
    stride = ((int)gridDim.x - k + x - 1) / x;
    next = n * k / x + blockIdx.x / x;
    end = n * (k + 1) / x;
  }
};

template <typename T, int P>
__global__ __launch_bounds__(kThreads) void dft_forward_mixed_kernel(
    const T* __restrict__ nodal, T* __restrict__ fourier, const T* __restrict__ tw,
    const T* __restrict__ qw, MixedArgs a) {
  using VT = typename vec16<T>::type;
  constexpr int C = 2 * P, V = 16 / sizeof(T), CV = C / V;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cplx<T>* buf = reinterpret_cast<cplx<T>*>(smem_raw);
  cplx<T>* tws = buf + a.N * P;
  T* lds = reinterpret_cast<T*>(buf);
  const int NT = blockDim.x, N = a.N, J = a.J;
  // tile elements of this thread: vectors (cv, n0 + q NT / CV), or scalars
  constexpr int IT = (kElems * 2 + V - 1) / V;
  VT pre[IT];
  auto issue = [&](int64_t t) {
    const int tid = opaque_tid(), cv = tid % CV, n0 = tid / CV;
    const int64_t b = t / a.tpf;
    const int j0 = (int)(t - b * a.tpf) * C;
    // columns past J (whole vectors, since J % V == 0) load the tile's first
    const T* s = nodal + b * (int64_t)N * J + j0 + (j0 + cv * V < J ? cv * V : 0);
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int n = n0 + q * (NT / CV);
      if (n < N) pre[q] = *reinterpret_cast<const VT*>(s + (int64_t)n * J);
    }
  };
  TileWalk walk(a.ntiles);
  if (walk.next >= walk.end) return;
  if (a.vec) issue(walk.next);
  for (int k = threadIdx.x; k < N; k += NT) tws[k] = cplx<T>{tw[2 * k], -tw[2 * k + 1]};
  for (int64_t tile = walk.next; tile < walk.end; tile += walk.stride) {
  const int tid = opaque_tid(), cv = tid % CV;
  const int64_t b = tile / a.tpf;
  const int j0 = (int)(tile - b * a.tpf) * C;
  if (a.vec) {
    const bool ok = j0 + cv * V < J;
    const int n0 = tid / CV;
    VT w = {};
    if (a.weighted) w = *reinterpret_cast<const VT*>(qw + (ok ? j0 + cv * V : 0));
    else w = w + (T)1;
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int n = n0 + q * (NT / CV);
      if (n < N) *reinterpret_cast<VT*>(lds + n * C + cv * V) = ok ? pre[q] * w : VT{};
    }
  } else {
    const int c = tid % C;
    const bool ok = j0 + c < J;
    const T* s = nodal + b * (int64_t)N * J + j0 + (ok ? c : 0);
    const T w = a.weighted ? qw[ok ? j0 + c : 0] : (T)1;
#pragma unroll 8
    for (int n = tid / C; n < N; n += NT / C) lds[n * C + c] = ok ? s[(int64_t)n * J] * w : (T)0;
  }
  __syncthreads();
  if (a.vec && tile + walk.stride < walk.end) issue(tile + walk.stride);
  mixed_fft<T, P, false>(buf, tws, a);
  const T inv_sqrt_2pi = (T)0.39894228040143267794;
  const T inv_sqrt_pi = (T)0.56418958354775628695;
  T* dst = fourier + b * (int64_t)a.R * J + j0;
  // entry (r, c) of the Fourier rows from the spectra of column pair c / 2
  auto entry = [&](int r, int c) -> T {
    const int m = (r + 1) / 2;
    const cplx<T> zm = buf[m * P + c / 2];
    const cplx<T> zn = buf[(m == 0 ? 0 : N - m) * P + c / 2];
    T re, im;
    if ((c & 1) == 0) {
      re = (zm.x + zn.x) * (T)0.5;
      im = (zm.y - zn.y) * (T)0.5;
    } else {
      re = (zm.y + zn.y) * (T)0.5;
      im = -(zm.x - zn.x) * (T)0.5;
    }
    return r == 0 ? re * inv_sqrt_2pi : ((r & 1) ? re * inv_sqrt_pi : -im * inv_sqrt_pi);
  };
  if (a.vec) {
    if (j0 + cv * V < J) {
      for (int r = tid / CV; r < a.R; r += NT / CV) {
        VT o;
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = entry(r, cv * V + e);
        *reinterpret_cast<VT*>(dst + (int64_t)r * J + cv * V) = o;
      }
    }
  } else {
    const int c = tid % C;
    if (j0 + c < J)
      for (int r = tid / C; r < a.R; r += NT / C) dst[(int64_t)r * J + c] = entry(r, c);
  }
  __syncthreads();  // buf is rewritten by the next tile
  }
}

template <typename T, int P>
__global__ __launch_bounds__(kThreads) void dft_inverse_mixed_kernel(
    const T* __restrict__ fourier, T* __restrict__ nodal, const T* __restrict__ tw,
    const T* __restrict__ qw, MixedArgs a) {
  using VT = typename vec16<T>::type;
  constexpr int C = 2 * P, V = 16 / sizeof(T), CV = C / V;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cplx<T>* buf = reinterpret_cast<cplx<T>*>(smem_raw);
  cplx<T>* tws = buf + a.N * P;
  T* lds = reinterpret_cast<T*>(buf);
  const int NT = blockDim.x, N = a.N, J = a.J, M = a.M;
  const T inv_sqrt_2pi = (T)0.39894228040143267794;
  const T half_inv_sqrt_pi = (T)0.28209479177387814347;
  // spectrum of a column pair from its cos and sin rows: entries m and N - m
  auto put = [&](int m, int p, T a1, T a2, T b1, T b2) {
    if (m == 0) {
      buf[p] = cplx<T>{a1 * inv_sqrt_2pi, b1 * inv_sqrt_2pi};
    } else {
      buf[m * P + p] = cplx<T>{(a1 + b2) * half_inv_sqrt_pi, (b1 - a2) * half_inv_sqrt_pi};
      buf[(N - m) * P + p] = cplx<T>{(a1 - b2) * half_inv_sqrt_pi, (a2 + b1) * half_inv_sqrt_pi};
    }
  };
  // M <= (N + 1) / 2 wavenumbers, two rows each
  constexpr int IT = kElems / V;
  VT g1[IT], g2[IT];
  auto issue = [&](int64_t t) {
    const int tid = opaque_tid(), cv = tid % CV, m0 = tid / CV;
    const int64_t b = t / a.tpf;
    const int j0 = (int)(t - b * a.tpf) * C;
    const T* s = fourier + b * (int64_t)a.R * J + j0 + (j0 + cv * V < J ? cv * V : 0);
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int m = m0 + q * (NT / CV);
      if (m < M) {
        g1[q] = *reinterpret_cast<const VT*>(s + (int64_t)(m == 0 ? 0 : 2 * m - 1) * J);
        g2[q] = *reinterpret_cast<const VT*>(s + (int64_t)(2 * m) * J);
      }
    }
  };
  TileWalk walk(a.ntiles);
  if (walk.next >= walk.end) return;
  if (a.vec) issue(walk.next);
  for (int k = threadIdx.x; k < N; k += NT) tws[k] = cplx<T>{tw[2 * k], -tw[2 * k + 1]};
  for (int64_t tile = walk.next; tile < walk.end; tile += walk.stride) {
  const int tid = opaque_tid(), cv = tid % CV;
  const int64_t b = tile / a.tpf;
  const int j0 = (int)(tile - b * a.tpf) * C;
  for (int idx = tid; idx < (N - 2 * M + 1) * P; idx += NT) buf[M * P + idx] = cplx<T>{0, 0};
  if (a.vec) {
    const bool ok = j0 + cv * V < J;
    const int m0 = tid / CV;
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int m = m0 + q * (NT / CV);
      if (m < M) {
        const VT x = ok ? g1[q] : VT{}, y = ok ? g2[q] : VT{};
#pragma unroll
        for (int e = 0; e < V; e += 2)
          put(m, (cv * V + e) / 2, x[e], y[e], x[e + 1], y[e + 1]);
      }
    }
  } else {
    const T* src = fourier + b * (int64_t)a.R * J + j0;
    const int p = tid % P;
    const bool oka = j0 + 2 * p < J, okb = j0 + 2 * p + 1 < J;
#pragma unroll 4
    for (int m = tid / P; m < M; m += NT / P) {
      const T* r1 = src + (int64_t)(m == 0 ? 0 : 2 * m - 1) * J + 2 * p;
      const T* r2 = src + (int64_t)(2 * m) * J + 2 * p;
      const T a1 = oka ? r1[0] : (T)0, a2 = oka ? r2[0] : (T)0;
      const T b1 = okb ? r1[1] : (T)0, b2 = okb ? r2[1] : (T)0;
      put(m, p, a1, a2, b1, b2);
    }
  }
  __syncthreads();
  if (a.vec && tile + walk.stride < walk.end) issue(tile + walk.stride);
  mixed_fft<T, P, true>(buf, tws, a);
  T* dst = nodal + b * (int64_t)N * J + j0;
  if (a.vec) {
    if (j0 + cv * V < J) {
      VT w = {};
      if (a.weighted) w = *reinterpret_cast<const VT*>(qw + j0 + cv * V);
      else w = w + (T)1;
      for (int n = tid / CV; n < N; n += NT / CV)
        *reinterpret_cast<VT*>(dst + (int64_t)n * J + cv * V) =
            *reinterpret_cast<const VT*>(lds + n * C + cv * V) * w;
    }
  } else {
    const int c = tid % C;
    if (j0 + c < J) {
      const T w = a.weighted ? qw[j0 + c] : (T)1;
      for (int n = tid / C; n < N; n += NT / C) dst[(int64_t)n * J + c] = lds[n * C + c] * w;
    }
  }
  __syncthreads();  // buf is rewritten by the next tile
  }
}

// Fewest radices from {2 .. 10} whose product is n (largest first among equal
// counts); 0 when n has a prime factor above 7.
int factor(int n, int* radix, int top = 10) {
  if (n == 1) return 0;
  int best = 0, cand[kMaxPasses];
  for (int r = std::min(top, n); r >= 2; --r) {
    if (n % r) continue;
    const int rest = n / r;
    const int c = rest == 1 ? 1 : factor(rest, cand, r);
    if (rest > 1) {
      if (c == 0) continue;
      if (best && c + 1 >= best) continue;
      radix[0] = r;
      std::copy(cand, cand + c, radix + 1);
      best = c + 1;
    } else {
      radix[0] = r;
      return 1;
    }
  }
  return best;
}

template <typename T, int P>
int launch(bool forward, const MixedArgs& a, const T* in, T* out, const T* tw, const T* qw,
           hipStream_t s) {
  const int threads = std::max((a.N * P + 64 * kElems - 1) / (64 * kElems) * 64, 64);
  const size_t lds = sizeof(cplx<T>) * (size_t)a.N * (P + 1);
  const void* k = forward ? (const void*)dft_forward_mixed_kernel<T, P>
                          : (const void*)dft_inverse_mixed_kernel<T, P>;
  if (lds > 65536)
    DINO_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  int per_cu = 0;
  DINO_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, threads, lds));
  const int64_t grid = std::min<int64_t>(a.ntiles, (int64_t)std::max(per_cu, 1) * device_cus());
  if (forward)
    dft_forward_mixed_kernel<T, P><<<(unsigned)grid, threads, lds, s>>>(in, out, tw, qw, a);
  else
    dft_inverse_mixed_kernel<T, P><<<(unsigned)grid, threads, lds, s>>>(in, out, tw, qw, a);
  DINO_LAUNCH_CHECK("mixed-radix dft kernel");
  return DINO_OK;
}

template <typename T, int P>
int launch_p(bool forward, MixedArgs a, int64_t B, const T* in, T* out, const T* tw, const T* qw,
             hipStream_t s) {
  constexpr int V = 16 / sizeof(T);
  a.tpf = (a.J + 2 * P - 1) / (2 * P);
  a.ntiles = B * a.tpf;
  a.vec = a.J % V == 0 && reinterpret_cast<uintptr_t>(in) % 16 == 0 &&
          reinterpret_cast<uintptr_t>(out) % 16 == 0;
  return launch<T, P>(forward, a, in, out, tw, qw, s);
}

// Column pairs per workgroup.  Several workgroups of 3 to 5 waves share a CU
// and overlap their phases best: about 2560 (FP32) or 1536 (FP64) complex
// elements each, in powers of two up to 16 pairs; but at least 4 pairs, since rows
// of 16 bytes (FP32, 2 pairs) cost more (I = 1280: 128 us against 111 forward)
// than a CU that holds one workgroup, while the tile fits kElems a thread.
// Measured at B fields, FP32 forward, pairs 16 / 8 / 4 / 2: I = 320, J = 160,
// B = 600: 65 / 61 / 69 / - us; I = 192, J = 96, B = 800: 40 / 35 / 42 / -; FP64:
// I = 320: - / 153 / 116 / -.
int pairs_for(int N, bool f64) {
  const int most = f64 ? 1536 : 2560;
  int P = 16;
  while (P > 4 && N * P > most) P /= 2;
  while (P > 2 && N * P > kThreads * kElems) P /= 2;
  return P;
}

}  // namespace

// Whether the mixed-radix kernels serve length N in this type: N factors into
// 2, 3, 5, 7 and a tile of two column pairs (24 or 48 bytes a longitude) fits
// the LDS.  In FP64 the limit is that of the direct transform (3 N doubles in
// 64 KiB), so lengths beyond it are refused as ever.
bool dft_mixed_available(int N, bool f64) {
  int radix[kMaxPasses];
  return N >= 8 && N <= (f64 ? 2730 : 4096) && factor(N, radix) > 0;
}

template <typename T>
int dft_mixed(bool forward, const dino_plan* pl, const T* in, T* out, const T* tw, const T* qw,
              int64_t B, int weighted, hipStream_t s) {
  MixedArgs a = {};
  a.N = pl->I;
  a.J = pl->J;
  a.R = pl->R;
  a.M = pl->M;
  a.weighted = weighted;
  a.npass = factor(a.N, a.radix);
  int64_t ns = 1;
  for (int i = 0; i < a.npass; ++i) {
    a.magic[i] = (unsigned)(((int64_t)1 << 32) / ns + (((int64_t)1 << 32) % ns != 0));
    ns *= a.radix[i];
  }
  switch (pairs_for(a.N, sizeof(T) == 8)) {
    case 16: return launch_p<T, 16>(forward, a, B, in, out, tw, qw, s);
    case 8: return launch_p<T, 8>(forward, a, B, in, out, tw, qw, s);
    case 4: return launch_p<T, 4>(forward, a, B, in, out, tw, qw, s);
    default: return launch_p<T, 2>(forward, a, B, in, out, tw, qw, s);
  }
}

template int dft_mixed<float>(bool, const dino_plan*, const float*, float*, const float*,
                              const float*, int64_t, int, hipStream_t);
template int dft_mixed<double>(bool, const dino_plan*, const double*, double*, const double*,
                               const double*, int64_t, int, hipStream_t);

}  // namespace dino
