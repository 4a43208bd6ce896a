// Legendre contractions of FP64 data on the FP64 matrix cores
// (v_mfma_f64_16x16x4f64); same sums as legendre.hip.
//
// The FP64 runs are parity and reference runs: modest batches of small and
// middle grids, where the tiled FMA kernels spend their time waiting (258
// workgroups and a barrier pair per 16 degrees at T85, 96 fields, for 23 MB and
// 0.09 GFLOP).  Here every wave works alone, with no LDS and no barriers: it
// owns 16 rows (field, cos / sin) of one zonal wavenumber and reads the table
// p64 (degree-major, 128-byte runs of 16 nodes) through the L1, which the
// waves of a block share.  The launch splits degrees (forward) or nodes
// (inverse) until the chip is full.  Forward / inverse, FMA tiles -> here:
// T85, 96 fields 34 / 25 -> 21 / 16 us; T106, 111 fields 56 / 42 -> 31 / 28; TL255,
// 10 fields 79 / 55 -> 43 / 32; TL255, 222 fields 413 -> 283 forward.  The bound on
// large batches is the L2: waves of a block drift apart and read the table
// again, so the inverse keeps the FMA tiles there (legendre_f64_inverse_pays).
#include <algorithm>

#include "dino_common.h"

namespace dino {

int device_cus();  // dft.hip

namespace {

typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 32;  // degrees per tile, from l = m: class q holds l - m = 2 i + q

__device__ __forceinline__ d4 mma64(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void row_field(int m, int q, int* b, int* r) {
  *b = m == 0 ? q : q >> 1;
  *r = m == 0 ? 0 : 2 * m - 1 + (q & 1);
}

// Forward: 4 waves = 2 strips of 16 rows x 2 fold parities.  A wave keeps its
// rows, folded for its parity (sum or difference of the hemispheres), as A operands and forms the degrees of its parity tile by tile;
// block z takes tiles z, z + gridDim.z, ....  kt node groups of KT are in use.
// Operand u = 2 h + i of group t is node 16 t + 8 h + 2 g + i in lane group g,
// so a table load covers 64 contiguous bytes of each of 16 degrees.
template <int KT>
__global__ __launch_bounds__(256) void leg_fwd_f64_kernel(
    const double* __restrict__ fourier, double* __restrict__ modal, const double* __restrict__ p64,
    const int64_t* __restrict__ m_off, int B, int L, int J, int Jh, int Jhp, int Rrows,
    int skip_zero) {
  const int m = blockIdx.y;
  const int nrows = (m == 0) ? B : 2 * B;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int par = wave & 1, g = lane >> 4, c16 = lane & 15;
  const int row0 = (blockIdx.x * 2 + (wave >> 1)) * 16;
  if (row0 >= nrows) return;  // no barriers below
  const int kt = (Jh + 15) / 16;
  const double sgn = par ? -1.0 : 1.0;
  double x[KT][4];
  {
    const int row = row0 + c16;
    const bool rok = row < nrows;
    int b, r;
    row_field(m, rok ? row : row0, &b, &r);
    const double* const f = fourier + ((int64_t)b * Rrows + r) * J;
#pragma unroll
    for (int t = 0; t < KT; ++t) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x[t][u] = 0;
        if (t >= kt) continue;
        const int jj = 16 * t + 8 * (u >> 1) + 2 * g + (u & 1);
        const bool ok = rok && jj < Jh;
        // odd J: node 0 is the equator, counted once
        const bool okd = ok && !((J & 1) && jj == 0);
        const double up = f[ok ? J - Jh + jj : 0];
        const double dn = f[okd ? Jh - 1 - jj : 0];
        x[t][u] = (ok ? up : 0.0) + sgn * (okd ? dn : 0.0);
      }
    }
  }
  // output rows 4 i + g of this lane
  auto out_row = [&](int i) -> double* {
    const int row = row0 + 4 * i + g;
    if (row >= nrows) return nullptr;
    int b, r;
    row_field(m, row, &b, &r);
    return modal + ((int64_t)b * Rrows + r) * L;
  };
  // zeros below the triangle; with skip_zero only from the first tile's degree on
  if (blockIdx.z == 0) {
    const int l0 = skip_zero ? leg_tile_start(m, L) : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      double* const o = out_row(i);
      if (o)
        for (int l = l0 + 2 * c16 + par; l < m; l += 32) o[l] = 0.0;
    }
  }
  const double* const pm = p64 + m_off[m];
  const int ntile = (L - m + kTile - 1) / kTile;
  for (int tt = blockIdx.z; tt < ntile; tt += gridDim.z) {
    const int d = kTile * tt + 2 * c16 + par;  // this lane's column: degree m + d
    const double* const pr = pm + (int64_t)(m + d < L ? d : L - 1 - m) * Jhp + 2 * g;
    d4 a0 = {0, 0, 0, 0}, a1 = a0;
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      if (t >= kt) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // Jhp is a multiple of 8; the half group past the padded row (x = 0
        // there) reads the row's first nodes
        const int j = 16 * t + 8 * h;
        const d2 p = *reinterpret_cast<const d2*>(pr + (j < Jhp ? j : 0));
        a0 = mma64(x[t][2 * h], p[0], a0);
        a1 = mma64(x[t][2 * h + 1], p[1], a1);
      }
    }
    if (m + d < L) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        double* const o = out_row(i);
        if (o) o[m + d] = a0[i] + a1[i];
      }
    }
  }
}

// Inverse: 4 waves = 4 strips of 16 rows; block z owns 16 NT
// nodes, whose two class sums a wave accumulates over all degrees.  Operand
// (s, q) is degree l0 + 8 s + 2 g + q in lane group g: a row load covers 64
// bytes of each of 16 rows.
template <int NT>
__global__ __launch_bounds__(256) void leg_inv_f64_kernel(
    const double* __restrict__ modal, double* __restrict__ fourier, const double* __restrict__ p64,
    const int64_t* __restrict__ m_off, int B, int L, int J, int Jh, int Jhp, int Rrows) {
  const int m = blockIdx.y;
  const int nrows = (m == 0) ? B : 2 * B;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c16 = lane & 15;
  const int row0 = blockIdx.x * 64 + wave * 16;
  if (row0 >= nrows) return;  // no barriers below
  const int jb = blockIdx.z * 16 * NT;
  d4 acc[NT][2];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n][0] = acc[n][1] = d4{0, 0, 0, 0};
  const bool rok = row0 + c16 < nrows;
  int b, r;
  row_field(m, rok ? row0 + c16 : row0, &b, &r);
  const double* const f = modal + ((int64_t)b * Rrows + r) * L;
  // node columns of this lane; those past the padded row read a valid one and are not stored
  const double* const pm = p64 + m_off[m];
  int jc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) jc[n] = jb + 16 * n + c16 < Jhp ? jb + 16 * n + c16 : 0;
  for (int l0 = m; l0 < L; l0 += kTile) {
    double a[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int l = l0 + 8 * (e >> 1) + 2 * g + (e & 1);
      const double v = f[l < L ? l : L - 1];
      a[e] = rok && l < L ? v : 0.0;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int l = l0 + 8 * (e >> 1) + 2 * g + (e & 1);
      const double* const pr = pm + (int64_t)((l < L ? l : L - 1) - m) * Jhp;
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[n][e & 1] = mma64(a[e], pr[jc[n]], acc[n][e & 1]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = row0 + 4 * i + g;
    if (row >= nrows) continue;
    row_field(m, row, &b, &r);
    double* const o = fourier + ((int64_t)b * Rrows + r) * J;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int jj = jb + 16 * n + c16;
      if (jj >= Jh) continue;
      const int jup = J - Jh + jj, jdn = Jh - 1 - jj;
      o[jup] = acc[n][0][i] + acc[n][1][i];
      if (jdn != jup) o[jdn] = acc[n][0][i] - acc[n][1][i];
    }
  }
}

template <int KT>
int launch_fwd(const dino_plan* pl, const double* in, double* out, int64_t B, int skip,
               hipStream_t s) {
  // up to four blocks a CU by splitting the degree tiles of a row block; its rows are
  // then read once per part, so no more (T85, 96 fields: 21.1 us in one part, 26.7 in two,
  // which would be 4.03 blocks a CU)
  const int64_t gx = (2 * B + 31) / 32, want = 4 * (int64_t)device_cus();
  const int tiles = (pl->L + kTile - 1) / kTile;
  const int z = (int)std::min<int64_t>(tiles, std::max<int64_t>(1, want / (gx * pl->M)));
  const dim3 grid((unsigned)gx, (unsigned)pl->M, (unsigned)z);
  leg_fwd_f64_kernel<KT><<<grid, 256, 0, s>>>(in, out, pl->p64, pl->m_offset, (int)B, pl->L,
                                              pl->J, pl->Jh, pl->Jhp, pl->R, skip);
  DINO_LAUNCH_CHECK("legendre forward f64 kernel");
  return DINO_OK;
}

template <int NT>
int launch_inv(const dino_plan* pl, const double* in, double* out, int64_t B, hipStream_t s) {
  const dim3 grid((unsigned)((2 * B + 63) / 64), (unsigned)pl->M,
                  (unsigned)((pl->Jh + 16 * NT - 1) / (16 * NT)));
  leg_inv_f64_kernel<NT><<<grid, 256, 0, s>>>(in, out, pl->p64, pl->m_offset, (int)B, pl->L,
                                              pl->J, pl->Jh, pl->Jhp, pl->R);
  DINO_LAUNCH_CHECK("legendre inverse f64 kernel");
  return DINO_OK;
}

}  // namespace

// By the grid alone: the two kernels add in another order, and a field's result does not
// depend on the batch.  FMA tiles / here, us: TL255, 222 fields 413 / 283; T213 (160
// nodes), 37 fields 143 / 66; small grids with many fields are even, T31 (24 nodes), 1000
// fields 23.6 / 24.5, T42 35 / 33, 80 longitudes x 40 nodes 54 / 56 (500 fields 35 / 38); TL639, 37
// fields, 1120 / 1200 (operands of 320 nodes leave one wave per SIMD).
bool legendre_f64_forward_pays(const dino_plan* pl, int64_t B) {
  return pl->Jh <= 256 && B < (int64_t)1 << 30;
}

// By the batch as well: both kernels add a class's products in the order of the degrees,
// so their results are bitwise the same.  FMA tiles / here, us: T85 (64 nodes), 1000
// fields, 2752 row blocks 98 / 87; TL255 (128 nodes), 8 fields, 256 row blocks 53 / 28, 64
// fields, 512, 78 / 59, 300 fields, 2560, 329 / 340.  Above 128 nodes the waves of a block
// re-read a table that the L2s do not hold (T213 29 MB, T340 119 MB), so only where a block
// has one wave with rows (8 fields) or the row blocks are few: T213 (160 nodes), 32
// fields, 214 row blocks 63 / 38, 37 fields, 428, 65 / 70; T340, 8 fields 79 / 59, 12 fields,
// 341, 84 / 89; TL639, 8 fields 310 / 228, 37 fields 674 / 874.
bool legendre_f64_inverse_pays(const dino_plan* pl, int64_t B) {
  const int64_t blocks = (2 * B + 63) / 64 * pl->M;
  if (B >= (int64_t)1 << 30) return false;
  return pl->Jh <= 96 || (pl->Jh <= 128 ? blocks <= 512 : B <= 8 || blocks <= 256);
}

int legendre_forward_f64(const dino_plan* pl, const double* in, double* out, int64_t B,
                         bool triangle_only, hipStream_t s) {
  if (B == 0) return DINO_OK;
  const int skip = triangle_only ? 1 : 0;
  if (pl->Jh <= 32) return launch_fwd<2>(pl, in, out, B, skip, s);
  if (pl->Jh <= 64) return launch_fwd<4>(pl, in, out, B, skip, s);
  if (pl->Jh <= 128) return launch_fwd<8>(pl, in, out, B, skip, s);
  return launch_fwd<16>(pl, in, out, B, skip, s);
}

int legendre_inverse_f64(const dino_plan* pl, const double* in, double* out, int64_t B,
                         hipStream_t s) {
  if (B == 0) return DINO_OK;
  // narrower node blocks re-read the modal rows but make more waves: T85, 96
  // fields (258 blocks of 64 nodes) 16.0 us with 32 nodes, 17.3 with 64; 1000
  // fields 108 and 99.  A grid of up to 32 nodes has no use for 64: T31, 1000 fields 13.3
  // and 19.7, T42 19.9 and 27.5
  const int64_t blocks = (2 * B + 63) / 64 * pl->M * ((pl->Jh + 63) / 64);
  if (pl->Jh <= 16) return launch_inv<1>(pl, in, out, B, s);
  if (pl->Jh <= 32 || blocks < 4 * (int64_t)device_cus()) return launch_inv<2>(pl, in, out, B, s);
  return launch_inv<4>(pl, in, out, B, s);
}

}  // namespace dino
