// Held-Suarez drag and relaxation (held_suarez.py:99-167) on the nodal buffers
// of the primitive equations' explicit terms, and their adjoint.
//
// The primitive equations already carry the nodal winds and temperature
// between their two transforms, so the forcing needs no transforms of its own
// but one field, ln ps, on the way in and the temperature tendency on the way
// out:
//   CU += kv / cos^2(lat) u,  CV += kv / cos^2(lat) v
//     (the combined flux enters the tendencies as -curl and -div, the drag
//     -kv u as curl and div),
//   HT = -kt (T_ref + T - T_eq),  T_eq = max(minT, p^kappa (maxT - dTy sin^2(lat)
//     - dThz ln(p) cos^2(lat))),  p = sigma exp(ln ps) / p0
//     (a group of its own: unlike TEMP it is not clipped at the top degree).
//
// Bound by HBM: 8 field passes of K levels forward (U, V, T read, CU, CV
// read and written, HT written).  A block owns 64 columns, its 4 waves a
// quarter of the levels each: the adjoint's sum over the levels (ln ps) is
// formed per wave and added through LDS in a fixed order.  Two forward and
// adjoint steps of TL127 L32, one member, composed with this forcing: 23.1 ms
// as separate tensor operations and transforms (2600 launches, host bound),
// 5.1 ms fused.
#include <vector>

#include "dino_common.h"

struct dino_held_suarez {
  int K, I, J;
  double min_t, max_t, dty, dthz, kappa, p0;
  // kv_cos2 (K, J), kt (K, J), sigma (K), tref (K), sin2 (J), cos2 (J)
  double* c64;
  float* c32;
};

namespace dino {
namespace {

struct HsArgs {
  int K, J;
  int64_t IJ;
  int64_t t, u, v, ln;  // nodal input groups (fields)
  int64_t cu, cv, ht;   // nodal output groups
  double min_t, max_t, dty, dthz, kappa, p0;
};

// Equilibrium temperature at ln ps and its derivative with respect to ln ps.
template <typename T>
__device__ __forceinline__ T equilibrium(const HsArgs& a, T sigma, T surface, T s2, T c2, T* dq) {
  const T p = sigma * surface;
  const T pk = pow(p, (T)a.kappa);
  const T q = pk * ((T)a.max_t - (T)a.dty * s2 - (T)a.dthz * log(p) * c2);
  const bool warm = !(q < (T)a.min_t);  // NaN passes through
  *dq = warm ? (T)a.kappa * q - pk * (T)a.dthz * c2 : (T)0;
  return warm ? q : (T)a.min_t;
}

constexpr int kWaves = 4;

template <typename T, bool ADJ>
__global__ __launch_bounds__(64 * kWaves) void held_suarez_kernel(
    const T* __restrict__ in, const T* __restrict__ gout, T* __restrict__ out,
    const T* __restrict__ cst, HsArgs a) {
  const int lane = threadIdx.x, wave = threadIdx.y;
  const int64_t col = (int64_t)blockIdx.x * 64 + lane;
  const int64_t e = blockIdx.y;
  const bool ok = col < a.IJ;
  const int64_t c = ok ? col : a.IJ - 1;
  const int K = a.K, J = a.J, j = (int)(c % J);
  const T* const kvc = cst + j;
  const T* const kt = cst + (int64_t)K * J + j;
  const T* const sigma = cst + (int64_t)2 * K * J;
  const T* const tref = sigma + K;
  const T s2 = tref[K + j], c2 = tref[K + J + j];
  auto field = [&](int64_t group, int lev, int k) { return (group + e * lev + k) * a.IJ + c; };
  // ln ps is about 45 in nondimensional units, so its exponential and the sum
  // of the adjoint are formed in FP64 (one of each per thread)
  const T surface = (T)(exp((double)in[field(a.ln, 1, 0)]) / a.p0);
  double sum = 0;
  const int k0 = K * wave / kWaves, k1 = K * (wave + 1) / kWaves;
  for (int k = k0; k < k1; ++k) {
    T dq;
    const T q = equilibrium(a, sigma[k], surface, s2, c2, &dq);
    const T drag = kvc[(int64_t)k * J], rate = kt[(int64_t)k * J];
    if (!ADJ) {
      const T u = in[field(a.u, K, k)], v = in[field(a.v, K, k)], t = in[field(a.t, K, k)];
      if (ok) {
        out[field(a.cu, K, k)] += drag * u;
        out[field(a.cv, K, k)] += drag * v;
        out[field(a.ht, K, k)] = -rate * (tref[k] + t - q);
      }
    } else {
      const T gt = gout[field(a.ht, K, k)];
      const T gu = gout[field(a.cu, K, k)], gv = gout[field(a.cv, K, k)];
      sum += (double)(rate * gt * dq);
      if (ok) {
        out[field(a.u, K, k)] += drag * gu;
        out[field(a.v, K, k)] += drag * gv;
        out[field(a.t, K, k)] -= rate * gt;
      }
    }
  }
  if (ADJ) {
    __shared__ double part[kWaves][64];
    part[wave][lane] = sum;
    __syncthreads();
    if (wave == 0 && ok)
      out[field(a.ln, 1, 0)] =
          (T)((part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]));
  }
}

template <typename T>
int run_held_suarez(const dino_held_suarez* h, const void* in, const void* gout, void* out,
                    const HsArgs& a, int64_t members, hipStream_t s) {
  const T* cst;
  if constexpr (sizeof(T) == 8) cst = h->c64;
  else cst = h->c32;
  const dim3 grid((unsigned)((a.IJ + 63) / 64), (unsigned)members), block(64, kWaves);
  if (gout)
    held_suarez_kernel<T, true><<<grid, block, 0, s>>>((const T*)in, (const T*)gout, (T*)out, cst, a);
  else
    held_suarez_kernel<T, false><<<grid, block, 0, s>>>((const T*)in, nullptr, (T*)out, cst, a);
  DINO_LAUNCH_CHECK("held-suarez kernel");
  return DINO_OK;
}

int held_suarez_entry(const dino_held_suarez* h, const void* in, const void* gout, void* out,
                      const int64_t* in_groups, const int64_t* out_groups, int64_t members,
                      int dtype, void* stream) {
  DINO_REQUIRE(members >= 1 && members <= 65535, DINO_EINVAL, "members must be in [1, 65535]");
  DINO_REQUIRE(dtype == DINO_F32 || dtype == DINO_F64, DINO_EINVAL, "unknown dtype %d", dtype);
  HsArgs a;
  a.K = h->K;
  a.J = h->J;
  a.IJ = (int64_t)h->I * h->J;
  a.t = in_groups[0];
  a.u = in_groups[1];
  a.v = in_groups[2];
  a.ln = in_groups[3];
  a.cu = out_groups[0];
  a.cv = out_groups[1];
  a.ht = out_groups[2];
  a.min_t = h->min_t;
  a.max_t = h->max_t;
  a.dty = h->dty;
  a.dthz = h->dthz;
  a.kappa = h->kappa;
  a.p0 = h->p0;
  if (dtype == DINO_F64)
    return run_held_suarez<double>(h, in, gout, out, a, members, as_stream(stream));
  return run_held_suarez<float>(h, in, gout, out, a, members, as_stream(stream));
}

}  // namespace
}  // namespace dino

using namespace dino;

extern "C" int dino_held_suarez_create(int K, int I, int J, const double* kv_cos2,
                                       const double* kt, const double* sigma, const double* tref,
                                       const double* sin2, const double* cos2, double min_t,
                                       double max_t, double dty, double dthz, double kappa,
                                       double p0, dino_held_suarez** out) {
  DINO_REQUIRE(out, DINO_EINVAL, "dino_held_suarez_create: out is NULL");
  *out = nullptr;
  DINO_REQUIRE(K >= 1 && I >= 1 && J >= 1, DINO_EINVAL, "invalid nodal shape");
  DINO_REQUIRE(kv_cos2 && kt && sigma && tref && sin2 && cos2, DINO_EINVAL, "NULL coefficient array");
  std::vector<double> h;
  h.insert(h.end(), kv_cos2, kv_cos2 + (size_t)K * J);
  h.insert(h.end(), kt, kt + (size_t)K * J);
  h.insert(h.end(), sigma, sigma + K);
  h.insert(h.end(), tref, tref + K);
  h.insert(h.end(), sin2, sin2 + J);
  h.insert(h.end(), cos2, cos2 + J);
  const std::vector<float> hf(h.begin(), h.end());
  dino_held_suarez* p = new dino_held_suarez{K, I, J, min_t, max_t, dty, dthz, kappa, p0, nullptr,
                                             nullptr};
  hipError_t e = hipMalloc(&p->c64, sizeof(double) * h.size());
  if (e == hipSuccess) e = hipMalloc(&p->c32, sizeof(float) * h.size());
  if (e == hipSuccess)
    e = hipMemcpy(p->c64, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(p->c32, hf.data(), sizeof(float) * h.size(), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)dino_held_suarez_destroy(p);
    return hip_fail(e, "dino_held_suarez_create");
  }
  *out = p;
  return DINO_OK;
}

extern "C" int dino_held_suarez_destroy(dino_held_suarez* p) {
  if (p) {
    if (p->c64) (void)hipFree(p->c64);
    if (p->c32) (void)hipFree(p->c32);
    delete p;
  }
  return DINO_OK;
}

extern "C" int dino_held_suarez_nodal(const dino_held_suarez* h, const void* nodal_in,
                                      void* nodal_out, const int64_t* in_groups,
                                      const int64_t* out_groups, int64_t members, int dtype,
                                      void* stream) {
  DINO_REQUIRE(h && nodal_in && nodal_out && in_groups && out_groups, DINO_EINVAL,
               "dino_held_suarez_nodal: NULL argument");
  return held_suarez_entry(h, nodal_in, nullptr, nodal_out, in_groups, out_groups, members, dtype,
                           stream);
}

extern "C" int dino_held_suarez_nodal_adjoint(const dino_held_suarez* h, const void* nodal_in,
                                              const void* out_cot, void* in_cot,
                                              const int64_t* in_groups, const int64_t* out_groups,
                                              int64_t members, int dtype, void* stream) {
  DINO_REQUIRE(h && nodal_in && out_cot && in_cot && in_groups && out_groups, DINO_EINVAL,
               "dino_held_suarez_nodal_adjoint: NULL argument");
  return held_suarez_entry(h, nodal_in, out_cot, in_cot, in_groups, out_groups, members, dtype,
                           stream);
}
