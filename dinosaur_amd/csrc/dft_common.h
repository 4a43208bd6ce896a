// Complex arithmetic and small fixed-length DFTs shared by the longitude
// transform kernels (dft.hip, dft_mixed.hip).
#pragma once

#include "dino_common.h"

namespace dino {

template <typename T>
struct cplx {
  T x, y;
};

template <typename T>
__device__ __forceinline__ cplx<T> cadd(cplx<T> a, cplx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ cplx<T> csub(cplx<T> a, cplx<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T>
__device__ __forceinline__ cplx<T> cmul(cplx<T> a, cplx<T> b) {
  return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
// multiply by -i (forward) or +i (inverse)
template <typename T, bool INV>
__device__ __forceinline__ cplx<T> mul_mi(cplx<T> a) {
  return INV ? cplx<T>{-a.y, a.x} : cplx<T>{a.y, -a.x};
}

template <typename T, bool INV>
__device__ __forceinline__ void dft2(cplx<T>* v) {
  cplx<T> a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}

template <typename T, bool INV>
__device__ __forceinline__ void dft4(cplx<T>& a0, cplx<T>& a1, cplx<T>& a2, cplx<T>& a3) {
  cplx<T> s02 = cadd(a0, a2), d02 = csub(a0, a2);
  cplx<T> s13 = cadd(a1, a3), d13 = mul_mi<T, INV>(csub(a1, a3));
  a0 = cadd(s02, s13);
  a2 = csub(s02, s13);
  a1 = cadd(d02, d13);
  a3 = csub(d02, d13);
}

template <typename T, bool INV>
__device__ __forceinline__ void dft4v(cplx<T>* v) { dft4<T, INV>(v[0], v[1], v[2], v[3]); }

template <typename T, bool INV>
__device__ __forceinline__ void dft8(cplx<T>* v) {
  const T c = (T)0.70710678118654752440;
  cplx<T> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
  cplx<T> o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
  dft4<T, INV>(e0, e1, e2, e3);
  dft4<T, INV>(o0, o1, o2, o3);
  // W8^k for k = 1, 2, 3 (conjugated for the inverse)
  cplx<T> w1 = INV ? cplx<T>{c, c} : cplx<T>{c, -c};
  cplx<T> w3 = INV ? cplx<T>{-c, c} : cplx<T>{-c, -c};
  o1 = cmul(o1, w1);
  o2 = mul_mi<T, INV>(o2);
  o3 = cmul(o3, w3);
  v[0] = cadd(e0, o0);
  v[4] = csub(e0, o0);
  v[1] = cadd(e1, o1);
  v[5] = csub(e1, o1);
  v[2] = cadd(e2, o2);
  v[6] = csub(e2, o2);
  v[3] = cadd(e3, o3);
  v[7] = csub(e3, o3);
}

// e^{-2 pi i r / R} (forward) or its conjugate (inverse) for the odd radices
template <typename T, bool INV>
__device__ __forceinline__ void dft3(cplx<T>* v) {
  const T h = (T)0.86602540378443864676;  // sin(2 pi / 3)
  const cplx<T> s = cadd(v[1], v[2]);
  const cplx<T> d = mul_mi<T, INV>(csub(v[1], v[2]));
  const cplx<T> a = v[0];
  const cplx<T> m = {a.x - (T)0.5 * s.x, a.y - (T)0.5 * s.y};
  v[0] = cadd(a, s);
  v[1] = {m.x + h * d.x, m.y + h * d.y};
  v[2] = {m.x - h * d.x, m.y - h * d.y};
}

// Odd prime radix by its real symmetry: with s_q = v_q + v_{R-q} and
// d_q = v_q - v_{R-q}, output +-k is v_0 + sum_q c_qk s_q -+ i sum_q s_qk d_q.
template <typename T, int R, bool INV>
__device__ __forceinline__ void dft_odd(cplx<T>* v) {
  constexpr int H = (R - 1) / 2;
  // cos and sin of 2 pi q / R, q = 1 .. H
  constexpr double C5[] = {0.30901699437494742410, -0.80901699437494742410};
  constexpr double S5[] = {0.95105651629515357212, 0.58778525229247312917};
  constexpr double C7[] = {0.62348980185873353053, -0.22252093395631440429,
                           -0.90096886790241912624};
  constexpr double S7[] = {0.78183148246802980871, 0.97492791218182360702,
                           0.43388373911755812048};
  cplx<T> s[H], d[H];
#pragma unroll
  for (int q = 0; q < H; ++q) {
    s[q] = cadd(v[1 + q], v[R - 1 - q]);
    d[q] = mul_mi<T, INV>(csub(v[1 + q], v[R - 1 - q]));
  }
  const cplx<T> a = v[0];
  cplx<T> sum = a;
#pragma unroll
  for (int q = 0; q < H; ++q) sum = cadd(sum, s[q]);
  v[0] = sum;
#pragma unroll
  for (int k = 1; k <= H; ++k) {
    cplx<T> e = a, o = {0, 0};
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      const int i = (q * k) % R, j = i <= H ? i : R - i;  // angle index, folded
      const T c = (T)(R == 5 ? C5[j - 1] : C7[j - 1]);
      const T z = (T)(R == 5 ? S5[j - 1] : S7[j - 1]) * (i <= H ? (T)1 : (T)-1);
      e.x += c * s[q - 1].x;
      e.y += c * s[q - 1].y;
      o.x += z * d[q - 1].x;
      o.y += z * d[q - 1].y;
    }
    v[k] = cadd(e, o);
    v[R - k] = csub(e, o);
  }
}

// Composite radix R = A * B: B-point DFTs over the stride-A subsequences,
// twiddles e^{-2 pi i a b / R}, A-point DFTs; outputs in natural order.
template <typename T, int R, bool INV>
__device__ __forceinline__ void dft_r(cplx<T>* v);

template <typename T, int A, int B, bool INV>
__device__ __forceinline__ void dft_ab(cplx<T>* v, const double* wc, const double* ws) {
  constexpr int R = A * B;
  cplx<T> t[R];
#pragma unroll
  for (int a = 0; a < A; ++a) {
    cplx<T> u[B];
#pragma unroll
    for (int b = 0; b < B; ++b) u[b] = v[a + A * b];
    dft_r<T, B, INV>(u);
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int i = a * b;
      t[a * B + b] = i == 0 ? u[b]
                            : cmul(u[b], cplx<T>{(T)wc[i], INV ? (T)ws[i] : (T)-ws[i]});
    }
  }
#pragma unroll
  for (int b = 0; b < B; ++b) {
    cplx<T> u[A];
#pragma unroll
    for (int a = 0; a < A; ++a) u[a] = t[a * B + b];
    dft_r<T, A, INV>(u);
#pragma unroll
    for (int a = 0; a < A; ++a) v[b + B * a] = u[a];
  }
}

template <typename T, int R, bool INV>
__device__ __forceinline__ void dft_r(cplx<T>* v) {
  if constexpr (R == 2) {
    dft2<T, INV>(v);
  } else if constexpr (R == 3) {
    dft3<T, INV>(v);
  } else if constexpr (R == 4) {
    dft4v<T, INV>(v);
  } else if constexpr (R == 5 || R == 7) {
    dft_odd<T, R, INV>(v);
  } else if constexpr (R == 6) {
    constexpr double wc[] = {1.0, 0.5, -0.5};
    constexpr double ws[] = {0.0, 0.86602540378443864676, 0.86602540378443864676};
    dft_ab<T, 2, 3, INV>(v, wc, ws);
  } else if constexpr (R == 8) {
    dft8<T, INV>(v);
  } else if constexpr (R == 9) {
    constexpr double wc[] = {1.0, 0.76604444311897803520, 0.17364817766693034885, 0.0,
                             -0.93969262078590838405};
    constexpr double ws[] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.0,
                             0.34202014332566873304};
    dft_ab<T, 3, 3, INV>(v, wc, ws);
  } else {
    static_assert(R == 10, "unsupported radix");
    constexpr double wc[] = {1.0, 0.80901699437494742410, 0.30901699437494742410,
                             -0.30901699437494742410, -0.80901699437494742410};
    constexpr double ws[] = {0.0, 0.58778525229247312917, 0.95105651629515357212,
                             0.95105651629515357212, 0.58778525229247312917};
    dft_ab<T, 2, 5, INV>(v, wc, ws);
  }
}

}  // namespace dino
