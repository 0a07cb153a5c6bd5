// In-register DFTs and the stage sequence of the Stockham passes, shared by
// the transform kernels (pw_fft.hip, pw_pencil.hip).
#pragma once
#include "pw_common.h"

namespace {

template <typename T2> struct Prec;
template <> struct Prec<double2> {
  typedef double T;
  static __device__ inline double2 from(double2 v) { return v; }
};
template <> struct Prec<float2> {
  typedef float T;
  static __device__ inline float2 from(double2 v) { return make_float2((float)v.x, (float)v.y); }
};

template <typename T2>
__device__ inline T2 czero() { T2 r; r.x = 0; r.y = 0; return r; }

// a * (sign * i)
template <typename T2>
__device__ inline T2 mul_si(T2 a, int sign) {
  T2 r;
  r.x = sign > 0 ? -a.y : a.y;
  r.y = sign > 0 ? a.x : -a.x;
  return r;
}

// cos/sin(2 pi m / R)
template <int R> struct Roots;
template <> struct Roots<3> {
  static constexpr double c[3] = {1.0, -0.5, -0.5};
  static constexpr double s[3] = {0.0, 0.86602540378443864676, -0.86602540378443864676};
};
template <> struct Roots<5> {
  static constexpr double c[5] = {1.0, 0.30901699437494742410, -0.80901699437494742410,
                                  -0.80901699437494742410, 0.30901699437494742410};
  static constexpr double s[5] = {0.0, 0.95105651629515357212, 0.58778525229247312917,
                                  -0.58778525229247312917, -0.95105651629515357212};
};
template <> struct Roots<7> {
  static constexpr double c[7] = {1.0, 0.62348980185873353053, -0.22252093395631440429,
                                  -0.90096886790241912624, -0.90096886790241912624,
                                  -0.22252093395631440429, 0.62348980185873353053};
  static constexpr double s[7] = {0.0, 0.78183148246802980871, 0.97492791218182360702,
                                  0.43388373911755812048, -0.43388373911755812048,
                                  -0.97492791218182360702, -0.78183148246802980871};
};
template <> struct Roots<11> {
  static constexpr double c[11] = {1.0, 0.84125353283118116886, 0.41541501300188642553,
                                   -0.14231483827328514044, -0.65486073394528506406,
                                   -0.95949297361449738989, -0.95949297361449738989,
                                   -0.65486073394528506406, -0.14231483827328514044,
                                   0.41541501300188642553, 0.84125353283118116886};
  static constexpr double s[11] = {0.0, 0.54064081745559758211, 0.90963199535451837141,
                                   0.98982144188093273238, 0.75574957435425828377,
                                   0.28173255684142969771, -0.28173255684142969771,
                                   -0.75574957435425828377, -0.98982144188093273238,
                                   -0.90963199535451837141, -0.54064081745559758211};
};

template <> struct Roots<9> {
  static constexpr double c[9] = {1.0, 0.766044443118978035202, 0.173648177666930348852, -0.5,
                                  -0.939692620785908384054, -0.939692620785908384054, -0.5,
                                  0.173648177666930348852, 0.766044443118978035202};
  static constexpr double s[9] = {0.0, 0.642787609686539326323, 0.984807753012208059367,
                                  0.866025403784438646764, 0.342020143325668733044,
                                  -0.342020143325668733044, -0.866025403784438646764,
                                  -0.984807753012208059367, -0.642787609686539326323};
};
template <> struct Roots<16> {
  static constexpr double c[16] = {1.0, 0.923879532511286756128, 0.707106781186547524401,
                                   0.382683432365089771728, 0.0, -0.382683432365089771728,
                                   -0.707106781186547524401, -0.923879532511286756128, -1.0,
                                   -0.923879532511286756128, -0.707106781186547524401,
                                   -0.382683432365089771728, 0.0, 0.382683432365089771728,
                                   0.707106781186547524401, 0.923879532511286756128};
  static constexpr double s[16] = {0.0, 0.382683432365089771728, 0.707106781186547524401,
                                   0.923879532511286756128, 1.0, 0.923879532511286756128,
                                   0.707106781186547524401, 0.382683432365089771728, 0.0,
                                   -0.382683432365089771728, -0.707106781186547524401,
                                   -0.923879532511286756128, -1.0, -0.923879532511286756128,
                                   -0.707106781186547524401, -0.382683432365089771728};
};

template <typename T2, int R>
__device__ inline void dft(T2 *v, int sign);

// DFT of size R = P Q from P-point and Q-point DFTs: input r = Q a + b,
// output q = q1 + P q2; Y_b = DFT_P over a, times exp(sign 2 pi i b q1 / R),
// then DFT_Q over b.
template <typename T2, int P, int Q>
__device__ inline void dft_pq(T2 *v, int sign) {
  typedef typename Prec<T2>::T T;
  constexpr int R = P * Q;
  T2 y[Q][P];
#pragma unroll
  for (int b = 0; b < Q; ++b) {
    T2 t[P];
#pragma unroll
    for (int a = 0; a < P; ++a) t[a] = v[Q * a + b];
    dft<T2, P>(t, sign);
#pragma unroll
    for (int q1 = 0; q1 < P; ++q1) y[b][q1] = t[q1];
  }
#pragma unroll
  for (int b = 1; b < Q; ++b)
#pragma unroll
    for (int q1 = 1; q1 < P; ++q1) {
      const int m = (b * q1) % R;
      T2 w;
      w.x = (T)Roots<R>::c[m];
      w.y = sign > 0 ? (T)Roots<R>::s[m] : -(T)Roots<R>::s[m];
      y[b][q1] = cmul(y[b][q1], w);
    }
#pragma unroll
  for (int q1 = 0; q1 < P; ++q1) {
    T2 t[Q];
#pragma unroll
    for (int b = 0; b < Q; ++b) t[b] = y[b][q1];
    dft<T2, Q>(t, sign);
#pragma unroll
    for (int q2 = 0; q2 < Q; ++q2) v[q1 + P * q2] = t[q2];
  }
}

// in-register DFT of size R: v[q] <- sum_r v[r] exp(sign 2 pi i r q / R)
template <typename T2, int R>
__device__ inline void dft(T2 *v, int sign) {
  typedef typename Prec<T2>::T T;
  if constexpr (R == 2) {
    T2 a = v[0], b = v[1];
    v[0] = cadd(a, b); v[1] = csub(a, b);
  } else if constexpr (R == 3) {
    // m = v0 - t/2, out(1,2) = m +- sign sin(2 pi/3) i d: 12 operations
    const T c = (T)-0.5, s = (T)0.86602540378443864676;
    const T2 t = cadd(v[1], v[2]), d = csub(v[1], v[2]);
    T2 m;
    m.x = v[0].x + c * t.x;
    m.y = v[0].y + c * t.y;
    v[0] = cadd(v[0], t);
    const T sx = sign > 0 ? s : -s;
    T2 o1, o2;
    o1.x = m.x - sx * d.y;
    o1.y = m.y + sx * d.x;
    o2.x = m.x + sx * d.y;
    o2.y = m.y - sx * d.x;
    v[1] = o1;
    v[2] = o2;
  } else if constexpr (R == 4) {
    T2 t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
    T2 t2 = cadd(v[1], v[3]), t3 = mul_si(csub(v[1], v[3]), sign);
    v[0] = cadd(t0, t2); v[2] = csub(t0, t2);
    v[1] = cadd(t1, t3); v[3] = csub(t1, t3);
  } else if constexpr (R == 9) {
    dft_pq<T2, 3, 3>(v, sign);
  } else if constexpr (R == 16) {
    dft_pq<T2, 4, 4>(v, sign);
  } else if constexpr (R == 8) {
    T2 e[4] = {v[0], v[2], v[4], v[6]};
    T2 o[4] = {v[1], v[3], v[5], v[7]};
    dft<T2, 4>(e, sign);
    dft<T2, 4>(o, sign);
    const T r2 = (T)0.70710678118654752440;
    // w^q, w = exp(sign 2 pi i/8)
    T2 w1; w1.x = r2; w1.y = sign > 0 ? r2 : -r2;
    T2 w3; w3.x = -r2; w3.y = sign > 0 ? r2 : -r2;
    T2 o1 = cmul(o[1], w1), o2 = mul_si(o[2], sign), o3 = cmul(o[3], w3);
    v[0] = cadd(e[0], o[0]); v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], o1);   v[5] = csub(e[1], o1);
    v[2] = cadd(e[2], o2);   v[6] = csub(e[2], o2);
    v[3] = cadd(e[3], o3);   v[7] = csub(e[3], o3);
  } else {
    constexpr int H = (R - 1) / 2;
    T2 sp[H], sm[H];
#pragma unroll
    for (int r = 1; r <= H; ++r) {
      sp[r - 1] = cadd(v[r], v[R - r]);
      sm[r - 1] = mul_si(csub(v[r], v[R - r]), sign);
    }
    // out[q], out[R-q] = a_q +- b_q with a_q = v0 + sum_r cos(2 pi r q/R) sp_r
    // and b_q = sum_r sin(2 pi r q/R) sm_r (cos even, sin odd in q)
    T2 out[R];
    out[0] = v[0];
#pragma unroll
    for (int r = 0; r < H; ++r) out[0] = cadd(out[0], sp[r]);
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      T2 a = v[0], b;
#pragma unroll
      for (int r = 1; r <= H; ++r) {
        const int m = (r * q) % R;
        const T c = (T)Roots<R>::c[m];
        a.x += sp[r - 1].x * c;
        a.y += sp[r - 1].y * c;
      }
      b.x = sm[0].x * (T)Roots<R>::s[q % R];
      b.y = sm[0].y * (T)Roots<R>::s[q % R];
#pragma unroll
      for (int r = 2; r <= H; ++r) {
        const T s = (T)Roots<R>::s[(r * q) % R];
        b.x += sm[r - 1].x * s;
        b.y += sm[r - 1].y * s;
      }
      out[q] = cadd(a, b);
      out[R - q] = csub(a, b);
    }
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = out[q];
  }
}

// stages of a Stockham transform of length n (fft_factor's rule for these
// passes): odd radices, then 16, 8, 4, 2
__host__ __device__ constexpr Fft1D fft_stockham_ct(int n) {
  Fft1D f{};
  f.n = n;
  int m = n;
  const int order[9] = {9, 3, 5, 7, 11, 16, 8, 4, 2};
  for (int io = 0; io < 9; ++io)
    while (m % order[io] == 0 && f.nstage < 12) {
      f.radix[f.nstage++] = order[io];
      m /= order[io];
    }
  return f;
}

}  // namespace
