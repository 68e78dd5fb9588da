// Direct M2L, M2M and L2L of the packed real basis (conventions of
// device_math.hpp), without rotations: every output coefficient is a sum over
// the input coefficients times solid harmonics of the separation, taken degree
// by degree so that only three degrees of harmonics are alive at a time.
//
// With R_n^m the regular harmonics, S_n^m = (n-m)! P_n^m(cos t) e^{i m phi} / r^{n+1}
// the irregular ones and R_n^{-m} = (-1)^m conj(R_n^m) (S likewise):
//   M2M  M'_n^m = sum_{k,l} M_k^l R_{n-k}^{m-l}(d)            (addition theorem)
//   L2L  the transpose of M2M at the same d
//   M2L  F_n^m = 2 Re L, F_n^{-m} = -2 Im L (F_n^0 = Re L),
//        L_n^m = sum_{k <= P-n, l} M_k^l conj(S_{n+k}^{m+l}(d))
// The terms of orders l and -l (l > 0) join in real sums and differences of two
// harmonics, which depend on (n -/+ k, m, l) only: they are formed once and then
// cost one multiply-add for every pair of a kept output and an input coefficient.
// Multiply-adds per translation: sum_{n+k<=P} (2n+1)(2k+1) = 155 / 532 / 1365 at
// order 4 / 6 / 8, for all three.  The rotation cascade (two Dz and two B_U
// applications each way) needs 475 / 1100 / 2110 instructions with its scalings.
#pragma once

#include "device_math.hpp"

namespace jfm {

// One degree of harmonics from the two before it; c/s: real and imaginary parts
// of orders 0..N (c[0..N], s[0] = 0).  c1/s1: degree N - 1, c2: degree N - 2.
template <typename T, int N>
__host__ __device__ __forceinline__ void regular_degree(T x, T y, T z, T r2, const T* c1, const T* s1, const T* c2,
                                                        const T* s2, T* c, T* s) {
  if constexpr (N == 0) {
    c[0] = T(1);
    s[0] = T(0);
  } else {
    constexpr T f = static_cast<T>(0.5 / N);
    c[N] = f * (x * c1[N - 1] - y * s1[N - 1]);
    s[N] = f * (x * s1[N - 1] + y * c1[N - 1]);
    c[N - 1] = z * c1[N - 1];
    s[N - 1] = z * s1[N - 1];
#pragma unroll
    for (int m = 0; m <= N - 2; ++m) {
      const T inv = static_cast<T>(1.0 / double((N - m) * (N + m)));
      const T a = static_cast<T>((2.0 * N - 1.0) / double((N - m) * (N + m))) * z, b = inv * r2;
      c[m] = a * c1[m] - b * c2[m];
      s[m] = a * s1[m] - b * s2[m];
    }
  }
}

// s0 times the irregular harmonics: (x, y, z) = d / r^2, ir2 = 1 / r^2, degree 0 = s0 / r.
template <typename T, int N>
__host__ __device__ __forceinline__ void irregular_degree(T x, T y, T z, T ir2, T start, const T* c1, const T* s1,
                                                          const T* c2, const T* s2, T* c, T* s) {
  if constexpr (N == 0) {
    c[0] = start;
    s[0] = T(0);
  } else {
    const T f = static_cast<T>(2 * N - 1);
    const T fx = f * x, fy = f * y, fz = f * z;
    c[N] = fx * c1[N - 1] - fy * s1[N - 1];
    s[N] = fx * s1[N - 1] + fy * c1[N - 1];
    c[N - 1] = fz * c1[N - 1];
    s[N - 1] = fz * s1[N - 1];
#pragma unroll
    for (int m = 0; m <= N - 2; ++m) {
      const T b = static_cast<T>((N - 1) * (N - 1) - m * m) * ir2;
      c[m] = fz * c1[m] - b * c2[m];
      s[m] = fz * s1[m] - b * s2[m];
    }
  }
}

// Contributions of degree N = n + k of the irregular harmonics (twice them) to
// w, inputs of degree k <= KMAX; degrees N + 1.. follow by recursion.  The monopole's
// share of degrees 0 and 1, which is most of them, is left to m2l_direct.
template <typename T, int P, int KMAX, int N>
__host__ __device__ __forceinline__ void m2l_degrees(const T* v, T* w, T x, T y, T z, T ir2, T start, const T* c1,
                                                     const T* s1, const T* c2, const T* s2) {
  if constexpr (N <= P) {
    T c[N + 1], s[N + 1];
    irregular_degree<T, N>(x, y, z, ir2, start, c1, s1, c2, s2, c, s);
    constexpr int KTOP = N < KMAX ? N : KMAX;
    // m = 0, l = 0
    const T h = T(0.5) * c[0];
#pragma unroll
    for (int k = N <= 1 ? 1 : 0; k <= KTOP; ++k) w[sh_idx(N - k, 0)] = fma(h, v[sh_idx(k, 0)], w[sh_idx(N - k, 0)]);
    // m > 0, l = 0 and m = 0, l > 0
#pragma unroll
    for (int m = 1; m <= N; ++m) {
#pragma unroll
      for (int k = 0; k <= KTOP; ++k) {
        const int n = N - k;
        if (m <= n && !(N == 1 && k == 0)) {
          w[sh_idx(n, m)] = fma(c[m], v[sh_idx(k, 0)], w[sh_idx(n, m)]);
          w[sh_idx(n, -m)] = fma(s[m], v[sh_idx(k, 0)], w[sh_idx(n, -m)]);
        }
        if (m <= k) w[sh_idx(n, 0)] = fma(c[m], v[sh_idx(k, m)], fma(s[m], v[sh_idx(k, -m)], w[sh_idx(n, 0)]));
      }
    }
    // m >= l > 0 and the mirrored (l, m): with A + iB of order m + l and
    // D + iE = (-1)^l (order m - l), out_m gets a (A + D) + b (B - E), out_-m
    // a (B + E) + b (D - A); for (l, m) B - E and B + E change places
#pragma unroll
    for (int m = 1; m < N; ++m)
#pragma unroll
      for (int l = 1; l <= m; ++l)
        if (m + l <= N) {
          const T sg = (l & 1) ? T(-1) : T(1);
          const T A = c[m + l], B = s[m + l];
          const T pp = fma(sg, c[m - l], A), tt = fma(sg, c[m - l], -A);
          const T qq = m == l ? B : fma(-sg, s[m - l], B), rr = m == l ? B : fma(sg, s[m - l], B);
#pragma unroll
          for (int k = 1; k <= KTOP; ++k) {
            const int n = N - k;
            if (l <= k && m <= n) {
              const T a = v[sh_idx(k, l)], b = v[sh_idx(k, -l)];
              w[sh_idx(n, m)] = fma(pp, a, fma(qq, b, w[sh_idx(n, m)]));
              w[sh_idx(n, -m)] = fma(rr, a, fma(tt, b, w[sh_idx(n, -m)]));
            }
            if (m != l && m <= k && l <= n) {
              const T a = v[sh_idx(k, m)], b = v[sh_idx(k, -m)];
              w[sh_idx(n, l)] = fma(pp, a, fma(rr, b, w[sh_idx(n, l)]));
              w[sh_idx(n, -l)] = fma(qq, a, fma(tt, b, w[sh_idx(n, -l)]));
            }
          }
        }
    m2l_degrees<T, P, KMAX, N + 1>(v, w, x, y, z, ir2, start, c, s, c1, s1);
  }
}

// Separations r at which the harmonics of degrees 0..P stay well inside T's range:
// r^-(P+1) between 2^-90 and 2^100 (float; the harmonics are at most 2 P! times
// that) or 2^-900 and 2^900 (double).
constexpr int safe_exponent(int p, int bytes, bool low) {
  const int e = bytes == 4 ? (low ? 100 : 90) : 900;
  return e / (p + 1);
}
constexpr double pow2(int e) {
  double v = 1.0;
  for (int i = 0; i < (e < 0 ? -e : e); ++i) v *= e < 0 ? 0.5 : 2.0;
  return v;
}

// w = m2l(v, d) at order P by the direct form (v is overwritten), input degrees above
// KMAX taken as zero.  Where some active lane's r leaves the safe range, every active
// lane scales its inputs by r^-k, takes the harmonics of the unit vector and scales
// the outputs by r^-(n+1).  Both branches are the same for a wave.
//
// Rounding in float32 against 64 bits, direct / cascade, of potential and gradient of
// 20 pairs summed: 7.0e-8 / 6.7e-8 and 1.45e-7 / 1.65e-7 at order 4, 6.6e-8 / 7.1e-8
// and 1.5e-7 / 1.6e-7 at 5.  It takes three things: a pair's w apart from the running
// sums (its (P + 1)^2 products a coefficient added to those one by one: 2.6e-7), the
// largest terms, the monopole's, added last (first: 1.0e-7 against 5.2e-8 of one pair),
// and a corrected 1 / r (the estimate alone: gradient 1.8e-7).
template <typename T, int P, int KMAX = P>
__host__ __device__ __forceinline__ void m2l_direct(T* v, T* w, T dx, T dy, T dz) {
  constexpr T lo = static_cast<T>(pow2(-safe_exponent(P, sizeof(T), true)));
  constexpr T hi = static_cast<T>(pow2(safe_exponent(P, sizeof(T), false)));
  const T r2 = fma(dx, dx, fma(dy, dy, dz * dz));
  const bool safe = r2 >= lo * lo && r2 <= hi * hi;
#if defined(__HIP_DEVICE_COMPILE__)
  const bool rescale = __builtin_expect(__any(!safe), 0);
#else
  const bool rescale = !safe;
#endif
  T rinv = T(0), ir;
  if (rescale) {
    if (r2 > T(0)) {
      const T r = dev_sqrt(r2);
      dx /= r;
      dy /= r;
      dz /= r;
      rinv = T(1) / (r > T(1e-30) ? r : T(1e-30));
    } else {  // coincident centres: unit vector z at the floor distance
      dx = dy = T(0);
      dz = T(1);
      rinv = T(1) / T(1e-30);
    }
    T f = rinv;
#pragma unroll
    for (int k = 1; k <= KMAX; ++k) {
#pragma unroll
      for (int m = -k; m <= k; ++m) v[sh_idx(k, m)] *= f;
      f *= rinv;
    }
    ir = T(1);
  } else {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (sizeof(T) == 4) {  // the hardware estimate (about 1 ulp; r2 is normal here), one Newton step
      const T y = __builtin_amdgcn_rsqf(r2);
      ir = fma(T(0.5) * y, fma(-(r2 * y), y, T(1)), y);
    } else
#endif
      ir = T(1) / dev_sqrt(r2);
  }
#pragma unroll
  for (int j = 0; j < ncoef(P); ++j) w[j] = T(0);
  const T ir2 = ir * ir, x = dx * ir2, y = dy * ir2, z = dz * ir2;
  const T zero[1] = {T(0)};
  m2l_degrees<T, P, KMAX, 0>(v, w, x, y, z, ir2, T(2) * ir, zero, zero, zero, zero);
  const T mono = ir * v[0];
  w[0] += mono;
  if constexpr (P >= 1) {
    w[sh_idx(1, 0)] = fma(z, mono, w[sh_idx(1, 0)]);
    w[sh_idx(1, 1)] = fma(x, T(2) * mono, w[sh_idx(1, 1)]);
    w[sh_idx(1, -1)] = fma(y, T(2) * mono, w[sh_idx(1, -1)]);
  }
  if (rescale) {
    T f = rinv;
#pragma unroll
    for (int n = 0; n <= P; ++n) {
#pragma unroll
      for (int m = -n; m <= n; ++m) w[sh_idx(n, m)] *= f;
      f *= rinv;
    }
  }
}

// w = m2l(v, d): the direct form up to order LINE, the rotation cascade above.
// Instructions of a float32 pair, direct / cascade: 340 / 500 at order 4, 600 / 720 at
// 5, about 850 / 980 at 6 and 1880 / 1740 at 8; registers 73 / 52, 93 / 68, 129 / 88,
// 263 / 128.  The line is that of the centre adjoints, which translate at the order
// above the expansions'; the M2L kernels have lines of their own (direct_line).
constexpr int kDirectM2L = 5;

template <typename T, int P, int KMAX = P, int LINE = kDirectM2L>
__host__ __device__ __forceinline__ void m2l(T* v, T* w, T dx, T dy, T dz) {
  if constexpr (P <= LINE) {
    m2l_direct<T, P, KMAX>(v, w, dx, dy, dz);
  } else {
    Align<T, P> a;
    a.init(dx, dy, dz);
    rotate_all<T, P, Rot::ToZMultipole>(v, a);
    zm2l<T, P>(v, w, a.r);
    rotate_all<T, P, Rot::FromZLocal>(w, a);
  }
}

// A shift's outputs in four parts of nearly equal work, by order |m|: {1, 7}, {2, 6},
// {3, 5}, {0, 4, 8} (20, 20, 20 and 21 of the 81 outputs at order 8, 12, 12, 12 and
// 13 of 49 at order 6).
__host__ __device__ constexpr int shift_part(int m) { return m == 0 || m == 4 || m == 8 ? 3 : (m < 4 ? m : 8 - m) - 1; }
// Whether part PART (-1: all of them) computes outputs of order m.
template <int PART>
__host__ __device__ constexpr bool in_part(int m) {
  return PART < 0 || shift_part(m) == PART;
}

// Contributions of degree N of the regular harmonics to w.  UP: M2M (input
// degree k, output degree N + k); else L2L, its transpose.  Only outputs of PART.
template <typename T, int P, bool UP, int N, int PART = -1>
__host__ __device__ __forceinline__ void shift_degrees(const T* v, T* w, T x, T y, T z, T r2, const T* c1,
                                                       const T* s1, const T* c2, const T* s2) {
  if constexpr (N <= P) {
    T c[N + 1], s[N + 1];
    regular_degree<T, N>(x, y, z, r2, c1, s1, c2, s2, c, s);
    if constexpr (N == 0) {
#pragma unroll
      for (int n = 0; n <= P; ++n)
#pragma unroll
        for (int m = -n; m <= n; ++m)
          if (in_part<PART>(m < 0 ? -m : m)) w[sh_idx(n, m)] = v[sh_idx(n, m)];
    } else {
      // rows: the higher degree n = N + k with order m, columns: degree k with order l
#pragma unroll
      for (int m = 0; m <= P; ++m)
#pragma unroll
        for (int l = 0; l <= P - N; ++l) {
          const int dm = m >= l ? m - l : l - m;
          if (dm > N || !in_part<PART>(UP ? m : l)) continue;
          const bool sum = m + l <= N;
          const T sg = (l & 1) ? T(-1) : T(1);
          const T fl = (m < l && (dm & 1)) ? T(-1) : T(1);
          // order m - l: e1 + i g1, (-1)^l order m + l: sg (c + i s)
          const T e1 = fl * c[dm];
          const T g1 = dm == 0 ? T(0) : (m < l ? -fl : fl) * s[dm];
          T ra, rb = T(0), ia = T(0), ib = T(0);  // row m from column +l / -l, row -m from +l / -l
          if (l == 0) {
            ra = c[dm];
            ia = dm == 0 ? T(0) : s[dm];
          } else if (m == 0) {
            ra = T(2) * sg * c[l <= N ? l : 0];
            rb = T(2) * sg * s[l <= N ? l : 0];
          } else {
            const T e2 = sum ? c[sum ? m + l : 0] : T(0), g2 = sum ? s[sum ? m + l : 0] : T(0);
            ra = sum ? fma(sg, e2, e1) : e1;
            ib = sum ? fma(-sg, e2, e1) : e1;
            rb = sum ? (dm == 0 ? sg * g2 : fma(sg, g2, -g1)) : -g1;
            ia = sum ? (dm == 0 ? sg * g2 : fma(sg, g2, g1)) : g1;
          }
          const bool has_s = !(dm == 0 && !sum);  // the -m/+l and +m/-l couplings vanish with s_0
#pragma unroll
          for (int k = 0; k <= P - N; ++k) {
            const int n = N + k;
            if (l > k || m > n) continue;
            const int rp = sh_idx(n, m), rm = sh_idx(n, -m), cp = sh_idx(k, l), cm = sh_idx(k, -l);
            if constexpr (UP) {
              w[rp] = fma(ra, v[cp], w[rp]);
              if (l > 0 && has_s) w[rp] = fma(rb, v[cm], w[rp]);
              if (m > 0) {
                if (has_s) w[rm] = fma(ia, v[cp], w[rm]);
                if (l > 0) w[rm] = fma(ib, v[cm], w[rm]);
              }
            } else {
              w[cp] = fma(ra, v[rp], w[cp]);
              if (l > 0 && has_s) w[cm] = fma(rb, v[rp], w[cm]);
              if (m > 0) {
                if (has_s) w[cp] = fma(ia, v[rm], w[cp]);
                if (l > 0) w[cm] = fma(ib, v[rm], w[cm]);
              }
            }
          }
        }
    }
    shift_degrees<T, P, UP, N + 1, PART>(v, w, x, y, z, r2, c, s, c1, s1);
  }
}

// One part of w = m2m(v, d) (UP) or l2l(v, d), direct at every order.
template <typename T, int P, bool UP, int PART>
__host__ __device__ __forceinline__ void shift_part_of(const T* v, T* w, T dx, T dy, T dz) {
  const T zero[1] = {T(0)};
  shift_degrees<T, P, UP, 0, PART>(v, w, dx, dy, dz, fma(dx, dx, fma(dy, dy, dz * dz)), zero, zero, zero, zero);
}

// w = m2m(v, d), d = source - destination.  Direct up to order kDirectShift: 258 /
// 520 / 846 / 2129 instructions at order 4 / 5 / 6 / 8 against 450 / 700 / 1020 /
// 2110 of the cascade.  At order 6 the direct L2L's 128 registers (cascade: 112) and
// the 260 of the float64 top levels wait longer for room beside the P2P (the 2M
// galaxy step 0.9% slower), so the line lies below it.
constexpr int kDirectShift = 5;

template <typename T, int P>
__host__ __device__ __forceinline__ void m2m(T* v, T* w, T dx, T dy, T dz) {
  if constexpr (P <= kDirectShift) {
    const T zero[1] = {T(0)};
    shift_degrees<T, P, true, 0>(v, w, dx, dy, dz, fma(dx, dx, fma(dy, dy, dz * dz)), zero, zero, zero, zero);
  } else {
    Align<T, P> a;
    a.init(dx, dy, dz);
    rotate_all<T, P, Rot::ToZMultipole>(v, a);
    zshift_m2m<T, P>(v, a.r);
    rotate_all<T, P, Rot::FromZMultipole>(v, a);
#pragma unroll
    for (int j = 0; j < ncoef(P); ++j) w[j] = v[j];
  }
}

// w = l2l(v, d), d = parent - child.
template <typename T, int P>
__host__ __device__ __forceinline__ void l2l(T* v, T* w, T dx, T dy, T dz) {
  if constexpr (P <= kDirectShift) {
    const T zero[1] = {T(0)};
    shift_degrees<T, P, false, 0>(v, w, dx, dy, dz, fma(dx, dx, fma(dy, dy, dz * dz)), zero, zero, zero, zero);
  } else {
    Align<T, P> a;
    a.init(dx, dy, dz);
    rotate_all<T, P, Rot::ToZLocal>(v, a);
    zshift_l2l<T, P>(v, a.r);
    rotate_all<T, P, Rot::FromZLocal>(v, a);
#pragma unroll
    for (int j = 0; j < ncoef(P); ++j) w[j] = v[j];
  }
}

}  // namespace jfm
