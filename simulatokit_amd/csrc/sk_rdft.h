// sk_rdft.h — unscaled DFTs of a compile-time length R in registers, for any R whose prime factors are at most 13:
// the building blocks of the two-stage line transforms (sk_pair.h). Everything folds at compile time: the index maps,
// the roots (float64-derived, rounded once) and the products with 1, i and (1 + i) / sqrt 2.
#pragma once

#include <hip/hip_runtime.h>

#include "sk_internal.h"

namespace sk {

// cos and sin of 2 pi m / r in float64 at compile time: reduced to [0, pi / 4] with integer octants, then the Taylor
// series (15 terms leave less than one ulp there).
namespace rootdetail {
constexpr double kPi = 3.14159265358979323846;
constexpr double taylor_sin(double x) {
  double t = x, s = x;
  for (int k = 1; k < 15; ++k) {
    t *= -x * x / double((2 * k) * (2 * k + 1));
    s += t;
  }
  return s;
}
constexpr double taylor_cos(double x) {
  double t = 1, s = 1;
  for (int k = 1; k < 15; ++k) {
    t *= -x * x / double((2 * k - 1) * (2 * k));
    s += t;
  }
  return s;
}
// 2 pi m / r = (pi / 4) (8 m / r): octant o and the remainder's numerator over r
constexpr double cos_of(int m, int r) {
  m %= r;
  const int e = 8 * m, o = e / r, f = e - o * r;  // angle = (pi / 4) (o + f / r)
  const double x = kPi / 4 * f / r, y = kPi / 4 * (r - f) / r;
  switch (o) {
    case 0: return taylor_cos(x);
    case 1: return taylor_sin(y);
    case 2: return -taylor_sin(x);
    case 3: return -taylor_cos(y);
    case 4: return -taylor_cos(x);
    case 5: return -taylor_sin(y);
    case 6: return taylor_sin(x);
    default: return taylor_cos(y);
  }
}
// sin(2 pi m / r) = cos(2 pi (4 m - r) / (4 r))
constexpr double sin_of(int m, int r) { return cos_of((4 * (m % r) + 3 * r) % (4 * r), 4 * r); }
}  // namespace rootdetail

// The float32 roots e^{2 pi i m / R}. A pass of the slice loop applies a transform one way and (conjugated) back, and
// the errors of the constants' rounding would add up: the way back (BACK) takes other roundings that cancel them as far
// as float32 goes. For a composite radix, whose roots are factors: the reciprocal conjugates of the first table's
// entries. For an odd prime, whose sines and cosines are summed: 2 x - (the first table's rounding of x).
// The cosines of an odd prime sum to -1/2 over half a turn, and so do their roundings here: what they miss (9e-8 for 13,
// each rounded by itself) would turn a constant line, the bulk of a wave that entered as a plane one, into other
// frequencies, the same way in every slice. The smallest cosine, which has the finest steps, takes the difference. Exit
// waves at lengths with a factor 7, 11 or 13 come to 0.72 of their error with it (geometric mean of 47 planes).
template <int R, bool BACK = false>
struct RootTable {
  float c[R], s[R];
  constexpr RootTable() : c(), s() {
    const bool prime = R == 3 || R == 5 || R == 7 || R == 11 || R == 13;
    for (int m = 0; m < R; ++m) {
      const double cx = rootdetail::cos_of(m, R), sx = rootdetail::sin_of(m, R);
      const float c0 = float(cx), s0 = float(sx);
      const double n = double(c0) * c0 + double(s0) * s0;
      c[m] = !BACK ? c0 : float(prime ? 2 * cx - c0 : c0 / n);
      s[m] = !BACK ? s0 : float(prime ? 2 * sx - s0 : s0 / n);
    }
    if (prime && R > 5) {  // 3: -1/2 itself; 5: written as -1/4 +- sqrt(5) / 4
      int least = 1;
      double sum = c[1];
      for (int m = 2; m <= R / 2; ++m) {
        sum += c[m];
        if ((c[m] < 0 ? -c[m] : c[m]) < (c[least] < 0 ? -c[least] : c[least])) least = m;
      }
      c[least] = c[R - least] = float(c[least] - (sum + 0.5));
    }
  }
};

// The transforms are templates on the complex type: float2 on the device; double2, with the same float32 constants, on
// the host, where the launch code measures what the constants' rounding does to a transform's gain (sk_pair.hip).
template <class V>
__host__ __device__ __forceinline__ V cx(decltype(V::x) x, decltype(V::x) y) {
  V v;
  v.x = x;
  v.y = y;
  return v;
}
template <class V>
__host__ __device__ __forceinline__ V vadd(V a, V b) { return cx<V>(a.x + b.x, a.y + b.y); }
template <class V>
__host__ __device__ __forceinline__ V vsub(V a, V b) { return cx<V>(a.x - b.x, a.y - b.y); }
__host__ __device__ __forceinline__ float vfma(float a, float b, float c) { return fmaf(a, b, c); }
__host__ __device__ __forceinline__ double vfma(double a, double b, double c) { return a * b + c; }

// a * e^{SIGN 2 pi i m / R}; m is a constant after unrolling
template <int R, int SIGN, bool BACK, class V>
__host__ __device__ __forceinline__ V mul_root(V a, int m) {
  constexpr RootTable<R, BACK> T{};
  m %= R;
  const float h = 0.70710678118654752f, g = SIGN < 0 ? -1.f : 1.f;
  if (m == 0) return a;
  if (2 * m == R) return cx<V>(-a.x, -a.y);
  if (4 * m == R) return cx<V>(-g * a.y, g * a.x);
  if (4 * m == 3 * R) return cx<V>(g * a.y, -g * a.x);
  if (8 * m == R) return cx<V>((a.x - g * a.y) * h, (a.y + g * a.x) * h);
  if (8 * m == 3 * R) return cx<V>((-a.x - g * a.y) * h, (-a.y + g * a.x) * h);
  if (8 * m == 5 * R) return cx<V>((-a.x + g * a.y) * h, (-a.y - g * a.x) * h);
  if (8 * m == 7 * R) return cx<V>((a.x + g * a.y) * h, (a.y - g * a.x) * h);
  const float c = T.c[m], s = g * T.s[m];
  return cx<V>(a.x * c - a.y * s, a.x * s + a.y * c);
}

constexpr bool is_prime(int r) {
  for (int p = 2; p * p <= r; ++p)
    if (r % p == 0) return false;
  return r > 1;
}
// The split R = a b of a composite radix: coprime (a the largest prime power, so the halves need no twiddles), or for
// a prime power its square-ish split (Cooley-Tukey with constant twiddles).
constexpr int prime_power_part(int r, int p) {
  int q = 1;
  while (r % p == 0) {
    r /= p;
    q *= p;
  }
  return q;
}
constexpr int split_of(int r) {
  int best = 1;
  for (int p = 2; p <= r; ++p)
    if (is_prime(p) && r % p == 0) {
      const int q = prime_power_part(r, p);
      if (q != r && q > best) best = q;
    }
  if (best > 1) return best;
  switch (r) {  // a prime power
    case 8: return 2;
    case 16: return 4;
    case 32: return 4;
    default: break;
  }
  for (int p = 3; p < r; ++p)
    if (r % p == 0) return p;
  return r;
}
constexpr int gcd_of(int a, int b) { return b == 0 ? a : gcd_of(b, a % b); }
constexpr int inverse_mod(int a, int m) {
  for (int x = 1; x < m; ++x)
    if (a * x % m == 1) return x;
  return 1 % m;
}

// u <- DFT_R(u): u_k = sum_j u_j e^{SIGN 2 pi i j k / R}, in natural order. TR: the transposed flow graph (every step
// backwards), whose matrix is the transpose of the other's, the rounding of its constants included.
template <int R, int SIGN, bool TR = false, class V>
__host__ __device__ __forceinline__ void rdft(V (&u)[R]) {
  if constexpr (R == 1) {
    return;
  } else if constexpr (R == 2) {
    const V a = u[0], b = u[1];
    u[0] = vadd(a, b);
    u[1] = vsub(a, b);
  } else if constexpr (R == 4) {
    const V t0 = vadd(u[0], u[2]), t1 = vsub(u[0], u[2]), t2 = vadd(u[1], u[3]);
    const V d = vsub(u[1], u[3]);
    const V t3 = SIGN < 0 ? cx<V>(d.y, -d.x) : cx<V>(-d.y, d.x);
    u[0] = vadd(t0, t2);
    u[2] = vsub(t0, t2);
    u[1] = vadd(t1, t3);
    u[3] = vsub(t1, t3);
  } else if constexpr (R == 5) {
    // the cosines of 2 pi / 5 and 4 pi / 5 are -1/4 +- sqrt(5) / 4: their sum is exact this way, where two rounded
    // cosines would make every fifth root's row carry a little of the constant
    constexpr RootTable<5, TR> T{};
    const decltype(V::x) h = 0.55901699437494742f, s1 = T.s[1], s2 = T.s[2];
    const V p1 = vadd(u[1], u[4]), p2 = vadd(u[2], u[3]), d1 = vsub(u[1], u[4]), d2 = vsub(u[2], u[3]);
    const V t = vadd(p1, p2), e = vsub(p1, p2), u0 = u[0];
    const V m = cx<V>(vfma(decltype(V::x)(-0.25f), t.x, u0.x), vfma(decltype(V::x)(-0.25f), t.y, u0.y));
    const V a1 = cx<V>(vfma(h, e.x, m.x), vfma(h, e.y, m.y)), a2 = cx<V>(vfma(-h, e.x, m.x), vfma(-h, e.y, m.y));
    const V b1 = cx<V>(vfma(s2, d2.x, s1 * d1.x), vfma(s2, d2.y, s1 * d1.y));
    const V b2 = cx<V>(vfma(-s1, d2.x, s2 * d1.x), vfma(-s1, d2.y, s2 * d1.y));
    const V i1 = SIGN < 0 ? cx<V>(b1.y, -b1.x) : cx<V>(-b1.y, b1.x);
    const V i2 = SIGN < 0 ? cx<V>(b2.y, -b2.x) : cx<V>(-b2.y, b2.x);
    u[0] = vadd(u0, t);
    u[1] = vadd(a1, i1);
    u[4] = vsub(a1, i1);
    u[2] = vadd(a2, i2);
    u[3] = vsub(a2, i2);
  } else if constexpr (is_prime(R)) {
    // an odd prime: with s_j = u_j + u_{R-j}, d_j = u_j - u_{R-j}, the pair (k, R - k) is
    // u_0 + sum_j cos(2 pi j k / R) s_j  +-  SIGN i sum_j sin(2 pi j k / R) d_j
    constexpr RootTable<R, TR> T{};
    constexpr int H = (R - 1) / 2;
    V s[H], d[H];
    V total = u[0];
#pragma unroll
    for (int j = 0; j < H; ++j) {
      s[j] = vadd(u[j + 1], u[R - 1 - j]);
      d[j] = vsub(u[j + 1], u[R - 1 - j]);
      total = vadd(total, s[j]);
    }
    const V u0 = u[0];
    u[0] = total;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      V a = u0, b = cx<V>(0, 0);
#pragma unroll
      for (int j = 0; j < H; ++j) {
        const int m = (j + 1) * k % R;
        const decltype(V::x) c = T.c[m], q = T.s[m];
        a.x = vfma(c, s[j].x, a.x);
        a.y = vfma(c, s[j].y, a.y);
        b.x = j == 0 ? q * d[j].x : vfma(q, d[j].x, b.x);
        b.y = j == 0 ? q * d[j].y : vfma(q, d[j].y, b.y);
      }
      // SIGN i b
      const V ib = SIGN < 0 ? cx<V>(b.y, -b.x) : cx<V>(-b.y, b.x);
      u[k] = vadd(a, ib);
      u[R - k] = vsub(a, ib);
    }
  } else {
    constexpr int A = split_of(R), B = R / A;
    if constexpr (gcd_of(A, B) == 1) {
      // prime-factor map: input n = (B n1 + A n2) mod R, output k = (e1 k1 + e2 k2) mod R with e1 = 1 mod A, 0 mod B
      constexpr int E1 = B * inverse_mod(B % A, A), E2 = A * inverse_mod(A % B, B);
      V w[R];  // [n2][k1]
      if constexpr (!TR) {
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
          V t[A];
#pragma unroll
          for (int n1 = 0; n1 < A; ++n1) t[n1] = u[(B * n1 + A * n2) % R];
          rdft<A, SIGN>(t);
#pragma unroll
          for (int k1 = 0; k1 < A; ++k1) w[n2 * A + k1] = t[k1];
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
          V t[B];
#pragma unroll
          for (int n2 = 0; n2 < B; ++n2) t[n2] = w[n2 * A + k1];
          rdft<B, SIGN>(t);
#pragma unroll
          for (int k2 = 0; k2 < B; ++k2) u[(E1 * k1 + E2 * k2) % R] = t[k2];
        }
      } else {
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
          V t[B];
#pragma unroll
          for (int k2 = 0; k2 < B; ++k2) t[k2] = u[(E1 * k1 + E2 * k2) % R];
          rdft<B, SIGN, true>(t);
#pragma unroll
          for (int n2 = 0; n2 < B; ++n2) w[n2 * A + k1] = t[n2];
        }
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
          V t[A];
#pragma unroll
          for (int k1 = 0; k1 < A; ++k1) t[k1] = w[n2 * A + k1];
          rdft<A, SIGN, true>(t);
#pragma unroll
          for (int n1 = 0; n1 < A; ++n1) u[(B * n1 + A * n2) % R] = t[n1];
        }
      }
    } else {
      // Cooley-Tukey: input n = B n1 + n2, output k = k1 + A k2, the twiddle e^{SIGN 2 pi i n2 k1 / R} between
      V w[R];
      if constexpr (!TR) {
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
          V t[A];
#pragma unroll
          for (int n1 = 0; n1 < A; ++n1) t[n1] = u[B * n1 + n2];
          rdft<A, SIGN>(t);
#pragma unroll
          for (int k1 = 0; k1 < A; ++k1) w[n2 * A + k1] = mul_root<R, SIGN, false>(t[k1], n2 * k1);
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
          V t[B];
#pragma unroll
          for (int n2 = 0; n2 < B; ++n2) t[n2] = w[n2 * A + k1];
          rdft<B, SIGN>(t);
#pragma unroll
          for (int k2 = 0; k2 < B; ++k2) u[k1 + A * k2] = t[k2];
        }
      } else {
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
          V t[B];
#pragma unroll
          for (int k2 = 0; k2 < B; ++k2) t[k2] = u[k1 + A * k2];
          rdft<B, SIGN, true>(t);
#pragma unroll
          for (int n2 = 0; n2 < B; ++n2) w[n2 * A + k1] = mul_root<R, SIGN, true>(t[n2], n2 * k1);
        }
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
          V t[A];
#pragma unroll
          for (int k1 = 0; k1 < A; ++k1) t[k1] = w[n2 * A + k1];
          rdft<A, SIGN, true>(t);
#pragma unroll
          for (int n1 = 0; n1 < A; ++n1) u[B * n1 + n2] = t[n1];
        }
      }
    }
  }
}

}  // namespace sk
