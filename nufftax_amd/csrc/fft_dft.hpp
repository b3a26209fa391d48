// Register DFTs of small lengths for the mixed-radix FFT passes (fftn.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace nufftx {

template <typename T>
struct alignas(2 * sizeof(T)) fcplx {
  T x, y;
};

template <typename T>
__host__ __device__ __forceinline__ fcplx<T> operator+(fcplx<T> a, fcplx<T> b) {
  return {a.x + b.x, a.y + b.y};
}
template <typename T>
__host__ __device__ __forceinline__ fcplx<T> operator-(fcplx<T> a, fcplx<T> b) {
  return {a.x - b.x, a.y - b.y};
}
template <typename T>
__host__ __device__ __forceinline__ fcplx<T> fmul(fcplx<T> a, fcplx<T> b) {
  return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
// -i a
template <typename T>
__host__ __device__ __forceinline__ fcplx<T> mul_mi(fcplx<T> a) {
  return {a.y, -a.x};
}

// cos and sin of 2 pi n / 16, n < 16, and of 2 pi n / 9.  Not recursive: the compiler folds these to literals only where it
// can inline them, and a function that calls itself stays a call (with a call per inner twiddle in the radix-8 and
// radix-16 columns, small type 1 calls on 240 x 240 FP32 and 1600 x 1600 FP64 grids took 50 and 152 us; now 42 and 97).
template <typename T>
__host__ __device__ __forceinline__ constexpr T cos16(int n) {
  const int m = (n & 15) > 8 ? 16 - (n & 15) : n & 15, q = m > 4 ? 8 - m : m;
  const T c = q == 0   ? T(1)
              : q == 1 ? T(0.92387953251128675613)
              : q == 2 ? T(0.70710678118654752440)
              : q == 3 ? T(0.38268343236508977173)
                       : T(0);
  return m > 4 ? -c : c;
}
template <typename T>
__host__ __device__ __forceinline__ constexpr T cos9(int n) {
  const int m = n % 9 > 4 ? 9 - n % 9 : n % 9;
  return m == 0   ? T(1)
         : m == 1 ? T(0.76604444311897803520)
         : m == 2 ? T(0.17364817766693034885)
         : m == 3 ? T(-0.5)
                  : T(-0.93969262078590838405);
}
template <typename T>
__host__ __device__ __forceinline__ constexpr T sin9(int n) {
  const int m = n % 9, q = m > 4 ? 9 - m : m;
  const T s = q == 0   ? T(0)
              : q == 1 ? T(0.64278760968653932632)
              : q == 2 ? T(0.98480775301220805937)
              : q == 3 ? T(0.86602540378443864676)
                       : T(0.34202014332566873304);
  return m > 4 ? -s : s;
}
// exp(-2 pi i n / R) for the inner twiddles of R = 8, 16 and 9
template <typename T, int R>
__host__ __device__ __forceinline__ constexpr fcplx<T> wconst(int n) {
  return R == 9 ? fcplx<T>{cos9<T>(n), -sin9<T>(n)}
                : fcplx<T>{cos16<T>(n * (16 / R)), -cos16<T>(n * (16 / R) + 12)};  // sin(a) = cos(a - pi/2)
}

// the k in [0, A B) with k = a mod A and k = b mod B (A, B coprime)
template <int A, int B>
__host__ __device__ constexpr int crt(int a, int b) {
  int k = a;
  while (k % B != b) k += A;
  return k;
}

// R-point forward DFT of v in place, natural order in and out.
template <typename T, int R>
struct Dft {
  // R = A B: prime factors (Good 1958) where A and B are coprime, no twiddles; else one Cooley-Tukey step
  static constexpr int A = R == 16 ? 4 : R == 12 ? 4 : R == 10 ? 2 : R == 9 ? 3 : R == 8 ? 4 : R == 6 ? 2 : 3;
  static constexpr int B = R / A;
  static constexpr bool kCoprime = R == 6 || R == 10 || R == 12 || R == 15;
  static __host__ __device__ __forceinline__ void run(fcplx<T> (&v)[R]) {
    static_assert(A * B == R, "");
    fcplx<T> t[B][A];  // t[n2][k1]
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) t[n2][n1] = v[kCoprime ? (B * n1 + A * n2) % R : B * n1 + n2];
      Dft<T, A>::run(t[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      fcplx<T> u[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2)
        u[n2] = kCoprime || n2 * k1 == 0 ? t[n2][k1] : fmul(t[n2][k1], wconst<T, R>(n2 * k1));
      Dft<T, B>::run(u);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[kCoprime ? crt<A, B>(k1, k2) : k1 + A * k2] = u[k2];
    }
  }
};
template <typename T>
struct Dft<T, 2> {
  static __host__ __device__ __forceinline__ void run(fcplx<T> (&v)[2]) {
    const fcplx<T> a = v[0], b = v[1];
    v[0] = a + b;
    v[1] = a - b;
  }
};
template <typename T>
struct Dft<T, 3> {
  static __host__ __device__ __forceinline__ void run(fcplx<T> (&v)[3]) {
    constexpr T h = T(0.5), s = T(0.86602540378443864676);
    const fcplx<T> p = v[1] + v[2], m = v[1] - v[2];
    const fcplx<T> q = {v[0].x - h * p.x, v[0].y - h * p.y}, r = {s * m.y, -s * m.x};
    v[0] = v[0] + p;
    v[1] = q + r;
    v[2] = q - r;
  }
};
template <typename T>
struct Dft<T, 4> {
  static __host__ __device__ __forceinline__ void run(fcplx<T> (&v)[4]) {
    const fcplx<T> a = v[0] + v[2], b = v[0] - v[2], c = v[1] + v[3], d = mul_mi(v[1] - v[3]);
    v[0] = a + c;
    v[1] = b + d;
    v[2] = a - c;
    v[3] = b - d;
  }
};
template <typename T>
struct Dft<T, 5> {
  static __host__ __device__ __forceinline__ void run(fcplx<T> (&v)[5]) {
    constexpr T c1 = T(0.30901699437494742410), c2 = T(-0.80901699437494742410);
    constexpr T s1 = T(0.95105651629515357212), s2 = T(0.58778525229247312917);
    const fcplx<T> p1 = v[1] + v[4], m1 = v[1] - v[4], p2 = v[2] + v[3], m2 = v[2] - v[3];
    const fcplx<T> a = {v[0].x + c1 * p1.x + c2 * p2.x, v[0].y + c1 * p1.y + c2 * p2.y};
    const fcplx<T> b = {v[0].x + c2 * p1.x + c1 * p2.x, v[0].y + c2 * p1.y + c1 * p2.y};
    const fcplx<T> d = {s1 * m1.y + s2 * m2.y, -(s1 * m1.x + s2 * m2.x)};
    const fcplx<T> e = {s2 * m1.y - s1 * m2.y, -(s2 * m1.x - s1 * m2.x)};
    v[0] = v[0] + p1 + p2;
    v[1] = a + d;
    v[2] = b + e;
    v[3] = b - e;
    v[4] = a - d;
  }
};

}  // namespace nufftx
