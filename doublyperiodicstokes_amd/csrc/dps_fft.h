// dps_fft.h -- register-resident complex DFTs of up to 35 points, shared by the
// FFT kernels and the host-side checks.
#pragma once
#include "dps_core.h"

namespace dps {

// cos(pi j / 16), j = 0..16
constexpr double kCos16[17] = {
    1.0,
    0.98078528040323044912618223613424,
    0.92387953251128675612818318939679,
    0.83146961230254523707878837761791,
    0.70710678118654752440084436210485,
    0.55557023301960222474283081394853,
    0.38268343236508977172845998403040,
    0.19509032201612826784828486847702,
    0.0,
    -0.19509032201612826784828486847702,
    -0.38268343236508977172845998403040,
    -0.55557023301960222474283081394853,
    -0.70710678118654752440084436210485,
    -0.83146961230254523707878837761791,
    -0.92387953251128675612818318939679,
    -0.98078528040323044912618223613424,
    -1.0};

// bit reversal of i over log2(R) bits
constexpr int fft_brev(int i, int R)
{
  int r = 0;
  for (int b = 1; b < R; b <<= 1) {
    r = (r << 1) | (i & 1);
    i >>= 1;
  }
  return r;
}

// cos(2 pi j / 24), j = 0..23
constexpr double kCos24[24] = {
    1.0,
    0.96592582628906828674974319972890,
    0.86602540378443864676372317075294,
    0.70710678118654752440084436210485,
    0.5,
    0.25881904510252076234889883762405,
    0.0,
    -0.25881904510252076234889883762405,
    -0.5,
    -0.70710678118654752440084436210485,
    -0.86602540378443864676372317075294,
    -0.96592582628906828674974319972890,
    -1.0,
    -0.96592582628906828674974319972890,
    -0.86602540378443864676372317075294,
    -0.70710678118654752440084436210485,
    -0.5,
    -0.25881904510252076234889883762405,
    0.0,
    0.25881904510252076234889883762405,
    0.5,
    0.70710678118654752440084436210485,
    0.86602540378443864676372317075294,
    0.96592582628906828674974319972890};

template <int R, int DIR, class T> DPS_HD void fft_reg(T (&re)[R], T (&im)[R]);

// DFT of R = 3 P points (P = 1, 2, 4 or 8) held in registers: the three
// P-point DFTs of the decimated sequences x[3 n2 + n1], then
//   X_k = sum_{n1 < 3} exp(DIR 2 pi i n1 k / R) A_{n1}[k mod P]
// with the twiddles cos/sin(2 pi m / 24), m = (24 / R) n1 k mod 24,
// compile-time constants once the loops are unrolled.
template <int R, int DIR, class T>
DPS_HD void dft_reg3(T (&re)[R], T (&im)[R])
{
  static_assert(R == 3 || R == 6 || R == 12 || R == 24, "R must be 3 times 1, 2, 4 or 8");
  constexpr int P = R / 3;
  T ar[3][P], ai[3][P];
#pragma unroll
  for (int n1 = 0; n1 < 3; ++n1)
#pragma unroll
    for (int n2 = 0; n2 < P; ++n2) {
      ar[n1][n2] = re[3 * n2 + n1];
      ai[n1][n2] = im[3 * n2 + n1];
    }
  if constexpr (P > 1) {
#pragma unroll
    for (int n1 = 0; n1 < 3; ++n1) fft_reg<P, DIR>(ar[n1], ai[n1]);
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    T xr = ar[0][k % P], xi = ai[0][k % P];
#pragma unroll
    for (int n1 = 1; n1 < 3; ++n1) {
      const int m = ((24 / R) * n1 * k) % 24;
      const T c = (T)kCos24[m];
      const T sn = (T)(DIR * kCos24[(m + 18) % 24]);   // sin(2 pi m / 24) = cos(2 pi (m - 6) / 24)
      const T yr = ar[n1][k % P], yi = ai[n1][k % P];
      xr += yr * c - yi * sn;
      xi += yr * sn + yi * c;
    }
    re[k] = xr;
    im[k] = xi;
  }
}

// In-place DFT of R points held in registers: X_k = sum_n x_n exp(DIR 2 pi
// i n k / R), DIR = -1 forward, +1 inverse (unnormalised).  R = 2, 4, 8, 16
// or 32: radix-2 decimation in time; every twiddle is a compile-time constant
// once the loops are unrolled, and the trivial ones are skipped.  R = 3, 6,
// 12 or 24: dft_reg3 (three R/3-point transforms and a radix-3 combination).
template <int R, int DIR, class T>
DPS_HD void fft_reg(T (&re)[R], T (&im)[R])
{
  if constexpr (R % 3 == 0) {
    dft_reg3<R, DIR>(re, im);
    return;
  } else {
  static_assert(R >= 2 && R <= 32 && (R & (R - 1)) == 0, "R must be a power of two <= 32");
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int j = fft_brev(i, R);
    if (i < j) {
      const T a = re[i], b = im[i];
      re[i] = re[j];
      im[i] = im[j];
      re[j] = a;
      im[j] = b;
    }
  }
#pragma unroll
  for (int len = 2; len <= R; len <<= 1) {
    const int half = len >> 1;
#pragma unroll
    for (int i = 0; i < R; i += len) {
#pragma unroll
      for (int k = 0; k < half; ++k) {
        // twiddle exp(DIR 2 pi i m / 32), m = 32 k / len in [0, 16)
        const int m = k * (32 / len);
        T br = re[i + k + half], bi = im[i + k + half];
        if (m != 0) {
          const T c = (T)kCos16[m];
          const T s = (T)(DIR * kCos16[m < 8 ? 8 - m : m - 8]);
          const T tr = br * c - bi * s;
          const T ti = br * s + bi * c;
          br = tr;
          bi = ti;
        }
        re[i + k + half] = re[i + k] - br;
        im[i + k + half] = im[i + k] - bi;
        re[i + k] += br;
        im[i + k] += bi;
      }
    }
  }
  }
}

// cos(2 pi m / n) evaluated by the compiler: reduced to an angle of at most
// pi / 4, then the Taylor series of cosine or sine (12 terms, below an ulp)
constexpr double kPi = 3.14159265358979323846264338327950288;
constexpr double taylor_cos(double x)
{
  double t = 1, s = 1;
  for (int i = 1; i < 12; ++i) {
    t *= -x * x / ((2 * i - 1) * (2 * i));
    s += t;
  }
  return s;
}
constexpr double taylor_sin(double x)
{
  double t = x, s = x;
  for (int i = 1; i < 12; ++i) {
    t *= -x * x / ((2 * i) * (2 * i + 1));
    s += t;
  }
  return s;
}
constexpr double cos_turn(int m, int n)
{
  m = ((m % n) + n) % n;
  if (2 * m > n) m = n - m;                              // cos(-a) = cos a
  if (4 * m > n) return -cos_turn(n - 2 * m, 2 * n);     // cos(pi - a) = -cos a
  return 8 * m <= n ? taylor_cos(2 * kPi * m / n) : taylor_sin(2 * kPi * (n - 4 * m) / (4 * n));
}
constexpr double sin_turn(int m, int n) { return cos_turn(4 * m - n, 4 * n); }

// the n-th roots of unity: constants once the loops that index it are unrolled
template <int N> struct Circle {
  double c[N], s[N];
  constexpr Circle() : c(), s()
  {
    for (int m = 0; m < N; ++m) {
      c[m] = cos_turn(m, N);
      s[m] = sin_turn(m, N);
    }
  }
};
template <int N> constexpr Circle<N> kCircle{};

// DFT of an odd prime P: the sums and differences of x_j and x_{P-j}, combined
// with cosines and sines
template <int P, int DIR, class T>
DPS_HD void dft_prime(T (&re)[P], T (&im)[P])
{
  constexpr int H = P / 2;
  T sr[H], si[H], dr[H], di[H];
#pragma unroll
  for (int j = 1; j <= H; ++j) {
    sr[j - 1] = re[j] + re[P - j];
    si[j - 1] = im[j] + im[P - j];
    dr[j - 1] = re[j] - re[P - j];
    di[j - 1] = im[j] - im[P - j];
  }
  const T r0 = re[0], i0 = im[0];
#pragma unroll
  for (int j = 0; j < H; ++j) {
    re[0] += sr[j];
    im[0] += si[j];
  }
#pragma unroll
  for (int k = 1; k <= H; ++k) {
    T ar = r0, ai = i0, br = 0, bi = 0;
#pragma unroll
    for (int j = 1; j <= H; ++j) {
      const T c = (T)kCircle<P>.c[(j * k) % P], s = (T)kCircle<P>.s[(j * k) % P];
      ar += c * sr[j - 1];
      ai += c * si[j - 1];
      br += s * dr[j - 1];
      bi += s * di[j - 1];
    }
    // exp(DIR i a) d: the difference part times DIR i
    re[k] = ar - (T)DIR * bi;
    im[k] = ai + (T)DIR * br;
    re[P - k] = ar + (T)DIR * bi;
    im[P - k] = ai - (T)DIR * br;
  }
}

// whether fft_reg above holds this length
constexpr bool fft_reg_has(int R) { return (R & (R - 1)) == 0 || R == 3 || R == 6 || R == 12 || R == 24; }
constexpr int largest_prime(int R) { return R % 7 == 0 ? 7 : (R % 5 == 0 ? 5 : (R % 3 == 0 ? 3 : 2)); }

// In-place DFT of R points (R = 1 or a product of 2, 3, 5 and 7 up to 35) held
// in registers, sign DIR, unnormalised.  Lengths that fft_reg lacks are split
// by their largest prime P, R = P Q: Q-point DFTs of the decimated sequences
// x[P q + p], twiddles, and P-point DFTs across them.
template <int R, int DIR, class T>
DPS_HD void dft(T (&re)[R], T (&im)[R])
{
  if constexpr (R == 1) {
    return;
  } else if constexpr (fft_reg_has(R)) {
    fft_reg<R, DIR>(re, im);
  } else if constexpr (R == 5 || R == 7) {
    dft_prime<R, DIR>(re, im);
  } else {
    constexpr int P = largest_prime(R), Q = R / P;
    T ar[P][Q], ai[P][Q];
#pragma unroll
    for (int a = 0; a < P; ++a) {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        ar[a][q] = re[P * q + a];
        ai[a][q] = im[P * q + a];
      }
      dft<Q, DIR>(ar[a], ai[a]);
    }
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      T br[P], bi[P];
#pragma unroll
      for (int a = 0; a < P; ++a) {
        br[a] = ar[a][k];
        bi[a] = ai[a][k];
        if (a * k != 0) {
          const T c = (T)kCircle<R>.c[a * k], s = (T)(DIR * kCircle<R>.s[a * k]);
          br[a] = ar[a][k] * c - ai[a][k] * s;
          bi[a] = ar[a][k] * s + ai[a][k] * c;
        }
      }
      if constexpr (P == 3) fft_reg<3, DIR>(br, bi);
      else dft_prime<P, DIR>(br, bi);
#pragma unroll
      for (int b = 0; b < P; ++b) {
        re[k + Q * b] = br[b];
        im[k + Q * b] = bi[b];
      }
    }
  }
}

}  // namespace dps
