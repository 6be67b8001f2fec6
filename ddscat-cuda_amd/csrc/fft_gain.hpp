// Gain of the FP32 transforms, on the host.
//
// Twiddle factors rounded to FP32 are no longer of modulus one, and a transform
// of a length with its inverse returns its input times 1 + g, g the mean of
// |w|^2 - 1 over the entries of the DFT matrix that the rounded factors make up:
// the sum of the butterflies' own and of the twiddles between the stages.  It
// is the same for every mode, so it adds up over the axes while rounding
// errors average out: up to 7e-8 an axis (400 points as 20 x 20; 256 points as 16 x
// 16 -5e-8), most of the error of a MATVEC.  Pass 5 divides it out of its scale.
// MATVECs of cubes against 64 bits, relative L2, without and with: 32^3 1.60e-7 ->
// 1.14e-7, 128^3 2.07e-7 -> 1.35e-7, 200^3 2.41e-7 -> 1.52e-7, 256^3 2.18e-7 -> 1.46e-7,
// 384^3 2.54e-7 -> 1.53e-7.
#pragma once
#include "common.hpp"
#include <cmath>

namespace ddhip {

// |w|^2 - 1 of w = e^{2 pi i m / N} with both parts rounded to FP32
inline double twiddle_excess(long m, long N) {
  const double a = 6.283185307179586476925286766559 * (double)(m % N) / (double)N;
  const double c = (double)(float)std::cos(a), s = (double)(float)std::sin(a);
  return c * c + s * s - 1.0;
}
// mean excess over r < R, k < P of w_{PR}^{r k}: the twiddles of a radix-R stage behind P points
inline double stage_excess(int P, int R) {
  double t = 0.0;
  for (int r = 1; r < R; ++r)
    for (int k = 1; k < P; ++k) t += twiddle_excess((long)r * k, (long)P * R);
  return t / ((double)P * R);
}
// R-point butterfly: the closed forms of fft_device.hpp, and compositions of
// them, split as dft_reg does (fft_reg.hpp)
inline double radix_gain(int R) {
  if (R == 1 || R == 2 || R == 4) return 0.0;  // exact factors
  if (R == 3 || R == 5 || R == 7) {            // (R - 1)^2 of R^2 entries, those of one row over and over
    double t = 0.0;
    for (int m = 1; m < R; ++m) {
      const int q = m < R - m ? m : R - m;  // the constants of the first half
      t += twiddle_excess(q, R);
    }
    return (R - 1) * t / ((double)R * R);
  }
  if (R == 8) return 16.0 / 64.0 * twiddle_excess(1, 8);  // odd row times odd column: (1 + i) / sqrt 2
  const int Q = R == 16 ? 4 : R % 8 == 0 ? 8 : R % 4 == 0 ? 4 : R % 5 == 0 ? 5 : R % 3 == 0 ? 3 : 2;
  return radix_gain(R / Q) + radix_gain(Q) + stage_excess(Q, R / Q);
}
// transform of the radices of p, in order
inline double fft_gain(const FftPlan& p) {
  double g = 0.0;
  for (int s = 0, P = 1; s < p.nst; P *= p.rad[s++]) g += radix_gain(p.rad[s]) + (s ? stage_excess(P, p.rad[s]) : 0.0);
  return g;
}

}  // namespace ddhip
