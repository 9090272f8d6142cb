// Host helper: FP64 unit-modulus value -> FP32 pair with the squared modulus
// nearest 1.
//
// Rounding the two components independently leaves |w|^2 - 1 of a few 1e-8 with
// a fixed sign per value.  Twiddles and propagator entries are applied hundreds
// of times to every probe, so such a bias adds up coherently; among the
// neighbouring floats of each component this picks the pair closest to the unit
// circle (ties: closest value), which is within one ulp of the FP64 value.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

namespace totem {

inline float2 unit_float2(double c, double s) {
  const float c0 = (float)c, s0 = (float)s;
  float best_c = c0, best_s = s0;
  double best = 1e300;
  for (int i = -1; i <= 1; ++i)
    for (int j = -1; j <= 1; ++j) {
      float cc = c0, ss = s0;
      if (i) cc = std::nextafter(c0, i < 0 ? -2.0f : 2.0f);
      if (j) ss = std::nextafter(s0, j < 0 ? -2.0f : 2.0f);
      const double dn = std::fabs((double)cc * cc + (double)ss * ss - 1.0);
      const double dv = std::fabs(cc - c) + std::fabs(ss - s);
      const double score = dn * 1e6 + dv;
      if (score < best) {
        best = score;
        best_c = cc;
        best_s = ss;
      }
    }
  return make_float2(best_c, best_s);
}

// Unit-modulus values of one table column (one factor for consecutive k), rounded so
// that their squared moduli average 1: of the neighbouring floats the pair taken for
// each value is the one that brings the running sum of |w|^2 - 1 nearest 0, its distance
// from the value counting 16 times.  The fused stages multiply at every level of a
// butterfly, so what the wave's norm sees is a column's mean modulus (near 45 degrees no
// single pair is on the circle: the nearest are off by -3.4e-8 and +5.0e-8), while each
// pair's own distance goes into the wave.  Exit waves of 80 slices against complex128 by
// weight, 4 / 8 / 16 / 32: 128^2 2.8e-6, 2.6e-6, 2.5e-6, 2.4e-6; 512^2 2.8, 2.7, 2.7, 2.8;
// 1024^2 3.3, 3.0, 3.1, 3.3 (4.5 at 1, 3.6 at 2); 1536^2 3.3, 3.3, 3.6, 3.9: flat from 8
// to 16, where the weight was taken.  The images' error (1e-7 to 4e-6) follows what is
// left of the norm's drift, which no weight orders; unit_float2 lets it drift to 6.9e-6 at
// 1024^2.
inline float2 balanced_float2(double c, double s, double& sum) {
  const float c0 = (float)c, s0 = (float)s;
  float best_c = c0, best_s = s0;
  double best = 1e300, best_d = 0.0;
  for (int i = -1; i <= 1; ++i)
    for (int j = -1; j <= 1; ++j) {
      float cc = c0, ss = s0;
      if (i) cc = std::nextafter(c0, i < 0 ? -2.0f : 2.0f);
      if (j) ss = std::nextafter(s0, j < 0 ? -2.0f : 2.0f);
      const double d = (double)cc * cc + (double)ss * ss - 1.0;
      const double score = std::fabs(sum + d) + 16.0 * std::hypot(cc - c, ss - s);
      if (score < best) {
        best = score;
        best_c = cc;
        best_s = ss;
        best_d = d;
      }
    }
  sum += best_d;
  return make_float2(best_c, best_s);
}

}  // namespace totem
