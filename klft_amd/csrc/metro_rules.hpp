// Rules of the Metropolis sweep, free of HIP calls: the kernels and the host
// code take them from here, and a host compiler can check them.
#pragma once
#include "philox.hpp"

namespace klft_metro {

// Whether a row v of an SU(3) proposal with |v|^2 = n2 is drawn again: the
// reference goes on while 1 + |v| rounds to 1 (SUN.hpp:198-233), which is |v| <=
// 2^-53.  The square root of the double after 2^-106 still rounds to 2^-53.  A NaN
// is not drawn again: it would never end, and a NaN proposal is rejected.
KLFT_HD bool row_redrawn(double n2) { return n2 <= 0x1.0000000000001p-106; }

// Whether the rows of SU(3) proposals with this delta can be expected to be
// kept: six uniforms of [0, |delta|) with a norm above 2^-53 (FP32 links: 2^-24) and
// a square that does not overflow.  At the limits, half the smallest norm and
// twice the largest, one row in about a thousand is kept; beyond them the kernels
// would draw for ever.  U(1), SU(2) and the symmetric law have no such loop, and a
// delta that is not finite is drawn once.
inline bool rows_kept(double delta, bool fp64) {
  const double d = fp64 ? delta : (double)(float)delta;
  const double a = d < 0.0 ? -d : d;
  if (!(a <= (fp64 ? 1.7976931348623157e308 : 3.4028234663852886e38))) return true;
  return fp64 ? (a >= 0x1p-54 && a <= 0x1p513) : (a >= 0x1p-25 && a <= 0x1p65);
}

// Whether a pass of Vh sites runs faster with a link's hits in parallel
// (metro_hits.hpp) than with site waves fed by staple waves.  The site-wave
// kernel's pass costs one block's serial chain however few blocks there are;
// the hit-parallel kernel's chain is up to six times shorter but spends up
// to ten lanes on a site, so it wins until the sites fill the GPU.  In SU(3) every
// accepted hit costs a round in which all lanes of the site judge again, so the
// limit falls with the acceptance, which beta stands for (4D, thermalised,
// beta 2.5 / 4 / 5 / 6: 33, 13, 6, 3 %; 3D and 2D accept more but have
// fewer directions a site, and their limits come out the same).
// Measured in runs (ms per sweep, hit-parallel / site waves, or their ratio), around
// the limits in sites of a pass per CU:
//   SU(3), 10 hits   16/CU (16^4) FP64 0.23 / 0.64, FP32 0.17 / 0.49
//     26/CU (18^4)   FP64 beta 1.5 1.09, 2.5 0.93, 3.5 0.73
//     39/CU (20^4)   FP64 beta 2.5 1.27, 3.5 1.01, 4 0.87, 5 0.73
//     57/CU (22^4)   FP64 beta 4 1.14, 4.5 1.02, 5 0.93, 6 0.82
//     81/CU (24^4)   FP64 beta 5 1.18, 6 1.03 (0.68 / 0.71 from an ordered start),
//                    FP32 beta 5 1.04, 6 0.91
//   SU(3), 4 hits    39/CU FP64 beta 3.5 1.09, 4 1.03, 5 0.92; 57/CU beta 6 1.04
//   SU(3), 1 hit     39/CU FP64 beta 4 1.07, 5 0.99, 6 0.95; 57/CU beta 6 1.12
//   symmetric law, delta 0.005 / 0.1 / 0.4 (99, 80, 27 % accepted), FP64:
//     12 hits        26/CU 1.06, 0.88, 0.59; 32/CU 1.20, 0.99, 0.65
//     4 hits         26/CU 1.03, 1.00, 0.77; 1 hit 20/CU 0.82, 0.87, 0.98, 26/CU
//                    0.94, 1.00, 1.09
//   SU(2)  16/CU FP64 0.32 / 0.52; 26/CU 0.48 / 0.52, FP32 0.29 / 0.35; 39/CU
//          0.67 / 0.52
//   U(1)   16/CU FP64 0.22 / 0.28; 26/CU 0.30 / 0.28, FP32 0.22 / 0.23; with 4
//          hits 39/CU 0.16 / 0.19
// (SU(2) and U(1) step through their hits, accepted or not: the limit holds for
// every beta), and in 2D with fewer than 4 hits the site waves' chain is as short
// (U(1) 32^2, 1 hit: 32 against 29 us).
inline bool hits_in_parallel(int nd, int nc, long long Vh, int cus, int nhits, double beta, bool symmetric) {
  if (nd == 2 && nhits < 4) return false;
  double per_cu;
  if (nc == 1) {
    per_cu = nhits < 5 ? 40 : 20;
  } else if (nc == 2) {
    per_cu = 27;
  } else if (symmetric) {
    per_cu = nhits < 4 ? 20 : 27;
  } else {
    const double most = nhits < 4 ? 40 : (nhits < 8 ? 48 : 81);
    const double at_beta = nhits < 8 ? 8 * beta : 18 * beta - 27;
    per_cu = at_beta > 20 ? (at_beta < most ? at_beta : most) : 20;
  }
  return (double)Vh <= per_cu * cus;
}

}  // namespace klft_metro
