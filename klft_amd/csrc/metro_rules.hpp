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

}  // namespace klft_metro
