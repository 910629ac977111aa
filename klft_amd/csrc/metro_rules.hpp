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

}  // namespace klft_metro
