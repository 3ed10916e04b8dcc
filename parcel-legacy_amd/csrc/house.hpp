// house.hpp -- the host half of TSQR (house.cpp).
#pragma once

namespace parcel {

// R (n x n, column-major) of the m x n matrix whose row j is S[j * n ..]
// (overwritten), bit for bit dense.hpp's house_r.  Returns false, with S
// untouched, where it does not run: n > 16, m < n or a CPU without FMA.
bool house_r_rows(int m, int n, double* S, double* R);

}  // namespace parcel
