// The device headers' per-cell functions over arrays of cells, on the host.
#include "mgpu_srrmhd.hpp"

using namespace mgpu;

extern "C" {

// srrmhd_secant from the starting values Z, which the results replace.
void secant(int n, const double *SbSq, const double *D, const double *tauBar, double gam, double *Z, int *its) {
  for (int k = 0; k < n; ++k) its[k] = srrmhd_secant(Z[k], SbSq[k], D[k], tauBar[k], gam);
}

}  // extern "C"
