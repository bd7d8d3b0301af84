// The device headers' per-cell functions over arrays of cells, on the host.
#include "mgpu_srrmhd.hpp"

using namespace mgpu;

extern "C" {

// srrmhd_secant from the starting values Z, which the results replace.
void secant(int n, const double *SbSq, const double *D, const double *tauBar, double gam, double *Z, int *its) {
  for (int k = 0; k < n; ++k) its[k] = srrmhd_secant(Z[k], SbSq[k], D[k], tauBar[k], gam);
}

// srmhd_recover (U [n][9], root [n][2] = v^2, Z) into P [n][8], A [n][13].
void recover(int n, const double *U, const double *root, double gam, double *P, double *A) {
  for (int k = 0; k < n; ++k) srmhd_recover(U + 9 * k, gam, root[2 * k], root[2 * k + 1], P + 8 * k, A + 13 * k);
}

// srrmhd_recover (U [n][14], root [n] = Z) into P [n][11], A [n][17].
void recover_resistive(int n, const double *U, const double *root, double gam, double sigma, double *P, double *A) {
  for (int k = 0; k < n; ++k) srrmhd_recover(U + 14 * k, gam, sigma, root[k], P + 11 * k, A + 17 * k);
}

}  // extern "C"
