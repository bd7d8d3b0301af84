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

// 1 / sqrt(b) alone, and with the root.
void rsqrt_refined(int n, const double *b, double *alone, double *w, double *root) {
  for (int k = 0; k < n; ++k) {
    alone[k] = rsqrt_pos(b[k]);
    w[k] = rsqrt_pos(b[k], root[k]);
  }
}

// The x flux of S and tau (U [n][9], P [n][8] -> f [n][4]), and the same formulas
// with 1/W an IEEE square root and W an IEEE division.
void flux_x(int n, const double *U, const double *P, double *out) {
  for (int k = 0; k < n; ++k) {
    double f[9];
    srmhd_flux<0, false>(U + 9 * k, P[8 * k + 1], P[8 * k + 2], P[8 * k + 3], P[8 * k + 4], f);
    for (int v = 0; v < 4; ++v) out[4 * k + v] = f[1 + v];
  }
}

void flux_x_ieee(int n, const double *U, const double *P, double *out) {
  for (int k = 0; k < n; ++k) {
    const double *u = U + 9 * k, *v = P + 8 * k + 1, *B = u + 5, p = P[8 * k + 4];
    const double iW = sqrt(1.0 - fma(v[2], v[2], fma(v[1], v[1], v[0] * v[0]))), W = 1.0 / iW;
    const double b0 = W * fma(v[2], B[2], fma(v[1], B[1], v[0] * B[0]));
    const double bsq = fma(b0, b0, fma(B[2], B[2], fma(B[1], B[1], B[0] * B[0]))) * (iW * iW);
    const double ptot = fma(0.5, bsq, p), BiW = B[0] * iW;
    for (int c = 0; c < 3; ++c) out[4 * k + c] = fma(u[1 + c], v[0], -fma(B[c], iW, b0 * v[c]) * BiW);
    out[4 * k] += ptot;
    out[4 * k + 3] = fma(u[4] + ptot, v[0], -b0 * BiW);
  }
}

}  // extern "C"
