// FP64 half-transform and exchange on the matrix cores (see fp64.hip).
#pragma once
#include "common.hpp"

#include <algorithm>

namespace nopt {
// X[r*ldx + c] = sum_n B[r*ld + n] Cp[c*ld + n] for the rows r = Q*nbf + m of
// all naux functions and c < ldx (an even count; column groups of 16 nt,
// half_f64_nt picks nt and their number), B's and Cp's columns nbf.. up to the
// next multiple of 16 zero. With nd > 0 also the gamma partials of the nd
// densities Dp + d*dstride (rows of ld), per tile of kHalfF64Rows pair rows (row
// m of the functions 2p and 2p + 1: pair row p*nbf + m): those of gamma_d[Q], p
// = Q / 2, are gpart[d*gstride + 2*(tile + p) + Q % 2] for the tiles that hold
// rows of the pair, tile = p*nbf / kHalfF64Rows .. (p*nbf + nbf - 1) / kHalfF64Rows.
constexpr int kHalfF64Rows = 64, kHalfF64Dens = 2;
static inline int half_f64_tiles(long naux, long nbf) {
  return (int)(((naux + 1) / 2 * nbf + kHalfF64Rows - 1) / kHalfF64Rows);
}
static inline long half_f64_gstride(long naux, long nbf) { return 2 * (half_f64_tiles(naux, nbf) + (naux + 1) / 2); }
int half_f64_nt(long ncol, int* groups);
hipError_t launch_half_f64(int nt, int groups, int nd, hipStream_t s, const double* B, long ld, int naux, int nbf,
                           const double* Cp, const double* Dp, long dstride, double* X, long ldx, double* gpart);

// R_Q[a2][a1] = sum_mn C2[a2][n] B_Q[m][n] C1[a1][m], na <= 32, B symmetric
// (rows of ld values, zero from nbf to the next multiple of 16): Cp holds the
// na rows of C2, then those of C1, ldc values each (ldc a multiple of 16, zero
// from nbf on). R[Q / G][a2*na + a1][Q % G], G = kActiveGroup, zero for
// Q >= naux: the X of launch_syrk_f64 with na*na rows, ldx = kpad = G and
// ceil(naux / G) functions.
constexpr int kActiveGroup = 32;
hipError_t launch_active_half(hipStream_t s, const double* B, long ld, int nbf, int naux, const double* Cp, int ldc,
                              int na, double* R);

// The J pass over FP64 rows: Jpart[d*jstride + (s*nbf + m)*nbf + n], n <= m, the
// sum over the functions Q of split s of gamma_d[Q] B[Q][m][n] (ld > nbf).
// gamma[d*gstride + Q], or with grows > 0 the partials of launch_half_f64
// (tiles of grows rows). launch_jpart_f64: up to four densities, nd*ceil(naux /
// nsplit) gamma values in LDS (at most 64 KB). jpart_rides_f64: whether the
// pass can go into the launch of an exchange: up to two densities, and a split's
// gamma values in what four exchange blocks leave of a CU's LDS.
struct JF64 {
  const double* B;
  long ld;
  int nbf, naux;
  const double* gamma;
  long gstride;
  int grows, nsplit;
  double* Jpart;
  long jstride;
};
constexpr int kRideGamma = 320;
hipError_t launch_jpart_f64(const JF64& a, int nd, hipStream_t s);
bool jpart_rides_f64(int nd, int naux, int nsplit);

constexpr int kSyrkF64Tile = 64;  // exchange tile edge

// Kpart[split][tile][r][c] = sum over the split's functions Q of
// sum_{i < kpad} X[Q][m][i] X[Q][n][i], m = 64 bi + r, n = 64 bj + c, for the
// ntiles lower-triangle tiles (elements above the diagonal and beyond nbf are
// not defined). X rows Q*nbf + m of ldx values (ldx even, X 16-byte aligned),
// kpad a multiple of 4. syrk_f64_splits: the splits to launch when nsplit are
// asked for, few enough that each has at least two slabs of 16 terms (a
// shorter one is over before its loads pay, and its partial tile has to be
// summed).
int syrk_f64_splits(int nsplit, int naux, int kpad);
// With j also the J pass of j's nd densities (jpart_rides_f64) in the same launch.
hipError_t launch_syrk_f64(int ntiles, int nsplit, hipStream_t s, const double* X, long ldx, int nbf, int naux,
                           int kpad, double* Kpart, const JF64* j = nullptr, int nd = 0);
}  // namespace nopt
