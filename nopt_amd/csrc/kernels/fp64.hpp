// FP64 exchange on the matrix cores (see fp64.hip).
#pragma once
#include "common.hpp"

#include <algorithm>

namespace nopt {
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
hipError_t launch_syrk_f64(int ntiles, int nsplit, hipStream_t s, const double* X, long ldx, int nbf, int naux,
                           int kpad, double* Kpart);
}  // namespace nopt
