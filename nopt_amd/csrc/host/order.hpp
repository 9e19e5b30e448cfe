// An order of the basis functions for B's integer forms.
#pragma once

namespace nopt {

// perm[new] = old: an order of the nbf functions in which functions whose
// products (m, n) carry weight sit close together. mx[m(m+1)/2 + n] (m >= n) is
// the weight of (m, n), max_P |T[P][mn]| of a packed three-index tensor T;
// (m, n) is an edge when it exceeds 2^-30 times the geometric mean of the
// weights of (m, m) and (n, n); the order is reverse Cuthill-McKee
// on that graph (breadth-first from a low-degree node at the end of a
// longest level structure, neighbours by increasing degree, then reversed),
// component after component. Deterministic (ties by index).
void band_order(const double* mx, long nbf, int* perm);

}  // namespace nopt
