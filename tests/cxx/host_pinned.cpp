// Pinned host memory is made by the first call that needs it, kept by the
// context and freed with it: a new geometry of the same shape asks for none.
#include "fake_hip.hpp"
#include "../../include/nopt_jk.h"

int main() {
  const long shapes[][2] = {{2, 2}, {24, 116}, {256, 130}};  // the last one: 34 MB, through the pinned pieces
  for (const auto& s : shapes) {
    const long nbf = s[0], naux = s[1];
    std::vector<double> T(naux * nbf * (nbf + 1) / 2, 1.0), V(naux * naux, 0.0);
    for (long i = 0; i < naux; ++i) V[i * naux + i] = 1.0;
    nopt_jk_ctx* c = nullptr;
    EXPECT(nopt_jk_create(0, nbf, naux, &c) == NOPT_OK);
    EXPECT(nopt_jk_set_B(c, T.data(), V.data()) == NOPT_OK);
    const int made = fake::pinned;
    EXPECT(nopt_jk_set_B(c, T.data(), V.data()) == NOPT_OK);
    std::printf("nbf %ld naux %ld: %d pinned allocations, %d in the second call\n", nbf, naux, made, fake::pinned - made);
    EXPECT(fake::pinned == made);
    nopt_jk_destroy(c);
    EXPECT(fake::pinned_live == 0);
    fake::pinned = 0;
  }
  std::puts("ok");
}
