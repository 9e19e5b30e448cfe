// The autotuner on a clock on which every candidate is faster than the last: it
// keeps the last candidate of each setting that it tries, and leaves alone a
// setting that the build it times does not look at. Where the Coulomb pair
// starts on the second stream (cplace) only means something for integer builds
// that use one: not for those that run in line (up to 288 MB of B's triangle).
#include "fake_hip.hpp"
#include "../../include/nopt_jk.h"

int main() {
  const struct {
    long nbf, naux;
    int cplace;
  } cases[] = {{24, 116, 1}, {72, 348, 1}, {250, 1206, 2}};
  for (const auto& x : cases) {
    const long npair = x.nbf * (x.nbf + 1) / 2;
    std::vector<double> T(x.naux * npair, 1.0);
    nopt_jk_ctx* c = nullptr;
    EXPECT(nopt_jk_create_ex(0, x.nbf, x.naux, NOPT_CTX_INT8_ONLY | NOPT_CTX_COMPACT, &c) == NOPT_OK);
    EXPECT(nopt_jk_set_B_fitted(c, T.data()) == NOPT_OK);
    int p[6];
    EXPECT(nopt_jk_get_tuning(c, p) == NOPT_OK);
    p[5] = 1;
    EXPECT(nopt_jk_set_tuning(c, p) == NOPT_OK);
    double* d = (double*)nopt_dev_malloc(0, sizeof(double) * x.nbf * x.nbf);
    EXPECT(nopt_jk_autotune(c, d, d, x.nbf / 4, NOPT_PREC_INT8, 1, nullptr, nopt_jk_stream(c)) == NOPT_OK);
    EXPECT(nopt_jk_get_tuning(c, p) == NOPT_OK);
    std::printf("nbf %ld: %d %d %d %d %d %d\n", x.nbf, p[0], p[1], p[2], p[3], p[4], p[5]);
    EXPECT(p[3] == 64 || p[3] == 32);  // the others move
    EXPECT(p[5] == x.cplace);
    nopt_dev_free(d);
    nopt_jk_destroy(c);
  }
  std::puts("ok");
}
