// Forming B where one device allocation fails: the call says so, a second call
// succeeds with every buffer in place, and nothing is left after destroy.
#include "fake_hip.hpp"
#include "../../include/nopt_jk.h"

int main() {
  const long nbf = 70, naux = 90, npair = nbf * (nbf + 1) / 2;
  std::vector<double> T(naux * npair, 1.0), V(naux * naux, 0.0);
  for (long i = 0; i < naux; ++i) V[i * naux + i] = 1.0;
  const int forms[] = {NOPT_CTX_DEFAULT, NOPT_CTX_FP64_ONLY, NOPT_CTX_INT8_ONLY, NOPT_CTX_DEFAULT | NOPT_CTX_COMPACT,
                       NOPT_CTX_INT8_ONLY | NOPT_CTX_COMPACT};
  for (int flags : forms)
    for (int fitted = 0; fitted < 2; ++fitted) {
      auto form = [&](nopt_jk_ctx* c) {
        return fitted ? nopt_jk_set_B_fitted(c, T.data()) : nopt_jk_set_B(c, T.data(), V.data());
      };
      nopt_jk_ctx* c = nullptr;
      EXPECT(nopt_jk_create_ex(0, nbf, naux, flags, &c) == NOPT_OK);
      fake::mallocs = 0;
      EXPECT(form(c) == NOPT_OK);
      const int total = fake::mallocs;
      const size_t whole = fake::live;
      nopt_jk_destroy(c);
      EXPECT(fake::live == 0);
      for (int k = 1; k <= total; ++k) {
        EXPECT(nopt_jk_create_ex(0, nbf, naux, flags, &c) == NOPT_OK);
        fake::mallocs = 0;
        fake::fail_at = k;
        const int rc = form(c);
        fake::fail_at = 0;
        std::printf("flags %d fitted %d allocation %d of %d: %d\n", flags, fitted, k, total, rc);
        EXPECT(rc == NOPT_ENOMEM);
        EXPECT(form(c) == NOPT_OK);
        EXPECT(fake::live == whole);
        nopt_jk_destroy(c);
        EXPECT(fake::live == 0);
      }
    }
  std::puts("ok");
}
