// nopt_jk_device_bytes against the allocations that are alive, through the calls
// that make buffers grow.
#include "fake_hip.hpp"
#include "../../include/nopt_jk.h"

int main() {
  const long shapes[][2] = {{1, 1}, {24, 116}, {70, 90}, {200, 40}};
  const int forms[] = {NOPT_CTX_DEFAULT, NOPT_CTX_FP64_ONLY, NOPT_CTX_INT8_ONLY, NOPT_CTX_INT8_ONLY | NOPT_CTX_COMPACT};
  for (const auto& s : shapes)
    for (int flags : forms) {
      const long nbf = s[0], naux = s[1], nocc = (nbf + 1) / 2;
      std::vector<double> T(naux * nbf * (nbf + 1) / 2, 1.0), V(naux * naux, 0.0), M(nbf * nbf), J(nbf * nbf),
          K(nbf * nbf), G(nbf * nbf), I(32 * 32 * 32 * 32);
      for (long i = 0; i < naux; ++i) V[i * naux + i] = 1.0;
      nopt_jk_ctx* c = nullptr;
      auto check = [&](const char* what) {
        std::printf("nbf %ld naux %ld flags %d %s: held %zu, reported %ld\n", nbf, naux, flags, what, fake::live,
                    nopt_jk_device_bytes(c));
        EXPECT(nopt_jk_device_bytes(c) == (long)fake::live);
      };
      EXPECT(nopt_jk_create_ex(0, nbf, naux, flags, &c) == NOPT_OK);
      check("created");
      EXPECT(nopt_jk_set_B(c, T.data(), V.data()) == NOPT_OK);
      check("B formed");
      const bool f64 = !(flags & NOPT_CTX_INT8_ONLY), i8 = !(flags & NOPT_CTX_FP64_ONLY);
      for (int prec = 0; prec <= 4; ++prec) {
        if (!(prec == NOPT_PREC_INT8 ? i8 : f64)) continue;
        EXPECT(nopt_jk_build(c, M.data(), M.data(), nocc, J.data(), K.data(), prec) == NOPT_OK);
        check("build");
      }
      const int prec = f64 ? NOPT_PREC_FP64 : NOPT_PREC_INT8;
      const double* in[4] = {M.data(), M.data(), M.data(), M.data()};
      double* out[4] = {J.data(), J.data(), J.data(), J.data()};
      const long n[4] = {nocc, 1, nbf, 0};
      EXPECT(nopt_jk_build_batch(c, 4, in, in, n, out, out, prec) == NOPT_OK);
      check("batch");
      EXPECT(nopt_jk_energy_gradient(c, M.data(), M.data(), nocc, prec, nullptr, G.data(), nullptr) == NOPT_OK);
      check("gradient");
      if (f64) {
        EXPECT(nopt_jk_active_ints(c, M.data(), M.data(), nbf < 20 ? 1 : 20, I.data()) == NOPT_OK);
        check("active integrals");
      }
      nopt_jk_destroy(c);
      EXPECT(fake::live == 0);
    }
  std::puts("ok");
}
