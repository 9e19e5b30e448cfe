// The exchange split count that a caller stores is the one that the FP32 and
// bf16 exchanges run with, and so is the FP64 one where every split keeps two
// slabs of terms; storing what get_tuning returned changes nothing.
#include "fake_hip.hpp"
#include "../../include/nopt_jk.h"

#include <algorithm>

int main() {
  const long shapes[][2] = {{24, 116}, {72, 348}, {130, 200}, {200, 500}, {300, 400}};
  for (const auto& s : shapes) {
    const long nbf = s[0], naux = s[1], nocc = nbf / 4;
    std::vector<double> T(naux * nbf * (nbf + 1) / 2, 1.0);
    nopt_jk_ctx* c = nullptr;
    EXPECT(nopt_jk_create_ex(0, nbf, naux, NOPT_CTX_FP64_ONLY, &c) == NOPT_OK);
    EXPECT(nopt_jk_set_B_fitted(c, T.data()) == NOPT_OK);
    double* d = (double*)nopt_dev_malloc(0, sizeof(double) * nbf * nbf);
    // the splits of the exchange of one K: the tiles are x blocks of a (tiles, splits) grid
    auto splits = [&](int prec) {
      fake::launches.clear();
      EXPECT(nopt_jk_build_device(c, nullptr, d, nocc, nullptr, d, prec, nopt_jk_stream(c)) == NOPT_OK);
      const long edge = prec == NOPT_PREC_FP64 ? 64 : 128, k = (nbf + edge - 1) / edge, tiles = k * (k + 1) / 2;
      for (const auto& l : fake::launches)
        if (l.name.find("syrk") != std::string::npos) {
          const long blocks = (long)l.grid.x * l.grid.y;
          EXPECT(blocks % tiles == 0);
          return blocks / tiles;
        }
      return 0L;
    };
    const int modes[] = {NOPT_PREC_FP64, NOPT_PREC_FP32, NOPT_PREC_BF16X3, NOPT_PREC_BF16X6};
    long before[4];
    int p[6];
    for (int m = 0; m < 4; ++m) before[m] = splits(modes[m]);
    EXPECT(nopt_jk_get_tuning(c, p) == NOPT_OK);
    std::printf("nbf %ld: stored %d, splits %ld %ld %ld %ld\n", nbf, p[0], before[0], before[1], before[2], before[3]);
    EXPECT(nopt_jk_set_tuning(c, p) == NOPT_OK);
    for (int m = 0; m < 4; ++m) EXPECT(splits(modes[m]) == before[m]);
    for (int v : {1, 3, 20, 64, (int)naux}) {
      p[0] = v;
      EXPECT(nopt_jk_set_tuning(c, p) == NOPT_OK);
      int q[6];
      EXPECT(nopt_jk_get_tuning(c, q) == NOPT_OK && std::equal(p, p + 6, q));
      const long kpad = (nocc + 3) / 4 * 4;
      EXPECT(splits(NOPT_PREC_FP64) == std::max(1L, std::min((long)v, naux * kpad / 32)));
      for (int m = 1; m < 4; ++m) EXPECT(splits(modes[m]) == v);
    }
    // the tuner's choice for one of these modes is that mode's own, and is what get_tuning returns
    EXPECT(nopt_jk_autotune(c, d, d, nocc, NOPT_PREC_FP32, 1, nullptr, nopt_jk_stream(c)) == NOPT_OK);
    EXPECT(nopt_jk_get_tuning(c, p) == NOPT_OK);
    std::printf("  tuned %d, splits %ld\n", p[0], splits(NOPT_PREC_FP32));
    EXPECT(splits(NOPT_PREC_FP32) == p[0] && p[0] == (naux < 128 ? 64 : 128));
    nopt_dev_free(d);
    nopt_jk_destroy(c);
  }
  std::puts("ok");
}
