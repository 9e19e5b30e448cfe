// A matrix product over no terms is an error, not a success that leaves C as it
// was; one without rows or columns has nothing to do.
#include "fake_hip.hpp"

struct ihipStream_t;
namespace nopt {
int gemm_f64(bool transB, int M, int N, int K, double alpha, const double* A, long lda, const double* B, long ldb,
             double beta, double* C, long ldc, ihipStream_t* s);
}

int main() {
  double m[16] = {};
  for (bool t : {false, true}) {
    EXPECT(nopt::gemm_f64(t, 4, 4, 4, 1.0, m, 4, m, 4, 0.0, m, 4, nullptr) == 0);
    EXPECT(fake::launches.size() == 1);
    EXPECT(nopt::gemm_f64(t, 4, 4, 0, 1.0, m, 4, m, 4, 0.0, m, 4, nullptr) != 0);
    EXPECT(nopt::gemm_f64(t, 0, 4, 4, 1.0, m, 4, m, 4, 0.0, m, 4, nullptr) == 0);
    EXPECT(nopt::gemm_f64(t, 4, 0, 4, 1.0, m, 4, m, 4, 0.0, m, 4, nullptr) == 0);
    EXPECT(fake::launches.size() == 1);
    fake::launches.clear();
  }
  std::puts("ok");
}
