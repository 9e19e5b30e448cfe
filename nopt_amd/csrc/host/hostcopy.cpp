// Threaded host copies (declared in hostcopy.hpp).
#include "hostcopy.hpp"

#include <omp.h>

#include <algorithm>
#include <cstring>

namespace nopt {

void copy_rows(char* dst, const char* src, size_t width, size_t pitch, long rows) {
  const size_t total = width * (size_t)rows;
  if (!total) return;
  const int nt = (int)std::min<size_t>((size_t)std::min(4, omp_get_max_threads()), (total >> 18) + 1);
#pragma omp parallel num_threads(nt)
  {
    // each thread a contiguous range of dst
    const size_t T = (size_t)omp_get_num_threads(), id = (size_t)omp_get_thread_num();
    size_t a = total * id / T;
    const size_t b = total * (id + 1) / T;
    while (a < b) {
      const size_t r = a / width, o = a % width, n = std::min(width - o, b - a);
      std::memcpy(dst + a, src + r * pitch + o, n);
      a += n;
    }
  }
}

}  // namespace nopt
