// What a test program sees of the HIP runtime in host memory (fake_hip.cpp).
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

namespace fake {
struct Dim3 {
  uint32_t x, y, z;
};
struct Launch {
  std::string name;  // mangled
  Dim3 grid;
  void* stream;
};
extern std::vector<Launch> launches;  // kernels launched so far
extern size_t live;                   // bytes allocated and not freed
extern int mallocs, fail_at;          // allocations so far; the one that fails (0: none)
extern int pinned, pinned_live;       // pinned host allocations so far, and those not freed
}  // namespace fake

#define EXPECT(cond)                                                          \
  do {                                                                        \
    if (!(cond)) {                                                            \
      std::printf("%s:%d: %s is false\n", __FILE__, __LINE__, #cond);         \
      std::exit(1);                                                           \
    }                                                                         \
  } while (0)
