// Host driver for the __host__ __device__ rules of tca/hip/gemm.h (test
// program): reads "m n k batch" lines on stdin and prints 1 for each whose
// whole 256x256 tiles the direct-to-LDS kernels take, else 0 (with any argument:
// in a plan without the small kernel, where no plane is too small). With the argument
// "steps": the 8-deep MFMA steps that the fp32 kernel takes over K = k in 32-deep
// slices dealt to `batch` groups of waves, largest group first.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <vector>

#include "tca/hip/gemm.h"

int main(int argc, char** argv) {
  unsigned m = 0, n = 0, k = 0, b = 0;
  if (argc > 1 && std::strcmp(argv[1], "steps") == 0) {
    while (std::scanf("%u %u %u %u", &m, &n, &k, &b) == 4) {
      std::vector<unsigned> group(b, 0u);
      const unsigned turns = (k / 32u + (k % 32u != 0u)) / b + 1u;
      for (unsigned s = 0; s < turns * b; ++s) group[s % b] += tca::hip::slice_steps32(k, 32u * s);
      std::sort(group.rbegin(), group.rend());
      for (unsigned g : group) std::printf("%u ", g);
      std::printf("\n");
    }
    return 0;
  }
  while (std::scanf("%u %u %u %u", &m, &n, &k, &b) == 4) {
    const bool whole = argc > 1 ? tca::hip::gemm16_on_whole_tiles<0u>(m, n, b) : tca::hip::gemm16_on_whole_tiles<8388608u>(m, n, b);
    std::printf("%d\n", whole && tca::hip::gemm16_direct_k(n, k) ? 1 : 0);
  }
  return 0;
}
