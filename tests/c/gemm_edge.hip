// Host driver for the __host__ __device__ rules of tca/hip/gemm.h (test
// program): reads "m n k batch" lines on stdin and prints 1 for each whose
// whole 256x256 tiles the direct-to-LDS kernels take, else 0.
#include <cstdio>

#include "tca/hip/gemm.h"

int main(int argc, char**) {
  unsigned m = 0, n = 0, k = 0, b = 0;
  while (std::scanf("%u %u %u %u", &m, &n, &k, &b) == 4) {
    const bool whole = argc > 1 ? tca::hip::gemm16_on_whole_tiles<0u>(m, n, b) : tca::hip::gemm16_on_whole_tiles<8388608u>(m, n, b);
    std::printf("%d\n", whole && tca::hip::gemm16_direct_k(n, k) ? 1 : 0);
  }
  return 0;
}
