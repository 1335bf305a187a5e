// The small contraction's k steps and wave sums as kernels of their own (test
// program): compiled for their code, never run.
#include "tca/hip/gemm.h"

using namespace tca::hip;

template <int IM, int D, bool B_NK>
__device__ __forceinline__ void steps16(const uint16_t* A, const uint16_t* B, float* C, uint32_t M, uint32_t N, uint32_t K,
                                        uint32_t n) {
  __shared__ __attribute__((aligned(16))) float red[kSmallWaves * 1024u];
  f32x4_t acc[IM][2];
  small16_steps<IM, D, B_NK, false>(A, B, M, N, K, 0u, 0u, 0u, n, reinterpret_cast<uint16_t*>(red) + (threadIdx.x >> 6) * 2048u,
                                    acc);
  small16_sum(acc, red, [&](uint32_t row, uint32_t col, float sum) { C[row * 32u + col] = sum; });
}

template <int IM, int D, bool B_NK>
__device__ __forceinline__ void steps32(const float* A, const float* B, float* C, uint32_t M, uint32_t N, uint32_t K, uint32_t n) {
  __shared__ __attribute__((aligned(16))) float red[kSmallWaves * 1024u];
  f32x16 acc[IM];
  small32_steps<IM, D, B_NK>(A, B, M, N, K, 0u, 0u, 0u, n, red + (threadIdx.x >> 6) * 1024u, acc);
  small32_sum(acc, red, [&](uint32_t row0, uint32_t t, float sum) { C[row0 * 32u + t] = sum; });
}

#define KERNEL(name, body, T)                                                                                        \
  extern "C" __global__ void __launch_bounds__(1024)                                                                 \
      name(const T* A, const T* B, float* C, uint32_t M, uint32_t N, uint32_t K, uint32_t n) {                       \
    body(A, B, C, M, N, K, n);                                                                                       \
  }
KERNEL(k16_32, (steps16<2, 4, false>), uint16_t)
KERNEL(k16_32_nt, (steps16<2, 4, true>), uint16_t)
KERNEL(k16_64, (steps16<4, 2, false>), uint16_t)
KERNEL(k16_64_nt, (steps16<4, 2, true>), uint16_t)
KERNEL(k32_32, (steps32<1, 2, false>), float)
KERNEL(k32_32_nt, (steps32<1, 2, true>), float)
KERNEL(k32_64, (steps32<2, 2, false>), float)
KERNEL(k32_64_nt, (steps32<2, 2, true>), float)
