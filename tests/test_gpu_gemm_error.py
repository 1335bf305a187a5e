"""Distance of the small contraction's tile shapes from 64 bits. A matrix
instruction that adds to a running sum rounds it worse than an addition, so the
order of the sums shows. The bounds are what sums dealt to 16 waves, 16 k (f32:
8 k) to an instruction chain, gave for the same distributions, over two seeds;
0.5% covers the choice of the seed (16000000 or 480000 results)."""
import pytest

from helpers import compiled, run

pytestmark = pytest.mark.gpu

CASES = [("bmm_bf16_nt", 32, 500, 500, 64, 4.02e-8), ("bmm_bf16_nt", 32, 500, 500, 128, 5.40e-8),
         ("bmm_bf16", 32, 500, 500, 100, 4.97e-8), ("bmm_bf16", 32, 500, 500, 256, 7.39e-8),
         ("bmm_bf16", 12, 1000, 1000, 2000, 9.78e-8), ("gemm_bf16", 1, 1000, 1000, 64, 4.02e-8),
         ("gemm_bf16_nt", 1, 1000, 1000, 500, 8.29e-8), ("gemm_bf16", 1, 1000, 1000, 1000, 8.87e-8),
         ("gemm_bf16", 1, 1000, 1000, 4096, 11.5e-8), ("gemm_f16", 1, 1000, 1000, 1000, 9.60e-8),
         ("gemm_f32", 1, 60, 8001, 64, 7.74e-8), ("gemm_f32_nt", 1, 60, 8001, 64, 7.74e-8),
         ("gemm_f32", 1, 60, 8001, 129, 9.37e-8), ("gemm_f32", 1, 60, 8001, 200, 10.7e-8),
         ("gemm_f32", 1, 1000, 1000, 1000, 16.2e-8), ("bmm_f32", 32, 500, 500, 64, 7.76e-8)]


@pytest.mark.parametrize("name,B,M,N,K,bound", CASES)
def test_no_further_from_64_bits(gpu, name, B, M, N, K, bound):
    import torch
    dtype = torch.bfloat16 if "bf16" in name else torch.float16 if "f16" in name else torch.float32
    nt, lead = name.endswith("_nt"), (B,) if name.startswith("bmm") else ()
    gen = torch.Generator(device=gpu)
    gen.manual_seed(K)

    def normal(shape, sigma):
        return torch.empty(shape, device=gpu).normal_(0, sigma, generator=gen).to(dtype)
    a, w = normal(lead + (M, K), 1.0), normal(lead + ((N, K) if nt else (K, N)), K ** -0.5)
    c = torch.empty(lead + (M, N), device=gpu)
    run(compiled(name), [a, w, c])
    want = torch.matmul(a.double(), w.double().transpose(-1, -2).contiguous() if nt else w.double())
    error = ((c.double() - want).norm() / want.norm()).item()
    print(name, B, M, N, K, error, flush=True)
    assert error <= 1.005 * bound
