"""The rules that choose a product's tile and its slices of K: plain host code, checked without a GPU
(the library counts 256 CUs where it cannot ask)."""

import pytest
import torch

from kllm_amd import kernels as K

BF16, F32 = torch.bfloat16, torch.float32
LONG = 1 << 23          # from this K on a lane's offset takes 64 bits


@pytest.mark.parametrize("n,m,k,dtype,slices", [
    (65, 3, LONG + 8, BF16, 8), (2000, 4096, LONG, BF16, 8), (2, 3, LONG + 8, F32, 8), (65, 3, LONG + 4, F32, 8),
    (64, 3, LONG + 8, BF16, 1), (2, 3, LONG + 8, BF16, 1), (64, 2048, 5632, BF16, 1), (1, 8, 8, BF16, 1),
    (0, 8, 8, BF16, 1),
])
def test_slices_where_the_times_are_not_estimated(n, m, k, dtype, slices):
    """Also right behind a product whose times are, which leaves its numbers on the stack."""
    for other in ((700, 2048, 5632), (64, 2048, 5632), (2048, 28672, 4096)):
        K.gemm_prompt_slices(*other, dtype)
        K.gemm_prompt_slices.cache_clear()
        assert K.gemm_prompt_slices(n, m, k, dtype) == slices
