"""How the kernel library cuts products of bfloat16 rows: what it says about a shape, asked without a GPU."""
import pytest
import torch

from imparo_amd.kernels import ops


@pytest.mark.parametrize("n,k", [(1024, 4608), (1024, 8192), (1536, 6912), (2048, 2048), (2048, 8192), (3072, 8192), (2048, 11008),
                                 (4096, 14336)])
def test_slices_of_k_are_equal_parts(n, k):
    """A slice's sum is rounded once more when the consumer adds it, so where K is cut is part of the result. A K in whole steps
    of the kernel is cut into equal parts only: three slices of 2,816, 2,816 and 2,560 in place of four equal ones were further
    from 64 bits (3.2e-7 against 2.7e-7 of the result at 1,100 rows of 2,048 by 8,192)."""
    for m in list(range(65, 600, 7)) + list(range(600, 4200, 61)):
        slices = ops.gemm_slices(m, n, k, torch.bfloat16)
        assert k % (128 * slices) == 0, (m, slices)
