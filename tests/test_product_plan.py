"""How the kernel library cuts products of bfloat16 rows: what it says about a shape, asked without a GPU."""
from ctypes import byref, c_int64

import pytest
import torch

from imparo_amd.kernels import library, ops
from imparo_amd.kernels.program import LinearDesc, StepArgs, SwigluDesc


@pytest.mark.parametrize("n,k", [(1024, 4608), (1024, 8192), (1536, 6912), (2048, 2048), (2048, 8192), (3072, 8192), (2048, 11008),
                                 (4096, 14336)])
def test_slices_of_k_are_equal_parts(n, k):
    """A slice's sum is rounded once more when the consumer adds it, so where K is cut is part of the result. A K in whole steps
    of the kernel is cut into equal parts only: three slices of 2,816, 2,816 and 2,560 in place of four equal ones were further
    from 64 bits (3.2e-7 against 2.7e-7 of the result at 1,100 rows of 2,048 by 8,192)."""
    for m in list(range(65, 600, 7)) + list(range(600, 4200, 61)):
        slices = ops.gemm_slices(m, n, k, torch.bfloat16)
        assert k % (128 * slices) == 0, (m, slices)


def _program(lib, width, ff, layers=2):
    """A step program of feed-forwards, whose addresses nothing reads (it is only asked what it needs)."""
    at, bf16, f32 = 1 << 20, 1, 0
    p = lib.imparo_program_new(bf16, 64)
    assert lib.imparo_program_embedding(p, at, bf16, 1000, width) == 0
    for _ in range(layers):
        desc = SwigluDesc(LinearDesc(at, None, bf16, 2 * ff, width), LinearDesc(at, None, bf16, width, ff))
        assert lib.imparo_program_norm(p, at, 1e-5, width, bf16) == 0 and lib.imparo_program_swiglu(p, byref(desc)) == 0
    return p, [lib.imparo_program_region_name(p, i).decode() for i in range(lib.imparo_program_n_regions(p))]


@pytest.mark.parametrize("width,ff,tokens", [(1024, 1024, 2048), (1024, 4608, 3000), (1536, 6912, 512), (2048, 2048, 512),
                                             (2048, 8192, 4096), (768, 3072, 4096)])
def test_what_steps_up_to_a_size_need_is_the_most_of_every_count(width, ff, tokens):
    """Slices times rows is largest at counts of no pattern (1,943 rows of 1,024 by 1,024, 2,681 of 1,024 by 4,608): asked once
    for all steps up to a size, the program says what the hungriest of them needs."""
    lib = library()
    p, names = _program(lib, width, ff)
    n = len(names)
    args, most, need = StepArgs(), (c_int64 * n)(), (c_int64 * n)()
    args.n_rows = args.n_portion = args.table_width = 1
    args.n_tokens = tokens
    assert lib.imparo_program_needs_up_to(p, byref(args), most) == 0
    want = [0] * n
    for t in range(1, tokens + 1):
        args.n_tokens = args.max_seg_len = t
        assert lib.imparo_program_needs(p, byref(args), need) == 0
        want = [max(a, b) for a, b in zip(want, need)]
    lib.imparo_program_delete(p)
    assert list(most) == want
    slices = [ops.gemm_slices(t, width, ff, torch.bfloat16) for t in range(1, tokens + 1)]
    assert most[names.index("ffn_out_sliced")] == 4 * width * max(s * (t + 1) if s > 1 else 0 for t, s in enumerate(slices))


@pytest.mark.parametrize("m", [65535 * 64 + 1, 2 ** 31 - 1])
@pytest.mark.parametrize("out_dtype", [0, 1])
def test_float32_product_refuses_more_rows_than_its_grid_takes(m, out_dtype):
    """Refused by its sizes, before anything is launched (the addresses are nobody's), also where rounding the rows up to tiles
    would pass 2^31."""
    at, refused = 1 << 20, 1
    assert library().imparo_gemm(at, at, None, at, 0, out_dtype, m, 64, 4, 0, 1, None) == refused
