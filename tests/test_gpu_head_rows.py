"""Products of 17 to 128 rows of a large plain weight, a head (csrc/gemm_blocks.hip: launch_shape; `HipKernels._one_row_of_tiles`)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kernels():
    from llmserve_amd.kernels import HipKernels

    return HipKernels(torch.bfloat16)


def near(got, x, w, bias, inner):
    """float32 sums of `inner` products, and a bfloat16 result's rounding."""
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    if bias is not None:
        want, size = want + bias.double(), size + bias.double().abs()
    allowed = (inner + 1) * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if got.dtype == torch.bfloat16 else 0.0)
    return bool(((got.double() - want).abs() <= allowed + 1e-6).all())


# rows about each shape's most; weight rows one under, at and past the line, inside a tile and a multiple of it; K of one stage, fewer than are asked for ahead and more
@pytest.mark.parametrize("rows", [1, 17, 32, 33, 64, 65, 96, 97])
@pytest.mark.parametrize("outer,inner", [(32768, 192), (32769, 64), (33024, 320), (65536, 128), (65801, 64), (66048, 448)])
def test_tiles_that_hold_all_rows(kernels, rows, outer, inner):
    generator = torch.Generator(device="cuda").manual_seed(rows + outer)
    x, w = (torch.randn(n, inner, generator=generator, device="cuda").bfloat16() for n in (rows, outer))
    bias = torch.randn(outer, generator=generator, device="cuda")
    for dtype, of in ((torch.float32, None), (torch.float32, bias), (torch.bfloat16, bias.bfloat16())):
        out = torch.full((rows + 1, outer), float("nan"), device="cuda", dtype=dtype)
        status = kernels._gemm_blocks.llmserve_gemm_blocks(x.data_ptr(), w.data_ptr(), of.data_ptr() if of is not None else None, int(of is not None and of.dtype == torch.float32),
                                                           out.data_ptr(), int(dtype == torch.float32), 0, rows, outer, inner, 1, kernels._stream)
        assert status == 0 and near(out[:rows], x, w, of, inner) and bool(out[rows].isnan().all())


@pytest.mark.parametrize("rows", [17, 64, 80, 128])
def test_a_head_through_linear(kernels, rows):
    from llmserve_amd.kernels.hip import LinearWeights

    outer, inner = 151_936, 1024
    generator = torch.Generator(device="cuda").manual_seed(rows)
    x, w = (torch.randn(n, inner, generator=generator, device="cuda").bfloat16() for n in (rows, outer))
    assert kernels._one_row_of_tiles(x, LinearWeights(w, None), False)
    got = kernels.linear(x, LinearWeights(w, None), out_dtype=torch.float32)
    assert got.shape == (rows, outer) and got.dtype == torch.float32
    some = torch.randint(0, outer, (4096,), generator=generator, device="cuda")
    assert near(got[:, some], x, w[some], None, inner)
    # rows that do not begin at 16 bytes keep their way
    moved = torch.empty(rows * inner + 1, device="cuda", dtype=torch.bfloat16)[1:].view(rows, inner).copy_(x)
    assert not kernels._one_row_of_tiles(moved, LinearWeights(w, None), False)
    assert near(kernels.linear(moved, LinearWeights(w, None), out_dtype=torch.float32)[:, some], x, w[some], None, inner)
