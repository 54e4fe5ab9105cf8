"""Tiled products whose weights one row of tiles alone reads, and which go past the caches (csrc/gemm_blocks.hip: ONCE)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kernels():
    from llmserve_amd.kernels import HipKernels

    return HipKernels(torch.bfloat16)


# rows up to a tile's and one more; weight rows that end inside a tile, a few over 8 MB and many; K of one stage, of few and of many, whole and in parts
@pytest.mark.parametrize("rows", [65, 96, 128, 129, 160, 256, 320])
@pytest.mark.parametrize("outer,inner,parts", [(65538, 64, 1), (4098, 1024, 1), (2206, 1920, 1), (17920, 512, 1), (1037, 4096, 4), (1536, 8960, 7)])
def test_products_past_the_caches(kernels, rows, outer, inner, parts):
    generator = torch.Generator(device="cuda").manual_seed(rows + outer)
    x, w = (torch.randn(n, inner, generator=generator, device="cuda").bfloat16() for n in (rows, outer))

    def product(weight, gated, is_float):
        width = weight.shape[0]
        out = torch.full((parts, rows, width // 2 if gated else width), float("nan"), device="cuda", dtype=torch.float32 if is_float else torch.bfloat16)
        status = kernels._gemm_blocks.llmserve_gemm_blocks(x.data_ptr(), weight.data_ptr(), None, 0, out.data_ptr(), int(is_float), int(gated), rows, width, inner, parts,
                                                           kernels._stream)
        assert status == 0
        return out

    assert outer * inner > 1 << 22
    some = w[: (1 << 22) // inner // 2 * 2 - 6].contiguous()  # (of no more than 8 MB: through the caches)
    for gated, is_float in ((False, True),) if parts > 1 or outer % 2 else ((False, True), (False, False), (True, False)):
        whole, part = product(w, gated, is_float), product(some, gated, is_float)
        assert torch.equal(whole[..., : part.shape[-1]], part)  # the same sums in the same order, in whichever tiles
        if is_float:  # float32 sums of `inner` products
            want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
            assert ((whole.double().sum(0) - want).abs() <= inner * 2.0 ** -24 * size + 1e-6).all()
