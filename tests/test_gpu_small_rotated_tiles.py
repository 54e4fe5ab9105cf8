"""The smallest tiles of the product whose heads are rotated on the way out (csrc/gemm_blocks.hip: launch_rotated): rows and pages are those of the tiled
product and of the kernel that rotates and stores behind it, bit for bit."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_kernels import kernels, on_gpu, paged_case  # noqa: F401

pytestmark = pytest.mark.gpu


# one stage of K, as many as are asked for ahead, and more; rows and columns that end inside a tile
@pytest.mark.parametrize("inner", [64, 512, 640])
@pytest.mark.parametrize("heads,kv_heads,dim,counts", [
    (12, 2, 128, [65]), (12, 2, 128, [64, 64]), (5, 3, 48, [70, 59]), (14, 2, 64, [1, 223]),   # 32 x 32
    (12, 2, 128, [129]), (12, 2, 128, [100, 61]), (12, 2, 128, [7, 217]), (5, 3, 144, [193]),  # 32 x 64
    (12, 2, 128, [255]), (12, 2, 128, [250, 6]), (14, 2, 64, [300, 150]),                      # 64 x 32
])
def test_small_tiles(kernels, monkeypatch, heads, kv_heads, dim, counts, inner):  # noqa: F811
    library, rows, generator = kernels[torch.bfloat16], sum(counts), torch.Generator().manual_seed(inner + dim)
    monkeypatch.setattr(type(library), "_rotated_ahead", staticmethod(lambda *sizes: True))
    x = torch.randn(rows, inner, generator=generator).bfloat16().cuda()
    width = (heads + 2 * kv_heads) * dim
    prepared = library.prepare_linear([on_gpu(torch.randn(width, inner, generator=generator) * inner ** -0.5, torch.bfloat16)],
                                      [on_gpu(torch.randn(width, generator=generator), torch.bfloat16)])
    inverse = on_gpu(1.0 / (3000.0 ** (torch.arange(0, dim, 2).float() / dim)))
    found = []
    for fused in (False, True):
        batch, cell, _, layout = paged_case([count + 5 for count in counts], counts, heads, kv_heads, dim, 16, torch.bfloat16, shuffle_seed=inner + dim)
        if fused:
            qkv = library.linear_rotated(x, prepared, layout, batch, cell, inverse, "adjacent")
        else:
            qkv = torch.empty(rows, width, dtype=torch.bfloat16, device="cuda")
            assert library._gemm_blocks.llmserve_gemm_blocks(x.data_ptr(), prepared.weight.data_ptr(), prepared.bias.data_ptr(), 0, qkv.data_ptr(), 0, 0, rows, width, inner, 1,
                                                             library._stream) == 0
            library.rotate_and_store(qkv, layout, batch, cell, inverse, "adjacent")
        found.append((qkv, cell.keys.float().nan_to_num(7e7), cell.values.float().nan_to_num(7e7)))
    assert all(torch.equal(apart, together) for apart, together in zip(*found))
