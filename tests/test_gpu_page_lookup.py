"""Pages of a fused decode step (csrc/attention_bf16.hip: a wave holds the request's row of the block table, 64 entries a register, as long as its registers hold all of it): at the
edges of a register, of all of them and beyond, over keys of which each head finds another one."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_kernels import TOLERANCE, _rewrite_cell, kernels, on_gpu, paged_case, rounded, step_rows  # noqa: F401

pytestmark = pytest.mark.gpu


# six registers of entries where a wave asks for two steps at once (heads up to 128 wide), else four; pages of 8 keys, of which a step of 32 has five, of 24, which are no power of
# two, and of 64, of which a step lies in one or two
@pytest.mark.parametrize("dim,page,pages", [
    (128, 8, 63), (128, 8, 64), (128, 8, 65), (128, 8, 128), (128, 8, 129), (128, 8, 320), (128, 8, 384), (128, 8, 385), (128, 8, 450), (128, 24, 64), (128, 24, 66), (128, 64, 65),
    (64, 8, 65), (64, 8, 384), (64, 24, 385), (192, 8, 65), (192, 8, 256), (192, 8, 257), (256, 24, 65), (256, 8, 256), (256, 8, 257),
])
@pytest.mark.parametrize("window", [None, 700])
def test_every_head_finds_its_key(kernels, dim, page, pages, window):  # noqa: F811
    heads, dtype = 8, torch.bfloat16
    length = pages * page - 3
    batch, cell, per_request, layout = paged_case([length, 20], [1, 1], heads, heads, dim, page, dtype, shuffle_seed=pages + dim)
    q, k, v = per_request[0]
    seen = max(0, length - window) if window else 0
    # keys at the edges of registers of pages, of a wave's first steps, and the last ones
    edges = [at * page + offset for at in (0, 1, 63, 64, 65, 127, 128, 255, 256, 319, 320, 383, 384) for offset in (0, page - 1)] + [32 * 8, 32 * 16, length - 2, length - 1, seen]
    edges = sorted({at for at in edges if seen <= at < length})
    for first in range(0, len(edges), heads):
        mine = [edges[min(first + head, len(edges) - 1)] for head in range(heads)]
        keys = k.clone()
        for head, at in enumerate(mine):
            keys[at, head] = 3.0 * q[-1, head] * (128 / dim) ** 0.5
        case = [(q, keys, v), per_request[1]]
        _rewrite_cell(batch, cell, case, page, dtype)
        qkv = on_gpu(step_rows(case, [1, 1], heads, heads, dim), dtype)
        out = kernels[dtype].rotate_store_attend(qkv, layout, batch, cell, None, "none", 1.0, window).cpu().double().view(2, heads, dim)
        scores = torch.einsum("hd,khd->hk", rounded(q, dtype)[-1], rounded(keys, dtype)[seen:])
        want = torch.einsum("hk,khd->hd", scores.softmax(-1), rounded(v, dtype)[seen:])
        torch.testing.assert_close(out[0], want, **TOLERANCE[dtype])
        for head, at in enumerate(mine):
            torch.testing.assert_close(out[0, head], rounded(v, dtype)[at, head], atol=5e-2, rtol=0)
