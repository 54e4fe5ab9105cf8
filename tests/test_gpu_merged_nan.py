"""NaN among key splits that the output projection merges (csrc/gemm_bf16.hip: gemm_merged): a run of keys that came out as no number is not a run
that saw no key.  It reaches its row, as it does where nothing is split or a kernel merges, and no other row."""

from __future__ import annotations

import math

import pytest
import torch

from tests.test_gpu_kernels import _rewrite_cell, kernels, on_gpu, paged_case, step_rows  # noqa: F401
from tests.test_gpu_linked_products import key_splits

pytestmark = pytest.mark.gpu


# heads for four, eight and twelve waves, one each and several; a sum of weights that is NaN, alone and under a score of +inf
@pytest.mark.parametrize("inner", [512, 1024, 1536, 2048])
@pytest.mark.parametrize("splits", [2, 3, 4, 6, 8])
def test_a_run_that_came_out_as_no_number(kernels, inner, splits):  # noqa: F811
    library, rows, width = kernels[torch.bfloat16], 7, 1536
    generator = torch.Generator(device="cuda").manual_seed(inner + splits)
    (pieces, pairs, _), _ = key_splits(rows, inner, splits, generator)
    weight = (inner ** -0.5 * torch.randn(width, inner, generator=generator, device="cuda")).bfloat16()
    project, hidden = library.prepare_linear([weight], None), torch.randn(rows, width, generator=generator, device="cuda")
    reader = library.prepare_gated_linear(*(torch.randn(1400, width, generator=generator, device="cuda").bfloat16() for _ in range(2)))

    def both(split):
        stream = hidden.clone()
        linked = library._linear_into_norm(None, split, project, library.norm_into(stream, torch.ones(width, device="cuda"), 1e-6, reader))
        out = torch.full((rows, width), 7.0, device="cuda")
        assert library._gemm_bf16.llmserve_gemm_merged(split[0].data_ptr(), split[1].data_ptr(), splits, weight.data_ptr(), None, 0, out.data_ptr(), rows, width, inner, 1,
                                                       library._stream) == 0
        return stream, linked.rows.float(), out

    sound = both((pieces, pairs, splits))
    assert all(bool(found.isfinite().all()) for found in sound)
    spoilt, hit = pairs.clone(), torch.zeros(rows, dtype=torch.bool, device="cuda")
    for row, head, top in ((0, 0, None), (3, inner // 128 - 1, math.inf), (6, inner // 256, None)):
        run = (splits - 1) * (row % 2 == 0)  # (of odd rows the last run has seen no key)
        spoilt[head, run, row, 1], hit[row] = math.nan, True
        if top is not None:
            spoilt[head, run, row, 0] = top
    for found, before in zip(both((pieces, spoilt, splits)), sound):
        assert bool(found[hit].isnan().all()) and torch.equal(found[~hit], before[~hit])


@pytest.mark.parametrize("planted", ["a key of NaN", "a score of +inf"])
@pytest.mark.parametrize("longest", [600, 2100])  # of which attention makes four runs and eight
def test_a_key_that_gives_no_number(kernels, planted, longest):  # noqa: F811
    """Through attention and the projection, merged by the product and by a kernel."""
    from llmserve_amd.kernels import HipKernels

    heads, kv_heads, dim, page, outer = 12, 2, 128, 16, 1536
    lengths, counts = [longest, longest - 77, 40], [1] * 3
    weight = torch.randn(outer, heads * dim) / math.sqrt(heads * dim)
    found = []
    for spoil in (False, True):
        batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, torch.bfloat16, shuffle_seed=longest)
        q, k, _ = per_request[1]
        if spoil:
            k[300, 1] = math.nan if planted == "a key of NaN" else 1e38 * q[-1, heads // kv_heads].sign()  # (of the second kv head, whose first head has this score)
        _rewrite_cell(batch, cell, per_request, page, torch.bfloat16)
        qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), torch.bfloat16)
        for merging in (True, False):
            library = HipKernels(torch.bfloat16)
            library.merge_in_product = merging
            out = library.rotate_store_attend(qkv.clone(), layout, batch, cell, None, "none", 0.3, None, project=library.prepare_linear([on_gpu(weight, torch.bfloat16)], None))
            found.append(out if out.ndim == 2 else out.sum(0))
    for merging, (before, after) in enumerate(zip(found[:2], found[2:])):
        assert bool(before.isfinite().all()) and bool(after[1].isnan().all()), merging
        assert torch.equal(after[[0, 2]], before[[0, 2]]), merging
