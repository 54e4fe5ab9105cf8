"""Whether more than 64 rows go through two products with a norm between them (`HipKernels._tiles_into_norm`) is asked once for each size: a step of more than 512 tokens is
launched kernel by kernel, and every question is the host's time in every layer."""

from __future__ import annotations

import pytest
import torch

from llmserve_amd.kernels.build import load_module
from llmserve_amd.kernels.hip import HipKernels, LinearWeights, _norm_pieces
from tests.test_routing import on_the_host


class Blocks:
    """The tiled kernel's host side, with what it is asked; its launches do nothing."""

    def __init__(self):
        self.asked, self.library = [], load_module("gemm_blocks")

    def __getattr__(self, name):
        def entry(*arguments):
            self.asked.append(name)
            return getattr(self.library, name)(*arguments) if "norm_" in name and "into" not in name else 0

        return entry


@pytest.mark.parametrize("rows,width,inner,taken", [(513, 1536, 8960, False), (640, 1536, 8960, True), (96, 1536, 8960, True), (96, 3584, 18944, False), (700, 896, 4864, False)])
def test_sizes_are_asked_for_once(rows, width, inner, taken):
    blocks = Blocks()
    kernels = on_the_host(_gemm_blocks=blocks)
    project, weight = LinearWeights(torch.empty(width, width, dtype=torch.bfloat16), None), torch.ones(width)
    reader = kernels.prepare_gated_linear(*(torch.empty(inner, width, dtype=torch.bfloat16) for _ in range(2)))
    x, hidden = torch.empty(rows, width, dtype=torch.bfloat16), torch.empty(rows, width)
    for again in range(3):
        linked = kernels.linear_into(x, project, kernels.norm_into(hidden, weight, 1e-6, reader))
        assert (linked is not None) == taken
        assert blocks.asked.count("llmserve_gemm_blocks_norm_cost") <= 1 and blocks.asked.count("llmserve_gemm_blocks_norm_pieces") <= 1
    assert blocks.asked.count("llmserve_gemm_blocks_into_norm") == 3 * taken


def test_answers_are_those_of_the_routes_apart():
    """Both products the tiled kernel's, as `_streaming` has it where the BLAS library is there."""
    library = load_module("gemm_blocks")
    for rows in (65, 96, 128, 129, 320, 513, 700, 2048):
        for width, inner, gated in ((1536, 1536, 17920), (2048, 2048, 22016), (896, 896, 9728), (3584, 3584, 37888), (1000, 1536, 4096)):
            both = HipKernels._tiled_ahead(rows, width, inner, False, True) and HipKernels._tiled_ahead(rows, gated, width, True, False) and width % 128 == 0
            for most in (-1, HipKernels._TILES_INTO_NORM, 1 << 29):
                pieces = _norm_pieces(library, rows, width, inner, gated, most)
                assert bool(pieces) == (both and library.llmserve_gemm_blocks_norm_cost(rows, width, inner) <= most)
                assert pieces in (0, library.llmserve_gemm_blocks_norm_pieces(rows, width, inner))


@pytest.mark.parametrize("rows,inner,taken", [(24, 2048, True), (32, 2048, True), (33, 2048, False), (64, 1664, False), (64, 1536, True), (40, 1280, True), (96, 1536, True)])
def test_steps_with_portions(rows, inner, taken):
    """Both sides of the line that `_links_beside_portions` draws; a step of single tokens links at these sizes of up to 64 rows whatever K."""
    kernels = on_the_host(_gemm_blocks=Blocks())
    width, gated = 1536, 8960
    project, weight = LinearWeights(torch.empty(width, inner, dtype=torch.bfloat16), None), torch.ones(width)
    reader = kernels.prepare_gated_linear(*(torch.empty(gated, width, dtype=torch.bfloat16) for _ in range(2)))
    into = kernels.norm_into(torch.empty(rows, width), weight, 1e-6, reader)
    x = torch.empty(rows, inner, dtype=torch.bfloat16)
    assert (kernels.linear_into(x, project, into) is not None) == taken
    assert rows > 64 or kernels._linear_into_norm(x, None, project, into) is not None
