"""What the fused decode step's loads of angles reach (csrc/attention_bf16.hip: angle_piece), asked of the built libraries (no GPU needed)."""

from __future__ import annotations

import pytest

from llmserve_amd.kernels.build import load_module
from llmserve_amd.kernels.variants import DEFAULT_VARIANTS


@pytest.mark.parametrize("dim", [defines["HEAD_DIM"] for defines in DEFAULT_VARIANTS["attention_bf16"]])
def test_angles_lie_in_their_rows(dim):
    """The table's rows are D / 2 pairs of float32.  A step that turns nothing makes the same loads of its rows of q, k and v, of which the narrowest are one head each."""
    library = load_module("attention_bf16", {"HEAD_DIM": dim})
    assert library.llmserve_attention_can_fuse(0) and library.llmserve_attention_angle_bytes(0) <= 3 * dim * 2
    for pairing in (1, 2):
        if library.llmserve_attention_can_fuse(pairing):
            assert library.llmserve_attention_angle_bytes(pairing) == 4 * dim
