"""How much of gate and up is brought beside the projection that merges key splits (`HipKernels._merging_ahead`), at sizes on both sides of its lines."""

from __future__ import annotations

import pytest

from llmserve_amd.kernels.hip import HipKernels


@pytest.mark.parametrize("width,heads,inner,each", [
    # KB a workgroup that brings; None: all of it
    (1152, 9, 6528, 128), (1280, 10, 7680, 128), (1536, 12, 8960, 132), (1792, 14, 7168, 154), (2048, 16, 8192, 176), (2560, 12, 9216, 132),
    (1536, 12, 5120, None), (1792, 14, 4352, None), (2048, 16, 3840, None), (768, 6, 4096, None), (2560, 12, 3072, 132),
])
def test_as_much_as_was_measured_to_pay(width, heads, inner, each):
    size, busy = 2 * 2 * inner * width, width // 16
    assert HipKernels._merging_ahead(busy, 128 * heads, size) == (size if each is None else (256 - busy) * (each << 10))


def test_nothing_where_no_workgroup_is_left():
    assert all(HipKernels._merging_ahead(busy, 1536, 1 << size) == 0 for busy in (256, 257, 400) for size in (1, 20, 30))
