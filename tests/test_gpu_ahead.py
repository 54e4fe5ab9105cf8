"""Weights brought into the caches by workgroups of the kernel before their product (csrc/common.h: Ahead): results are the same bits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kernels():
    from llmserve_amd.kernels import HipKernels

    return HipKernels(torch.bfloat16)


# weights of fewer runs than there are chiplets, of a run that no row fills, of runs of 16 bytes' multiples that are no power of two, and
# one too large to be brought whole; rows up to where it ends
@pytest.mark.parametrize("rows", [1, 8, 63, 64, 65, 300])
@pytest.mark.parametrize("out_features,in_features", [(8, 64), (16, 72), (120, 1000), (2048, 1536), (4608, 3584)])
def test_norm_with_a_weight_ahead(kernels, rows, out_features, in_features):
    generator = torch.Generator(device="cuda").manual_seed(rows + in_features)
    hidden, parts = (torch.randn(shape, generator=generator, device="cuda") for shape in ((rows, in_features), (3, rows, in_features)))
    norm = torch.ones(in_features, device="cuda", dtype=torch.bfloat16)
    weight = torch.randn(out_features, in_features, generator=generator, device="cuda").bfloat16()
    ahead, kept = kernels.prepare_linear([weight.clone()], None), weight
    brought = kernels._whole_ahead(ahead, rows, rows)[0]
    assert (brought > 0) == (rows <= 64 and 16 <= out_features and out_features * in_features <= 1 << 22)
    results = []
    for told in (None, ahead):
        stream = hidden.clone()
        results.append((kernels.add_rms_norm(stream, parts, norm, 1e-6, ahead=told), stream))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    assert torch.equal(ahead.weight, kept)


def test_refused(kernels):
    from llmserve_amd.kernels.hip import _pointer

    hidden, out = torch.randn(2, 64, device="cuda"), torch.empty(2, 64, device="cuda", dtype=torch.bfloat16)
    norm, weight = (torch.ones(n, device="cuda", dtype=torch.bfloat16) for n in (64, 4096))

    def status(*ahead):
        return kernels._elementwise.llmserve_add_rms_norm(_pointer(hidden), None, 1, _pointer(norm), 0, _pointer(out), 0, 2, 64, 1e-6, *ahead, kernels._stream)

    assert status(0, None, 0, 0) == 0
    assert status(4, weight.data_ptr(), 64, 128) == 0
    for ahead in ((-1, weight.data_ptr(), 64, 128), (4, None, 64, 128), (4, weight.data_ptr() + 8, 64, 1), (4, weight.data_ptr(), 24, 1),
                  (4, weight.data_ptr(), 0, 1), (4, weight.data_ptr(), 64, 0), (4, weight.data_ptr(), 1 << 30, 2)):
        assert status(*ahead) == 1001
