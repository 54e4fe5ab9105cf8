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


def told_or_not(monkeypatch, kernels, run):
    """What `run` gives where the kernels are told of the next weight and where they are not; and how many workgroups brought it."""
    found, brought = [], []
    for told in (True, False):
        with monkeypatch.context() as patch:
            own = type(kernels)._ahead

            def ahead(self, *arguments):
                answer = own(self, *arguments) if told else (0, None, 0, 0)
                brought.append(answer[0])
                return answer

            patch.setattr(type(kernels), "_ahead", ahead)
            found.append(run())
    return found, max(brought, default=0)


# the fused step of single tokens: splits that are merged by a kernel and by the projection, sinks and chunks; few and many workgroups (fewer than the
# chip's 256, or nothing is brought), a weight of fewer runs than chiplets, and one that is too large
@pytest.mark.parametrize("heads,kv_heads,dim,width,lengths,options", [
    (12, 2, 128, 1536, [640], {}), (12, 2, 128, 1536, [640, 3, 17, 1, 90, 33, 200, 11], {}), (12, 2, 128, 1536, list(range(1, 65)), {}),
    (4, 1, 64, 96, [5, 300, 41], {}), (2, 2, 96, 3000, [70] * 5, {}), (28, 4, 128, 3584, [100, 7], {}), (8, 2, 64, 512, [20, 200], {"sinks": True}),
    (8, 2, 64, 512, [20, 200], {"chunk": 64}),
])
def test_attention_with_a_weight_ahead(kernels, monkeypatch, heads, kv_heads, dim, width, lengths, options):
    from tests.test_gpu_kernels import paged_case, step_rows

    dtype, counts = torch.bfloat16, [1] * len(lengths)
    generator = torch.Generator(device="cuda").manual_seed(width + len(lengths))
    project = kernels.prepare_linear([(torch.randn(width, heads * dim, generator=generator, device="cuda") * (heads * dim) ** -0.5).bfloat16()], None)
    inverse = (1.0 / (3000.0 ** (torch.arange(0, dim, 2).float() / dim))).cuda()
    options = dict(options, sinks=torch.randn(heads, generator=generator, device="cuda")) if "sinks" in options else options

    def run():
        batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, 16, dtype, shuffle_seed=dim)
        qkv = step_rows(per_request, counts, heads, kv_heads, dim).to("cuda", dtype)
        out = kernels.rotate_store_attend(qkv, layout, batch, cell, inverse, "adjacent", dim ** -0.5, None, project=project, **options)
        return out, cell.keys.float().nan_to_num(7e7), cell.values.float().nan_to_num(7e7)

    (told, not_told), brought = told_or_not(monkeypatch, kernels, run)
    assert all(torch.equal(a, b) for a, b in zip(told, not_told))
    assert (brought > 0) == (width * heads * dim <= 1 << 22)


@pytest.mark.parametrize("rows", [1, 8, 16])
@pytest.mark.parametrize("width,inner,gated,splits", [(128, 128, 96, 2), (1536, 1536, 8960, 8), (384, 256, 200, 3), (1536, 1536, 1380, 6)])
def test_merging_projection_with_a_weight_ahead(kernels, monkeypatch, rows, width, inner, gated, splits):
    from tests.test_gpu_linked_products import key_splits

    generator = torch.Generator(device="cuda").manual_seed(rows + width)
    some = lambda *shape: (torch.randn(shape, generator=generator, device="cuda") * shape[-1] ** -0.5).bfloat16()
    project, reader = kernels.prepare_linear([some(width, inner)], None), kernels.prepare_gated_linear(some(gated, width), some(gated, width))
    hidden, norm = torch.randn(rows, width, generator=generator, device="cuda"), torch.ones(width, device="cuda")
    split, _ = key_splits(rows, inner, splits, generator)

    def run():
        stream = hidden.clone()
        scaled = kernels._linear_into_norm(None, split, project, kernels.norm_into(stream, norm, 1e-6, reader))
        return stream, scaled.rows, scaled.sums[: width // 16, :rows], kernels.gated_linear(scaled, reader)

    (told, not_told), brought = told_or_not(monkeypatch, kernels, run)
    assert all(torch.equal(a, b) for a, b in zip(told, not_told)) and brought > 0


def test_refused_by_the_merging_projection(kernels):
    """Bad runs, and workgroups that bring beside the projection that merges nothing."""
    from llmserve_amd.kernels.hip import _pointer
    from tests.test_gpu_linked_products import key_splits

    rows, width, inner = 2, 128, 128
    generator = torch.Generator(device="cuda").manual_seed(5)
    (split_x, split_ml, splits), _ = key_splits(rows, inner, 2, generator)
    x, weight, scaled = (torch.zeros(n, inner, device="cuda", dtype=torch.bfloat16) for n in (rows, width, rows))
    hidden, norm, sums = torch.zeros(rows, width, device="cuda"), torch.ones(width, device="cuda"), torch.zeros(16, 16, device="cuda")

    def status(merging, *ahead):
        return kernels._gemm_bf16.llmserve_gemm_into_norm(
            None if merging else _pointer(x), _pointer(split_x) if merging else None, _pointer(split_ml) if merging else None, splits if merging else 0,
            _pointer(weight), None, 0, _pointer(hidden), _pointer(norm), 1, _pointer(scaled), _pointer(sums), rows, width, inner, *ahead, kernels._stream)

    good = (3, weight.data_ptr(), 512, 64)
    assert status(True, *good) == 0 and status(False, 0, None, 0, 0) == 0 and status(False, *good) == 1001
    for wrong in ((-1, *good[1:]), (3, None, 512, 64), (3, weight.data_ptr() + 8, 512, 1), (3, weight.data_ptr(), 24, 1), (3, weight.data_ptr(), 512, 0)):
        assert status(True, *wrong) == 1001
