"""Operands of a product into a norm that begin inside a piece of 16 bytes (`HipKernels._linear_into_norm`): its kernels, and its reader's, bring whole
pieces, so such operands go to the steps apart."""

from __future__ import annotations

import pytest
import torch

from llmserve_amd.kernels.hip import LinearWeights
from tests.test_routing import on_the_host

FORMS = ["x", "a view of x", "weight", "stream", "norm", "reader"]


def operands(form, rows, width, inner, gated, device, generator=None):
    """x, the first product's weight, the stream, the norm's weight, gate and up in one, all in whole pieces but for `form`."""
    def some(name, *shape, dtype=torch.bfloat16):
        count = shape[0] * shape[1] if len(shape) == 2 else shape[0]
        values = torch.randn(count + 8, generator=generator, device=device).mul_(shape[-1] ** -0.5 if name in ("weight", "reader") else 1.0).to(dtype)
        return (values[1:-7] if form == name else values[:-8]).view(shape)

    x = some("x", rows, inner)
    if form == "a view of x":
        x = torch.cat([x, x], 1)[:, :inner]
    return x, some("weight", width, inner), some("stream", rows, width, dtype=torch.float32), some("norm", width, dtype=torch.float32), some("reader", 2 * gated, width)


def linked(kernels, x, weight, stream, norm, both):
    reader = kernels.prepare_gated_linear(both[::2], both[1::2])
    reader.both.weight = both
    return kernels._linear_into_norm(x, None, LinearWeights(weight, None), kernels.norm_into(stream, norm, 1e-6, reader)), reader


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("rows", [3, 24])
def test_such_operands_are_left_to_the_steps_apart(rows, form):
    kernels = on_the_host()
    assert linked(kernels, *operands(None, rows, 1536, 1280, 1400, "cpu"))[0] is not None and kernels._gemm_bf16.count == 1
    assert linked(kernels, *operands(form, rows, 1536, 1280, 1400, "cpu"))[0] is None and kernels._gemm_bf16.count == 1


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS[2:])  # (the entry points take pointers, so a view is the caller's to see)
def test_the_entry_points_refuse_them(form):
    from llmserve_amd.kernels import HipKernels

    kernels, width, inner, gated = HipKernels(torch.bfloat16), 1536, 1280, 1400
    for rows in (3, 24):
        x, weight, stream, norm, both = operands(form, rows, width, inner, gated, "cuda")
        before, scaled, sums = stream.clone(), torch.zeros(rows, width, device="cuda", dtype=torch.bfloat16), torch.zeros(width // 16, 32, device="cuda")
        out = torch.zeros(rows, gated, device="cuda", dtype=torch.bfloat16)
        library = kernels._gemm_bf16
        status = library.llmserve_gemm_into_norm(x.data_ptr(), None, None, 0, weight.data_ptr(), None, 0, stream.data_ptr(), norm.data_ptr(), 1, scaled.data_ptr(), sums.data_ptr(),
                                                 rows, width, inner, 0, None, 0, 0, kernels._stream)
        assert (status == 1001) == (form != "reader") and (form == "reader" or torch.equal(stream, before))
        status = library.llmserve_gemm_scaled(scaled.data_ptr(), sums.data_ptr(), 1e-6, both.data_ptr(), out.data_ptr(), 0 if rows <= 16 else 2, rows, 2 * gated, width, kernels._stream)
        assert (status == 1001) == (form == "reader")
        torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["x", "weight", "stream", "norm"])
@pytest.mark.parametrize("rows", [3, 24])
def test_the_steps_apart_take_them(rows, form):
    """What a model's step then computes, against 64 bits, where the library behind `linear` has a way for them."""
    from llmserve_amd.kernels import HipKernels

    kernels, width, inner, gated = HipKernels(torch.bfloat16), 1536, 1280, 1400
    x, weight, stream, norm, both = operands(form, rows, width, inner, gated, "cuda", torch.Generator(device="cuda").manual_seed(rows))
    after = stream.double() + x.double() @ weight.double().T
    scaled, reader = linked(kernels, x, weight, stream, norm, both)
    assert scaled is None
    got = kernels.gated_linear(kernels.add_rms_norm(stream, kernels.linear(x, LinearWeights(weight, None), out_dtype=torch.float32, partial=True), norm, 1e-6), reader).double()
    # float32 sums of `inner` products of values of size 1
    assert ((stream.double() - after).abs() <= 8 * inner ** 0.5 * 2.0 ** -24 + 1e-6 * after.abs()).all()
    normed = after * torch.rsqrt(after.square().mean(-1, keepdim=True) + 1e-6) * norm.double()
    want = torch.nn.functional.silu(normed @ both[::2].double().T) * (normed @ both[1::2].double().T)
    # three roundings to bfloat16, each of at most 2^-9 of its value
    assert (got - want).norm() < 3 * 2.0 ** -9 * want.norm()
