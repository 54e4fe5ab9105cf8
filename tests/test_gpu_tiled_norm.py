"""Tiled products of more than 64 rows with a norm between them and no kernel for it (csrc/gemm_blocks.hip: OUT_NORM, OUT_SCALED), against the steps apart in 64 bits."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kernels():
    from llmserve_amd.kernels import HipKernels

    return HipKernels(torch.bfloat16)


def check(kernels, rows, width, inner, gated, bias=None, norm=torch.float32):
    """Both entries at these sizes, whatever the route takes; which shape the second has."""
    generator = torch.Generator(device="cuda").manual_seed(rows + width + gated)

    def some(*shape, scale=1.0):
        return scale * torch.randn(shape, generator=generator, device="cuda")

    entries = kernels._gemm_blocks
    x, hidden = some(rows, inner).bfloat16(), some(rows, width)
    w, weight = some(width, inner, scale=inner ** -0.5).bfloat16(), (1.0 + some(width, scale=0.1)).to(norm)
    b = some(width).to(bias) if bias else None
    both = some(2 * gated, width, scale=width ** -0.5).bfloat16()
    pieces, stride = entries.llmserve_gemm_blocks_norm_pieces(rows, width, inner), -(-rows // 4) * 4
    stream = torch.cat([hidden, torch.full((1, width), 7.0, device="cuda")])
    scaled = torch.full((rows + 1, width), float("nan"), device="cuda", dtype=torch.bfloat16)
    sums = torch.full((pieces + 1, stride), float("nan"), device="cuda")
    assert entries.llmserve_gemm_blocks_into_norm(
        x.data_ptr(), w.data_ptr(), b.data_ptr() if bias else None, int(bias == torch.float32), stream.data_ptr(), weight.data_ptr(), int(norm == torch.float32),
        scaled.data_ptr(), sums.data_ptr(), rows, width, inner, kernels._stream) == 0
    after = hidden.double() + x.double() @ w.double().T + (b.double() if bias else 0.0)
    assert ((stream[:rows].double() - after).abs() <= 8 * inner ** 0.5 * 2.0 ** -24 + 1e-6 * after.abs()).all() and (stream[rows] == 7.0).all()
    assert torch.equal(scaled[:rows], (stream[:rows] * weight.float()).bfloat16()) and scaled[rows].isnan().all()
    torch.testing.assert_close(sums[:pieces, :rows].double().sum(0), stream[:rows].double().square().sum(1), atol=0, rtol=64 * 2.0 ** -24)
    assert sums[pieces].isnan().all() and sums[:, rows:].isnan().all()
    out = torch.full((rows + 1, gated), float("nan"), device="cuda", dtype=torch.bfloat16)
    assert entries.llmserve_gemm_blocks_scaled(scaled.data_ptr(), sums.data_ptr(), pieces, 1e-6, both.data_ptr(), out.data_ptr(), rows, 2 * gated, width, kernels._stream) == 0
    after = stream[:rows].double()
    normed = after * torch.rsqrt(after.square().mean(-1, keepdim=True) + 1e-6) * weight.double()
    want, got = F.silu(normed @ both[::2].double().T) * (normed @ both[1::2].double().T), out[:rows].double()
    # three roundings to bfloat16, each of at most 2^-9 of its value: the rows into the gate (silu's slope is near one), into up, and the result
    assert (got - want).norm() < 3 * 2.0 ** -9 * want.norm()
    torch.testing.assert_close(got, want, atol=3e-2, rtol=3e-2)
    assert out[rows].isnan().all()
    return entries.llmserve_gemm_blocks_shape(rows, 2 * gated, width, 1, 2)


# rows at the edges of the tiles and of four; widths of one tile, of parts of one and of many, so that a thread adds up a few pieces or many; first products of
# every shape; gated widths that end inside a tile and a group
@pytest.mark.parametrize("rows", [65, 66, 96, 127, 160, 163, 321, 1030])
@pytest.mark.parametrize("width,inner,gated,bias,norm", [
    (128, 64, 96, torch.float32, torch.float32), (640, 320, 1001, None, torch.bfloat16), (1536, 1536, 8960, torch.bfloat16, torch.bfloat16), (2816, 448, 2004, None, torch.float32),
    (5120, 128, 520, None, torch.float32),
])
def test_linked(kernels, rows, width, inner, gated, bias, norm):
    check(kernels, rows, width, inner, gated, bias, norm)


# of every shape one, with rows and weights that leave remainders in it
@pytest.mark.parametrize("shape,rows,gated,width", [
    (0, 385, 12001, 128), (1, 2049, 4099, 128), (2, 641, 4099, 512), (3, 321, 6001, 512), (4, 129, 16389, 256), (5, 129, 12001, 512),
    (6, 97, 8197, 512), (7, 65, 8197, 256), (8, 65, 4099, 128), (9, 65, 131, 128), (10, 321, 4099, 512), (11, 321, 16389, 256),
])
def test_shapes_of_the_second_product(kernels, shape, rows, gated, width):
    assert check(kernels, rows, width, 128, gated) == shape


@pytest.mark.parametrize("columns,rows,width,inner", [(32, 159, 1536, 1536), (64, 319, 1536, 1536), (64, 323, 1536, 1536), (64, 1500, 2816, 1536), (96, 2047, 1536, 1536), (96, 639, 4096, 1536), (128, 1030, 3584, 1536), (128, 639, 5120, 1536)])
def test_shapes_of_the_first_product(kernels, columns, rows, width, inner):
    assert -(-width // kernels._gemm_blocks.llmserve_gemm_blocks_norm_pieces(rows, width, inner)) == columns
    check(kernels, rows, width, inner, 131)


@pytest.mark.parametrize("rows", [65, 128, 320, 2048])
def test_the_route(kernels, rows):
    """What `linear`, `add_rms_norm` and `gated_linear` give, within the roundings above; what the two refuse goes on to the three."""
    width, inner, gated = 1536, 1536, 8960
    generator = torch.Generator(device="cuda").manual_seed(rows)
    x, hidden = torch.randn(rows, inner, generator=generator, device="cuda").bfloat16(), torch.randn(rows, width, generator=generator, device="cuda")
    weight = torch.ones(width, device="cuda")
    project = kernels.prepare_linear([(torch.randn(width, inner, generator=generator, device="cuda") * inner ** -0.5).bfloat16()], None)
    reader = kernels.prepare_gated_linear(*((torch.randn(gated, width, generator=generator, device="cuda") * width ** -0.5).bfloat16() for _ in range(2)))
    apart = hidden.clone()
    want = kernels.gated_linear(kernels.add_rms_norm(apart, kernels.linear(x, project, out_dtype=torch.float32, partial=True), weight, 1e-6), reader).double()
    stream = hidden.clone()
    linked = kernels._linear_into_norm(x, None, project, kernels.norm_into(stream, weight, 1e-6, reader))
    assert linked is not None
    got = kernels.gated_linear(linked, reader).double()
    torch.testing.assert_close(stream, apart, atol=2e-5, rtol=1e-5)
    assert (got - want).norm() < 6 * 2.0 ** -9 * want.norm()
    for refused in (x.float(), x[:-1], x[:, :1408].contiguous(), torch.empty(rows * inner + 1, device="cuda", dtype=torch.bfloat16)[1:].view(rows, inner).copy_(x)):
        before = hidden.clone()
        assert kernels._linear_into_norm(refused, None, project, kernels.norm_into(before, weight, 1e-6, reader)) is None and torch.equal(before, hidden)
    assert kernels._linear_into_norm(x, None, project, kernels.norm_into(hidden.bfloat16(), weight, 1e-6, reader)) is None
