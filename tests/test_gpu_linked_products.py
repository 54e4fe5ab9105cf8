"""Two products with a norm between them and no kernel for it (`HipKernels._linear_into_norm`), against the three apart in 64 bits."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kernels():
    from llmserve_amd.kernels import HipKernels

    return HipKernels(torch.bfloat16)


def check_linked(kernels, rows, width, inner, gated, bias=False, norm=torch.float32):
    """The two linked products against the three steps apart in 64 bits; False where they are of other kernels (and nothing has been done)."""
    generator = torch.Generator(device="cuda").manual_seed(rows + width)

    def some(*shape, scale=1.0):
        return scale * torch.randn(shape, generator=generator, device="cuda")

    x, hidden = some(rows, inner).bfloat16(), some(rows, width)
    w, b = some(width, inner, scale=inner ** -0.5).bfloat16(), some(width).bfloat16() if bias else None
    weight = (1.0 + some(width, scale=0.1)).to(norm)
    gate, up = (some(gated, width, scale=width ** -0.5).bfloat16() for _ in range(2))
    project = kernels.prepare_linear([w], [b] if bias else None)
    reader = kernels.prepare_gated_linear(gate, up)
    stream = hidden.clone()
    scaled = kernels._linear_into_norm(x, None, project, kernels.norm_into(stream, weight, 1e-6, reader))
    if scaled is None:
        assert torch.equal(stream, hidden)
        return False
    got = kernels.gated_linear(scaled, reader).double()
    after = hidden.double() + x.double() @ w.double().T + (b.double() if bias else 0.0)
    # float32 sums of `inner` products of values of size 1
    torch.testing.assert_close(stream.double(), after, atol=8 * inner ** 0.5 * 2.0 ** -24, rtol=1e-6)
    normed = after * torch.rsqrt((after * after).mean(-1, keepdim=True) + 1e-6) * weight.double()
    want = F.silu(normed @ gate.double().T) * (normed @ up.double().T)
    # three roundings to bfloat16, each of at most 2^-9 of its value: the rows into the gate (silu's slope is near one), into up, and
    # the result; in norm no more than their sum
    assert (got - want).norm() < 3 * 2.0 ** -9 * want.norm()
    torch.testing.assert_close(got, want, atol=3e-2, rtol=3e-2)
    return True


# rows at the edges of the kernels' tiles; widths whose tiles of 16 columns divide evenly over the threads and not; gated products for
# the kernel for few rows (short and long K), and for the ring with four, five and ten tiles a workgroup
@pytest.mark.parametrize("rows", [1, 3, 8, 15, 16, 17, 31, 33, 64])
@pytest.mark.parametrize("width,inner,gated,bias,norm", [
    (128, 128, 96, True, torch.float32), (384, 256, 200, False, torch.bfloat16), (1536, 1536, 8960, False, torch.bfloat16),
    (1664, 896, 9000, True, torch.bfloat16), (3584, 3584, 18944, False, torch.bfloat16),
])
def test_linked_products(kernels, rows, width, inner, gated, bias, norm):
    taken = check_linked(kernels, rows, width, inner, gated, bias, norm)
    assert taken or rows > 16 or gated > 10000 or width == 3584


@pytest.mark.parametrize("rows", [33, 48, 64])
@pytest.mark.parametrize("width,inner,gated", [(256, 128, 10336), (2048, 2048, 11008)])
def test_six_weight_tiles_beside_four_of_x(kernels, rows, width, inner, gated):
    """The ring whose stages fill a CU's LDS to the last byte: the second product has no more of it than without a norm."""
    assert kernels._ring_shape(rows, 2 * gated, width, False)[0] == 6
    assert check_linked(kernels, rows, width, inner, gated)


def test_what_is_not_linked(kernels):
    """Rows, widths and activations that the linked kernels do not take: nothing is done, and the caller goes on as before."""
    def linked(rows, width, inner, gated, activation="silu"):
        x, hidden = torch.randn(rows, inner, device="cuda").bfloat16(), torch.randn(rows, width, device="cuda")
        project = kernels.prepare_linear([torch.randn(width, inner, device="cuda").bfloat16()], None)
        reader = kernels.prepare_gated_linear(*(torch.randn(gated, width, device="cuda").bfloat16() for _ in range(2)), activation)
        before = hidden.clone()
        result = kernels._linear_into_norm(x, None, project, kernels.norm_into(hidden, torch.ones(width, device="cuda"), 1e-6, reader))
        assert result is not None or torch.equal(hidden, before)
        return result

    assert linked(4, 256, 128, 96) is not None
    assert linked(65, 256, 128, 96) is None
    assert linked(4, 200, 128, 96) is None
    assert linked(4, 256, 96, 96) is None
    assert linked(4, 256, 128, 96, "relu") is None
