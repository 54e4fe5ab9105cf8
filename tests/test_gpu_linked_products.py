"""Two products with a norm between them and no kernel for it (`HipKernels._linear_into_norm`), against the three apart in 64 bits."""

from __future__ import annotations

import math

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kernels():
    from llmserve_amd.kernels import HipKernels

    return HipKernels(torch.bfloat16)


def key_splits(rows, inner, splits, generator):
    """What decode attention leaves of `rows` rows of inner / 128 heads in `splits` runs of keys, as the product reads it, and the rows
    that they merge to in 64 bits.  The last run of every second row has seen no key, and holds whatever was there."""
    heads = inner // 128
    x = torch.randn(heads, splits, rows, 128, generator=generator, device="cuda").bfloat16()
    highest = 4.0 * torch.randn(heads, splits, rows, generator=generator, device="cuda")
    weight = 0.5 + 20.0 * torch.rand(heads, splits, rows, generator=generator, device="cuda")
    highest[:, -1, 1::2] = -math.inf
    x[:, -1, 1::2] = math.nan
    held = torch.full((heads, splits, 16, 128), math.nan, dtype=torch.bfloat16, device="cuda")
    held[:, :, :rows] = x
    pairs = torch.full((heads, splits, 16, 2), math.nan, device="cuda")
    pairs[:, :, :rows] = torch.stack([highest, weight], -1)
    shares = weight.double() * torch.exp2(highest.double() - highest.double().amax(1, keepdim=True))
    merged = (x.double().nan_to_num() * (shares / shares.sum(1, keepdim=True))[..., None]).sum(1)
    pieces = held.unflatten(-1, (16, 8)).transpose(2, 3).contiguous()  # [heads, splits, 16 pieces, 16 rows, 8]
    return (pieces, pairs, splits), merged.transpose(0, 1).flatten(1)


def check_linked(kernels, rows, width, inner, gated, bias=False, norm=torch.float32, splits=0):
    """The two linked products against the three steps apart in 64 bits; the shape of the second's kernel (0: the one for few rows, else
    weight tiles of the ring's), or None where the products are of other kernels and nothing has been done."""
    generator = torch.Generator(device="cuda").manual_seed(rows + width)

    def some(*shape, scale=1.0):
        return scale * torch.randn(shape, generator=generator, device="cuda")

    x, hidden = some(rows, inner).bfloat16(), some(rows, width)
    w, b = some(width, inner, scale=inner ** -0.5).bfloat16(), some(width).bfloat16() if bias else None
    weight = (1.0 + some(width, scale=0.1)).to(norm)
    gate, up = (some(gated, width, scale=width ** -0.5).bfloat16() for _ in range(2))
    project = kernels.prepare_linear([w], [b] if bias else None)
    reader = kernels.prepare_gated_linear(gate, up)
    split, merged = key_splits(rows, inner, splits, generator) if splits else (None, x.double())
    stream = hidden.clone()
    scaled = kernels._linear_into_norm(None if splits else x, split, project, kernels.norm_into(stream, weight, 1e-6, reader))
    if scaled is None:
        assert torch.equal(stream, hidden)
        return None
    after = hidden.double() + merged @ w.double().T + (b.double() if bias else 0.0)
    # float32 sums of `inner` products of values of size 1; merged rows are rounded to bfloat16 besides, by 2^-9 of a value at the most: that
    # bounds a result's error by 2^-9 of the sum of its products' sizes, and, the roundings being independent, all results' errors
    # together by 2^-9 of the roots of their squares' sums
    error = (stream.double() - after).abs()
    sums = 8 * inner ** 0.5 * 2.0 ** -24 + 1e-6 * after.abs()
    if splits:
        assert (error <= sums + 1.001 * 2.0 ** -9 * (merged.abs() @ w.double().abs().T)).all()
        assert error.norm() < 2.0 ** -9 * (merged.square() @ w.double().square().T).sqrt().norm()
    else:
        assert (error <= sums).all()
    assert torch.equal(scaled.rows, (stream * weight.float()).bfloat16())
    squares = (stream.double() ** 2).unflatten(1, (-1, 16)).sum(-1).T
    torch.testing.assert_close(scaled.sums[: width // 16, :rows].double(), squares, atol=0, rtol=16 * 2.0 ** -24)
    got = kernels.gated_linear(scaled, reader).double()
    after = stream.double()
    normed = after * torch.rsqrt((after * after).mean(-1, keepdim=True) + 1e-6) * weight.double()
    want = F.silu(normed @ gate.double().T) * (normed @ up.double().T)
    # three roundings to bfloat16, each of at most 2^-9 of its value: the rows into the gate (silu's slope is near one), into up, and
    # the result; in norm no more than their sum
    assert (got - want).norm() < 3 * 2.0 ** -9 * want.norm()
    torch.testing.assert_close(got, want, atol=3e-2, rtol=3e-2)
    return scaled.tiles


ROWS = [1, 3, 8, 15, 16, 17, 31, 33, 64]  # at the edges of the kernels' tiles


# widths whose tiles of 16 columns divide evenly over the threads and not; gated products for the kernel for few rows (short and long K)
# and for the ring with five, six and ten tiles a workgroup; small ones over more than 16 rows and large first products are of other kernels
@pytest.mark.parametrize("rows,at", [(rows, at) for at, rows in enumerate(ROWS)])
@pytest.mark.parametrize("width,inner,gated,bias,norm,taken", [
    (128, 128, 96, True, torch.float32, [0] * 5 + [None] * 4),
    (384, 256, 200, False, torch.bfloat16, [0] * 5 + [None] * 4),
    (1536, 1536, 8960, False, torch.bfloat16, [0, 0, 0, 6, 6, 6, 6, 5, 5]),
    (1664, 896, 9000, True, torch.bfloat16, [0, 0, 0, 6, 6, 6, 6, 5, 5]),
    (3584, 3584, 18944, False, torch.bfloat16, [0, 0, 10, 10, 10] + [None] * 4),
])
def test_linked_products(kernels, rows, at, width, inner, gated, bias, norm, taken):
    assert check_linked(kernels, rows, width, inner, gated, bias, norm) == taken[at]


# every shape of the ring that the second product can have, with two tiles of x and with four, at gated products that leave remainders
@pytest.mark.parametrize("width,gated,tiles", [
    (3584, 2500, (2, 2, 2)), (1536, 5540, (4, 4, 4)), (1024, 8260, (6, 6, 5)), (1024, 12420, (8, 8, 8)), (512, 16420, (10, 10, 10)),
    (512, 20580, (12, 12, 12)), (512, 24740, (14, 14, 14)), (1536, 1380, (0, 2, 2)), (512, 4258, (0, 4, 4)), (256, 8262, (0, 6, 5)),
    (256, 12418, (0, 8, 8)), (128, 16422, (0, 10, 10)), (128, 20581, (0, 12, 12)), (128, 24741, (0, 14, 14)), (256, 10341, (0, 6, 6)),
])
def test_linked_products_of_every_ring_shape(kernels, width, gated, tiles):
    for rows, expected in zip((16, 17, 32, 33, 64), (tiles[0], tiles[1], tiles[1], tiles[2], tiles[2])):
        assert check_linked(kernels, rows, width, 128, gated) == expected, rows


@pytest.mark.parametrize("rows", [33, 48, 64])
@pytest.mark.parametrize("width,inner,gated", [(256, 128, 10336), (2048, 2048, 11008)])
def test_six_weight_tiles_beside_four_of_x(kernels, rows, width, inner, gated):
    """The ring whose stages fill a CU's LDS to the last byte: the second product has no more of it than without a norm."""
    assert check_linked(kernels, rows, width, inner, gated) == 6


# up to four heads of K (four waves), eight (eight waves), more (twelve, a head each or two and three)
@pytest.mark.parametrize("inner", [128, 512, 640, 1024, 1536, 3584])
@pytest.mark.parametrize("splits", [2, 3, 4, 6, 8])
def test_linked_products_of_unmerged_key_splits(kernels, inner, splits):
    for rows in (1, 3, 15, 16):
        assert check_linked(kernels, rows, 1536, inner, 1400, bias=rows % 3 == 0, splits=splits) == 0, rows


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
