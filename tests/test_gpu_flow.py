"""Products of up to 16 rows that stream whole cache lines of the weight (csrc/gemm_bf16.hip: gemm_flow), against the plain product in 64 bits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kernels():
    from llmserve_amd.kernels import HipKernels

    return HipKernels(torch.bfloat16)


# rows of x at the edges of one and two eights; weight rows that leave every number of eights a workgroup (8 to 40 rows each), an odd last one, fewer
# than eight, small weights and large; K of fewer units than waves, and units that the waves share unevenly; parts of K
@pytest.mark.parametrize("rows", [1, 7, 8, 9, 16])
@pytest.mark.parametrize("outer,inner,splits", [
    (5, 64, 1), (1001, 128, 1), (2049, 192, 1), (4098, 1088, 1), (17921, 320, 1), (6146, 1536, 1), (9219, 960, 1), (20000, 832, 1), (38402, 576, 1), (300, 8960, 5), (1536, 5120, 8),
])
def test_flowing_products(kernels, rows, outer, inner, splits):
    generator = torch.Generator(device="cuda").manual_seed(rows + outer)
    x, w = (torch.randn(n, inner, generator=generator, device="cuda").bfloat16() for n in (rows, outer))
    bias = torch.randn(outer, generator=generator, device="cuda")
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    entry = kernels._gemm_bf16.llmserve_gemm_skinny
    # float32 sums of `inner` products, each rounding of at most 2^-24 of a partial sum, itself at most the sum of sizes: by far less than so many in a row
    bound = inner * 2.0 ** -24 * size

    out = torch.full((splits, rows, outer), float("nan"), device="cuda")
    assert entry(x.data_ptr(), w.data_ptr(), bias.data_ptr(), 1, out.data_ptr(), 1, 0, rows, outer, inner, splits, kernels._stream) == 0
    assert ((out.double().sum(0) - want - bias.double()).abs() <= bound + 2.0 ** -22 * (want + bias.double()).abs() + 1e-6).all()
    if splits > 1:
        return
    rounding = lambda exact: 2.0 ** -8 * exact.abs() + 1e-6  # half a unit of bfloat16's eight bits, twice over for the sums' own error
    short = torch.full((rows, outer), float("nan"), device="cuda", dtype=torch.bfloat16)
    assert entry(x.data_ptr(), w.data_ptr(), None, 0, short.data_ptr(), 0, 0, rows, outer, inner, 1, kernels._stream) == 0
    assert ((short.double() - want).abs() <= bound + rounding(want)).all()
    even = outer // 2 * 2
    gate, up = want[:, 0:even:2], want[:, 1:even:2]
    for gated, exact in ((1, torch.nn.functional.silu(gate) * up), (2, gate.relu() * up)):
        short = torch.full((rows, even // 2), float("nan"), device="cuda", dtype=torch.bfloat16)
        assert entry(x.data_ptr(), w.data_ptr(), None, 0, short.data_ptr(), 0, gated, rows, even, inner, 1, kernels._stream) == 0
        # (silu's slope is at most 1.1)
        moved = 1.1 * bound[:, 0:even:2] * (up.abs() + bound[:, 1:even:2]) + bound[:, 1:even:2] * gate.abs()
        assert ((short.double() - exact).abs() <= moved + rounding(exact)).all()
    first = outer // 3
    left, right = torch.full((rows, first), float("nan"), device="cuda", dtype=torch.bfloat16), torch.full((rows, outer - first + 3), 7.0, device="cuda", dtype=torch.bfloat16)
    status = kernels._gemm_bf16.llmserve_gemm_skinny_tail(x.data_ptr(), w.data_ptr(), None, 0, left.data_ptr() if first else None, first, right.data_ptr(), right.shape[1],
                                                          rows, outer, inner, kernels._stream)
    assert status == 0 and (right[:, outer - first :] == 7.0).all()
    assert ((left.double() - want[:, :first]).abs() <= (bound + rounding(want))[:, :first]).all()
    squared, off = want[:, first:].relu() ** 2, bound[:, first:]
    assert ((right[:, : outer - first].double() - squared).abs() <= off * (2 * want[:, first:].abs() + off) + rounding(squared)).all()


@pytest.mark.parametrize("shift_x,shift_w", [(4, 0), (0, 2)])
def test_operands_that_begin_inside_a_piece_go_to_the_other_kernel(kernels, shift_x, shift_w):
    rows, outer, inner = 3, 530, 640
    x, w = (torch.randn(n * inner + 8, device="cuda").bfloat16()[shift : shift + n * inner].view(n, inner) for n, shift in ((rows, shift_x), (outer, shift_w)))
    got = kernels.linear(x, kernels.prepare_linear([w], None), out_dtype=torch.float32)
    torch.testing.assert_close(got.double(), x.double() @ w.double().T, atol=1e-3, rtol=1e-4)


def test_a_row_has_the_same_bits_beside_others(kernels):
    """Among up to eight rows, and among nine to sixteen (the workgroups' rows differ, not a result's sum)."""
    for outer, inner in ((4610, 1536), (20000, 1536)):
        x, weights = torch.randn(16, inner, device="cuda").bfloat16(), kernels.prepare_linear([torch.randn(outer, inner, device="cuda").bfloat16()], None)
        whole = kernels.linear(x, weights, out_dtype=torch.float32)
        for rows in (1, 5, 8, 9, 15):
            assert torch.equal(kernels.linear(x[:rows].contiguous(), weights, out_dtype=torch.float32), whole[:rows]), rows


@pytest.mark.parametrize("outer,inner", [(1536, 8960), (1024, 3072), (1152, 6912), (2560, 4096)])
def test_a_row_has_the_same_bits_beside_others_in_parts(kernels, outer, inner):
    x, weights = torch.randn(16, inner, device="cuda").bfloat16(), kernels.prepare_linear([torch.randn(outer, inner, device="cuda").bfloat16()], None)
    whole = kernels.linear(x, weights, out_dtype=torch.float32, partial=True)
    assert whole.ndim == 3 and whole.shape[0] > 1
    for rows in range(1, 16):
        assert torch.equal(kernels.linear(x[:rows].contiguous(), weights, out_dtype=torch.float32, partial=True), whole[:, :rows]), rows


@pytest.mark.parametrize("width", [2048, 2176, 4096, 4224, 8192])
def test_scaled_rows_at_the_edges_of_the_sums(kernels, width):
    """Widths at which a thread holds another number of pieces of the rows' sums."""
    from tests.test_gpu_linked_products import check_linked

    for rows in (1, 8, 9, 16):
        assert check_linked(kernels, rows, width, 128, 330) is not None
