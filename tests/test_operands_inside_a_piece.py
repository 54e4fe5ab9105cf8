"""Operands that begin inside a piece of 16 bytes: kernels that bring pieces into LDS do not take them (`HipKernels._instead_of_ring`)."""

from __future__ import annotations

import pytest
import torch

from llmserve_amd.kernels.hip import LinearWeights
from tests.test_routing import on_the_host


class Calls:
    """Takes the place of a kernel library: notes which entry points are called."""

    def __init__(self):
        self.names = []

    def __getattr__(self, name):
        def entry(*arguments):
            if name.endswith("parts"):
                return 1
            self.names.append(name.removeprefix("llmserve_"))
            return 0

        return entry


def called(rows, outer, inner, gated, moved, **changes):
    library = Calls()
    kernels = on_the_host(_gemm_bf16=library, _gemm_blocks=library, _gemm_generic=library, _elementwise=library, _gemm_f32=None, **changes)
    x, weight = (torch.zeros(n * inner + 8, dtype=torch.bfloat16) for n in (rows, outer))
    x, weight = ((t[1:-7] if name in moved else t[:-8]).view(-1, inner) for name, t in (("x", x), ("weight", weight)))
    weights = LinearWeights(weight, None)
    if gated:
        prepared = kernels.prepare_gated_linear(weight[::2].clone(), weight[1::2].clone())
        prepared.both = weights
        kernels.gated_linear(x, prepared)
    else:
        kernels.linear(x, weights)
    return library.names


@pytest.mark.parametrize("moved", ["x", "weight"])
@pytest.mark.parametrize("rows,outer,inner,gated,there,instead", [
    (24, 4096, 1152, False, "gemm_ring", ["gemm_medium"]), (64, 8192, 1024, True, "gemm_ring", ["gemm_medium"]),
    (128, 8192, 1024, True, "gemm_blocks", ["silu_mul"]),  # (behind the BLAS library's product)
])
def test_products_of_17_to_128_rows(rows, outer, inner, gated, there, instead, moved):
    assert called(rows, outer, inner, gated, ()) == [there]
    assert called(rows, outer, inner, gated, moved) == instead


@pytest.mark.parametrize("moved", ["x", "weight"])
@pytest.mark.parametrize("rows,gated,instead", [(200, False, ["gemm_generic"]), (96, True, ["gemm_generic", "silu_mul"])])
def test_products_of_many_rows_without_the_blas_library(rows, gated, instead, moved):
    assert called(rows, 8192, 1024, gated, (), library_products=False) == ["gemm_blocks"]
    assert called(rows, 8192, 1024, gated, moved, library_products=False) == instead


@pytest.mark.gpu
@pytest.mark.parametrize("moved", ["x", "weight"])
@pytest.mark.parametrize("for_replay", [True, False])
@pytest.mark.parametrize("rows,outer,inner,gated", [(24, 1536, 1536, False), (64, 1210, 640, False), (24, 4096, 1152, False), (64, 8192, 1024, True), (128, 8192, 1024, True)])
def test_their_results(rows, outer, inner, gated, for_replay, moved):
    from llmserve_amd.kernels import HipKernels

    kernels, generator = HipKernels(torch.bfloat16), torch.Generator(device="cuda").manual_seed(rows + inner)
    kernels._for_replay = for_replay
    x, weight = (torch.randn(n * inner + 8, generator=generator, device="cuda").mul_(scale).bfloat16() for n, scale in ((rows, 1.0), (outer, inner ** -0.5)))
    x, weight = ((t[1:-7] if name == moved else t[:-8]).view(-1, inner) for name, t in (("x", x), ("weight", weight)))
    want = x.double() @ weight.double().T
    if gated:
        prepared = kernels.prepare_gated_linear(weight[::2], weight[1::2])
        prepared.both = LinearWeights(weight, None)
        got, want = kernels.gated_linear(x, prepared).double(), torch.nn.functional.silu(want[:, ::2]) * want[:, 1::2]
        assert (got - want).norm() < 3 * 2.0 ** -9 * want.norm()  # (gate and up may be rounded to bfloat16, and the result is)
    else:
        for partial in (False, True):
            got = kernels.linear(x, LinearWeights(weight, None), out_dtype=torch.float32, partial=partial).double()
            got = got if got.ndim == 2 else got.sum(0)
            assert ((got - want).abs() <= inner * 2.0 ** -24 * (x.double().abs() @ weight.double().abs().T) + 1e-6).all()


@pytest.mark.gpu
def test_entry_points_refuse_them():
    from llmserve_amd.kernels import HipKernels

    kernels = HipKernels(torch.bfloat16)
    x, w, out = (torch.zeros(n, device="cuda", dtype=torch.bfloat16) for n in (128 * 1024 + 8, 8192 * 1024 + 8, 128 * 8192))
    for a, b in ((x[1:], w), (x, w[4:])):
        assert kernels._gemm_bf16.llmserve_gemm_ring(a.data_ptr(), b.data_ptr(), None, 0, out.data_ptr(), 0, 0, 24, 8192, 1024, 1, 4, kernels._stream) == 1001
        assert kernels._gemm_bf16.llmserve_gemm_stream(a.data_ptr(), b.data_ptr(), None, 0, out.data_ptr(), 0, 0, 24, 512, 1024, 1, kernels._stream) == 1001
        assert kernels._gemm_blocks.llmserve_gemm_blocks(a.data_ptr(), b.data_ptr(), None, 0, out.data_ptr(), 0, 0, 128, 8192, 1024, 1, kernels._stream) == 1001


@pytest.mark.gpu
def test_the_rotated_product_refuses_them():
    from llmserve_amd.kernels import HipKernels

    kernels, rows, inner, heads, kv_heads, dim, page = HipKernels(torch.bfloat16), 96, 1536, 12, 2, 128, 16
    x, w, out, keys, values = (torch.zeros(n + 8, device="cuda", dtype=torch.bfloat16) for n in (rows * inner, 2048 * inner, rows * 2048, 8 * page * kv_heads * dim, 8 * page * kv_heads * dim))
    table, slots = torch.zeros(rows * dim, device="cuda"), torch.full((rows,), -1, device="cuda", dtype=torch.int32)
    for a, b, status in ((x, w, 0), (x[1:], w, 1001), (x, w[4:], 1001)):
        assert kernels._gemm_blocks.llmserve_gemm_rotated(a.data_ptr(), b.data_ptr(), None, 0, out.data_ptr(), rows, inner, table.data_ptr(), heads, kv_heads, dim, keys.data_ptr(),
                                                          values.data_ptr(), slots.data_ptr(), page, kernels._stream) == status
    torch.cuda.synchronize()
