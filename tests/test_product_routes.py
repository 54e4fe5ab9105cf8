"""What the host decides for products of many rows, asked of the built libraries (no GPU needed)."""

from __future__ import annotations

import re

import pytest

from llmserve_amd.kernels.build import build_module, load_module

# (weight rows, K): parts of K by rows of x.  Sums of parts meet in another order, so a product whose number of parts changes gives other bits.
PARTS = {
    (1536, 8960): {65: 10, 96: 10, 128: 10, 160: 7, 192: 7, 224: 7, 256: 7, 320: 5, 384: 5, 448: 4, 512: 4, 640: 4, 960: 2, 1031: 4, 1536: 4, 2048: 2},
    (1536, 1536): {65: 6, 96: 6, 128: 4, 160: 4, 192: 3, 224: 3, 256: 3, 320: 2, 384: 2, 448: 2, 512: 2, 640: 1, 960: 2, 1031: 1, 1536: 1, 2048: 1},
    (3584, 18944): {65: 8, 96: 8, 128: 8, 160: 8, 192: 8, 224: 8, 256: 8, 320: 4, 384: 4, 448: 4, 512: 4, 640: 8, 960: 4, 1031: 4, 1536: 2, 2048: 2},
    (3584, 3584): {65: 4, 96: 4, 128: 4, 160: 4, 192: 2, 224: 4, 256: 4, 320: 2, 384: 2, 448: 2, 512: 2, 640: 2, 960: 1, 1031: 1, 1536: 1, 2048: 1},
    (1536, 6144): {65: 8, 96: 8, 128: 8, 160: 6, 192: 6, 224: 8, 256: 8, 320: 4, 384: 6, 448: 4, 512: 4, 640: 3, 960: 2, 1031: 3, 1536: 3, 2048: 2},
    (1536, 480): {97: 3, 300: 3, 1000: 1}, (4096, 1568): {97: 7, 300: 1},
}


@pytest.mark.parametrize("weight", PARTS)
def test_parts_of_a_product_stay_what_they_are(weight):
    parts = load_module("gemm_blocks").llmserve_gemm_blocks_parts
    assert {rows: parts(rows, *weight) for rows in PARTS[weight]} == PARTS[weight]


# the same in float32 where an operand begins inside a piece of 16 bytes: the kernel that brings its operands through registers, in the parts that are best for it
FLOAT32_PARTS_ANYWHERE = {
    (1536, 8960): {65: 7, 96: 7, 128: 8, 160: 8, 192: 7, 224: 6, 256: 8, 384: 7, 512: 8, 777: 8, 2048: 4},
    (1536, 1536): {65: 5, 96: 5, 128: 5, 160: 6, 192: 5, 224: 6, 256: 5, 384: 5, 512: 4, 777: 4, 2048: 1},
    (3584, 3584): {65: 6, 96: 6, 128: 8, 160: 8, 192: 6, 224: 5, 256: 8, 384: 3, 512: 4, 777: 4, 2048: 2},
}


@pytest.mark.parametrize("weight", FLOAT32_PARTS_ANYWHERE)
def test_parts_of_a_float32_product_whose_operands_begin_anywhere(weight):
    parts = load_module("gemm_f32").llmserve_gemm_f32_parts
    assert {rows: parts(rows, *weight, 0) for rows in FLOAT32_PARTS_ANYWHERE[weight]} == FLOAT32_PARTS_ANYWHERE[weight]


@pytest.mark.parametrize("rows,outer,inner,parts,kind", [
    (400, 4608, 3584, 1, 0), (400, 4608, 3584, 1, 2), (448, 4608, 3584, 1, 2), (224, 4608, 3584, 2, 1), (640, 11008, 2048, 1, 1), (129, 9728, 896, 1, 1),
    (160, 9728, 896, 1, 0), (513, 896, 4864, 4, 1), (366, 5712, 4608, 3, 1), (378, 5712, 4608, 3, 1),
])
def test_no_tiles_that_share_a_few_compute_units(rows, outer, inner, parts, kind):
    """Tiles of 64 x 128 that come to a few more than 256 workgroups: those that share a CU take nearly twice as long, and the product with them (measured
    20 to 40 percent behind the other shapes)."""
    picked = load_module("gemm_blocks").llmserve_gemm_blocks_shape(rows, outer, inner, parts, kind)
    assert picked >= 0 and not (picked == 8 and 256 < -(-outer // 64) * -(-rows // 128) * parts < 512)  # (8: 64 x 128)


@pytest.mark.parametrize("rows,outer,inner", [(200, 17920, 1536), (256, 17920, 1536), (160, 37888, 3584), (200, 37888, 3584), (224, 37888, 3584)])
def test_no_whole_tiles_where_the_other_float32_kernel_is_ahead(rows, outer, inner):
    """Sizes at which whole tiles were measured 3 to 6 percent behind."""
    assert 0 <= load_module("gemm_f32").llmserve_gemm_f32_tile(rows, outer, inner, 1) < 5


@pytest.mark.parametrize("rows,outer,inner", [(160, 3584, 3584), (224, 1536, 8960)])
def test_no_whole_tiles_in_parts_where_the_other_float32_kernel_is_ahead(rows, outer, inner):
    """Sizes at which whole tiles were measured 8 to 10 percent behind in the parts that the product has."""
    library = load_module("gemm_f32")
    assert 0 <= library.llmserve_gemm_f32_tile(rows, outer, inner, library.llmserve_gemm_f32_parts(rows, outer, inner, 1)) < 5


@pytest.mark.parametrize("rows,outer,inner", [(128, 2048, 1536), (512, 2048, 1536), (160, 17920, 1536), (96, 17920, 1536), (512, 3584, 3584)])
def test_whole_tiles_where_they_are_ahead_of_the_other_float32_kernel(rows, outer, inner):
    """Sizes of few rounds of workgroups, at which whole tiles were measured 5 to 30 percent ahead."""
    assert load_module("gemm_f32").llmserve_gemm_f32_tile(rows, outer, inner, 1) >= 5


@pytest.mark.parametrize("module,kernel", [("gemm_blocks", "gemm_block_kernel"), ("gemm_f32", "gemm_f32_whole_kernel"),
                                           ("gemm_bf16", "gemm_stream_kernel"), ("gemm_bf16", "gemm_ring_kernel"), ("gemm_bf16", "gemm_merged_kernel")])
def test_kernels_that_read_ahead_keep_their_registers(module, kernel):
    """Kernels whose reads of LDS are instructions with waits of their own have no memory of a lane's: a register put away there before its read has come
    would come back with what it held before.  As the built library's own description of its kernels has it."""
    described = re.findall(rb"\.private_segment_fixed_size(.).*?\.symbol.*?(_Z\w+)\.kd", build_module(module).read_bytes(), re.S)
    sizes = {name.decode(): size for size, name in described if kernel.encode() in name}
    assert sizes and {name: size for name, size in sizes.items() if size != b"\0"} == {}
