"""The rules that shape products of up to 16 rows (csrc/gemm_bf16.hip: flow_shape, llmserve_gemm_flow_parts), at random sizes and at measured ones."""

from __future__ import annotations

import random
import re

from llmserve_amd.kernels.build import build_module, load_module

SMALL, MOST, SMALL_MOST = 1 << 22, 40, 16


def test_rows_and_parts_are_ones_that_the_kernel_takes():
    library, draw = load_module("gemm_bf16"), random.Random(11)
    for _ in range(20000):
        rows, inner = draw.randint(1, 16), 64 * draw.randint(1, 500)
        outer = draw.choice([draw.randint(1, 400), draw.randint(1, 40000), draw.randint(1, 300000)])
        parts = library.llmserve_gemm_flow_parts(rows, outer, inner)
        assert 1 <= parts <= 8 and inner % parts == 0 and inner // parts % 64 == 0 and (parts == 1 or inner // parts >= 512)
        for splits in (1, parts):
            each = library.llmserve_gemm_flow_rows(rows, outer, inner, splits)
            assert each % 2 == 0 and 8 <= each <= (SMALL_MOST if outer * inner <= SMALL else MOST)
    assert library.llmserve_gemm_flow_parts(1, 1536, 8960 + 32) == 1  # (not a K of whole units: another kernel's)


def test_parts_are_the_same_for_every_number_of_rows():
    """Parts decide in which order a row's sums meet: a row has the same bits whatever stands beside it."""
    library, draw = load_module("gemm_bf16"), random.Random(12)
    for outer, inner in [(1536, 8960), (1024, 3072), (1152, 6912)] + [(draw.randint(1, 8000), 64 * draw.randint(1, 400)) for _ in range(3000)]:
        assert len({library.llmserve_gemm_flow_parts(rows, outer, inner) for rows in range(1, 17)}) == 1, (outer, inner)


def test_sizes_that_were_measured():
    """Workgroups that come out even on 256 CUs, or within a few percent of the best of what was measured."""
    library = load_module("gemm_bf16")
    for rows in (1, 8, 16):
        assert library.llmserve_gemm_flow_rows(rows, 17920, 1536, 1) in (24, 36, 38, 40)  # not 32: three workgroups a CU of 32
        assert library.llmserve_gemm_flow_rows(rows, 4608, 3584, 1) == 18
        assert library.llmserve_gemm_flow_parts(rows, 1536, 8960) in (4, 5)
        assert library.llmserve_gemm_flow_parts(rows, 3584, 18944) in (1, 2)


def test_workgroups_do_not_walk_the_same_channels():
    """Weights of neighbouring workgroups 256 or 512 KB apart were measured 15 to 40 percent behind, where there are many; not where there are few, or a power of two is
    a smaller or larger one."""
    library = load_module("gemm_bf16")
    for outer, inner in [(57344, 8192), (24576, 4096), (28672, 4096), (128256, 4096), (8192, 8192), (32000, 4096), (16384, 4096)]:
        for rows in (1, 2, 8, 9, 16):
            assert library.llmserve_gemm_flow_rows(rows, outer, inner, 1) * 2 * inner not in (256 << 10, 512 << 10), (outer, inner, rows)
    for outer, inner, parts in [(2048, 8192, 4), (128256, 2048, 1), (40000, 12288, 1)]:
        assert library.llmserve_gemm_flow_rows(1, outer, inner, parts) == 32


def test_the_kernel_keeps_its_registers():
    """Its reads of LDS are instructions with waits of their own: a register put away into a lane's memory before its read has come would come back with
    what it held before.  As the built library's own description of its kernels has it."""
    described = re.findall(rb"\.private_segment_fixed_size(.).*?\.symbol.*?(_Z\w+)\.kd", build_module("gemm_bf16").read_bytes(), re.S)
    sizes = {name.decode(): size for size, name in described if b"gemm_flow_kernel" in name}
    assert sizes and {name: size for name, size in sizes.items() if size != b"\0"} == {}
