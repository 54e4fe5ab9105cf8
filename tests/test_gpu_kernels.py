"""Each kernel alone against a plain float32 reference of the same operation, at sizes
other than the tiny models': widths and vocabularies that are no power of two, head sizes
in steps of 16, odd numbers of heads and groups, pages of several sizes, shuffled pages."""

from __future__ import annotations

import contextlib
import math
import random
import types

import pytest
import torch
import torch.nn.functional as F

from tests.plain import qwen2_plain as plain

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]
TOLERANCE = {torch.float32: dict(atol=2e-5, rtol=2e-5), torch.bfloat16: dict(atol=2e-2, rtol=2e-2)}


@pytest.fixture(scope="module")
def kernels():
    from llmserve_amd.kernels import HipKernels

    return {dtype: HipKernels(dtype) for dtype in DTYPES}


@pytest.fixture(scope="module")
def own_kernels():
    """The library with every product on the hand-written kernels (none sent to the BLAS library)."""
    from llmserve_amd.kernels import HipKernels

    return HipKernels(torch.bfloat16, library_products=False)


def on_gpu(tensor, dtype=None):
    return tensor.to("cuda", dtype) if dtype else tensor.to("cuda")


def rounded(tensor, dtype):
    """What the kernel sees: the reference's inputs rounded to the run dtype."""
    return tensor.to(dtype).double()


@pytest.mark.parametrize("dtype", DTYPES)
def test_embedding(kernels, dtype):
    table = torch.randn(301, 72)
    ids = torch.tensor([0, 300, 17, 17, 5], dtype=torch.int32)
    out = kernels[dtype].embedding(on_gpu(table, dtype), on_gpu(ids))
    assert out.dtype == torch.float32
    torch.testing.assert_close(out.cpu().double(), rounded(table, dtype)[ids.long()], atol=0, rtol=0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,eps", [(72, 1e-6), (1000, 1e-2), (4099, 1e-5)])
def test_add_rms_norm(kernels, dtype, width, eps):
    hidden, delta = torch.randn(7, width), 0.3 * torch.randn(7, width)
    weight = 1 + 0.2 * torch.randn(width)
    for weight_dtype in (dtype, torch.float32):
        device_hidden = on_gpu(hidden.clone())
        out = kernels[dtype].add_rms_norm(device_hidden, on_gpu(delta), on_gpu(weight, weight_dtype), eps)
        summed = hidden.double() + delta.double()
        torch.testing.assert_close(device_hidden.cpu().double(), summed, atol=1e-6, rtol=1e-6)
        expected = plain.rms_norm(summed, rounded(weight, weight_dtype), eps)
        assert out.dtype == dtype
        torch.testing.assert_close(out.cpu().double(), expected, **TOLERANCE[dtype])
    alone = kernels[dtype].add_rms_norm(on_gpu(hidden.clone()), None, on_gpu(weight, dtype), eps)
    torch.testing.assert_close(alone.cpu().double(), plain.rms_norm(hidden.double(), rounded(weight, dtype), eps), **TOLERANCE[dtype])
    small = 1e-4 * hidden  # eps decides here
    tiny = kernels[dtype].add_rms_norm(on_gpu(small.clone()), None, on_gpu(torch.ones(width), dtype), eps)
    torch.testing.assert_close(tiny.cpu().double(), plain.rms_norm(small.double(), torch.ones(width).double(), eps), **TOLERANCE[dtype])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,inner,outer", [(1, 72, 50), (5, 200, 333), (70, 129, 65), (130, 64, 1000),
                                              (1, 256, 48), (8, 1536, 272), (16, 96, 1000), (17, 1184, 50), (33, 512, 24),
                                              (64, 4480, 130), (64, 160, 2048),
                                              # up to 16 rows with two or four weight tiles a wave: a long K, all 16 rows, a vocabulary-sized N
                                              (8, 4096, 8192), (13, 512, 16400), (5, 1536, 66000)])
def test_linear_and_gated_linear(kernels, dtype, rows, inner, outer):
    k = kernels[dtype]
    # weights scaled so that every output is of order one, whatever `inner` is
    x, w, b = torch.randn(rows, inner), torch.randn(outer, inner) / math.sqrt(inner), torch.randn(outer)
    expected = rounded(x, dtype) @ rounded(w, dtype).T + rounded(b, dtype)
    parts = [w[: outer // 3], w[outer // 3 :]], [b[: outer // 3], b[outer // 3 :]]
    handle = k.prepare_linear([on_gpu(p, dtype) for p in parts[0]], [on_gpu(p, dtype) for p in parts[1]])
    for out_dtype in (None, torch.float32):
        out = k.linear(on_gpu(x, dtype), handle, out_dtype=out_dtype)
        assert out.dtype == (out_dtype or dtype)
        tolerance = TOLERANCE[dtype] if out_dtype is None else dict(atol=1e-4, rtol=1e-4)
        torch.testing.assert_close(out.cpu().double(), expected, **tolerance)
    no_bias = k.linear(on_gpu(x, dtype), k.prepare_linear([on_gpu(w, dtype)], None), out_dtype=torch.float32)
    torch.testing.assert_close(no_bias.cpu().double(), expected - rounded(b, dtype), atol=1e-4, rtol=1e-4)
    # a weight kept in 32-bit under a bfloat16 run
    wide = k.linear(on_gpu(x, dtype), k.prepare_linear([on_gpu(w)], None), out_dtype=torch.float32)
    torch.testing.assert_close(wide.cpu().double(), rounded(x, dtype) @ w.double().T, atol=1e-4, rtol=1e-4)
    up = torch.randn(outer, inner) / math.sqrt(inner)
    gated = k.gated_linear(on_gpu(x, dtype), k.prepare_gated_linear(on_gpu(w, dtype), on_gpu(up, dtype)))
    want = F.silu(rounded(x, dtype) @ rounded(w, dtype).T) * (rounded(x, dtype) @ rounded(up, dtype).T)
    torch.testing.assert_close(gated.cpu().double(), want, **TOLERANCE[dtype])


@pytest.mark.parametrize("rows,inner,outer", [(17, 128, 64), (32, 256, 100), (33, 1536, 272), (64, 1280, 130), (64, 8960, 48),
                                              (40, 96, 77), (64, 160, 2048), (100, 256, 40), (65, 32, 128), (130, 1536, 272),
                                              (300, 96, 1000), (2048, 512, 384), (129, 129, 50), (2000, 64, 6500), (2048, 2048, 1500),
                                              (1100, 2048, 700), (2048, 416, 6400), (1000, 160, 12900), (2040, 96, 6401), (8, 18944, 3584)])
def test_products_without_the_library(own_kernels, rows, inner, outer):
    """17 to 64 rows: the kernel that shares x through LDS (K a multiple of 128), else the
    weight-streaming one with several tiles of x; more rows: the tiled one (K a multiple of 32; its
    256 x 256 tiles where there are 200 of them, with K steps that are and are not a multiple of its
    four stages, K cut into partial sums where a float32 result may stay in parts); else the generic one."""
    k, dtype = own_kernels, torch.bfloat16
    x, w, b = torch.randn(rows, inner), torch.randn(outer, inner) / math.sqrt(inner), torch.randn(outer)
    expected = rounded(x, dtype) @ rounded(w, dtype).T + rounded(b, dtype)
    handle = k.prepare_linear([on_gpu(w, dtype)], [on_gpu(b, dtype)])
    torch.testing.assert_close(k.linear(on_gpu(x, dtype), handle).cpu().double(), expected, **TOLERANCE[dtype])
    parts = k.linear(on_gpu(x, dtype), handle, out_dtype=torch.float32, partial=True)
    summed = parts if parts.ndim == 2 else parts.sum(0)
    torch.testing.assert_close(summed.cpu().double(), expected, atol=1e-4, rtol=1e-4)
    up = torch.randn(outer, inner) / math.sqrt(inner)
    gated = k.gated_linear(on_gpu(x, dtype), k.prepare_gated_linear(on_gpu(w, dtype), on_gpu(up, dtype)))
    want = F.silu(rounded(x, dtype) @ rounded(w, dtype).T) * (rounded(x, dtype) @ rounded(up, dtype).T)
    torch.testing.assert_close(gated.cpu().double(), want, **TOLERANCE[dtype])


@pytest.mark.parametrize("rows,inner,outer", [(65, 64, 1536), (96, 1536, 17920), (129, 128, 2050), (200, 192, 40), (257, 1024, 4100), (384, 8960, 1536),
                                              (511, 640, 9000), (640, 320, 20000), (1100, 1536, 6400), (2048, 256, 17920)])
def test_tiles_of_many_rows(own_kernels, rows, inner, outer):
    """The LDS-tiled product, from one stage of K on, at rows and weight rows that leave remainders (each of its shapes and their stages:
    `test_every_shape_of_a_tile`): plain, gated, and in every number of parts that K allows.  Partial sums are float32 sums of
    `inner` products of bfloat16 values: a few times sqrt(K) * 2^-24 of a result of size 1."""
    k, dtype = own_kernels, torch.bfloat16
    generator = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, inner, generator=generator, device="cuda").to(dtype)
    w, up = (torch.randn(outer, inner, generator=generator, device="cuda").div_(math.sqrt(inner)).to(dtype) for _ in range(2))
    b = torch.randn(outer, generator=generator, device="cuda").to(dtype)
    expected = x.double() @ w.double().T + b.double()
    torch.testing.assert_close(k.linear(x, k.prepare_linear([w], [b])).double(), expected, **TOLERANCE[dtype])
    want = F.silu(x.double() @ w.double().T) * (x.double() @ up.double().T)
    torch.testing.assert_close(k.gated_linear(x, k.prepare_gated_linear(w, up)).double(), want, **TOLERANCE[dtype])
    bound = dict(atol=8 * math.sqrt(inner) * 2.0 ** -24, rtol=1e-5)
    for splits in range(1, 13):
        if inner % (32 * splits):
            continue
        parts = torch.full((splits, rows, outer), float("nan"), device="cuda")
        status = k._gemm_blocks.llmserve_gemm_blocks(x.data_ptr(), w.data_ptr(), b.data_ptr(), 0, parts.data_ptr(), 1, 0, rows, outer, inner, splits,
                                                     torch.cuda.current_stream().cuda_stream)
        assert status == 0
        torch.testing.assert_close(parts.double().sum(0), expected, **bound)


@pytest.mark.parametrize("shape,rows,plain,float32,gated,inner", [
    (0, 700, 15681, 13070, None, 512), (0, 1300, None, None, 8964, 512), (1, 1025, 13057, 13059, None, 512), (1, 1300, None, None, 10892, 512),
    (2, 700, 8200, None, 8212, 512), (2, 700, None, 8167, None, 576), (3, 200, 16817, None, None, 512), (3, 161, None, 19309, None, 512), (3, 195, None, None, 16830, 512), (4, 513, 9798, 9796, None, 512),
    (4, 194, None, None, 16590, 512), (5, 260, 12517, None, None, 512), (5, 265, None, 11301, None, 512), (5, 264, None, None, 13070, 512), (6, 2047, 1421, None, 1420, 512),
    (6, 195, None, 10796, None, 512),
    (7, 135, 10461, None, None, 512), (7, 130, None, 10525, None, 512), (7, 135, None, None, 10386, 512), (8, 97, 9985, 10565, 9666, 512), (9, 97, 614, 603, 612, 512),
    (10, 193, 13273, None, None, 512), (10, 388, None, 8104, None, 512), (10, 205, None, None, 12482, 512), (11, 513, 11133, None, None, 512), (11, 324, None, 16577, None, 512),
    (11, 514, None, None, 11510, 512),
])
def test_every_shape_of_a_tile(kernels, shape, rows, plain, float32, gated, inner):
    """Each shape of the LDS-tiled product where it is picked, at rows and weight rows that leave remainders, in each kind of result.  Bounds as in
    `test_tiles_of_many_rows`; the hardware's 2^x and 1/x are within a few 2^-23."""
    for kind, outer in enumerate((plain, float32, gated)):
        if outer is not None:
            check_shape(kernels[torch.bfloat16], shape, rows, outer, kind, inner)


def check_shape(k, shape, rows, outer, kind, inner):
    assert k._gemm_blocks.llmserve_gemm_blocks_shape(rows, outer, inner, 1, kind) == shape
    generator = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, inner, generator=generator, device="cuda").to(torch.bfloat16)
    w = torch.randn(outer, inner, generator=generator, device="cuda").div_(math.sqrt(inner)).to(torch.bfloat16)
    b = torch.randn(outer, generator=generator, device="cuda")
    out = torch.full((rows, outer // 2 if kind == 2 else outer), float("nan"), device="cuda", dtype=torch.float32 if kind == 1 else torch.bfloat16)
    status = k._gemm_blocks.llmserve_gemm_blocks(
        x.data_ptr(), w.data_ptr(), b.data_ptr(), 1, out.data_ptr(), int(kind == 1), int(kind == 2), rows, outer, inner, 1, torch.cuda.current_stream().cuda_stream)
    assert status == 0
    expected = x.double() @ w.double().T + b.double()
    if kind == 2:
        expected = F.silu(expected[:, 0::2]) * expected[:, 1::2]
    bound = dict(atol=8 * math.sqrt(inner) * 2.0 ** -24, rtol=1e-5) if kind == 1 else TOLERANCE[torch.bfloat16]
    torch.testing.assert_close(out.double(), expected, **bound)


TILES = [(256, 256), (256, 320), (128, 256), (192, 128), (160, 160), (128, 160), (96, 128), (128, 96), (64, 128), (64, 64), (128, 128), (256, 128)]


def sizes_of_a_shape(k, shape, kind, inner, multiple):
    """The smallest of many products that a shape is picked for: more rows and weight rows than a tile has, a remainder of both, weight rows a multiple of `multiple`."""
    n, m = TILES[shape]
    draw, best = random.Random(inner + 10 * shape + kind), None
    for _ in range(20000):
        rows, outer = draw.randrange(65, 2100), multiple * draw.randrange(1, 20000 // multiple)
        if rows < m or outer < n or rows % m == 0 or outer % n == 0 or (best and rows * outer >= best[0] * best[1]):
            continue
        if k._gemm_blocks.llmserve_gemm_blocks_shape(rows, outer, inner, 1, kind) == shape:
            best = rows, outer
    assert best
    return best


@pytest.mark.parametrize("kind", range(3))
@pytest.mark.parametrize("shape", range(len(TILES)))
def test_every_shape_of_a_tile_in_whole_pieces(kernels, shape, kind):
    """Results whose rows are whole pieces of 16 bytes, which leave in such pieces, inside a tile and at both edges (bounds as above)."""
    k = kernels[torch.bfloat16]
    check_shape(k, shape, *sizes_of_a_shape(k, shape, kind, 512, 16), kind, 512)


# (shape, kind): the K of as few stages of 64 as it is picked with, up to one more than it keeps in LDS
FEW_STAGES = {(0, 0): (64, 128, 192), (0, 1): (64, 128, 192), (1, 2): (64, 128, 192), (2, 1): (128, 192, 256), (3, 0): (128, 192, 256, 320), (3, 2): (192, 256, 320),
              (4, 2): (192, 256, 320), (4, 1): (192, 256, 320), (5, 0): (256, 320), (6, 2): (256, 320, 384), (7, 2): (192, 256, 320, 384), (7, 0): (256, 320, 384),
              (8, 0): (64, 128, 192, 256), (8, 1): (64, 128, 192, 256), (9, 0): (64, 128, 192, 256, 320, 384), (9, 2): (64, 128, 192, 256, 320, 384),
              (10, 2): (384,), (11, 1): (128, 192, 256), (11, 0): (192, 256)}


@pytest.mark.parametrize("shape,kind", FEW_STAGES)
def test_every_shape_of_a_tile_over_few_stages(kernels, shape, kind):
    """A K of fewer stages than a shape keeps in LDS, of as many and of one more (bounds as above)."""
    k = kernels[torch.bfloat16]
    for inner in FEW_STAGES[shape, kind]:
        check_shape(k, shape, *sizes_of_a_shape(k, shape, kind, inner, 2 if kind == 2 else 1), kind, inner)


@pytest.mark.parametrize("shape,inner", [(0, 96), (0, 160), (0, 480), (7, 288), (7, 352), (7, 544), (8, 32), (8, 96), (8, 224), (9, 32), (9, 96), (9, 352), (10, 544), (10, 800)])
def test_every_shape_that_takes_half_a_stage(kernels, shape, inner):
    """A K that ends in half a stage, one of half a stage alone among them: rows of the result in whole pieces and not (bounds as above)."""
    k = kernels[torch.bfloat16]
    for kind, multiple in ((0, 16), (1, 1), (2, 2)):
        check_shape(k, shape, *sizes_of_a_shape(k, shape, kind, inner, multiple), kind, inner)


@pytest.mark.parametrize("rows,inner,width", [(130, 128, 44), (300, 192, 1092), (1000, 256, 4860), (700, 512, 4100), (2048, 128, 8956)])
def test_gated_widths_of_four_mod_eight(own_kernels, rows, inner, width):
    """A gated result whose rows begin in the middle of 16 bytes every other time: each value in its place and nothing outside (bound as in `test_tiles_of_many_rows`)."""
    k, dtype = own_kernels, torch.bfloat16
    generator = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, inner, generator=generator, device="cuda").to(dtype)
    w = torch.randn(2 * width, inner, generator=generator, device="cuda").div_(math.sqrt(inner)).to(dtype)
    around = torch.full((rows * width + 128,), float("nan"), device="cuda", dtype=dtype)
    out = around[64 : 64 + rows * width].view(rows, width)
    assert k._gemm_blocks.llmserve_gemm_blocks(x.data_ptr(), w.data_ptr(), None, 0, out.data_ptr(), 0, 1, rows, 2 * width, inner, 1,
                                               torch.cuda.current_stream().cuda_stream) == 0
    expected = x.double() @ w.double().T
    torch.testing.assert_close(out.double(), F.silu(expected[:, 0::2]) * expected[:, 1::2], **TOLERANCE[dtype])
    assert around[:64].isnan().all() and around[64 + rows * width :].isnan().all()


@pytest.mark.parametrize("rows,inner,outer", [(512, 1536, 2048), (513, 1536, 2048), (2048, 1536, 2048), (2049, 1536, 2048), (513, 64, 1024), (777, 320, 1030), (600, 1536, 1536)])
def test_small_weights_over_many_rows(kernels, rows, inner, outer):
    """Both sides of the line from which small plain products are the tiled kernel's, with and without leave to split: a route that takes
    one and not the other would leave a product to the generic kernel.  Float32 results as in `test_tiles_of_many_rows`."""
    k, dtype = kernels[torch.bfloat16], torch.bfloat16
    generator = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, inner, generator=generator, device="cuda").to(dtype)
    w = torch.randn(outer, inner, generator=generator, device="cuda").div_(math.sqrt(inner)).to(dtype)
    b = torch.randn(outer, generator=generator, device="cuda").to(dtype)
    expected, handle = x.double() @ w.double().T + b.double(), k.prepare_linear([w], [b])
    taken = 512 < rows and rows * outer <= 1 << 22
    assert (k._streaming(x, handle) == "tiled") == taken and (not taken or k._streaming(x, handle, may_split=True) == "tiled")
    torch.testing.assert_close(k.linear(x, handle).double(), expected, **TOLERANCE[dtype])
    parts = k.linear(x, handle, out_dtype=torch.float32, partial=True)
    summed = parts.double() if parts.ndim == 2 else parts.double().sum(0)
    torch.testing.assert_close(summed, expected, atol=8 * math.sqrt(inner) * 2.0 ** -24, rtol=1e-5)


def key_pieces(rows):
    """Key pages written as rows [pages, kv, offset, dim] -> as the cache keeps them, in pieces of eight
    elements, the same piece of all the keys of a page side by side: [pages, kv, dim / w, offset, w]
    (a head size that is no multiple of 8 is one piece)."""
    pages, kv, page, dim = rows.shape
    width = 8 if dim % 8 == 0 else dim
    return rows.view(pages, kv, page, dim // width, width).permute(0, 1, 3, 2, 4).contiguous()


def key_rows(pieces):
    """The inverse of `key_pieces`."""
    pages, kv, count, page, width = pieces.shape
    return pieces.permute(0, 1, 3, 2, 4).reshape(pages, kv, page, count * width)


def value_pieces(rows):
    """Value pages written transposed [pages, kv, dim, page] -> as the cache keeps them, in pieces of eight keys,
    the same piece of all dimensions side by side: [pages, kv, page / v, dim, v] (a page size that is no
    multiple of 8 is one piece)."""
    pages, kv, dim, page = rows.shape
    width = 8 if page % 8 == 0 else page
    return rows.view(pages, kv, dim, page // width, width).permute(0, 1, 3, 2, 4).contiguous()


def value_rows(pieces):
    """The inverse of `value_pieces`."""
    pages, kv, count, dim, width = pieces.shape
    return pieces.permute(0, 1, 3, 2, 4).reshape(pages, kv, dim, count * width)


def paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=0, spare_pages=3):
    """Requests with `lengths[i]` cached tokens of which the last `counts[i]` are this step's.
    Returns the step's batch, the cell with garbage in every unused slot, and per-request q, k, v."""
    from llmserve_amd.cache import CacheCell
    from llmserve_amd.engine.batch import GroupBatch, SequenceChunk, StepBatch
    from llmserve_amd.parts import HeadLayout, PagedKeyValue

    generator = torch.Generator().manual_seed(shuffle_seed)
    blocks = [math.ceil(n / page) for n in lengths]
    pages = sum(blocks) + spare_pages
    order = torch.randperm(pages, generator=generator).tolist()
    width = max(blocks)
    tables = torch.full((len(lengths), width), -1, dtype=torch.int32)
    keys = torch.full((pages, kv_heads, page, dim), float("nan"))
    values = torch.full((pages, kv_heads, dim, page), float("nan"))  # value pages are stored transposed
    per_request, slot_mapping, positions, token_sequence, chunks = [], [], [], [], []
    for index, (length, count) in enumerate(zip(lengths, counts)):
        mine = [order.pop() for _ in range(blocks[index])]
        tables[index, : len(mine)] = torch.tensor(mine, dtype=torch.int32)
        q = torch.randn(length, heads, dim, generator=generator)
        k = torch.randn(length, kv_heads, dim, generator=generator)
        v = torch.randn(length, kv_heads, dim, generator=generator)
        per_request.append((q, k, v))
        for position in range(length):
            keys[mine[position // page], :, position % page] = k[position]
            values[mine[position // page], :, :, position % page] = v[position]
        for position in range(length - count, length):
            slot_mapping.append(mine[position // page] * page + position % page)
            positions.append(position)
            token_sequence.append(index)
        chunks.append(SequenceChunk(f"r{index}", index, length - count, count))
    starts = [0]
    for count in counts:
        starts.append(starts[-1] + count)
    ints = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    group = GroupBatch(page, tables.cuda(), ints(slot_mapping), width)
    batch = StepBatch(
        num_tokens=sum(counts), chunks=chunks, token_ids=ints([0] * sum(counts)), positions=ints(positions),
        token_sequence=ints(token_sequence), query_start=ints(starts), context_lengths=ints(lengths),
        state_slots=ints(list(range(len(lengths)))), groups=[group], logit_rows=ints([]), num_logit_rows=0,
        max_query_length=max(counts), max_context_length=max(lengths),
    )
    cell = CacheCell(PagedKeyValue(kv_heads, dim), True, 0, key_pieces(keys).to("cuda", dtype), value_pieces(values).to("cuda", dtype))
    return batch, cell, per_request, HeadLayout(heads, kv_heads, dim)


def step_rows(per_request, counts, heads, kv_heads, dim):
    """The step's qkv rows [T, (heads + 2 kv) * dim] from the per-request tensors."""
    rows = []
    for (q, k, v), count in zip(per_request, counts):
        rows.append(torch.cat([q[-count:].flatten(1), k[-count:].flatten(1), v[-count:].flatten(1)], dim=1))
    return torch.cat(rows)


ATTENTION_SHAPES = [  # heads, kv_heads, dim, page
    (12, 2, 32, 16),  # the reference's own test shape (tests/test_triton_paged_attention.py:24)
    (6, 1, 48, 8),
    (5, 5, 80, 24),  # a page that is no power of two
    (8, 2, 128, 16),
    (3, 1, 112, 64),
    (4, 2, 256, 16),  # the widest head the matrix-core kernel takes: one column tile a wave
    (4, 4, 16, 1),
    (40, 8, 128, 16),  # the 32B sizes: five query heads a kv head
    (10, 2, 128, 16),
    (28, 4, 128, 16),  # the 7B sizes: seven
]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,dim,page", ATTENTION_SHAPES)
def test_paged_attention_at_page_edges(kernels, dtype, heads, kv_heads, dim, page):
    """Lengths around page edges (the reference's 1, 15, 16, 17, 31, 32, 33, scaled to the page),
    single decoded tokens beside portions, shuffled pages, garbage in unused slots."""
    lengths = [1, page - 1 or 1, page, page + 1, 2 * page - 1, 2 * page, 2 * page + 1, 5 * page + 3, 150]
    counts = [1, 1, page, 1, 3, 2 * page, 1, 2 * page + 2, 1]
    counts = [min(count, length) for count, length in zip(counts, lengths)]
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=dim)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    scale = 0.37
    out = kernels[dtype].paged_attention(qkv, layout, batch, cell, scale, None).cpu().double()
    expected = []
    for (q, k, v), count in zip(per_request, counts):
        full = plain.causal_attention(rounded(q, dtype), rounded(k, dtype), rounded(v, dtype), scale)
        expected.append(full[-count:].flatten(1))
    torch.testing.assert_close(out, torch.cat(expected), **TOLERANCE[dtype])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window", [1, 5, 16, 17, 40])
def test_paged_attention_window_edge(kernels, dtype, window):
    """One key far back is made to stand out: it must count exactly while it is inside the window."""
    heads, kv_heads, dim, page = 4, 2, 32, 8
    lengths, counts = [70, 41], [30, 1]
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=window)
    for q, k, v in per_request:  # the key at the window's far edge of the last query dominates its scores
        edge = q.shape[0] - window
        if edge >= 0:
            k[edge] = 4.0 * q[-1, ::2]
    batch, cell, _, _ = _rewrite_cell(batch, cell, per_request, page, dtype)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    out = kernels[dtype].paged_attention(qkv, layout, batch, cell, 0.25, window).cpu().double()
    expected = []
    for (q, k, v), count in zip(per_request, counts):
        full = plain.causal_attention(rounded(q, dtype), rounded(k, dtype), rounded(v, dtype), 0.25, window)
        expected.append(full[-count:].flatten(1))
    torch.testing.assert_close(out, torch.cat(expected), **TOLERANCE[dtype])
    wider = kernels[dtype].paged_attention(qkv, layout, batch, cell, 0.25, window + 1).cpu().double()
    assert not torch.allclose(wider, out, atol=1e-2)


def _rewrite_cell(batch, cell, per_request, page, dtype):
    keys, values = key_rows(cell.keys.cpu().float()), value_rows(cell.values.cpu().float())
    tables = batch.groups[0].block_tables.cpu()
    for index, (q, k, v) in enumerate(per_request):
        for position in range(k.shape[0]):
            keys[tables[index, position // page], :, position % page] = k[position]
            values[tables[index, position // page], :, :, position % page] = v[position]
    cell.keys, cell.values = key_pieces(keys).to("cuda", dtype), value_pieces(values).to("cuda", dtype)
    return batch, cell, per_request, None


@pytest.mark.parametrize("dtype", DTYPES)
def test_paged_attention_finds_a_far_key_among_hundreds(kernels, dtype):
    heads, kv_heads, dim, page = 6, 2, 64, 16
    lengths, counts = [700], [1]
    for far in (0, 15, 16, 337, 698):
        batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=far)
        q, k, v = per_request[0]
        k[far] = 3.0 * q[-1, ::3]  # for heads 0 and 3 this key dominates; v[far] must come out
        _rewrite_cell(batch, cell, per_request, page, dtype)
        qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
        out = kernels[dtype].paged_attention(qkv, layout, batch, cell, 1.0, None).cpu().double().view(heads, dim)
        full = plain.causal_attention(rounded(q, dtype), rounded(k, dtype), rounded(v, dtype), 1.0)[-1]
        torch.testing.assert_close(out, full, **TOLERANCE[dtype])
        torch.testing.assert_close(out[0], rounded(v, dtype)[far, 0], atol=5e-2, rtol=0)


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("window", [None, 21, 64])
@pytest.mark.parametrize("heads,kv_heads,page", [(12, 2, 16), (28, 4, 8), (40, 2, 16), (5, 5, 24), (3, 1, 32), (40, 8, 16), (10, 2, 16), (12, 2, 64), (7, 1, 128)])
def test_prompt_portions_that_share_keys_through_lds(heads, kv_heads, page, window, splits):
    """At head size 128 prompt portions may go to the kernel whose four waves share each step's K and V
    through LDS (pages of a power of two from 16 keys on; the others stay with the kernel above): portions that
    fill its workgroups, that leave waves empty, that end inside a step of 32 keys and that begin long after the
    sequence's start, with and without a window, whole or in three runs of keys that a second kernel merges
    (some of them empty: a request of five keys has one step)."""
    from llmserve_amd.kernels import HipKernels

    dim, dtype = 128, torch.bfloat16
    shared = HipKernels(dtype, shared_portions="always")
    shared.portion_splits = splits
    apart = HipKernels(dtype, shared_portions="never")
    lengths = [130, 97, 33, 300, 64, 5]
    counts = [130, 40, 33, 70, 17, 3]
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=heads)
    if window:
        # blocks that the window has passed are given back in the engine: here their table entries name a page
        # nobody wrote (all NaN), which a kernel that looked there would carry into its sums
        tables = batch.groups[0].block_tables.cpu()
        unwritten = int(torch.isnan(cell.keys.float()).flatten(1).all(dim=1).nonzero()[0])
        for index, (length, count) in enumerate(zip(lengths, counts)):
            tables[index, : max(0, length - count - window + 1) // page] = unwritten
        batch.groups[0].block_tables.copy_(tables)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    scale = 0.11
    out = shared.paged_attention(qkv, layout, batch, cell, scale, window).cpu().double()
    expected = []
    for (q, k, v), count in zip(per_request, counts):
        full = plain.causal_attention(rounded(q, dtype), rounded(k, dtype), rounded(v, dtype), scale, window)
        expected.append(full[-count:].flatten(1))
    torch.testing.assert_close(out, torch.cat(expected), **TOLERANCE[dtype])
    other = apart.paged_attention(qkv, layout, batch, cell, scale, window).cpu().double()
    torch.testing.assert_close(out, other, **TOLERANCE[dtype])


@pytest.mark.parametrize("heads,kv_heads", [(12, 2), (40, 2), (7, 7)])
def test_decoded_tokens_beside_portions_that_share_keys_through_lds(heads, kv_heads):
    """A step of long portions beside single decoded tokens over long contexts: the portions go to the kernel
    that shares K and V through LDS, the decoded tokens to a launch of their own whose keys are cut into runs
    (partial results kept by work item, merged for those rows only); a far key dominates one decoded token."""
    from llmserve_amd.kernels import HipKernels

    dim, page, dtype = 128, 16, torch.bfloat16
    shared = HipKernels(dtype, shared_portions="always")
    lengths, counts = [3100, 4200, 600, 2500, 90], [1, 600, 300, 1, 1]
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=5)
    q, k, v = per_request[0]
    k[40] = 3.0 * q[-1, :: heads // kv_heads]  # for the first query head of every kv head this key dominates
    _rewrite_cell(batch, cell, per_request, page, dtype)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    out = shared.paged_attention(qkv, layout, batch, cell, 1.0, None).cpu().double()
    expected = []
    for (q, k, v), count in zip(per_request, counts):
        full = plain.causal_attention(rounded(q, dtype), rounded(k, dtype), rounded(v, dtype), 1.0, None)
        expected.append(full[-count:].flatten(1))
    torch.testing.assert_close(out, torch.cat(expected), **TOLERANCE[dtype])
    torch.testing.assert_close(out[0].view(heads, dim)[0], rounded(per_request[0][2], dtype)[40, 0], atol=5e-2, rtol=0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("window", [None, 1500])
def test_paged_attention_portion_of_a_long_context(kernels, window, dtype):
    """A portion at the end of a context of more than 4,096 keys (hundreds of steps a wave, many
    pages; in float32 the keys are cut into splits that a second kernel merges), with a far key that
    dominates and, with a window, lies just inside it."""
    heads, kv_heads, dim, page = 6, 2, 64, 16
    lengths, counts = [4200, 37], [150, 37]
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=3)
    q, k, v = per_request[0]
    far = 4199 - 1499 if window else 1
    k[far] = 3.0 * q[-1, ::3]  # for heads 0 and 3 of the last query this key dominates
    _rewrite_cell(batch, cell, per_request, page, dtype)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    out = kernels[dtype].paged_attention(qkv, layout, batch, cell, 1.0, window).cpu().double()
    expected = []
    for (q, k, v), count in zip(per_request, counts):
        full = plain.causal_attention(rounded(q, dtype), rounded(k, dtype), rounded(v, dtype), 1.0, window)
        expected.append(full[-count:].flatten(1))
    torch.testing.assert_close(out, torch.cat(expected), **TOLERANCE[dtype])
    torch.testing.assert_close(out[149].view(heads, dim)[0], rounded(per_request[0][2], dtype)[far, 0], atol=5e-2, rtol=0)


@pytest.mark.parametrize("window", [None, 3000])
def test_float32_decode_attention_over_many_key_splits(kernels, window):
    """Two requests decode over 9,000 and 5,003 keys in float32: few items, so each is cut into several key
    splits (some of them empty for the shorter request, some wholly outside the window) that the merging
    kernel adds up; a far key per request dominates one head."""
    heads, kv_heads, dim, page, dtype = 10, 2, 128, 16, torch.float32
    lengths, counts = [9000, 5003], [1, 1]
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=11)
    fars = [6500, 2100]
    for (q, k, v), far in zip(per_request, fars):
        k[far] = 2.0 * q[-1, ::5]  # heads 0 and 5 share kv heads 0 and 1
    _rewrite_cell(batch, cell, per_request, page, dtype)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    out = kernels[dtype].paged_attention(qkv, layout, batch, cell, 0.5, window).cpu().double()
    for row, ((q, k, v), far) in enumerate(zip(per_request, fars)):
        full = plain.causal_attention(q.double(), k.double(), v.double(), 0.5, window)[-1]
        torch.testing.assert_close(out[row].view(heads, dim), full, **TOLERANCE[dtype])
        torch.testing.assert_close(out[row].view(heads, dim)[0], v.double()[far, 0], atol=5e-2, rtol=0)


@pytest.mark.parametrize("rows,inner,outer", [(3, 100, 77), (8, 8960, 1536), (16, 1536, 48), (11, 2052, 130),
                                              (40, 8960, 200), (200, 4480, 130), (130, 100, 77), (2048, 264, 384),
                                              (129, 2048, 1030)])
def test_float32_products_in_parts_and_at_odd_sizes(kernels, rows, inner, outer):
    """The 32-bit path's products on the matrix cores: K that is a multiple of 4 but not of 16 or 64, rows and
    weight rows that fill no tile, and K cut into partial sums where the result may stay in parts (up to 16 rows:
    the weight-streaming kernel; more: the tiled one), with bias, and with SiLU(gate) * up over interleaved rows.
    The bound is that of a float32 sum of K terms in any order: a few times sqrt(K) * 2^-24 of its size."""
    k = kernels[torch.float32]
    x, w, b = torch.randn(rows, inner), torch.randn(outer, inner) / math.sqrt(inner), torch.randn(outer)
    expected = x.double() @ w.double().T + b.double()
    bound = dict(atol=8 * math.sqrt(inner) * 2.0 ** -24, rtol=1e-5)
    handle = k.prepare_linear([on_gpu(w)], [on_gpu(b)])
    torch.testing.assert_close(k.linear(on_gpu(x), handle).cpu().double(), expected, **bound)
    parts = k.linear(on_gpu(x), handle, out_dtype=torch.float32, partial=True)
    cut = k._float32_splits(rows, outer, inner)
    assert parts.shape == ((cut, rows, outer) if cut > 1 else (rows, outer)) and (cut > 1 or inner < 2048 or rows > 200 or outer > 1000)
    summed = parts if parts.ndim == 2 else parts.double().sum(0)
    torch.testing.assert_close(summed.cpu().double(), expected, **bound)
    up = torch.randn(outer, inner) / math.sqrt(inner)
    gated = k.gated_linear(on_gpu(x), k.prepare_gated_linear(on_gpu(w), on_gpu(up)))
    want = F.silu(x.double() @ w.double().T) * (x.double() @ up.double().T)
    torch.testing.assert_close(gated.cpu().double(), want, **bound)


@pytest.mark.parametrize("inner,outer", [(1536, 2048), (1540, 4098), (260, 9002), (4100, 1030)])
def test_a_float32_row_has_the_same_bits_in_every_batch_of_few_rows(kernels, inner, outer):
    """Up to 64 rows the waves' walks and the order of their sums follow the weight alone: with four, eight and sixteen waves a
    workgroup, a K and weight rows that leave remainders, whole, in parts and gated."""
    k = kernels[torch.float32]
    x, w = on_gpu(torch.randn(64, inner)), on_gpu(torch.randn(outer, inner) / math.sqrt(inner))
    handle, gated = k.prepare_linear([w], [on_gpu(torch.randn(outer))]), k.prepare_gated_linear(w[: outer // 2], w[outer // 2 : outer // 2 * 2])
    forms = [lambda rows: k.linear(rows, handle), lambda rows: k.linear(rows, handle, out_dtype=torch.float32, partial=True), lambda rows: k.gated_linear(rows, gated)]
    for form in forms:
        alone = form(x[:7])
        for rows in (1, 16, 17, 32, 33, 48, 49, 64):
            assert torch.equal(form(x[:rows])[..., : min(rows, 7), :], alone[..., : min(rows, 7), :]), rows
    expected = x.double() @ w.double().T + handle.bias.double()
    torch.testing.assert_close(k.linear(x, handle).double(), expected, atol=8 * math.sqrt(inner) * 2.0 ** -24, rtol=1e-5)


@pytest.mark.parametrize("tile,rows,inner,outer,gated,splits", [
    (0, 70, 512, 42, False, 1), (0, 70, 512, 42, True, 1), (0, 70, 1536, 42, False, 2), (1, 65, 320, 2723, False, 1),
    (1, 65, 320, 2724, True, 1), (1, 65, 512, 6818, False, 2), (2, 66, 512, 2078, False, 1), (2, 97, 512, 1368, True, 1),
    (2, 97, 1536, 690, False, 2), (3, 129, 256, 10887, False, 1), (3, 129, 256, 10888, True, 1), (3, 81, 256, 1590, False, 4),
    (4, 161, 256, 6108, True, 1), (4, 161, 320, 2740, False, 1), (4, 87, 256, 1418, False, 4), (5, 98, 256, 6134, False, 1),
    (5, 98, 256, 6134, True, 1), (5, 97, 512, 3033, False, 2), (6, 65, 256, 19128, True, 1), (6, 65, 320, 18435, False, 1),
    (6, 65, 512, 9270, False, 2),
])
def test_float32_whole_tiles(kernels, tile, rows, inner, outer, gated, splits):
    """The 32-bit product in whole tiles with each of its tiles, where it is picked, over more stages of K than it keeps in LDS (fewer: `test_float32_whole_tiles_over_few_stages`),
    at rows and weight rows that leave remainders: plain, gated and in parts (the bound as above; a gated result's error is that of its two sums)."""
    k = kernels[torch.float32]
    assert k._gemm_f32.llmserve_gemm_f32_tile(rows, outer, inner, splits) == 5 + tile
    generator = torch.Generator(device="cuda").manual_seed(rows + outer)
    x, w = torch.randn(rows, inner, generator=generator, device="cuda"), torch.randn(outer, inner, generator=generator, device="cuda") / math.sqrt(inner)
    bias = torch.randn(outer, generator=generator, device="cuda")
    out = torch.full((splits, rows, outer // 2 if gated else outer), float("nan"), device="cuda")
    status = k._gemm_f32.llmserve_gemm_f32(x.data_ptr(), w.data_ptr(), bias.data_ptr(), out.data_ptr(), int(gated), rows, outer, inner, splits,
                                           torch.cuda.current_stream().cuda_stream)
    assert status == 0
    expected = x.double() @ w.double().T + bias.double()
    if gated:
        expected = F.silu(expected[:, 0::2]) * expected[:, 1::2]
    bound = dict(atol=8 * math.sqrt(inner) * 2.0 ** -24 * (4 if gated else 1), rtol=1e-5)
    torch.testing.assert_close(out.double().sum(0), expected, **bound)


WHOLE_TILES = [(16, 48), (16, 80), (32, 32), (32, 48), (48, 48), (48, 80), (80, 80)]
FEW_FLOAT32_STAGES = [(0, 192), (0, 256), (0, 320), (1, 64), (1, 128), (1, 192), (1, 256), (2, 128), (2, 192), (2, 256), (2, 320),
    (3, 64), (3, 128), (3, 192), (3, 256), (4, 64), (4, 128), (4, 192), (4, 256), (5, 128), (5, 192), (5, 256), (6, 64), (6, 128), (6, 192), (6, 256)]


@pytest.mark.parametrize("tile,inner", FEW_FLOAT32_STAGES)
def test_float32_whole_tiles_over_few_stages(kernels, tile, inner):
    """The whole tiles over as few stages of 64 k as each is picked with, up to one more than it keeps in LDS: result rows that leave in pieces of 16 bytes and rows that
    do not (bound as in `test_float32_whole_tiles`)."""
    k = kernels[torch.float32]
    for multiple in (1, 4):
        rows, outer = sizes_of_a_whole_tile(k, tile, inner, multiple)
        generator = torch.Generator(device="cuda").manual_seed(rows)
        x = torch.randn(rows, inner, generator=generator, device="cuda")
        w = torch.randn(outer, inner, generator=generator, device="cuda") / math.sqrt(inner)
        b = torch.randn(outer, generator=generator, device="cuda")
        out = torch.full((rows, outer), float("nan"), device="cuda")
        status = k._gemm_f32.llmserve_gemm_f32(x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), 0, rows, outer, inner, 1, torch.cuda.current_stream().cuda_stream)
        assert status == 0
        torch.testing.assert_close(out.double(), x.double() @ w.double().T + b.double(), atol=8 * math.sqrt(inner) * 2.0 ** -24, rtol=1e-5)


def sizes_of_a_whole_tile(k, tile, inner, multiple):
    """The smallest of many products that a whole tile is picked for, with a remainder of rows and of weight rows."""
    n, m = WHOLE_TILES[tile]
    draw, best = random.Random(inner + 10 * tile), None
    for _ in range(20000):
        rows, outer = draw.randrange(65, 513), multiple * draw.randrange(17, draw.choice((3000, 20000)) // multiple)
        if rows % m == 0 or outer % n == 0 or (best and rows * outer >= best[0] * best[1]):
            continue
        if k._gemm_f32.llmserve_gemm_f32_tile(rows, outer, inner, 1) == 5 + tile:
            best = rows, outer
    assert best
    return best


@pytest.mark.parametrize("x_from,w_from", [(1, 0), (0, 2), (3, 1)])
@pytest.mark.parametrize("rows,inner,outer", [(70, 512, 48), (129, 256, 10888), (200, 1536, 1536)])
def test_float32_operands_that_begin_inside_a_piece(kernels, rows, inner, outer, x_from, w_from):
    """Contiguous views that begin 4, 8 or 12 bytes into a piece of 16, at sizes of whole tiles, which need whole pieces: plain, gated and in the parts that the library
    takes (the bound as above)."""
    k = kernels[torch.float32]
    generator = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows * inner + 4, generator=generator, device="cuda")[x_from : x_from + rows * inner].view(rows, inner)
    w = torch.randn(outer * inner + 4, generator=generator, device="cuda").div_(math.sqrt(inner))[w_from : w_from + outer * inner].view(outer, inner)
    assert (x.data_ptr() | w.data_ptr()) % 16 and k._gemm_f32.llmserve_gemm_f32_tile(rows, outer, inner, 1) >= 5
    handle = k.prepare_linear([w], None)
    assert handle.weight.data_ptr() == w.data_ptr()
    expected = x.double() @ w.double().T
    bound = dict(atol=8 * math.sqrt(inner) * 2.0 ** -24, rtol=1e-5)
    torch.testing.assert_close(k.linear(x, handle).double(), expected, **bound)
    parts = k.linear(x, handle, out_dtype=torch.float32, partial=True)
    torch.testing.assert_close((parts if parts.ndim == 2 else parts.double().sum(0)), expected, check_dtype=False, **bound)
    out = torch.full((rows, outer // 2), float("nan"), device="cuda")
    assert k._gemm_f32.llmserve_gemm_f32(x.data_ptr(), w.data_ptr(), None, out.data_ptr(), 1, rows, outer, inner, 1, torch.cuda.current_stream().cuda_stream) == 0
    torch.testing.assert_close(out.double(), F.silu(expected[:, 0::2]) * expected[:, 1::2], atol=4 * bound["atol"], rtol=1e-5)


@pytest.mark.parametrize("inner,outer", [(1536, 1536), (8960, 1536), (3584, 3584), (4864, 896)])
@pytest.mark.parametrize("rows", [65, 96, 160, 192, 224, 384, 512])
def test_float32_parts_keep_their_sums_as_short(kernels, rows, inner, outer):
    """A product left in parts is no further from 64 bits than from the kernel that views which begin inside a piece go to, in that one's own parts: an error
    goes with the root of how many k one sum runs over, which parts of K have to keep as short.  (Over a result of 58,000 values and more the norm of the
    error of one and the same order of sums varies by less than 1 percent from draw to draw.)"""
    k = kernels[torch.float32]
    generator = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, inner, generator=generator, device="cuda")
    w = torch.randn(outer, inner, generator=generator, device="cuda") / math.sqrt(inner)
    apart = torch.empty(rows * inner + 1, device="cuda")[1:].view(rows, inner).copy_(x)
    handle, expected = k.prepare_linear([w], None), x.double() @ w.double().T

    def error(rows_of_x):
        parts = k.linear(rows_of_x, handle, out_dtype=torch.float32, partial=True)
        total = parts if parts.ndim == 2 else parts[0].clone()
        for part in parts[1:] if parts.ndim == 3 else ():
            total += part
        return ((total.double() - expected).norm() / expected.norm()).item()

    assert error(x) <= 1.03 * error(apart)


@pytest.mark.parametrize("rows,inner,outer", [(33, 1540, 96), (64, 260, 2050), (65, 1540, 98), (67, 260, 2050), (97, 516, 7003), (129, 1028, 9001), (230, 260, 37890),
                                              (509, 300, 16001), (1000, 300, 8197)])
def test_float32_tiles(kernels, rows, inner, outer):
    """The tiled 32-bit product with each of its five tiles, at rows, weight rows and K that leave remainders (the bound as above)."""
    k = kernels[torch.float32]
    x, w = torch.randn(rows, inner), torch.randn(outer, inner) / math.sqrt(inner)
    expected = x.double() @ w.double().T
    bound = dict(atol=8 * math.sqrt(inner) * 2.0 ** -24, rtol=1e-5)
    handle = k.prepare_linear([on_gpu(w)], None)
    torch.testing.assert_close(k.linear(on_gpu(x), handle).cpu().double(), expected, **bound)
    parts = k.linear(on_gpu(x), handle, out_dtype=torch.float32, partial=True)
    torch.testing.assert_close((parts if parts.ndim == 2 else parts.double().sum(0)).cpu().double(), expected, **bound)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("pairing", ["adjacent", "half", "none"])
@pytest.mark.parametrize("heads,kv_heads,dim,page", [(6, 2, 32, 8), (5, 1, 48, 16), (2, 2, 128, 4)])
def test_rotate_and_store(kernels, dtype, pairing, heads, kv_heads, dim, page):
    lengths, counts = [9, 40, 1], [9, 3, 1]
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype)
    before_keys, before_values = cell.keys.clone(), cell.values.clone()
    rows = step_rows(per_request, counts, heads, kv_heads, dim)
    qkv = on_gpu(rows, dtype)
    theta = 5000.0
    inverse = 1.0 / (theta ** (torch.arange(0, dim, 2).float() / dim))
    kernels[dtype].rotate_and_store(qkv, layout, batch, cell, None if pairing == "none" else on_gpu(inverse), pairing)
    positions = batch.positions.cpu().long()
    view = rounded(rows, dtype).view(-1, heads + 2 * kv_heads, dim)
    angles = plain.rope_angles(dim, theta, positions)
    rotate = {"adjacent": plain.rope_adjacent, "half": plain.rope_half, "none": lambda x, a: x}[pairing]
    expected = torch.cat([rotate(view[:, : heads + kv_heads], angles), view[:, heads + kv_heads :]], dim=1)
    torch.testing.assert_close(qkv.cpu().double().view_as(expected), expected, **TOLERANCE[dtype])
    slots = batch.groups[0].slot_mapping.cpu().long()
    stored_k = key_rows(cell.keys.cpu().double())[slots // page, :, slots % page]
    stored_v = value_rows(cell.values.cpu().double())[slots // page, :, :, slots % page]
    torch.testing.assert_close(stored_k, expected[:, heads : heads + kv_heads], **TOLERANCE[dtype])
    torch.testing.assert_close(stored_v, expected[:, heads + kv_heads :], atol=0, rtol=0)
    untouched = torch.ones(cell.keys.shape[0], page, dtype=torch.bool)
    untouched[slots // page, slots % page] = False
    same = lambda a, b: torch.equal(torch.nan_to_num(a.float().cpu(), nan=7.0), torch.nan_to_num(b.float().cpu(), nan=7.0))
    assert same(key_rows(cell.keys).transpose(1, 2)[untouched], key_rows(before_keys).transpose(1, 2)[untouched])
    assert same(value_rows(cell.values).permute(0, 3, 1, 2)[untouched], value_rows(before_values).permute(0, 3, 1, 2)[untouched])
    # a cell that is only read stores nothing
    readonly = types.SimpleNamespace(writable=False)
    again = on_gpu(rows, dtype)
    kernels[dtype].rotate_and_store(again, layout, batch, readonly, None if pairing == "none" else on_gpu(inverse), pairing)
    torch.testing.assert_close(again, qkv)


@pytest.mark.parametrize("width,parts", [(64, 1), (1536, 3), (4096, 8), (5120, 11), (12292, 2), (16384, 17), (4102, 9)])
def test_add_rms_norm_of_partial_sums(kernels, width, parts):
    """What a product cut over K leaves: [parts, rows, width] partial sums, added in order.  Widths
    with one, two and four pieces a thread, the widest the register-resident kernel takes, and one
    that is no multiple of four (the plain kernel)."""
    rows = 5
    hidden, delta = torch.randn(rows, width), 0.3 * torch.randn(parts, rows, width)
    weight = 1 + 0.2 * torch.randn(width)
    k = kernels[torch.bfloat16]
    device_hidden = on_gpu(hidden.clone())
    out = k.add_rms_norm(device_hidden, on_gpu(delta), on_gpu(weight, torch.bfloat16), 1e-6)
    summed = hidden.double() + delta.double().sum(0)
    torch.testing.assert_close(device_hidden.cpu().double(), summed, atol=2e-6, rtol=1e-6)
    expected = plain.rms_norm(summed, rounded(weight, torch.bfloat16), 1e-6)
    torch.testing.assert_close(out.cpu().double(), expected, **TOLERANCE[torch.bfloat16])
    # a row's result does not depend on how many rows there are
    one = on_gpu(hidden[2:3].clone())
    alone = k.add_rms_norm(one, on_gpu(delta[:, 2:3].contiguous()), on_gpu(weight, torch.bfloat16), 1e-6)
    assert torch.equal(alone[0], out[2]) and torch.equal(one[0], device_hidden[2])


@pytest.mark.parametrize("dtype", DTYPES)
def test_gather_rows(kernels, dtype):
    hidden, delta = torch.randn(9, 100), torch.randn(9, 100)
    rows = torch.tensor([8, 0, 3, 3], dtype=torch.int32)
    out = kernels[dtype].gather_rows(on_gpu(hidden), on_gpu(delta), on_gpu(rows))
    torch.testing.assert_close(out.cpu(), (hidden + delta)[rows.long()])
    torch.testing.assert_close(kernels[dtype].gather_rows(on_gpu(hidden), None, on_gpu(rows)).cpu(), hidden[rows.long()])


@pytest.mark.parametrize("vocab", [5, 1000, 1025, 151936])
def test_argmax_and_sampling(kernels, vocab):
    k = kernels[torch.float32]
    torch.manual_seed(vocab)
    rows = 6
    logits = 3.0 * torch.randn(rows, vocab)
    logits[1, vocab // 2] = logits[1].max() + 1
    logits[2, [3, vocab - 1]] = 50.0  # a tie: the first wins
    assert k.argmax(on_gpu(logits)).cpu().tolist() == logits.argmax(-1).tolist()
    assert k.argmax(on_gpu(logits)).cpu().tolist()[2] == 3
    cases = [(0.0, 1.0), (0.8, 1.0), (0.7, 0.8), (1.5, 0.3), (0.2, 0.95), (1.0, 1.0)]
    for draw in range(12):
        uniforms = [plain.uniform_for(draw, row) for row in range(rows)]
        got = k.sample(
            on_gpu(logits), on_gpu(torch.tensor([c[0] for c in cases])), on_gpu(torch.tensor([c[1] for c in cases])),
            on_gpu(torch.tensor(uniforms)),
        ).cpu().tolist()
        want = [plain.sample(logits[row], cases[row][0], cases[row][1], uniforms[row]) for row in range(rows)]
        assert got == want, (draw, got, want)


def test_sampling_edges(kernels):
    k = kernels[torch.float32]
    logits = torch.tensor([[0.0, 0.0, 0.0, 0.0], [5.0, 1.0, 5.0, 5.0], [1.0, 2.0, 3.0, 4.0]])
    for u, want in ((0.0, [0, 0, 0]), (0.26, [1, 0, 0]), (0.9999, [3, 3, 3])):
        got = k.sample(on_gpu(logits), on_gpu(torch.full((3,), 1.0)), on_gpu(torch.ones(3)), on_gpu(torch.full((3,), u))).cpu().tolist()
        assert got[0] == want[0] and got[2] == plain.sample(logits[2], 1.0, 1.0, u)
    # top-p with ties: equal entries are kept in index order until the mass is reached
    for u in (0.0, 0.3, 0.4, 0.7, 0.99):
        got = k.sample(on_gpu(logits), on_gpu(torch.full((3,), 1.0)), on_gpu(torch.full((3,), 0.6)), on_gpu(torch.full((3,), u))).cpu().tolist()
        want = [plain.sample(logits[row], 1.0, 0.6, u) for row in range(3)]
        assert got == want, (u, got, want)


def test_sampling_refuses_a_workspace_that_is_too_small(kernels):
    from llmserve_amd.kernels.hip import _pointer

    k = kernels[torch.float32]
    library = k._sampling_library()
    rows, vocab = 5, 1000
    kib = library.llmserve_sample_workspace_kib(rows, vocab)
    assert kib > rows * vocab * 4 // 1024 and library.llmserve_sample_workspace_kib(0, vocab) < 0
    logits, values, out = torch.randn(rows, vocab).cuda(), torch.full((rows,), 0.5).cuda(), torch.zeros(rows, dtype=torch.int32).cuda()
    workspace = torch.empty(kib * 1024, dtype=torch.uint8, device="cuda")
    arguments = lambda space, size: (_pointer(logits), _pointer(values), _pointer(values), _pointer(values), space, size, _pointer(out), rows, vocab, 1, k._stream)
    assert library.llmserve_sample(*arguments(_pointer(workspace), kib - 1)) == 1001
    assert library.llmserve_sample(*arguments(None, kib)) == 1001
    assert library.llmserve_sample(*arguments(_pointer(workspace) + 16, kib)) == 1001  # not aligned to 256 bytes
    assert library.llmserve_sample(*arguments(_pointer(workspace), kib)) == 0
    torch.cuda.synchronize()
    assert all(0 <= token < vocab for token in out.cpu().tolist())


@pytest.mark.parametrize("rows,vocab", [(70, 1025), (300, 130), (3, 40000)])
def test_sampling_of_many_rows_and_hard_rows(kernels, rows, vocab):
    """The stages cut a row into fewer pieces when there are many rows; rows whose entries are all
    equal, tie in groups, underflow to zero or to subnormal numbers, or hold one entry far above the
    rest must come out as the plain rule says; and leaving the top-p stages out changes nothing for
    rows without top-p."""
    k = kernels[torch.float32]
    torch.manual_seed(rows + vocab)
    logits = 2.0 * torch.randn(rows, vocab)
    # all equal, as many as a power of two (the plain rule rounds p = 1 / n to float32 before it adds, the kernel
    # divides nothing: with every entry tied they agree only where 1 / n is exact); the rest can never come
    equal = 1 << (vocab.bit_length() - 1)
    logits[0] = 1.5
    logits[0, equal:] = -float("inf")
    if vocab <= 2048:
        # four values, many ties.  Not at the large size: float32 softmax, which the plain rule starts from, is
        # off from a sum of 1 by a few parts in a million there, and among ten thousand tied entries that
        # moves the end of the kept set by an entry; the kernel normalises nothing and has no such error
        logits[1] = torch.randint(0, 4, (vocab,)).float()
    logits[2, 1:] -= 200.0  # everything but one entry underflows
    logits[2, 0] = 3.0
    if rows > 3:
        logits[3] = torch.linspace(-180.0, 0.0, vocab)  # the low end is subnormal or zero after exp
        logits[4, vocab // 3] += 30.0
    temperatures = [(0.0, 0.6, 1.0, 1.7)[row % 4] for row in range(rows)]
    temperatures[0], temperatures[1], temperatures[2] = 1.0, 0.9, 1.0
    top_ps = [(1.0, 0.9, 0.5, 0.05, 0.999)[row % 5] for row in range(rows)]
    top_ps[0], top_ps[1] = 0.5, 0.7
    for draw in range(3):
        uniforms = [plain.uniform_for(draw + 20, row) for row in range(rows)]
        if draw == 2:
            uniforms[0], uniforms[1] = 0.0, 0.999999
        got = k.sample(on_gpu(logits), on_gpu(torch.tensor(temperatures)), on_gpu(torch.tensor(top_ps)), on_gpu(torch.tensor(uniforms))).cpu().tolist()
        want = [plain.sample(logits[row], temperatures[row], top_ps[row], uniforms[row]) for row in range(rows)]
        assert got == want, (draw, [(row, a, b) for row, (a, b) in enumerate(zip(got, want)) if a != b])
        ones = [1.0] * rows
        got = k.sample(on_gpu(logits), on_gpu(torch.tensor(temperatures)), on_gpu(torch.tensor(ones)), on_gpu(torch.tensor(uniforms)), False).cpu().tolist()
        want = k.sample(on_gpu(logits), on_gpu(torch.tensor(temperatures)), on_gpu(torch.tensor(ones)), on_gpu(torch.tensor(uniforms))).cpu().tolist()
        assert got == want
        assert got == [plain.sample(logits[row], temperatures[row], 1.0, uniforms[row]) for row in range(rows)]


@pytest.mark.parametrize("pairing", ["adjacent", "half", "none"])
@pytest.mark.parametrize("heads,kv_heads,dim,page", [(12, 2, 128, 16), (6, 1, 64, 8), (5, 5, 32, 4), (4, 2, 48, 16), (40, 2, 64, 16), (2, 1, 256, 16), (40, 8, 128, 16), (10, 2, 128, 16), (28, 4, 128, 16)])
def test_fused_decode_attention(kernels, pairing, heads, kv_heads, dim, page):
    """A step of single tokens: rotation, the store of the new key and value, attention and the
    merge of key splits in one kernel (or, where the sizes do not allow it, in the separate ones):
    the result and the pages must be what the separate steps give."""
    dtype = torch.bfloat16
    lengths = [1, 2, page, page + 1, 33, 64, 65, 700, 301]
    counts = [1] * len(lengths)
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=dim + page)
    theta = 800.0
    inverse = 1.0 / (theta ** (torch.arange(0, dim, 2).float() / dim))
    rotate = {"adjacent": plain.rope_adjacent, "half": plain.rope_half, "none": lambda x, a: x}[pairing]
    # the pages hold the earlier tokens' keys already rotated; the new token's slot holds garbage
    expected = []
    for index, (q, k, v) in enumerate(per_request):
        angles = plain.rope_angles(dim, theta, torch.arange(q.shape[0]))
        k_rot = rotate(rounded(k, dtype), angles).to(dtype).double()
        q_rot = rotate(rounded(q, dtype), angles).to(dtype).double()
        per_request[index] = (q, k_rot.float(), v)
        full = plain.causal_attention(q_rot, k_rot, rounded(v, dtype), 0.2)
        expected.append(full[-1:].flatten(1))
    _rewrite_cell(batch, cell, per_request, page, dtype)
    slots = batch.groups[0].slot_mapping.cpu().long()
    cell.keys[slots // page, :, :, slots % page] = float("nan")
    cell.put_value_rows(slots // page, slots % page, torch.full((len(slots), cell.values.shape[1], cell.values.shape[3]), float("nan"), device=cell.values.device))
    rows = []  # the step's rows carry unrotated q and k
    for (q, k, v), original in zip(per_request, [p[1] for p in paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=dim + page)[2]]):
        rows.append(torch.cat([q[-1:].flatten(1), original[-1:].flatten(1), v[-1:].flatten(1)], dim=1))
    qkv = on_gpu(torch.cat(rows), dtype)
    out = kernels[dtype].rotate_store_attend(qkv, layout, batch, cell, None if pairing == "none" else on_gpu(inverse), pairing, 0.2, None)
    torch.testing.assert_close(out.cpu().double(), torch.cat(expected), **TOLERANCE[dtype])
    stored_k = key_rows(cell.keys.cpu().double())[slots // page, :, slots % page]
    stored_v = value_rows(cell.values.cpu().double())[slots // page, :, :, slots % page]
    want_k = torch.stack([p[1][-1].double() for p in per_request])
    want_v = torch.stack([rounded(p[2][-1], dtype) for p in per_request])
    torch.testing.assert_close(stored_k, want_k, **TOLERANCE[dtype])
    torch.testing.assert_close(stored_v, want_v, atol=0, rtol=0)


@pytest.mark.parametrize("requests", [3, 12])
def test_fused_decode_attention_over_long_contexts(kernels, requests):
    """Single tokens against thousands of keys: the one-kernel decode step cuts the keys over several
    workgroups and merges them.  Every request has one far key made to dominate two of its heads (the
    value stored there must come out), at a place that differs from request to request, first and
    last keys and the edges of the cuts among them; the other heads are compared with plain attention."""
    dtype, heads, kv_heads, dim, page = torch.bfloat16, 12, 2, 128, 16
    lengths = [4100, 2049, 3333] + [1500 + 37 * i for i in range(requests - 3)]
    counts = [1] * len(lengths)
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=requests)
    places = [0, 2048, 3332] + [(211 * i) % 1500 for i in range(requests - 3)]
    for (q, k, v), far in zip(per_request, places):
        k[far] = 3.0 * q[-1, ::6]  # kv head g takes the query of its first head: heads 0 and 6 find this key
    _rewrite_cell(batch, cell, per_request, page, dtype)
    slots = batch.groups[0].slot_mapping.cpu().long()
    cell.keys[slots // page, :, :, slots % page] = float("nan")  # the step itself stores the newest key and value
    cell.put_value_rows(slots // page, slots % page, torch.full((len(slots), cell.values.shape[1], cell.values.shape[3]), float("nan"), device=cell.values.device))
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    out = kernels[dtype].rotate_store_attend(qkv, layout, batch, cell, None, "none", 1.0, None).cpu().double()
    for index, ((q, k, v), far) in enumerate(zip(per_request, places)):
        full = plain.causal_attention(rounded(q, dtype), rounded(k, dtype), rounded(v, dtype), 1.0)[-1]
        got = out[index].view(heads, dim)
        torch.testing.assert_close(got, full, **TOLERANCE[dtype])
        for head in (0, 6):
            torch.testing.assert_close(got[head], rounded(v, dtype)[far, head // 6], atol=0.05, rtol=0.05)


def test_fused_decode_attention_over_tens_of_thousands_of_keys(kernels):
    """Beyond 4,096 keys a decode step cuts the keys into five to sixty-four parts and a kernel of its own
    merges them (up to there, at up to 16 rows, the output projection does).  Two requests of 30,000 and 9,000 keys, a
    far key planted to dominate heads 0 and 6 of each (deep inside the long one, near the start of the
    other): the value stored there must come out, and every head must agree with plain attention of the
    last token over all keys."""
    dtype, heads, kv_heads, dim, page = torch.bfloat16, 12, 2, 128, 16
    lengths, counts, places = [30000, 9000] + [30000 - 100 * i for i in range(6)], [1] * 8, [23456, 100] + [29000 - 4000 * i for i in range(6)]
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=30)
    for (q, k, v), far in zip(per_request, places):
        k[far] = 3.0 * q[-1, ::6]
    _rewrite_cell(batch, cell, per_request, page, dtype)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    out = kernels[dtype].rotate_store_attend(qkv, layout, batch, cell, None, "none", 1.0, None).cpu().double()
    for index, ((q, k, v), far) in enumerate(zip(per_request, places)):
        last = rounded(q, dtype)[-1]  # [heads, dim]
        all_keys = rounded(k, dtype).repeat_interleave(heads // kv_heads, dim=1)  # [T, heads, dim]
        all_values = rounded(v, dtype).repeat_interleave(heads // kv_heads, dim=1)
        weights = torch.softmax(torch.einsum("hd,thd->ht", last, all_keys), dim=-1)
        want = torch.einsum("ht,thd->hd", weights, all_values)
        got = out[index].view(heads, dim)
        torch.testing.assert_close(got, want, **TOLERANCE[dtype])
        for head in (0, 6):
            torch.testing.assert_close(got[head], rounded(v, dtype)[far, head // 6], atol=0.05, rtol=0.05)
    # Keys of zero: every key weighs the same and the result is the mean of all values, which the
    # kernel's arithmetic gives almost exactly (weights of 1, sums in float32), so that thirty-two keys
    # left out anywhere would show (a value is of order one, the mean of 30,000 of order 0.006).
    for q, k, v in per_request:
        k.zero_()
    _rewrite_cell(batch, cell, per_request, page, dtype)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    out = kernels[dtype].rotate_store_attend(qkv, layout, batch, cell, None, "none", 1.0, None).cpu().double()
    for index, (q, k, v) in enumerate(per_request):
        want = rounded(v, dtype).mean(0).repeat_interleave(heads // kv_heads, dim=0)  # [heads, dim]
        torch.testing.assert_close(out[index].view(heads, dim), want, atol=6e-5, rtol=5e-3)


@pytest.mark.parametrize("heads,kv_heads,outer,requests", [(12, 2, 1536, 8), (40, 8, 272, 16), (28, 4, 1000, 3), (2, 1, 100, 1)])
def test_decode_attention_whose_key_splits_the_output_projection_merges(kernels, heads, kv_heads, outer, requests):
    """A step of up to 16 single tokens at head size 128 followed by the output projection: the attention
    leaves its key splits unmerged and the product merges them while it loads its x.  Contexts from one
    key (all splits but one see no key) to thousands, a far key planted to dominate a head; against
    plain attention followed by the plain product, and against the library's own unfused pair."""
    from llmserve_amd.kernels import HipKernels

    dtype, dim, page = torch.bfloat16, 128, 16
    lengths = ([1, 2, 700, 33, 2049, 301, 64, 17, 4100, 530, 65, 1500, 5, 999, 129, 48])[:requests]
    counts = [1] * requests
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=heads)
    for q, k, v in per_request:
        if k.shape[0] > 40:
            k[k.shape[0] // 3] = 3.0 * q[-1, :: heads // kv_heads]  # the first head of every kv head finds this key
    _rewrite_cell(batch, cell, per_request, page, dtype)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    weight, bias = torch.randn(outer, heads * dim) / math.sqrt(heads * dim), torch.randn(outer)
    k = kernels[dtype]
    project = k.prepare_linear([on_gpu(weight, dtype)], [on_gpu(bias, dtype)])
    got = k.rotate_store_attend(qkv.clone(), layout, batch, cell, None, "none", 0.3, None, project=project)
    got = (got if got.ndim == 2 else got.sum(0)).cpu().double()
    attended = torch.cat([
        plain.causal_attention(rounded(q, dtype), rounded(key, dtype), rounded(v, dtype), 0.3)[-1:].flatten(1)
        for q, key, v in per_request
    ])
    expected = attended @ rounded(weight, dtype).T + rounded(bias, dtype)
    # the attention's output is rounded to bfloat16 on its way into the product (once, or twice where splits
    # are merged): 2^-8 of values of order 1, through a product whose weights have unit row norm
    torch.testing.assert_close(got, expected, atol=2e-2, rtol=2e-2)
    apart = HipKernels(dtype)
    apart.merge_in_product = False
    other = apart.rotate_store_attend(qkv.clone(), layout, batch, cell, None, "none", 0.3, None, project=project)
    other = (other if other.ndim == 2 else other.sum(0)).cpu().double()
    torch.testing.assert_close(got, other, atol=1e-2, rtol=1e-2)
    assert float((got - expected).abs().mean()) < 1.5 * float((other - expected).abs().mean()) + 1e-4


@pytest.mark.parametrize("rows,inner,outer", [(130, 16384, 72), (600, 8960, 200), (70, 16448, 40)])
def test_library_products_cut_over_a_long_k(kernels, rows, inner, outer):
    """A product with a long K beside few weight rows goes to the library as a strided batch over slices of K
    and comes back as partial sums for the reader to add; the sum is the product."""
    from llmserve_amd.kernels import HipKernels

    dtype = torch.bfloat16
    k = kernels[dtype]
    assert HipKernels._library_splits(rows, outer, inner) > 1
    x, w = torch.randn(rows, inner), torch.randn(outer, inner) / math.sqrt(inner)
    handle = k.prepare_linear([on_gpu(w, dtype)], None)
    parts = k.linear(on_gpu(x, dtype), handle, out_dtype=torch.float32, partial=True)
    assert parts.ndim == 3 and parts.shape[1:] == (rows, outer)
    expected = rounded(x, dtype) @ rounded(w, dtype).T
    torch.testing.assert_close(parts.sum(0).cpu().double(), expected, atol=1e-3, rtol=1e-3)
    whole = k.linear(on_gpu(x, dtype), handle, out_dtype=torch.float32)
    assert whole.ndim == 2
    torch.testing.assert_close(whole.cpu().double(), expected, atol=1e-3, rtol=1e-3)
    # the norm that follows adds the parts in order
    hidden = torch.randn(rows, outer)
    device_hidden = hidden.cuda()
    normed = k.add_rms_norm(device_hidden, parts, on_gpu(torch.ones(outer), dtype), 1e-6)
    torch.testing.assert_close(device_hidden.cpu().double(), hidden.double() + expected, atol=2e-3, rtol=1e-3)
    torch.testing.assert_close(normed.cpu().double(), plain.rms_norm(hidden.double() + expected, torch.ones(outer).double(), 1e-6), **TOLERANCE[dtype])


@pytest.mark.parametrize("rows", [1, 7, 16, 17, 40, 64])
@pytest.mark.parametrize("outer,inner,gated,splits,bias", [
    (40, 128, False, 1, None), (1000, 384, False, 1, "bfloat16"), (4610, 3584, False, 1, "float32"),  # two tiles a wave
    (154, 2560, False, 5, None), (318, 256, True, 1, None), (6000, 1536, True, 1, None),
])
def test_products_streamed_through_lds(kernels, rows, outer, inner, gated, splits, bias):
    """The product for up to 64 rows that brings weights and x through LDS, quad by quad, alone: odd
    numbers of weight rows (the last tile is cut), one and two tiles a wave, one, two and four tiles of
    x (the last one cut), a bias of either type, K cut into partial sums, SiLU(gate) * up over
    interleaved rows; against the plain product."""
    from llmserve_amd.kernels.hip import _check, _pointer

    k = kernels[torch.bfloat16]
    x, w = torch.randn(rows, inner), torch.randn(outer, inner) / math.sqrt(inner)
    b = None if bias is None else torch.randn(outer)
    device_x, device_w = on_gpu(x, torch.bfloat16), on_gpu(w, torch.bfloat16)
    device_b = None if b is None else on_gpu(b, getattr(torch, bias))
    float_out = splits > 1 or bias == "float32"
    out = torch.full((splits, rows, outer // 2 if gated else outer), float("nan"), device="cuda",
                     dtype=torch.float32 if float_out else torch.bfloat16)
    status = k._gemm_bf16.llmserve_gemm_stream(
        _pointer(device_x), _pointer(device_w), _pointer(device_b), int(bias == "float32"), _pointer(out), int(float_out),
        int(gated), rows, outer, inner, splits, k._stream,
    )
    _check(status, "gemm_stream")
    expected = rounded(x, torch.bfloat16) @ rounded(w, torch.bfloat16).T
    if b is not None:
        expected = expected + rounded(b, getattr(torch, bias))
    if gated:
        expected = torch.nn.functional.silu(expected[:, 0::2]) * expected[:, 1::2]  # weight rows alternate gate, up
    got = out.sum(0).cpu().double()
    tolerance = dict(atol=2e-3, rtol=2e-3) if float_out else TOLERANCE[torch.bfloat16]
    torch.testing.assert_close(got, expected, **tolerance)
    # and it refuses what it cannot take: more than 64 rows, a K that is no multiple of 128
    assert k._gemm_bf16.llmserve_gemm_stream(_pointer(device_x), _pointer(device_w), None, 0, _pointer(out), int(float_out),
                                             0, 65, outer, inner, 1, k._stream) != 0
    assert k._gemm_bf16.llmserve_gemm_stream(_pointer(device_x), _pointer(device_w), None, 0, _pointer(out), int(float_out),
                                             0, rows, outer, inner - 32, 1, k._stream) != 0


@pytest.mark.parametrize("rows", [24, 33, 64])
@pytest.mark.parametrize("tiles,steps", [(1, 1), (1, 2), (2, 1), (2, 2), (4, 1)])
def test_streamed_products_of_many_rows_in_every_shape(kernels, rows, tiles, steps):
    """The same kernel at 17 to 64 rows with every shape it is built in (weight tiles a workgroup, steps
    a group), plain with a bias and gated, and through the entry point that the engine's small products
    of such steps take."""
    from llmserve_amd.kernels.hip import _check, _pointer

    k = kernels[torch.bfloat16]
    outer, inner = 1210, 640
    x, w, b = torch.randn(rows, inner), torch.randn(outer, inner) / math.sqrt(inner), torch.randn(outer)
    device_x, device_w, device_b = on_gpu(x, torch.bfloat16), on_gpu(w, torch.bfloat16), on_gpu(b, torch.bfloat16)
    expected = rounded(x, torch.bfloat16) @ rounded(w, torch.bfloat16).T
    for gated in (False, True):
        want = expected + rounded(b, torch.bfloat16)
        if gated:
            want = torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2]
        out = torch.full((rows, outer // 2 if gated else outer), float("nan"), device="cuda", dtype=torch.bfloat16)
        status = k._gemm_bf16.llmserve_gemm_stream_shaped(
            _pointer(device_x), _pointer(device_w), _pointer(device_b), 0, _pointer(out), 0, int(gated), rows, outer,
            inner, 1, tiles, steps, k._stream,
        )
        _check(status, "gemm_stream_shaped")
        torch.testing.assert_close(out.cpu().double(), want, **TOLERANCE[torch.bfloat16])
    out = torch.full((rows, outer), float("nan"), device="cuda", dtype=torch.bfloat16)
    status = k._gemm_bf16.llmserve_gemm_skinny(
        _pointer(device_x), _pointer(device_w), _pointer(device_b), 0, _pointer(out), 0, 0, rows, outer, inner, 1, k._stream,
    )
    _check(status, "gemm_skinny")
    torch.testing.assert_close(out.cpu().double(), expected + rounded(b, torch.bfloat16), **TOLERANCE[torch.bfloat16])
    # and with K cut into partial sums (what the output projection of such a step asks for)
    for splits in (2, 5):
        parts = torch.full((splits, rows, outer), float("nan"), device="cuda", dtype=torch.float32)
        status = k._gemm_bf16.llmserve_gemm_skinny(
            _pointer(device_x), _pointer(device_w), None, 0, _pointer(parts), 1, 0, rows, outer, inner, splits, k._stream,
        )
        _check(status, "gemm_skinny in parts")
        torch.testing.assert_close(parts.sum(0).cpu().double(), expected, atol=2e-3, rtol=2e-3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("pairing", ["adjacent", "half"])
@pytest.mark.parametrize("heads,kv_heads,dim,page,lengths,counts", [
    (12, 2, 128, 16, [700, 301, 40, 2100], [150, 1, 40, 33]),   # portions beside a decoded token, packed columns
    (28, 4, 128, 16, [512] * 9, [512] * 9),                     # many whole prompts: the kernel that shares K and V through LDS
    (6, 1, 64, 8, [90, 17], [90, 2]),
    (40, 2, 64, 16, [130, 64], [30, 64]),                       # more than 16 query heads a kv head
    (4, 2, 48, 16, [70, 5], [70, 5]),
])
def test_rotation_store_and_attention_of_prompt_portions(kernels, dtype, pairing, heads, kv_heads, dim, page, lengths, counts):
    """`rotate_store_attend` on steps that are not single tokens (rotation and store, then attention).
    The step's rows carry unrotated q and k, the pages hold the earlier tokens' rotated keys and garbage
    where the step's will go; results and pages against the plain implementation."""
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=dim + heads)
    originals = [(q.clone(), k.clone(), v.clone()) for q, k, v in per_request]
    theta = 3000.0
    inverse = 1.0 / (theta ** (torch.arange(0, dim, 2).float() / dim))
    rotate = {"adjacent": plain.rope_adjacent, "half": plain.rope_half}[pairing]
    expected, rotated_keys = [], []
    for index, (q, k, v) in enumerate(per_request):
        angles = plain.rope_angles(dim, theta, torch.arange(q.shape[0]))
        k_rot = rotate(rounded(k, dtype), angles).to(dtype).double()
        q_rot = rotate(rounded(q, dtype), angles).to(dtype).double()
        per_request[index] = (q, k_rot.float(), v)
        rotated_keys.append(k_rot)
        full = plain.causal_attention(q_rot, k_rot, rounded(v, dtype), 0.2)
        expected.append(full[-counts[index]:].flatten(1))
    _rewrite_cell(batch, cell, per_request, page, dtype)
    slots = batch.groups[0].slot_mapping.cpu().long()
    cell.keys[slots // page, :, :, slots % page] = float("nan")  # the step stores these itself
    cell.put_value_rows(slots // page, slots % page, torch.full((len(slots), cell.values.shape[1], cell.values.shape[3]), float("nan"), device=cell.values.device))
    qkv = on_gpu(step_rows(originals, counts, heads, kv_heads, dim), dtype)
    out = kernels[dtype].rotate_store_attend(qkv, layout, batch, cell, on_gpu(inverse), pairing, 0.2, None)
    torch.testing.assert_close(out.cpu().double(), torch.cat(expected), **TOLERANCE[dtype])
    stored_k = key_rows(cell.keys.cpu().double())[slots // page, :, slots % page]
    stored_v = value_rows(cell.values.cpu().double())[slots // page, :, :, slots % page]
    want_k = torch.cat([k_rot[-count:] for k_rot, count in zip(rotated_keys, counts)])
    want_v = torch.cat([rounded(v, dtype)[-count:] for (q, k, v), count in zip(originals, counts)])
    torch.testing.assert_close(stored_k, want_k, **TOLERANCE[dtype])
    torch.testing.assert_close(stored_v, want_v, atol=0, rtol=0)


@pytest.mark.parametrize("with_bias", [torch.bfloat16, torch.float32, None])
@pytest.mark.parametrize("heads,kv_heads,dim,page,inner,counts", [
    (12, 2, 128, 16, 1536, [65]),              # tiles of 64 x 32, the last of one row
    (12, 2, 128, 16, 256, [33, 1, 223]),       # nine of them down, then too many: 64 x 64
    (2, 1, 16, 8, 64, [90, 7]),                # fewer columns than a tile, one stage
    (5, 3, 48, 24, 128, [70, 50]),             # heads across the tiles' edges, a page that is no power of two
    (4, 2, 80, 4, 192, [66, 3]),               # pages of less than a piece of values
    (14, 2, 64, 16, 896, [40, 9, 980]),        # 128 x 64
    (12, 2, 128, 16, 128, [7, 1026]),          # 128 x 128
    (12, 2, 128, 16, 96, [130, 30]),           # half a stage at the end of K
])
def test_product_rotated_and_stored_in_one_kernel(kernels, monkeypatch, heads, kv_heads, dim, page, inner, counts, with_bias):
    """`linear_rotated` against the product in 64 bits, rounded to bfloat16, rotated.  The sums are float32, so what is rotated may be the
    neighbouring bfloat16 (2^-7 of it), which a rotation keeps within 2^-7 of the pair's length, and the result is rounded once more (2^-8):
    together below 2^-6.  Values are rounded once.  Pages hold the rows' keys and values bit for bit; slots of no token stay as they were."""
    dtype = torch.bfloat16
    lengths = [count + 5 * index for index, count in enumerate(counts)]
    batch, cell, _, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=dim + heads)
    rows, generator = sum(counts), torch.Generator().manual_seed(inner)
    x = torch.randn(rows, inner, generator=generator).to(dtype)
    weight = (torch.randn(layout.width, inner, generator=generator) * inner ** -0.5).to(dtype)
    bias = None if with_bias is None else torch.randn(layout.width, generator=generator).to(with_bias)
    batch.groups[0].slot_mapping[3] = -1  # (a row that is not stored)
    slots = batch.groups[0].slot_mapping.cpu().long()
    before_k, before_v = key_rows(cell.keys.cpu().float()).clone(), value_rows(cell.values.cpu().float()).clone()
    library = kernels[dtype]
    prepared = library.prepare_linear([on_gpu(weight, dtype)], [on_gpu(bias, with_bias)] if bias is not None else None)
    inverse = 1.0 / (3000.0 ** (torch.arange(0, dim, 2).float() / dim))
    monkeypatch.setattr(type(library), "_rotated_ahead", staticmethod(lambda *sizes: True))  # every size, not only where it is ahead
    got = library.linear_rotated(x.cuda(), prepared, layout, batch, cell, on_gpu(inverse), "adjacent")
    assert got is not None
    got = got.cpu().double()
    exact = x.double() @ weight.double().T + (bias.double() if bias is not None else 0)
    split = (heads + kv_heads) * dim
    turned = exact.to(dtype).double()[:, :split].unflatten(1, (-1, dim))
    angles = plain.rope_angles(dim, 3000.0, batch.positions.cpu().long())
    turned = plain.rope_adjacent(turned, angles)
    lengths_of_pairs = turned.unflatten(2, (-1, 2)).norm(dim=-1, keepdim=True).expand(-1, -1, -1, 2).flatten(2)
    assert ((got[:, :split].unflatten(1, (-1, dim)) - turned).abs() <= lengths_of_pairs * 2.0 ** -6 + 1e-4).all()
    assert ((got[:, split:] - exact[:, split:]).abs() <= exact[:, split:].abs() * 2.0 ** -8 + 1e-4).all()
    stored = slots >= 0
    k, v = got[:, heads * dim : split].unflatten(1, (-1, dim)), got[:, split:].unflatten(1, (-1, dim))
    now_k, now_v = key_rows(cell.keys.cpu().float()), value_rows(cell.values.cpu().float())
    before_k[slots[stored] // page, :, slots[stored] % page] = k[stored].float()
    before_v[slots[stored] // page, :, :, slots[stored] % page] = v[stored].float()
    assert torch.equal(now_k.nan_to_num(7e7), before_k.nan_to_num(7e7)) and torch.equal(now_v.nan_to_num(7e7), before_v.nan_to_num(7e7))


@pytest.mark.parametrize("heads,kv_heads,dim,inner,counts", [
    (12, 2, 128, 256, [65, 448]),      # 64 x 64
    (12, 2, 128, 128, [7, 1026]),      # 128 x 128
    (5, 3, 48, 128, [700]),            # heads across the tiles' edges
    (14, 2, 64, 896, [40, 9, 980]),    # 128 x 64
])
def test_product_rotated_and_stored_has_the_bits_of_its_two_kernels(kernels, monkeypatch, heads, kv_heads, dim, inner, counts):
    """The tiled product's sums are the same in every tile, and a rotation rounds in the same places in either kernel, so that rows and pages
    are those of the product and of the kernel behind it, bit for bit."""
    dtype, page = torch.bfloat16, 16
    library, rows, generator = kernels[dtype], sum(counts), torch.Generator().manual_seed(rows_seed := inner + dim)
    x = torch.randn(rows, inner, generator=generator).to(dtype).cuda()
    monkeypatch.setattr(type(library), "_rotated_ahead", staticmethod(lambda *sizes: True))
    inverse = on_gpu(1.0 / (3000.0 ** (torch.arange(0, dim, 2).float() / dim)))
    found = []
    for fused in (False, True):
        batch, cell, _, layout = paged_case([count + 5 for count in counts], counts, heads, kv_heads, dim, page, dtype, shuffle_seed=rows_seed)
        generator.manual_seed(rows_seed)
        weight = (torch.randn(layout.width, inner, generator=generator) * inner ** -0.5).to(dtype)
        prepared = library.prepare_linear([on_gpu(weight, dtype)], [on_gpu(torch.randn(layout.width, generator=generator), dtype)])
        if fused:
            qkv = library.linear_rotated(x, prepared, layout, batch, cell, inverse, "adjacent")
        else:
            qkv = torch.empty(rows, layout.width, dtype=dtype, device="cuda")
            assert library._gemm_blocks.llmserve_gemm_blocks(
                x.data_ptr(), prepared.weight.data_ptr(), prepared.bias.data_ptr(), 0, qkv.data_ptr(), 0, 0, rows, layout.width, inner, 1, library._stream) == 0
            library.rotate_and_store(qkv, layout, batch, cell, inverse, "adjacent")
        found.append((qkv, cell.keys.float().nan_to_num(7e7), cell.values.float().nan_to_num(7e7)))
    assert all(torch.equal(apart, together) for apart, together in zip(*found))


def test_product_rotated_and_stored_refuses_bad_sizes(kernels):
    from llmserve_amd.kernels.hip import _pointer

    k = kernels[torch.bfloat16]
    x, w, out, table, pages = (torch.zeros(4096, device="cuda") for _ in range(5))
    slots = torch.zeros(4, dtype=torch.int32, device="cuda")

    def status(inner=64, heads=1, kv_heads=1, dim=16, page=16, keys=pages.data_ptr(), angles=table.data_ptr()):
        return k._gemm_blocks.llmserve_gemm_rotated(_pointer(x), _pointer(w), None, 0, _pointer(out), 1, inner, angles, heads, kv_heads, dim,
                                                    keys, pages.data_ptr(), _pointer(slots), page, k._stream)

    for wrong in (dict(inner=48), dict(inner=0), dict(heads=0), dict(kv_heads=0), dict(dim=24), dict(dim=0), dict(page=0), dict(keys=None),
                  dict(angles=None), dict(keys=pages.data_ptr() + 8)):
        assert status(**wrong) == 1001
    assert status() == 0


@pytest.mark.parametrize("heads,kv_heads,dim,window", [(6, 2, 64, None), (6, 1, 128, None), (8, 4, 128, 2048), (5, 1, 32, None), (4, 2, 160, None)])
@pytest.mark.parametrize("lengths,counts", [([3000, 20, 2100, 700, 1], [1, 20, 60, 1, 1]), ([520, 9, 300], [200, 9, 1]), ([4200, 2050], [1, 33])])
def test_portions_beside_long_contexts(kernels, heads, kv_heads, dim, window, lengths, counts):
    """A step of portions and decoded tokens whose longest walks are cut into runs that a second kernel merges (short requests
    in it have no key in the later runs), and whose tiles are walked by eight waves; against the plain attention."""
    dtype, page = torch.bfloat16, 16
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=dim)
    out = kernels[dtype].paged_attention(on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype), layout, batch, cell, dim ** -0.5, window)
    expected = []
    for (q, k, v), count in zip(per_request, counts):
        q, k, v = (rounded(rows, dtype).double() for rows in (q[-count:], k, v))
        k, v = (rows.repeat_interleave(heads // kv_heads, 1).transpose(0, 1) for rows in (k, v))
        distance = torch.arange(k.shape[1] - count, k.shape[1])[:, None] - torch.arange(k.shape[1])[None]
        scores = (q.transpose(0, 1) @ k.transpose(1, 2) * dim ** -0.5).masked_fill((distance < 0) | (distance >= (window or 1 << 30)), -math.inf)
        expected.append((scores.softmax(-1) @ v).transpose(0, 1).flatten(1))
    torch.testing.assert_close(out.cpu().double(), torch.cat(expected), **TOLERANCE[dtype])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("activation", ["silu", "gelu", "gelu_tanh", "relu"])
@pytest.mark.parametrize("rows,inner,outer", [(5, 96, 200), (16, 512, 520), (40, 128, 264), (70, 64, 333), (300, 128, 1000)])
def test_gated_products_with_every_gate_activation(kernels, dtype, activation, rows, inner, outer):
    """The gate's activation is a parameter of the gated product: SiLU is applied in the products' own epilogues (relu
    too in those for a few rows), the others by the activation kernel behind a plain product; one that has no kernel
    is refused by name."""
    k = kernels[dtype]
    acts = {"silu": F.silu, "gelu": F.gelu, "gelu_tanh": lambda z: F.gelu(z, approximate="tanh"), "relu": torch.relu}
    x, gate, up = torch.randn(rows, inner), torch.randn(outer, inner) / math.sqrt(inner), torch.randn(outer, inner) / math.sqrt(inner)
    weights = k.prepare_gated_linear(on_gpu(gate, dtype), on_gpu(up, dtype), activation)
    out = k.gated_linear(on_gpu(x, dtype), weights)
    want = acts[activation](rounded(x, dtype) @ rounded(gate, dtype).T) * (rounded(x, dtype) @ rounded(up, dtype).T)
    torch.testing.assert_close(out.cpu().double(), want, **TOLERANCE[dtype])
    from llmserve_amd.kernels.hip import KernelError

    with pytest.raises(KernelError, match="swish7"):
        k.prepare_gated_linear(on_gpu(gate, dtype), on_gpu(up, dtype), "swish7")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,dim,page,cap", [(6, 2, 32, 8, 1.5), (4, 1, 128, 16, None), (5, 5, 48, 4, 0.7)])
def test_paged_attention_with_a_distance_bias_and_a_soft_cap(kernels, dtype, heads, kv_heads, dim, page, cap):
    """Scores squashed to cap * tanh(score / cap), then lowered by slope[head] * distance: portions beside decoded
    tokens, on the matrix-core kernels of both precisions (pages of 4 in bfloat16: the generic one), against the
    formula."""
    lengths, counts = [45, 17, 70], [20, 1, 70]
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, page, dtype, shuffle_seed=heads)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    slopes = torch.tensor([0.3 / 2.0 ** head for head in range(heads)], dtype=torch.float32)
    scale = 1.0 / math.sqrt(dim)
    out = kernels[dtype].paged_attention(qkv, layout, batch, cell, scale, None, score_slopes=on_gpu(slopes), soft_cap=cap).cpu().double()
    expected = []
    for (q, k, v), count in zip(per_request, counts):
        q, k, v = rounded(q, dtype), rounded(k, dtype), rounded(v, dtype)
        length = q.shape[0]
        k, v = k.repeat_interleave(heads // kv_heads, dim=1), v.repeat_interleave(heads // kv_heads, dim=1)
        scores = torch.einsum("ihd,jhd->hij", q, k) * scale
        if cap:
            scores = cap * torch.tanh(scores / cap)
        distance = (torch.arange(length).unsqueeze(1) - torch.arange(length).unsqueeze(0)).double()
        scores = (scores - slopes.double().view(-1, 1, 1) * distance).masked_fill(distance < 0, float("-inf"))
        full = torch.einsum("hij,jhd->ihd", torch.softmax(scores, dim=-1), v)
        expected.append(full[-count:].flatten(1))
    torch.testing.assert_close(out, torch.cat(expected), **TOLERANCE[dtype])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lengths,counts,window", [([2100, 700, 5], [1, 1, 1], None), ([300, 2100, 900], [300, 64, 1], 512)])
@pytest.mark.parametrize("heads,kv_heads,dim,cap", [(12, 2, 128, 4.0), (7, 7, 64, None)])
def test_changed_scores_over_long_contexts(kernels, dtype, lengths, counts, window, heads, kv_heads, dim, cap):
    """The same change of the scores where the keys are split over workgroups and merged (single tokens over long
    contexts), in long portions, and under a window; slopes small enough that far keys still count, one head's zero."""
    batch, cell, per_request, layout = paged_case(lengths, counts, heads, kv_heads, dim, 16, dtype, shuffle_seed=3)
    qkv = on_gpu(step_rows(per_request, counts, heads, kv_heads, dim), dtype)
    slopes = torch.tensor([0.0 if head == 1 else 0.004 * (1 + head % 3) for head in range(heads)], dtype=torch.float32)
    scale = 1.0 / math.sqrt(dim)
    out = kernels[dtype].paged_attention(qkv, layout, batch, cell, scale, window, score_slopes=on_gpu(slopes), soft_cap=cap).cpu().double()
    expected = []
    for (q, k, v), count in zip(per_request, counts):
        q, k, v = rounded(q, dtype)[-count:], rounded(k, dtype), rounded(v, dtype)
        length = k.shape[0]
        k, v = k.repeat_interleave(heads // kv_heads, dim=1), v.repeat_interleave(heads // kv_heads, dim=1)
        scores = torch.einsum("ihd,jhd->hij", q, k) * scale
        if cap:
            scores = cap * torch.tanh(scores / cap)
        distance = (torch.arange(length - count, length).unsqueeze(1) - torch.arange(length).unsqueeze(0)).double()
        unseen = (distance < 0) | (distance >= window if window else torch.zeros_like(distance, dtype=torch.bool))
        scores = (scores - slopes.double().view(-1, 1, 1) * distance).masked_fill(unseen, float("-inf"))
        expected.append(torch.einsum("hij,jhd->ihd", torch.softmax(scores, dim=-1), v).flatten(1))
    torch.testing.assert_close(out, torch.cat(expected), **TOLERANCE[dtype])


def device_paged_case(requests, heads, kv_heads, dim, page, dtype, seed):
    """As `paged_case`, made on the device without a loop over positions, for contexts of thousands of keys:
    `requests` = [(cached tokens, of which this step's)].  Returns the batch, the cell (NaN in every slot that no
    token owns) and per request its step's queries and all its keys and values, as the kernel sees them."""
    from llmserve_amd.cache import CacheCell
    from llmserve_amd.engine.batch import GroupBatch, SequenceChunk, StepBatch
    from llmserve_amd.parts import HeadLayout, PagedKeyValue

    generator = torch.Generator(device="cuda").manual_seed(seed)
    blocks = [math.ceil(length / page) for length, _ in requests]
    pages = sum(blocks) + 3
    order = torch.randperm(pages, generator=torch.Generator().manual_seed(seed)).cuda()
    width = max(blocks)
    tables = torch.full((len(requests), width), -1, dtype=torch.int32, device="cuda")
    keys = torch.full((pages, kv_heads, page, dim), float("nan"), dtype=dtype, device="cuda")
    values = torch.full((pages, kv_heads, dim, page), float("nan"), dtype=dtype, device="cuda")
    per_request, rows, slot_mapping, positions, token_sequence, chunks, taken = [], [], [], [], [], [], 0
    for index, (length, count) in enumerate(requests):
        mine = order[taken : taken + blocks[index]]
        taken += blocks[index]
        tables[index, : blocks[index]] = mine.int()
        q = torch.randn(count, heads, dim, generator=generator, device="cuda").to(dtype)
        k = torch.randn(length, kv_heads, dim, generator=generator, device="cuda").to(dtype)
        v = torch.randn(length, kv_heads, dim, generator=generator, device="cuda").to(dtype)
        where = torch.arange(length, device="cuda")
        keys[mine[where // page], :, where % page] = k
        values[mine[where // page], :, :, where % page] = v
        per_request.append((q, k, v))
        rows.append(torch.cat([q.flatten(1), k[-count:].flatten(1), v[-count:].flatten(1)], dim=1))
        mine_cpu = mine.cpu().tolist()
        for position in range(length - count, length):
            slot_mapping.append(mine_cpu[position // page] * page + position % page)
            positions.append(position)
            token_sequence.append(index)
        chunks.append(SequenceChunk(f"r{index}", index, length - count, count))
    counts = [count for _, count in requests]
    starts = [0]
    for count in counts:
        starts.append(starts[-1] + count)
    ints = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    batch = StepBatch(
        num_tokens=sum(counts), chunks=chunks, token_ids=ints([0] * sum(counts)), positions=ints(positions),
        token_sequence=ints(token_sequence), query_start=ints(starts), context_lengths=ints([length for length, _ in requests]),
        state_slots=ints(list(range(len(requests)))), groups=[GroupBatch(page, tables, ints(slot_mapping), width)],
        logit_rows=ints([]), num_logit_rows=0, max_query_length=max(counts), max_context_length=max(length for length, _ in requests),
    )
    cell = CacheCell(PagedKeyValue(kv_heads, dim), True, 0, key_pieces(keys), value_pieces(values))
    return batch, cell, per_request, torch.cat(rows), HeadLayout(heads, kv_heads, dim)


def device_attention(q, k, v, scale, window):
    """softmax(q k^T * scale) v of a request's last rows over all its keys, causal (and windowed), float32 on the
    device with torch's own operations, one kv head at a time."""
    count, heads, dim = q.shape
    length, kv_heads = k.shape[0], k.shape[1]
    group = heads // kv_heads
    position = torch.arange(length - count, length, device=q.device).view(1, -1, 1)
    key = torch.arange(length, device=q.device).view(1, 1, -1)
    unseen = key > position
    if window:
        unseen = unseen | (key <= position - window)
    out = torch.empty(count, heads, dim, dtype=torch.float32, device=q.device)
    for kv_head in range(kv_heads):
        mine = q[:, kv_head * group : (kv_head + 1) * group].float()
        scores = torch.einsum("igd,jd->gij", mine, k[:, kv_head].float()) * scale
        weights = torch.softmax(scores.masked_fill(unseen, float("-inf")), dim=-1)
        out[:, kv_head * group : (kv_head + 1) * group] = torch.einsum("gij,jd->igd", weights, v[:, kv_head].float())
    return out.flatten(1)


@pytest.mark.parametrize("dtype,draws", [(torch.bfloat16, 100), (torch.float32, 30)])
def test_attention_at_random_step_shapes(dtype, draws):
    """What a step holds decides which attention kernel it goes to and how its keys are cut (the kernel that shares
    keys through LDS whole or in runs, the tiles kernel with one or two column tiles, key splits merged by row or
    by work item): steps drawn at random around those rules (long portions far into their prompts, few or many
    decoded tokens over short and long contexts, several head counts and pages, windows), each against torch's own
    operations, and the bfloat16 draws together must have taken every way; the float32 kernel under the same draws."""
    import random

    from llmserve_amd.kernels import HipKernels

    kernels = HipKernels(dtype)
    library = kernels._attention_library(128)
    ways = {"shared whole": 0, "shared in runs": 0, "tiles": 0, "tiles split": 0, "by item": 0}
    shared_entry, tiles_entry = library.llmserve_attention_portions, library.llmserve_attention_tiles

    def counted_shared(*arguments):
        ways["shared in runs" if arguments[19] > 1 else "shared whole"] += 1  # (splits)
        return shared_entry(*arguments)

    def counted_tiles(*arguments):
        splits, fuse = arguments[20], arguments[21]
        ways["by item" if fuse & 4 and splits > 1 else "tiles split" if splits > 1 else "tiles"] += 1
        return tiles_entry(*arguments)

    library.llmserve_attention_portions, library.llmserve_attention_tiles = counted_shared, counted_tiles
    try:
        for seed in range(draws):
            draw = random.Random(seed)
            heads, kv_heads = draw.choice([(12, 2), (28, 4), (40, 8), (16, 2), (64, 8), (7, 7)])
            page = draw.choice([16, 16, 32, 8, 64])
            window = draw.choice([None, None, 700, 4096])
            requests = []
            for _ in range(draw.choice([0, 1, 1, 2, 3])):
                count = draw.choice([64, 300, 512, 1024, 2048])
                requests.append((count + draw.choice([0, 0, 700, 3000, 9000, 17000]), count))
            for _ in range(draw.choice([0, 1, 5, 20, 40]) if requests else draw.choice([1, 5, 20, 40])):
                requests.append((draw.randint(1, draw.choice([300, 3000, 12000])), 1))
            draw.shuffle(requests)
            batch, cell, per_request, qkv, layout = device_paged_case(requests, heads, kv_heads, 128, page, dtype, seed)
            scale = 1.0 / math.sqrt(128)
            out = kernels.paged_attention(qkv, layout, batch, cell, scale, window).float()
            expected = torch.cat([device_attention(q, k, v, scale, window) for q, k, v in per_request])
            torch.testing.assert_close(out, expected, **TOLERANCE[dtype], msg=lambda m: f"seed {seed}, {heads}/{kv_heads} heads, pages of {page}, window {window}, {requests}: {m}")
            del batch, cell, per_request, qkv, out, expected
    finally:
        library.llmserve_attention_portions, library.llmserve_attention_tiles = shared_entry, tiles_entry
    assert dtype == torch.float32 or all(ways.values()), ways


@pytest.mark.parametrize("own", [False, True])
def test_products_at_random_shapes(own):
    """Rows, K and N decide which product kernel runs (weight-streaming with one, two or four tiles a wave, through
    registers or LDS, K cut into partial sums, the kernels for 17 to 64 rows, the library or the tiled kernels beyond,
    inside and outside a step that a graph will replay): shapes drawn at random around those rules, plain, with a
    bias, as float32 partial sums and gated, against torch's float32 product of the same rounded operands."""
    import random

    from llmserve_amd.kernels import HipKernels

    dtype = torch.bfloat16
    k = HipKernels(dtype, library_products=not own)
    generator = torch.Generator(device="cuda").manual_seed(5)
    for seed in range(200):
        draw = random.Random(1000 + seed)
        rows = draw.choice([1, 2, 3, 5, 8, 13, 16, 17, 24, 32, 33, 48, 64, 65, 100, 128, 130, 300])
        inner = 32 * draw.choice([1, 3, 4, 8, 12, 16, 28, 40, 48, 64, 70, 112, 148, 160, 216, 280])
        outer = draw.choice([16, 48, 100, 256, 272, 1000, 1536, 2048, 4099, 5120, 17920])
        if rows > 64 and inner * outer > 1 << 24:
            outer = 1000
        x = torch.randn(rows, inner, generator=generator, device="cuda").to(dtype)
        w = (torch.randn(outer, inner, generator=generator, device="cuda") / math.sqrt(inner)).to(dtype)
        up = (torch.randn(outer, inner, generator=generator, device="cuda") / math.sqrt(inner)).to(dtype)
        b = torch.randn(outer, generator=generator, device="cuda").to(dtype)
        said = f"draw {seed}: {rows} rows, K {inner}, N {outer}"
        want = x.float() @ w.float().T
        plain_weights, biased = k.prepare_linear([w], None), k.prepare_linear([w], [b])
        gated_weights = k.prepare_gated_linear(w, up)
        want_gated = F.silu(want) * (x.float() @ up.float().T)
        for replayed in (False, True):
            with k.replay_scope() if replayed else contextlib.nullcontext():
                torch.testing.assert_close(k.linear(x, plain_weights).float(), want, **TOLERANCE[dtype], msg=lambda m: f"{said}, plain, replay {replayed}: {m}")
                torch.testing.assert_close(k.linear(x, biased).float(), want + b.float(), **TOLERANCE[dtype], msg=lambda m: f"{said}, bias, replay {replayed}: {m}")
                parts = k.linear(x, plain_weights, out_dtype=torch.float32, partial=True)
                summed = parts if parts.ndim == 2 else parts.sum(0)
                torch.testing.assert_close(summed, want, atol=2e-4, rtol=2e-4, msg=lambda m: f"{said}, partial sums, replay {replayed}: {m}")
                torch.testing.assert_close(k.gated_linear(x, gated_weights).float(), want_gated, **TOLERANCE[dtype], msg=lambda m: f"{said}, gated, replay {replayed}: {m}")


@pytest.mark.parametrize("tiles", [2, 4, 5, 6, 8, 10, 12, 14])
@pytest.mark.parametrize("rows,inner,outer,parts", [(17, 128, 48, 1), (33, 1536, 1000, 3), (64, 8960, 272, 10), (50, 384, 4099, 1), (32, 512, 130, 2),
                                                    (8, 1024, 300, 2), (65, 256, 100, 1), (100, 1536, 1000, 4), (128, 3584, 272, 7)])
def test_product_through_the_ring(kernels, tiles, rows, inner, outer, parts):
    """The product for up to 128 rows whose weights and x go through a ring of stages in LDS, in every shape of
    workgroup it has (2 to 14 tiles of 16 weight rows; 5 for more than 32 rows only, 6, 12 and 14 for up to 64): rows
    and weight rows that end inside a tile, a K of one stage and of fewer stages than the ring has, with a bias, as float32
    partial sums and gated."""
    from llmserve_amd.kernels.hip import KernelError, _check, _is_float, _pointer

    k, dtype = kernels[torch.bfloat16], torch.bfloat16
    library = k._gemm_bf16
    x, w, b = torch.randn(rows, inner), torch.randn(outer, inner) / math.sqrt(inner), torch.randn(outer)
    up = torch.randn(outer, inner) / math.sqrt(inner)
    want = rounded(x, dtype) @ rounded(w, dtype).T

    def run(weight, bias, out, gated, splits):
        return library.llmserve_gemm_ring(
            _pointer(on_gpu(x, dtype)), _pointer(weight), _pointer(bias), _is_float(bias) if bias is not None else 0, _pointer(out),
            _is_float(out), 1 if gated else 0, rows, weight.shape[0], inner, splits, tiles, k._stream)

    weight, bias = on_gpu(w, dtype), on_gpu(b, dtype)
    out = torch.empty(rows, outer, dtype=dtype, device="cuda")
    if (tiles == 5 and rows <= 32) or (tiles in (6, 12, 14) and rows > 64):
        with pytest.raises(KernelError):
            _check(run(weight, bias, out, False, 1), "ring")
        return
    _check(run(weight, bias, out, False, 1), "ring")
    torch.testing.assert_close(out.cpu().double(), want + rounded(b, dtype), **TOLERANCE[dtype])
    float_bias = on_gpu(b, torch.float32)
    partial = torch.empty(parts, rows, outer, dtype=torch.float32, device="cuda")
    _check(run(weight, float_bias, partial, False, parts), "ring")
    torch.testing.assert_close(partial.sum(0).cpu().double(), want + b.double(), atol=1e-4, rtol=1e-4)
    both = torch.stack([on_gpu(w, dtype), on_gpu(up, dtype)], dim=1).reshape(2 * outer, inner).contiguous()
    gated = torch.empty(rows, outer, dtype=dtype, device="cuda")
    _check(run(both, None, gated, True, 1), "ring")
    torch.testing.assert_close(gated.cpu().double(), F.silu(want) * (rounded(x, dtype) @ rounded(up, dtype).T), **TOLERANCE[dtype])


@pytest.mark.parametrize("vocab", [9000, 8193, 40961])
def test_top_p_over_more_entries_than_a_block_keeps(kernels, vocab):
    """The row's block keeps 8,192 listed entries in registers: rows that list as many or more (a spread so small that all lie in two bins of
    the first level, nothing but one value, two values side by side, many ties) against the rule in 64 bits."""
    k = kernels[torch.float32]
    generator = torch.Generator().manual_seed(vocab)
    logits = torch.stack([
        0.01 * torch.randn(vocab, generator=generator), torch.full((vocab,), 2.5), torch.randint(0, 2, (vocab,), generator=generator) * 0.03,
        torch.randint(0, 9, (vocab,), generator=generator) * 0.005, torch.cat([torch.full((8192,), 1.0), torch.full((vocab - 8192,), -9.0)]),
    ])
    rows = logits.shape[0]
    p = torch.exp(logits - logits.amax(1, keepdim=True))  # float32, as the rule has it
    for draw, top_p in enumerate((0.1, 0.5, 0.93)):
        uniforms = [plain.uniform_for(draw, row) for row in range(rows)]
        got = k.sample(on_gpu(logits), on_gpu(torch.ones(rows)), on_gpu(torch.full((rows,), top_p)), on_gpu(torch.tensor(uniforms))).cpu().tolist()
        for row in range(rows):
            order = torch.argsort(p[row], descending=True, stable=True)
            mass = p[row].double()[order].cumsum(0)
            limit = float(torch.tensor(top_p)) * float(mass[-1])
            kept = int((mass - p[row].double()[order] < limit).sum())
            target = float(torch.tensor(uniforms[row])) * float(mass[kept - 1])
            # the kernel's exp may be off torch's in the last place: the place of the token in the order is right to as much of the mass
            place = int((order == got[row]).nonzero())
            slack = 4 * 2.0 ** -23 * float(mass[-1])
            assert place < kept + 1 and mass[place] > target - slack and (place == 0 or mass[place - 1] <= target + slack), (row, top_p)


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("rows", [65, 79, 80, 81, 95, 96, 97])
def test_ring_of_six_tiles_of_rows_has_the_bits_of_eight(kernels, rows, gated):
    """Up to 96 rows the ring has six tiles of x, beyond eight: a row's sums are the same products in the same order.  A last workgroup of
    weight rows that are not all there, rows that end inside a tile, and nothing written behind the last row."""
    from llmserve_amd.kernels.hip import _pointer

    k, inner, outer = kernels[torch.bfloat16], 640, 5 * 16 * 7 + 48
    generator = torch.Generator(device="cuda").manual_seed(rows)
    x, w = (torch.randn(shape, generator=generator, device="cuda").bfloat16() for shape in ((128, inner), (outer, inner)))
    results = []
    for count in (rows, 128):
        out = torch.full((130, outer // 2 if gated else outer), 7.0, device="cuda", dtype=torch.bfloat16)
        assert k._gemm_bf16.llmserve_gemm_ring(_pointer(x), _pointer(w), None, 0, _pointer(out), 0, int(gated), count, outer, inner, 1, 5, k._stream) == 0
        assert (out[count:] == 7.0).all()
        results.append(out[:rows])
    assert torch.equal(*results)
    exact = x[:rows].double() @ w.double().T
    if gated:
        exact = torch.nn.functional.silu(exact[:, ::2]) * exact[:, 1::2]
    torch.testing.assert_close(results[0].double(), exact, **TOLERANCE[torch.bfloat16])


@pytest.mark.parametrize("tiles,inner", [(2, 384), (4, 640), (8, 640), (8, 192), (10, 320)])
@pytest.mark.parametrize("rows", [65, 81, 96, 97])
def test_ring_of_six_tiles_of_rows_beside_any_weight_tiles(kernels, rows, tiles, inner):
    """As above beside two, four, eight and ten weight tiles (five: above), gated, whole and in parts."""
    from llmserve_amd.kernels.hip import _pointer

    k, outer = kernels[torch.bfloat16], tiles * 16 * 3 + 16
    generator = torch.Generator(device="cuda").manual_seed(rows + tiles)
    x, w = (torch.randn(shape, generator=generator, device="cuda").bfloat16() for shape in ((128, inner), (outer, inner)))
    exact = x.double() @ w.double().T
    for gated, parts in ((1, 1), (0, 1), (0, inner // 128 if inner % 128 == 0 else 1)):
        results, split = [], parts > 1
        for count in (rows, 128):
            out = torch.full((parts, 130, outer // 2 if gated else outer), 7.0, device="cuda", dtype=torch.float32 if split else torch.bfloat16)
            flat = out.view(-1)[: parts * count * out.shape[2]].view(parts, count, out.shape[2])
            assert k._gemm_bf16.llmserve_gemm_ring(_pointer(x), _pointer(w), None, 0, _pointer(out), int(split), gated, count, outer, inner, parts, tiles, k._stream) == 0
            assert (out.view(-1)[flat.numel() :] == 7.0).all()
            results.append(flat[:, :rows])
        assert torch.equal(*results)
        want = torch.nn.functional.silu(exact[:, ::2]) * exact[:, 1::2] if gated else exact
        torch.testing.assert_close(results[0].double().sum(0), want[:rows], **TOLERANCE[torch.bfloat16])


@pytest.mark.parametrize("rows", [1, 33, 257])
@pytest.mark.parametrize("vocab", [8191, 8193, 20003])
def test_top_p_of_rows_with_more_candidates_than_a_list_holds(kernels, rows, vocab):
    """Around 8,192 candidates, and far more; rows of a length that is no multiple of four, in sixteen parts, in seven and in one; more equal
    entries of one value and of several than what is gathered of a row holds.  Against the rule in 64 bits: the kernel's exp may be off by two
    units in the last place (2^-22 of the value), which moves every mass by as much of the whole, and logits that lie so close may tie in p."""
    k = kernels[torch.float32]
    generator = torch.Generator().manual_seed(vocab + rows)
    kinds = [lambda: torch.full((vocab,), 2.5), lambda: torch.randint(0, 3, (vocab,), generator=generator) * 0.003,
             lambda: 0.3 * torch.randn(vocab, generator=generator).bfloat16().float(), lambda: 0.01 * torch.randn(vocab, generator=generator),
             lambda: 4.0 * torch.randn(vocab, generator=generator)]
    logits = torch.stack([kinds[(row + vocab) % 5]() for row in range(rows)])
    p = torch.exp(logits.double() - logits.amax(1, keepdim=True).double())
    ranked, order = torch.sort(p, dim=1, descending=True, stable=True)
    mass = ranked.cumsum(1)
    for draw, top_p in enumerate((0.2, 0.95, 0.9999)):
        uniforms = torch.tensor([plain.uniform_for(draw, row) for row in range(rows)], dtype=torch.float32)
        if rows > 1:
            uniforms[0], uniforms[-1] = 0.0, 1.0 - 2.0 ** -24
        got = k.sample(on_gpu(logits), on_gpu(torch.ones(rows)), on_gpu(torch.full((rows,), top_p)), on_gpu(uniforms)).cpu().long()
        limit = float(torch.tensor(top_p)) * mass[:, -1]
        kept = (mass - ranked < limit[:, None]).sum(1)
        target = uniforms.double() * mass.gather(1, kept[:, None] - 1)[:, 0]
        place, value = (order == got[:, None]).int().argmax(1), p.gather(1, got[:, None])
        slack = 2.0 ** -21 * mass[:, -1]
        above = torch.where(p > value * (1 + 2.0 ** -21), p, 0.0).sum(1)  # certainly ranked before, and perhaps
        not_below = torch.where(p >= value * (1 - 2.0 ** -21), p, 0.0).sum(1)
        right = (above < limit + slack) & (above <= target + slack) & (not_below > target - slack)
        # values far apart, and equal ones in the order of their indices: the very entry, where the end of the kept set is not in question
        after, before = mass.gather(1, place[:, None])[:, 0], (mass - ranked).gather(1, place[:, None])[:, 0]
        exact = torch.tensor([(row + vocab) % 5 < 3 for row in range(rows)])
        right &= ~exact | ((after > target - slack) & (before <= target + slack) & (before < limit + slack + 1))
        assert not (wrong := (~right).nonzero()[:, 0].tolist()), (top_p, wrong[:9], got[wrong[:9]].tolist())


def test_the_samplers_memory(kernels):
    """A list holds 8,192 entries of a row and no longer the whole row: not beyond what a row's histograms and counts of its pieces took before."""
    library = kernels[torch.float32]._sampling_library()
    for rows in (1, 8, 64, 512):
        assert library.llmserve_sample_workspace_kib(rows, 151936) * 1024 < rows * (151936 * 4 + 96 * 1024) + 4096


def test_sampling_without_top_p_needs_no_memory_for_it(kernels):
    """The workspace of a call whose rows have no top-p is p and little else, one smaller is refused, and tokens are those with the rest around it."""
    from llmserve_amd.kernels.hip import _pointer

    k = kernels[torch.float32]
    library = k._sampling_library()
    rows, vocab = 9, 20001
    kib = library.llmserve_sample_plain_workspace_kib(rows, vocab)
    assert rows * vocab * 4 // 1024 < kib < rows * vocab * 4 // 1024 + 32 and library.llmserve_sample_plain_workspace_kib(0, vocab) < 0
    assert library.llmserve_sample_workspace_kib(rows, vocab) > kib
    generator = torch.Generator().manual_seed(3)
    logits, ones, uniforms = on_gpu(torch.randn(rows, vocab, generator=generator)), on_gpu(torch.ones(rows)), on_gpu(torch.rand(rows, generator=generator))
    workspace, out = torch.full((kib * 1024 + 256,), 7, dtype=torch.uint8, device="cuda"), torch.zeros(rows, dtype=torch.int32, device="cuda")

    def status(size, with_top_p):
        return library.llmserve_sample(_pointer(logits), _pointer(ones), _pointer(ones), _pointer(uniforms), _pointer(workspace), size, _pointer(out),
                                       rows, vocab, with_top_p, k._stream)

    assert status(kib - 1, 0) == 1001 and status(kib, 1) == 1001 and status(kib, 0) == 0
    assert (workspace[kib * 1024 :] == 7).all()
    assert torch.equal(out, k.sample(logits, ones, ones, uniforms)) and torch.equal(out, k.sample(logits, ones, ones, uniforms, with_top_p=False))
