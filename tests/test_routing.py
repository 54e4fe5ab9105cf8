"""Which kernel a product goes to, and in what shape, is decided on the host from its sizes alone
(`HipKernels._streaming`, `_ring_shape` and the other rules of `kernels/hip.py`); the kernels refuse what they
were not built for.  This walks the rules over the layer sizes of every configuration shipped here, over tiny
and odd sizes and over every number of rows up to 130, and checks each answer against what the entry points
in `csrc/gemm_bf16.hip` take (`pick_ring`, `launch_ring`; read from the source, restated here), so that a rule
cannot send a step to a refusal that only some batch size would meet.  No GPU needed: the tensors are `meta`."""

from __future__ import annotations

import json
import random
from pathlib import Path
from types import SimpleNamespace

import pytest
import torch

from llmserve_amd.kernels.hip import HipKernels, KernelError, LinearWeights

ROOT = Path(__file__).resolve().parents[1]
LDS_KB = 160
STAGE_KB = 1  # sixteen rows of thirty-two bfloat16 k


def products_of_the_shipped_configurations():
    """(out_features, in_features, gated, may_split) of every product of every configuration under configs/."""
    found = set()
    for path in sorted((ROOT / "configs").glob("*.json")):
        sizes = json.loads(path.read_text())
        if "hidden_size" not in sizes:  # another architecture: every matrix of its own list of tensors, whole and cut over K
            from llmserve_amd.registry import resolve_architecture

            architecture = resolve_architecture(sizes)
            spec = architecture.build_spec(architecture.config_class.from_dict(sizes))
            for name, tensor in spec.tensors().items():
                if len(tensor.shape) == 2 and name != spec.embedding_name:
                    found.add((tensor.shape[0], tensor.shape[1], False, False))
                    found.add((tensor.shape[0], tensor.shape[1], False, True))
                    if name.endswith("mlp.gate"):
                        found.add((2 * tensor.shape[0], tensor.shape[1], True, False))
            continue
        hidden, heads, kv_heads = sizes["hidden_size"], sizes["num_attention_heads"], sizes["num_key_value_heads"]
        head_dim = sizes.get("head_dim") or hidden // heads
        found.add(((heads + 2 * kv_heads) * head_dim, hidden, False, False))
        found.add((hidden, heads * head_dim, False, True))
        found.add((2 * sizes["intermediate_size"], hidden, True, False))
        found.add((hidden, sizes["intermediate_size"], False, True))
        found.add((sizes["vocab_size"], hidden, False, False))
    return sorted(found)


def ring_takes(tiles: int, rows: int) -> tuple[int, int, int] | None:
    """(tiles of x, k-steps a stage, stages) of the ring kernel that `pick_ring` launches, or None where it refuses."""
    if rows <= 64:
        x_tiles = 2 if rows <= 32 else 4
        if tiles in (2, 4, 6) or (tiles == 5 and rows > 32):
            return x_tiles, 4, 4
        if tiles in (8, 10, 12, 14):
            return x_tiles, 2, 4
        return None
    if rows <= 128:
        if tiles in (2, 4, 5):
            return 8, 4, 3
        if tiles in (8, 10):
            return 8, 2, 4
    return None


def check_ring(rows: int, out_features: int, in_features: int, may_split: bool) -> None:
    tiles, splits, rounds = HipKernels._ring_shape(rows, out_features, in_features, may_split)
    taken = ring_takes(tiles, rows)
    assert taken is not None, (rows, out_features, in_features, may_split, tiles)
    x_tiles, k_steps, depth = taken
    assert may_split or splits == 1
    assert in_features % splits == 0 and (in_features // splits) % (32 * k_steps) == 0, (rows, out_features, in_features, splits, tiles)
    assert depth * (tiles + x_tiles) * k_steps * STAGE_KB <= LDS_KB
    assert rounds >= 1 and splits <= 65535


def stand_in(**changes):
    settings = dict(ring_products=True, ring_rows_from=4, library_products=True, _for_replay=True, _ring_shape=HipKernels._ring_shape)
    settings.update(changes)
    return SimpleNamespace(**settings)


def route(kernels, rows: int, out_features: int, in_features: int, gated: bool, may_split: bool):
    x = torch.empty((rows, in_features), dtype=torch.bfloat16, device="meta")
    weights = LinearWeights(torch.empty((out_features, in_features), dtype=torch.bfloat16, device="meta"), None)
    return HipKernels._streaming(kernels, x, weights, gated=gated, may_split=may_split)


@pytest.mark.parametrize("for_replay", [True, False])
@pytest.mark.parametrize("library_products", [True, False])
def test_every_route_of_the_shipped_sizes_is_one_its_kernel_takes(for_replay, library_products):
    kernels = stand_in(_for_replay=for_replay, library_products=library_products)
    routes = set()
    for out_features, in_features, gated, may_split in products_of_the_shipped_configurations():
        for rows in list(range(1, 131)) + [192, 256, 2048]:
            way = route(kernels, rows, out_features, in_features, gated, may_split)
            routes.add(way)
            assert way in ("skinny", "ring", "medium", "tiled", None)
            if way == "ring":
                assert rows <= 128 and in_features % 128 == 0
                check_ring(rows, out_features, in_features, may_split and not gated)
            if way == "skinny":
                assert rows <= 64 and in_features % 32 == 0
            if way == "medium":
                assert 16 < rows <= 64 and in_features % 128 == 0
            if way == "tiled":
                assert rows > 64 and in_features % 32 == 0
            if way is None:  # the library, or (without it, and for sizes no matrix-core kernel takes) the generic kernel
                assert (library_products and rows > 16) or in_features % 32 != 0 or rows <= 0
    assert "ring" in routes and "skinny" in routes


def test_ring_shapes_at_random_sizes():
    draw = random.Random(5)
    for _ in range(20000):
        rows = draw.randint(1, 128)
        in_features = 128 * draw.randint(1, 260)
        out_features = draw.choice([draw.randint(1, 400), 16 * draw.randint(1, 4000), draw.randint(1, 160000)])
        check_ring(rows, out_features, in_features, draw.random() < 0.5)


def test_routes_at_random_sizes():
    draw = random.Random(6)
    kernels = [stand_in(_for_replay=a, library_products=b) for a in (True, False) for b in (True, False)]
    for _ in range(20000):
        rows = draw.choice([draw.randint(1, 130), draw.randint(1, 4096)])
        in_features = draw.choice([128 * draw.randint(1, 260), 32 * draw.randint(1, 900), draw.randint(1, 30000)])
        out_features = draw.choice([draw.randint(1, 400), 16 * draw.randint(1, 4000), draw.randint(1, 160000)])
        gated = draw.random() < 0.3
        if gated:
            out_features += out_features % 2
        may_split = not gated and draw.random() < 0.5
        way = route(draw.choice(kernels), rows, out_features, in_features, gated, may_split)
        if way == "ring":
            assert rows <= 128 and in_features % 128 == 0
            check_ring(rows, out_features, in_features, may_split)
        elif way in ("skinny", "medium"):
            assert rows <= 64 and in_features % 32 == 0
        elif way == "tiled":
            assert in_features % 32 == 0
        else:
            assert way is None


def test_attention_work_lists_cover_every_column_once_and_fit_the_padded_shape():
    """The attention kernels take their work from a list of (request, first token, first head of it, columns)
    items made on the host; a captured step's list has room for the most items its padded shape can hold.
    Steps drawn at random: the items cover every (token, head) column of the chosen chunks exactly once, no
    item is longer than the kernel's tile, and no step of a shape has more items than the shape's room."""
    from llmserve_amd.engine.batch import SequenceChunk

    draw = random.Random(9)
    for _ in range(3000):
        group = draw.choice([1, 2, 5, 6, 7, 8, 16, 17, 28])
        column_tiles = draw.choice([1, 2])
        packed = draw.choice([None, True, False])
        requests = draw.randint(1, 12)
        counts = [draw.choice([1, 1, 1, 2, 3, 16, 17, draw.randint(1, 700)]) for _ in range(requests)]
        chunks = [SequenceChunk(f"r{i}", i, draw.randint(0, 5000), count) for i, count in enumerate(counts)]
        longer_than, up_to = draw.choice([(0, None), (0, 16), (16, None), (1, None), (0, 1)])
        work, steps = HipKernels._work_items(chunks, group, column_tiles, longer_than, up_to, packed)
        is_packed = group <= 16 if packed is None else packed
        per_token = group if is_packed else 1
        per_item = column_tiles * (16 if is_packed else 1)
        chosen = [i for i, count in enumerate(counts) if count > longer_than and (up_to is None or count <= up_to)]
        starts = [sum(counts[:i]) for i in range(requests)]
        seen = set()
        for request, token, head, columns in work.tolist():
            assert request in chosen and 0 < columns <= per_item and 0 <= head < per_token
            for column in range(columns):
                at = (token - starts[request]) * per_token + head + column
                assert 0 <= at < counts[request] * per_token and (request, at) not in seen
                seen.add((request, at))
        assert len(seen) == sum(counts[i] * per_token for i in chosen)
        assert steps >= 0
        padded_tokens = sum(counts) + draw.randint(0, 64)
        assert len(work) <= HipKernels._work_capacity((padded_tokens, requests + draw.randint(0, 3)), group, column_tiles, packed)


class Launches:
    """Takes the place of a kernel library: counts the launches of the product into a norm."""

    def __init__(self) -> None:
        self.count = 0

    def llmserve_gemm_scaled_streams(self, rows, out_features, in_features):
        return 1

    def llmserve_gemm_into_norm(self, *arguments):
        self.count += 1
        return 0


def on_the_host(**changes):
    """`HipKernels` without a GPU: its rules and checks, on CPU tensors, with `Launches` for the kernels."""
    kernels = object.__new__(HipKernels)
    settings = dict(dtype=torch.bfloat16, device=torch.device("cpu"), ring_products=True, ring_rows_from=4, library_products=True,
                    _for_replay=True, _pinned_stream=0, _gemm_bf16=Launches())
    kernels.__dict__.update(settings | changes)
    return kernels


@pytest.mark.parametrize("rows", [4, 33])
def test_a_product_into_a_norm_takes_no_form_that_the_steps_apart_refuse(rows):
    """`linear` refuses an x that is not as wide as the weight, `add_rms_norm` a stream that is not float32: where the two are one
    product the same forms are left to them, and nothing is launched."""
    width, inner = 1536, 1280
    kernels = on_the_host()
    project = LinearWeights(torch.zeros(width, inner, dtype=torch.bfloat16), None)
    reader = kernels.prepare_gated_linear(*(torch.zeros(1400, width, dtype=torch.bfloat16) for _ in range(2)))

    def linked(x, hidden, weight=torch.ones(width)):
        before = kernels._gemm_bf16.count
        result = kernels._linear_into_norm(x, None, project, kernels.norm_into(hidden, weight, 1e-6, reader))
        assert kernels._gemm_bf16.count - before == (result is not None)
        return result

    x, hidden = torch.zeros(rows, inner, dtype=torch.bfloat16), torch.zeros(rows, width)
    assert linked(x, hidden) is not None
    assert linked(x[:, :1152].contiguous(), hidden) is None
    assert linked(torch.zeros(rows, width, dtype=torch.bfloat16), hidden) is None  # as wide as the stream
    assert linked(x[:-1], hidden) is None
    assert linked(x.float(), hidden) is None
    assert linked(x, hidden.bfloat16()) is None
    assert linked(x, hidden, torch.ones(width + 16)) is None
    with pytest.raises(KernelError):
        kernels.gated_linear(linked(x, hidden), kernels.prepare_gated_linear(*(torch.zeros(1400, width, dtype=torch.bfloat16) for _ in range(2))))


@pytest.mark.parametrize("rows,out_features,in_features,gated,may_split", [(96, 1536, 8960, False, True), (384, 1536, 8960, False, True),
                                                                            (600, 2048, 1536, False, False), (300, 9728, 896, True, False)])
def test_rows_that_are_views_go_to_the_library(rows, out_features, in_features, gated, may_split):
    """The library takes rows of any stride and at any address; the tiled kernel brings 16-byte pieces of whole rows, so such rows stay
    with the library (up to 128 rows with the kernel before it in line, which has always refused strides)."""
    kernels = stand_in()
    flat = torch.empty(rows * in_features + 8, dtype=torch.bfloat16)
    weight = torch.empty(out_features * in_features + 8, dtype=torch.bfloat16)
    forms = {
        "rows": flat[:-8].view(rows, in_features),
        "every second row": torch.empty((2 * rows, in_features), dtype=torch.bfloat16)[::2],
        "columns of wider rows": torch.empty((rows, in_features + 64), dtype=torch.bfloat16)[:, 64:],
        "rows that begin inside a piece": flat[1:-7].view(rows, in_features),
    }

    def way(x, w):
        return HipKernels._streaming(kernels, x, LinearWeights(w.view(out_features, in_features), None), gated=gated, may_split=may_split)

    assert way(forms["rows"], weight[:-8]) == "tiled"
    other = "ring" if rows <= 128 else None
    assert all(way(x, weight[:-8]) == other for name, x in forms.items() if name != "rows")
    assert way(forms["rows"], weight[1:-7]) == other


@pytest.mark.parametrize("rows,out_features,in_features,gated,may_split,tiled", [
    # gated: a round of tiles, a second one half empty, long K
    (384, 17920, 1536, True, False, True), (416, 17920, 1536, True, False, False), (576, 17920, 1536, True, False, False),
    (704, 17920, 1536, True, False, True), (600, 11264, 2048, True, False, True), (900, 12288, 2048, True, False, False),
    (520, 16384, 2048, True, False, False), (2048, 17920, 1536, True, False, True), (1536, 19456, 2560, True, False, False),
    (2048, 37888, 3584, True, False, True), (1024, 24576, 4096, True, False, False), (2048, 59136, 8192, True, False, False),
    # in parts: few rows, very large weights, large results, a K as long as the result is wide
    (128, 5120, 27648, False, True, True), (160, 5120, 27648, False, True, False), (320, 5120, 13824, False, True, True),
    (512, 4096, 14336, False, True, True), (576, 4096, 14336, False, True, False), (1280, 1536, 8960, False, True, True),
    (1536, 1536, 10496, False, True, False), (512, 3584, 3584, False, True, True), (576, 3584, 3584, False, True, False),
    # plain, small weights
    (512, 2048, 1536, False, False, False), (513, 2048, 1536, False, False, True), (2048, 2048, 1536, False, False, True),
])
def test_products_of_many_rows_go_where_they_were_measured_ahead(rows, out_features, in_features, gated, may_split, tiled):
    """Both sides of the lines that `_tiled_ahead` draws, at sizes that were measured there."""
    assert (route(stand_in(), rows, out_features, in_features, gated, may_split) == "tiled") == tiled


@pytest.mark.parametrize("rows,out_features,in_features,ahead", [
    (65, 2048, 1536, True), (2048, 2048, 1536, True), (2112, 2048, 1536, False), (1024, 1152, 896, True), (192, 4608, 3584, True),
    (256, 4608, 3584, False), (128, 7168, 5120, True), (192, 7168, 5120, False), (768, 2560, 2048, True), (1024, 2560, 2048, False), (96, 2048, 96, False),
])
def test_rotated_products_are_fused_where_it_was_measured_ahead(rows, out_features, in_features, ahead):
    """Both sides of the lines that `_rotated_ahead` draws."""
    assert HipKernels._rotated_ahead(rows, out_features, in_features) == ahead


@pytest.mark.parametrize("keys,blocks,runs", [
    (1024, 20, 1), (2048, 28, 2), (2048, 100, 2), (2048, 128, 2), (2048, 148, 1), (2048, 184, 1), (2048, 232, 1), (2048, 296, 1),
    (4096, 28, 4), (4096, 148, 3), (4096, 184, 1), (8192, 184, 2), (8192, 28, 8), (8192, 300, 1), (65536, 10, 8),
])
def test_walks_of_portions_are_cut_where_it_was_measured_to_pay(keys, blocks, runs):
    """Two runs for more workgroups than eight waves walk for cost a short context more than they save."""
    assert HipKernels._portion_runs(keys, blocks) == runs


@pytest.mark.parametrize("blocks,keys,padded,eight", [
    (88, 1024, False, True), (256, 704, False, True), (264, 608, False, False), (288, 2000, False, False), (100, 256, False, False),
    (288, 1024, True, True), (296, 1024, True, False),
])
def test_eight_waves_walk_where_a_workgroup_has_a_cu(blocks, keys, padded, eight):
    assert HipKernels._portion_eight_waves(blocks, keys, padded) == eight


def steps_with_portions(requests: int, chunk: int, longest: int, seed: int, steps: int):
    """(tokens, requests, longest context) of the steps with a portion in a run of ragged prompts beside decoded tokens."""
    rng = random.Random(seed)
    running, left, done = [], 0, 0
    for _ in range(steps):
        if not left and len(running) < requests and rng.random() < 0.15:
            left, done = int(2 ** rng.uniform(4, longest)), 0
        portion = min(chunk, left)
        context = max([length for length, _ in running] + [done + portion])
        if portion:
            yield len(running) + portion, len(running) + 1, context, bool(running) or portion == left
        running = [(length + 1, more - 1) for length, more in running if more > 1]
        if portion:
            left, done = left - portion, done + portion
            if not left:
                running.append((done, int(2 ** rng.uniform(3, 9))))


@pytest.mark.parametrize("requests,chunk,longest", [(8, 512, 11), (32, 256, 11), (64, 256, 12), (64, 480, 12), (32, 512, 13)])
def test_ragged_steps_seldom_capture_a_shape_again(requests, chunk, longest):
    """A captured step's shape is dropped when too many others have come since.  The graphs kept have to go with the shapes that
    the buckets make: a shape that is captured anew costs as much as many steps."""
    from llmserve_amd.engine.runner import ModelRunner

    seen, kept, captured = {}, {}, 0
    for tokens, present, context, wanted in steps_with_portions(requests, chunk, longest, 1, 20_000):
        if tokens > 512:  # (launched kernel by kernel)
            continue
        padded = ModelRunner._bucket(present + 1)
        key = (ModelRunner._token_bucket(tokens), padded, ModelRunner._bucket(-(-context // 16)), padded if wanted else 0)
        seen[key] = seen.get(key, 0) + 1
        if kept.pop(key, None) is None:
            if seen[key] < 2:
                continue
            captured += 1
            if len(kept) >= ModelRunner.max_step_graphs:
                kept.pop(next(iter(kept)))
        kept[key] = True
    again = captured - sum(1 for times in seen.values() if times >= 2)
    assert again <= captured // 4, f"{again} of {captured} captures were of shapes captured before"
