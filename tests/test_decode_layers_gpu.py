"""All layers of a step of single tokens in one launch against the same layers run part by part."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _model(layers=3, dtype="bfloat16", scales=None, sharp=1.0, turned=True, components=None, **sizes):
    """`scales`: the type of the norms' weights; `sharp`: a factor on the queries' norm weights, so that a row looks at few keys; `turned`:
    whether queries and keys are."""
    from qwen3_from_scratch_amd.config import ModelConfig
    from qwen3_from_scratch_amd.models.decoder import build_model
    from qwen3_from_scratch_amd.parts.base import Precision
    from qwen3_from_scratch_amd.weights import RandomWeights

    shape = dict(hidden_size=1024, num_attention_heads=16, num_key_value_heads=8, head_dim=128, intermediate_size=2048)
    config = ModelConfig.from_dict(dict(
        dict(shape, **sizes), architectures=["Qwen3ForCausalLM"], vocab_size=512, hidden_act="silu", num_hidden_layers=layers,
        max_position_embeddings=8192, rms_norm_eps=1e-6, rope_theta=1e6, tie_word_embeddings=False))
    class Source(RandomWeights):
        def get(self, name, device):
            t = super().get(name, device)
            if "q_norm" in name:
                t = t * sharp
            return t.float() * (1 + 2 ** -12) if scales == torch.float32 and "norm" in name else t

    model = build_model(config, Precision.named(dtype), "cuda:0", components=components)
    for step in model.spec.order if not turned else ():
        model.layers[step.layer].block.mixer.attach_position(None)
    model.load(Source(model.tensors(), seed=5, std=0.02, norm_jitter=0.1, generate_on="cuda:0"))
    return model


def _logits(model, lengths, steps, graphs=False, page=16, launch=True):
    """Per step the logits of a request of each length that decodes a token."""
    from qwen3_from_scratch_amd.engine import ModelRunner, StepEntry

    g = torch.Generator().manual_seed(3)
    runner = ModelRunner(model, page, sum(n // page + 2 for n in lengths) + 1, max_requests=len(lengths), use_graphs=graphs)
    ids = [torch.randint(0, 512, (n + steps,), generator=g).tolist() for n in lengths]
    run = model.decode_run
    for i, n in enumerate(lengths):
        runner.step([StepEntry(i, ids[i][:n], [])])
    model.decode_run = run if launch else None
    try:
        return torch.stack([runner.step([StepEntry(i, [ids[i][n + s]], [0]) for i, n in enumerate(lengths)]).clone()
                            for s in range(steps)])
    finally:
        model.decode_run = run


# the fewest and the most rows and those around the ways they are asked for; contexts without old keys, of a tile's edges and of several
# splits; steps of K that are no multiple of a wavefront's sixteen; one key head and as many as heads; a page of 32
@pytest.mark.parametrize("rows,longest,sizes,page", [
    (1, 1, {}, 16), (1, 32, {}, 16), (1, 700, dict(intermediate_size=3072), 16), (2, 2100, dict(hidden_size=640, intermediate_size=1408), 16),
    (3, 65, dict(num_attention_heads=8, num_key_value_heads=1), 32), (4, 300, dict(num_attention_heads=4, num_key_value_heads=4), 16),
    (5, 97, dict(hidden_size=2560, intermediate_size=9728), 16), (8, 513, {}, 16), (9, 40, dict(hidden_size=256, intermediate_size=384, num_attention_heads=2, num_key_value_heads=1), 16),
    (16, 260, dict(intermediate_size=5120), 16), (17, 90, {}, 16), (24, 400, dict(intermediate_size=3072), 16),
    (32, 35, dict(hidden_size=384, num_attention_heads=6, num_key_value_heads=2, intermediate_size=640), 16)])
def test_against_the_parts(rows, longest, sizes, page):
    model = _model(**sizes)
    assert model.decode_run is not None
    lengths = [max(1, longest - 13 * i) for i in range(rows)]
    want = _logits(model, lengths, 3, page=page, launch=False)
    got = _logits(model, lengths, 3, page=page)
    # both round every product and row to bfloat16 (each some 0.008 off exact numbers over these layers), at sums in other orders
    assert (got - want).norm() <= 0.02 * want.norm()
    assert not torch.equal(got, want)                    # (it was another kernel)
    if rows in (1, 2, 3, 8, 16, 24):                        # (sizes that graphs are captured for: no row fills up)
        replayed = _logits(model, lengths, 3, page=page, graphs=True, launch=True)
        assert (replayed - want).norm() <= 0.02 * want.norm()


# rows side by side in ones, twos, fours, eights and sixteens, one less and one more than a group holds, and two groups of wider models
@pytest.mark.parametrize("rows,sizes", [
    (2, {}), (3, {}), (4, {}), (6, {}), (7, {}), (10, {}), (15, {}), (18, {}), (31, {}), (17, dict(hidden_size=1536, intermediate_size=2304)),
    (32, dict(hidden_size=2048, intermediate_size=6144)), (19, dict(hidden_size=4096, num_attention_heads=32, intermediate_size=12288)),
    (32, dict(hidden_size=2176, intermediate_size=18944))])
def test_rows_side_by_side(rows, sizes):
    model = _model(layers=2, **sizes)
    lengths = [1 + (41 * i) % 150 for i in range(rows)]
    want = _logits(model, lengths, 2, launch=False)
    got = _logits(model, lengths, 2)
    # as in the test above; of each row by itself: one that another's numbers came into would be off by its own size
    assert ((got - want).norm(dim=-1) <= 0.03 * want.norm(dim=-1)).all()
    assert not torch.equal(got, want)


def test_any_number_of_blocks_gives_the_same_bits(monkeypatch):
    """Fewer blocks than there is work for, one alone, and more than find room at once, where those that are there go on by themselves."""
    from qwen3_from_scratch_amd.ops.layers import DecodeLayers

    model = _model()
    lengths = [400, 77, 1]
    want = _logits(model, lengths, 2)
    run = DecodeLayers.run
    for blocks, patience in ((1, 64), (7, 64), (100, 64), (300, 64), (300, 1)):
        monkeypatch.setattr(DecodeLayers, "run", lambda self, *args, **named: run(self, *args, **dict(named, blocks=blocks, patience=patience)))
        assert torch.equal(_logits(model, lengths, 2), want), blocks


def test_what_is_not_taken():
    from qwen3_from_scratch_amd import ops

    model = _model()
    native = model.decode_run.native
    rows = torch.zeros(33, 1024, device="cuda")
    caches = [(torch.zeros(4, 8, 16, 128, dtype=torch.bfloat16, device="cuda"), torch.zeros(4, 8, 128, 16, dtype=torch.bfloat16, device="cuda"))] * 3
    table, lens = torch.zeros(33, 4, dtype=torch.int32, device="cuda"), torch.ones(33, dtype=torch.int32, device="cuda")
    assert not native.run(rows, caches, table, lens, 1, None)                # more rows than there are registers for
    wide = _model(hidden_size=1152).decode_run.native
    assert not wide.run(torch.zeros(17, 1152, device="cuda"), caches, table, lens[:17], 1, None)      # or than it is the faster way for
    with pytest.raises(ops.OperandError):
        native.run(rows[:4], caches[:2], table, lens[:4], 1, None)
    with pytest.raises(ops.OperandError):
        native.run(rows[:4], caches, table, lens[:4], 65, None)              # longer than the block table
    assert _model(head_dim=64).decode_run is None
    for small in (dict(hidden_size=128), dict(intermediate_size=128), dict(num_attention_heads=1, num_key_value_heads=1)):
        assert _model(**small).decode_run is None        # (wavefronts without a step of K: their loads would start before the weights)
    layer = dict(native.layers[0], down_tiles=native.layers[0]["down_tiles"][:-1])
    sizes = dict(heads=16, kv_heads=8, dim=128, width=1024, inner=2048, qk_eps=1e-6, scale=1.0)
    assert type(native).of([native.layers[0]], window=0, **sizes) is not None
    assert type(native).of([native.layers[0]], window=8, **sizes) is None and type(native).of([layer], window=0, **sizes) is None


def _layer(heads, kv_heads, inner=256):
    """A layer whose product into the stream passes the attention on as it is and whose other weights are zeros: every key weighs the same."""
    from qwen3_from_scratch_amd import ops
    from qwen3_from_scratch_amd.ops.layers import DecodeLayers

    width = heads * 128
    layer = dict(q_norm=None, k_norm=None, entry_norm=torch.ones(width, device="cuda"), middle_norm=torch.ones(width, device="cuda"),
                 entry_eps=1e-6, middle_eps=1e-6)
    for name, shape in (("qkv", ((heads + 2 * kv_heads) * 128, width)), ("out", None), ("gate_up", (2 * inner, width)), ("down", (width, inner))):
        layer[name] = (torch.eye(width, device="cuda") if shape is None else torch.zeros(shape, device="cuda")).to(torch.bfloat16)
        layer[name + "_tiles"] = ops.tile_weight(layer[name])
    native = DecodeLayers.of([layer], heads, kv_heads, 128, width, inner, 1e-6, 128 ** -0.5, 0)
    assert native is not None
    return native


def _marked_caches(lengths, kv_heads, page, absent=()):
    """Caches where the keys of tile t (of 32) have a one in place t % 128 of their value and zeros elsewhere, in pages in no order, those of the table entries
    `absent` (row, entry) missing; what lies behind a sequence's end is not a number. And what every row's attention over them is."""
    g = torch.Generator().manual_seed(7)
    entries = [-(-n // page) for n in lengths]
    order = torch.randperm(sum(entries), generator=g).tolist()
    keys = torch.full((len(order), kv_heads, page, 128), float("nan"), dtype=torch.bfloat16)
    values = torch.full((len(order), kv_heads, 128, page), float("nan"), dtype=torch.bfloat16)
    table = torch.full((len(lengths), max(entries)), -1, dtype=torch.int32)
    want = torch.zeros(len(lengths), 128, dtype=torch.float64)
    for b, n in enumerate(lengths):
        for e in range(entries[b]):
            at = order.pop()
            held = min(n - 1 - e * page, page)            # (the last token comes with the step)
            if held > 0:
                keys[at, :, :held] = 0
                values[at, :, :, :held] = 0
                for slot in range(held):
                    values[at, :, (e * page + slot) // 32 % 128, slot] = 1
            if (b, e) in absent:
                continue
            table[b, e] = at
            for slot in range(max(held, 0)):
                want[b, (e * page + slot) // 32 % 128] += 1 / n
    return keys.cuda(), values.cuda(), table.cuda(), want


# contexts all alike and one long one among short ones: whole, in as many parts as there are blocks, in two rounds of pieces; rows that bring
# their first token; many key heads and one
UNEVEN = [([1], 8, 8), ([2050], 8, 8), ([1, 4100], 8, 2), ([3000, 31, 33, 64, 1], 8, 1), ([9000] + [40] * 5, 8, 8), ([600] * 8, 16, 16),
          ([50, 700, 5] * 4 + [6000], 16, 16), ([500] * 15 + [8000], 8, 8), ([30 + i for i in range(23)] + [9000], 8, 8), ([257] * 32, 8, 8),
          ([9000] * 2 + [300] * 30, 8, 4), ([2100 - 130 * i for i in range(16)], 32, 32)]


@pytest.mark.parametrize("lengths,heads,kv_heads", UNEVEN)
def test_every_key_counts_once(lengths, heads, kv_heads):
    native = _layer(heads, kv_heads)
    keys, values, table, want = _marked_caches(lengths, kv_heads, 16)
    lens = torch.tensor(lengths, dtype=torch.int32, device="cuda")
    stream = torch.zeros(len(lengths), heads * 128, device="cuda")
    assert native.run(stream, [(keys, values)], table, lens, max(lengths), None)
    got = stream.view(len(lengths), heads, 128).double().cpu()
    # ones and whole sums are exact, the quotient is rounded to bfloat16; a key more or less is 1 / 32 of a place that one tile has
    assert ((got - want[:, None]).abs() <= 2 ** -8 * want[:, None] + 1e-30).all()
    for b, n in enumerate(lengths):                          # the token's own key and value: zeros, where nothing was
        at, slot = int(table[b, (n - 1) // 16]), (n - 1) % 16
        assert not keys[at, :, slot].any() and not values[at, :, :, slot].any()


def test_uneven_keys_go_over_many_blocks():
    """A long sequence among short ones is in as many parts at least as attention of its own kernel would cut it into, pieces are numbered one
    behind the other, and where there are several a sequence, no more of them than the exchange has room for."""
    from qwen3_from_scratch_amd import ops

    native = _layer(8, 8)
    for rows in (1, 6, 8, 12, 16, 24, 32):
        for long in (2000, 8000, 30000):
            lens = torch.full((rows,), 500, dtype=torch.int32, device="cuda")
            lens[rows // 2] = long
            shares = native.shares(lens, long).cpu()
            assert shares[rows // 2, 1] >= (ops._splits(rows, 8, long) if long > 2000 else 1)
            order = shares[:, 0].argsort()
            assert shares[order[0], 0] == 0 and (shares[order][1:, 0] == (shares[order][:-1, 0] + 8 * shares[order][:-1, 1])).all()
            items = 8 * int(shares[:, 1].sum())
            assert items <= 512 and (shares[:, 1] <= 32).all()
            alike = native.shares(torch.full_like(lens, long), long).cpu()
            assert (alike[:, 1] == alike[0, 1]).all() and (alike[0, 1] == 1 or 8 * rows * int(alike[0, 1]) <= 512)


@pytest.mark.parametrize("width,heads,inner,rows", [(1024, 16, 4096, 32), (1024, 16, 8192, 24), (1024, 33, 4096, 24), (1024, 16, 8320, 16), (1152, 9, 3072, 16),
                                                    (4096, 32, 25600, 16), (4608, 36, 14336, 3), (5120, 40, 17408, 3), (5120, 64, 25600, 3),
                                                    (6144, 48, 16384, 8), (8192, 64, 28672, 8)])
def test_rows_that_other_kernels_are_faster_for(width, heads, inner, rows):
    from qwen3_from_scratch_amd.ops import library

    lib = library("decode_layers")
    lib.q3_decode_layers_workspace.restype = ctypes.c_long
    taken = [n for n in range(1, 40) if lib.q3_decode_layers_workspace(4, n, width, heads, heads, 128, inner, 2) > 0]
    assert taken == list(range(1, rows + 1))


def test_a_wait_that_is_given_up_leaves_no_numbers():
    """One look more than none at what other blocks pass on, which is too few for most: the stream is not numbers from end to end, whichever blocks
    and wavefronts gave up, and the launch ends."""
    for sizes, rows in (({}, 1), ({}, 3), ({}, 24), (dict(hidden_size=2560, intermediate_size=4096), 1), (dict(hidden_size=2560, intermediate_size=4096), 16)):
        model = _model(**sizes)
        native, width = model.decode_run.native, sizes.get("hidden_size", 1024)
        lengths = [500 - 7 * i for i in range(rows)]
        keys, values, table, _ = _marked_caches(lengths, 8, 16)
        caches = [(keys.clone(), values.clone()) for _ in native.layers]
        lens = torch.tensor(lengths, dtype=torch.int32, device="cuda")
        g = torch.Generator(device="cuda").manual_seed(2)
        first = torch.randn(rows, width, generator=g, device="cuda")
        rotation = model.position.rotation_table()

        def result(**named):
            stream = first.clone()
            assert native.run(stream, caches, table, lens, max(lengths), rotation, **named)
            return stream

        want = result()
        assert torch.isfinite(want).all()
        assert torch.isnan(result(limit=1)).all()
        assert torch.equal(result(), want)


def test_graphs_share_what_they_need_between_kernels():
    """Captured for one size after another, the launches' exchanges lie in the same memory, and each graph goes on giving what the parts give,
    whichever ran in between."""
    from qwen3_from_scratch_amd.engine import ModelRunner, StepEntry

    model = _model(layers=64)
    runs, sizes, steps = model.decode_run, (24, 16, 12, 8, 6, 4), 3
    g = torch.Generator().manual_seed(3)
    ids = [torch.randint(0, 512, (300 + steps * len(sizes),), generator=g).tolist() for _ in range(sizes[0])]
    taken, logits = [], {}
    for launch in (True, False):
        model.decode_run = runs if launch else None
        runner = ModelRunner(model, 16, 24 * 24, max_requests=24, use_graphs=launch)
        at = [200 + 3 * i for i in range(24)]
        for i, n in enumerate(at):
            runner.step([StepEntry(i, ids[i][:n], [])])
        out = []
        for _ in range(steps):
            for rows in sizes:
                out.append(runner.step([StepEntry(i, [ids[i][at[i]]], [0]) for i in range(rows)]).clone())
                at = [n + (i < rows) for i, n in enumerate(at)]
                if launch and len(taken) < len(sizes):
                    torch.cuda.synchronize()
                    taken.append(torch.cuda.memory_reserved())
        logits[launch] = out
    model.decode_run = runs
    for got, want in zip(logits[True], logits[False]):
        assert (got - want).norm() <= 0.04 * want.norm()
    own = [runs.native._workspace(64, rows, 1024, 16, 8, 128, 2048, 1) for rows in sizes[1:]]
    assert taken[-1] - taken[0] < sum(own) // 4, (taken, own)


NO_QK_NORM = {"mixer": {"name": "attention", "kwargs": dict(qk_norm=False)}}


# float32 weights of the norms, heads without norms, without a rotation, more layers than the launch's table takes at a time, by rows that take other
# instantiations; contexts far apart
@pytest.mark.parametrize("lengths,named", [
    ([300], dict(scales=torch.float32)), ([90, 5] * 5, dict(scales=torch.float32)), ([40 + i for i in range(20)], dict(scales=torch.float32)),
    ([300, 20], dict(components=NO_QK_NORM)), ([77] * 12, dict(components=NO_QK_NORM)), ([64] * 18, dict(components=NO_QK_NORM)),
    ([300, 20], dict(turned=False)), ([33, 600] * 9, dict(turned=False, scales=torch.float32)),
    ([70], dict(layers=43, hidden_size=256, num_attention_heads=2, num_key_value_heads=1, intermediate_size=256)),
    ([6000] + [40, 300, 5] * 3, {}), ([4, 2500] + [90] * 20, {})])
def test_other_layers_against_the_parts(lengths, named):
    model = _model(**named)
    assert model.decode_run is not None
    want = _logits(model, lengths, 2, launch=False)
    got = _logits(model, lengths, 2)
    # as in `test_against_the_parts`, whose three layers are off by 0.008 each side; rounding adds up with the root of the depth
    bound = 0.02 * max(1.0, (named.get("layers", 3) / 3) ** 0.5)
    assert (got - want).norm() <= bound * want.norm() and not torch.equal(got, want)


@pytest.mark.parametrize("lengths", [[700], [2100, 40], [90, 400, 33, 260] * 2, [1000 - 60 * i for i in range(14)], [35 * i + 5 for i in range(24)]])
def test_as_near_to_float32_as_the_parts(lengths):
    """Queries that look at few keys, row by row: the launch is as far from the same layers in float32 as the parts are. A tile of keys left out or
    counted twice shows in the rows that look at it."""
    exact = _logits(_model(dtype="float32", sharp=4.0), lengths, 2)
    model = _model(sharp=4.0)
    away = [(_logits(model, lengths, 2, launch=launch) - exact).norm(dim=-1) / exact.norm(dim=-1) for launch in (False, True)]
    assert away[1].max() <= 2 * away[0].max(), away
    assert away[1].pow(2).mean().sqrt() <= 1.25 * away[0].pow(2).mean().sqrt(), away


@pytest.mark.parametrize("rows", [5, 9, 17, 25])
def test_rows_that_fill_a_captured_step_up(rows):
    """Captured for the next larger size, with rows that stand for nobody: the requests' logits are those of a step without them."""
    model = _model()
    lengths = [50 + 11 * i for i in range(rows)]
    eager, replayed = _logits(model, lengths, 3), _logits(model, lengths, 3, graphs=True)
    want = _logits(model, lengths, 3, launch=False)
    assert (replayed - want).norm() <= 0.02 * want.norm()
    # (the same kernel, or another one of two groups of rows or of how rows are asked for: sums in the same order)
    assert torch.equal(eager, replayed)


@pytest.mark.parametrize("page", [16, 32])
def test_table_entries_without_a_page(page):
    """Keys of a page that is not there count as zeros with values of zeros: first, last old and inner ones, whole tiles and halves."""
    lengths, heads, kv_heads = [600, 97, 40], 8, 4
    absent = {(0, 0), (0, 7), (0, 8), (0, 600 // page - 1), (1, 1), (2, 0)}
    native = _layer(heads, kv_heads)
    keys, values, table, want = _marked_caches(lengths, kv_heads, page, absent)
    lens = torch.tensor(lengths, dtype=torch.int32, device="cuda")
    stream = torch.zeros(3, heads * 128, device="cuda")
    assert native.run(stream, [(keys, values)], table, lens, max(lengths), None)
    got = stream.view(3, heads, 128).double().cpu()
    assert ((got - want[:, None]).abs() <= 2 ** -8 * want[:, None] + 1e-30).all()


@pytest.mark.parametrize("lengths", [[40, 70, 33], [900, 500, 1200]])
@pytest.mark.parametrize("which,bad", [("keys", float("inf")), ("keys", float("nan")), ("values", float("inf")), ("values", float("nan"))])
def test_what_is_no_number_in_the_caches(lengths, which, bad):
    """One number of the middle request's keys or values that is none: its logits are none, as the parts have it, and the others' are unharmed."""
    from qwen3_from_scratch_amd.engine import ModelRunner, StepEntry

    model = _model()
    run, logits = model.decode_run, {}
    for launch in (True, False):
        for harmed in (False, True):
            model.decode_run = run if launch else None
            runner = ModelRunner(model, 16, 400, max_requests=3, use_graphs=False)
            for i, n in enumerate(lengths):
                runner.step([StepEntry(i, [(7 * j + i) % 512 for j in range(n)], [])])
            if harmed:
                at = runner.manager.block_table(1, 0)[1]
                runner.storage.paged[0][which][1][at, 3].view(-1)[200] = bad
            logits[launch, harmed] = runner.step([StepEntry(i, [9], [0]) for i in range(3)]).clone()
    model.decode_run = run
    for launch in (True, False):
        assert not torch.isfinite(logits[launch, True][1]).any(), launch
        assert torch.equal(logits[launch, True][[0, 2]], logits[launch, False][[0, 2]]), launch


def test_two_launches_on_two_streams():
    """Both in flight at once, each on whatever processors it finds: each gives what it gives alone."""
    model = _model()
    native, rotation, g = model.decode_run.native, model.position.rotation_table(), torch.Generator(device="cuda").manual_seed(4)
    steps = []
    for lengths in ([700, 90, 300], [400 + 9 * i for i in range(20)]):
        keys, values, table, _ = _marked_caches(lengths, 8, 16)
        steps.append((torch.randn(len(lengths), 1024, generator=g, device="cuda"), [(keys.clone(), values.clone()) for _ in native.layers], table,
                      torch.tensor(lengths, dtype=torch.int32, device="cuda"), max(lengths)))

    def launch(first, caches, table, lens, longest):
        stream = first.clone()
        assert native.run(stream, caches, table, lens, longest, rotation)
        return stream

    want = [launch(*step) for step in steps]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = []
    for turn in range(10):
        for on, step in zip(streams, steps):
            with torch.cuda.stream(on):
                got.append(launch(*step))
    torch.cuda.synchronize()
    for i, stream in enumerate(got):
        assert torch.equal(stream, want[i % 2]), i


def test_steps_over_nothing_are_left_to_the_parts():
    """Caches without a page, and sequences without a length: refused by neither."""
    from types import SimpleNamespace

    model = _model(layers=1)
    native, rotation = model.decode_run.native, model.position.rotation_table()
    stream, lens, table = torch.ones(2, 1024, device="cuda"), torch.ones(2, dtype=torch.int32, device="cuda"), torch.zeros(2, 4, dtype=torch.int32, device="cuda")
    for pages, longest in ((0, 1), (3, 0)):
        caches = [(torch.zeros(pages, 8, 16, 128, dtype=torch.bfloat16, device="cuda"), torch.zeros(pages, 8, 128, 16, dtype=torch.bfloat16, device="cuda"))]
        assert not native.run(stream, caches, table, lens * longest, longest, rotation)
        view = SimpleNamespace(paged=dict(keys=caches[0][0], values=caches[0][1]), block_table=table, writes=True)
        cache = SimpleNamespace(pages_of=lambda planes, names: (caches, table), view=lambda plane, writes=True: view)
        batch = SimpleNamespace(token_ids=torch.zeros(2, dtype=torch.int32, device="cuda"), max_q_len=1, min_q_len=1, kv_lens=lens * longest, max_kv_len=longest,
                                cu_seqlens_q=torch.arange(3, dtype=torch.int32, device="cuda"), logits_rows=None)
        assert torch.isfinite(model.forward(batch, cache)).all()
