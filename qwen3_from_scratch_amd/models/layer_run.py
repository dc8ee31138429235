"""Stretches of equal layers that a step may run as one native call."""

from ..ops.layers import DECODE_ROWS_MOST, Declined, DecodeLayers, DecoderLayers
from ..parts.base import UnscaledRows


class LayerRun:
    """The steps `begin` .. `end - 1` of a model's run order, whose layers `ops.layers.DecoderLayers` takes: layers of one shape,
    each with a cache plane of its own to write, each followed by one whose entry norm its last product prepares."""

    def __init__(self, begin, end, native, position, planes, blocks, exit_norm):
        self.begin, self.end = begin, end
        self.native, self.position, self.planes, self.blocks, self.exit_norm = native, position, planes, blocks, exit_norm

    def forward(self, first, x, pending, batch, cache):
        """The layers from step `first` on, from UnscaledRows, as their blocks would run them: (stream, what it still lacks, the
        first step that is not done yet), or None, with nothing done, for a step that is another kernel's: of single tokens alone
        (attention with its own preparation), of rows that a product does not take in the form that carries its norm, or over
        pages that the matrix cores do not take."""
        if batch.max_q_len == 1 or not self.native.rows_fit(x.shape[0]) or not hasattr(cache, "pages_of"):
            return None
        caches, block_table = cache.pages_of(self.planes[first - self.begin:], ("keys", "values"))
        if caches is None:
            return None
        table = self.position.rotation_table() if self.position is not None else None
        done = self.native.run(first - self.begin, self.end - first, x, pending.values, pending.sums, caches, block_table,
                               batch.positions, batch.seq_index, batch.cu_seqlens_q, batch.kv_lens, batch.max_q_len,
                               batch.min_q_len, batch.max_kv_len, getattr(batch, "max_kv_len_portions", None), table)
        if done is None:
            return None
        if isinstance(done, Declined):
            step = first + done.layer
            block = self.blocks[step - self.begin]
            if not done.of_attention:
                return x, block.feed_forward.down.forward(done.rows), step + 1
            h = block.feed_forward_norm.forward(x, delta=block.mixer.out.forward(done.rows))
            return x, block.feed_forward.forward(h, batch), step + 1
        return x, UnscaledRows(done[0], done[1], self.exit_norm.eps, self.exit_norm.size), self.end


def layer_runs(model):
    """{step of the run order: the LayerRun it belongs to} for every step that belongs to one."""
    order, found, runs = model.spec.order, [], {}
    for i, step in enumerate(order):
        block, entry = model.layers[step.layer].block, None
        if step.enters is None and step.reads_cache_of is None and i + 1 < len(order) and order[i + 1].enters is None:
            after = getattr(model.layers[order[i + 1].layer].block, "entry_norm", None)
            entry = after() if after else None
        found.append(block.native_layer(entry) if entry is not None and hasattr(block, "native_layer") else None)
    at = 0
    while at < len(order):
        end = at
        while end < len(order) and found[at] and found[end] and found[end][1:] == found[at][1:]:
            end += 1
        if end > at:
            native = DecoderLayers.of([f[0] for f in found[at:end]], **found[at][1])
            if native is not None:
                exit_norm = model.layers[order[end].layer].block.entry_norm()
                run = LayerRun(at, end, native, found[at][2], [model.plane_of_step[i] for i in range(at, end)],
                               [model.layers[order[i].layer].block for i in range(at, end)], exit_norm)
                runs.update((i, run) for i in range(at, end))
        at = max(end, at + 1)
    return runs


class DecodeRun:
    """All steps of a model's run order, of layers that `ops.layers.DecodeLayers` takes, each with a cache plane of its own to write."""

    def __init__(self, native, position, planes):
        self.native, self.position, self.planes = native, position, planes

    def forward(self, x, batch, cache):
        """The layers over the stream x, in place, if the step is one of single tokens that the launch takes; whether it was.
        (It takes the rows, widths and inner sizes for which it was measured to be the faster way: csrc/decode_layers.hip, `rows_most`.)"""
        if batch.max_q_len != 1 or not 1 <= x.shape[0] <= DECODE_ROWS_MOST or batch.kv_lens.shape[0] != x.shape[0]:
            return False
        if not hasattr(cache, "pages_of"):
            return False
        caches, block_table = cache.pages_of(self.planes, ("keys", "values"))
        if caches is None:
            return False
        table = self.position.rotation_table() if self.position is not None else None
        return self.native.run(x, caches, block_table, batch.kv_lens, batch.max_kv_len, table)


def decode_run(model):
    """The DecodeRun of a model, or None for one with other layers."""
    order, found = model.spec.order, []
    if getattr(model.pass_vectors, "wants_start", False):
        return None
    for step in order:
        block = model.layers[step.layer].block
        if step.enters is not None or step.reads_cache_of is not None or not hasattr(block, "native_layer"):
            return None
        found.append(block.native_layer())
    if not found or None in found or any(f[1:] != found[0][1:] for f in found):
        return None
    native = DecodeLayers.of([f[0] for f in found], **found[0][1])
    return None if native is None else DecodeRun(native, found[0][2], [model.plane_of_step[i] for i in range(len(order))])
