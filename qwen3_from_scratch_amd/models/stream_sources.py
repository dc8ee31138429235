"""A residual in several streams as the sums that its streams are.

Every stream is a weighted sum of the embedding's rows and of the sublayers' results so far, with weights that follow from the
layers' `in`, `out` and `mix` tables alone. While the results take no more memory than the streams and the next result would, a pass keeps the sources and
reads the weighted sum that a norm wants of them in one kernel (`ops.read_sources`); from the first sublayer on for which the
streams are the smaller, it goes on with them (`ops.streams_from_sources`, for whose length both are there).
"""

import math

import torch

from .. import ops
from ..parts.base import writes_to
from ..parts.block import HyperConnectionBlock
from ..parts.embedding import TokenEmbedding
from ..parts.norm import LayerNorm


class StreamPlan:
    """Per read of a pass (one per sublayer, and the last norm's) the sources' coefficients; `until` reads are made of sources,
    and `streams` (streams, sources) are the coefficients of the streams themselves in front of the read that is not."""

    def __init__(self, reads, until, streams, blocks=()):
        self.reads, self.until, self.streams = reads, until, streams
        # what the coefficients were made of: per block its tables, and how often each of them had been written
        self._made_of = [(block, dict(block.tables)) for block in blocks]
        self._writes = [(t, writes_to(t)) for _, held in self._made_of for of_sublayer in held.values() for t in of_sublayer]

    def current(self):
        """Whether the tables are still those, and as they were, that the coefficients were made of."""
        return (all(writes_to(t) == n for t, n in self._writes)
                and all(block.tables.get(q) is of_sublayer for block, held in self._made_of for q, of_sublayer in held.items()))

    def start(self, token_ids, table):
        return StreamSources(self, token_ids, table)


class StreamSources:
    """The residual of one pass: the embedding's rows, as table and ids, and the sublayers' results. Stands where the stream
    tensor does between blocks and norms."""

    def __init__(self, plan, ids, table):
        self.plan, self.ids, self.table = plan, ids, table
        self.values, self.at, self.streams = [], 0, None

    def join(self, delta):
        """What a sublayer gave (a HyperAddend, of one result or of several with a scale each) is a source from here on."""
        for values in delta.values if isinstance(delta.values, tuple) else (delta.values,):
            self.values.append(values if values.data_ptr() % 16 == 0 else values.clone())

    def read(self, norm, delta, read, rows):
        """`norm` of what its sublayer reads, behind `delta`."""
        if self.streams is not None:
            return ops.hyper_norm(self.streams, norm.weight, norm.eps, norm.precision.act, read=read,
                                  delta=None if delta is None else delta.joined(), mix=None if delta is None else delta.mix,
                                  write=None if delta is None else delta.write, rows=rows, write_back=rows is None)
        if delta is not None:
            self.join(delta)
        at, self.at = self.at, self.at + 1
        if at < self.plan.until:
            return ops.read_sources(self.ids, self.table, self.values, self.plan.reads[at], norm.weight, norm.eps, rows=rows)
        self.streams = ops.streams_from_sources(self.ids, self.table, self.values, self.plan.streams)
        self.values = []
        return ops.hyper_norm(self.streams, norm.weight, norm.eps, norm.precision.act, read=read, rows=rows)


def results_most(streams, size):
    """How many sublayers' results, of `size` bytes a number, are kept in the place of `streams` streams of float32 numbers: as many as
    take the memory of the streams and of the result that joins them next, and no more than 20 bytes a number, since results and streams are both
    there where one gives way to the other, beside less than what a mixer needs for itself. (By what a sublayer moves it would be twice as many; but
    a long prompt then needs more memory than with the streams: 24 layers of a width of 1,024 in four streams over 8,192 tokens 369 MB, so 330 as
    with them.)"""
    return min(ops.SOURCES_MOST - 3, 4 * streams // size + 1, 20 // size)


def stream_plan(model):
    """The plan of a loaded model on the GPU whose residual is in several streams from its embedding to its last norm, or None."""
    order, blocks = model.spec.order, [layer.block for layer in model.layers]
    streams = getattr(model.embedding, "copies", 0)
    if model.device.type != "cuda" or streams < 2 or type(model.embedding) is not TokenEmbedding:
        return None
    if model.spec.position.name != "none" or any(step.enters is not None for step in order):
        return None
    if not all(type(block) is HyperConnectionBlock and block.streams == streams for block in blocks):
        return None
    norms = [model.final_norm] + [n for block in blocks for n in (block.mixer_norm, block.feed_forward_norm) if n is not None]
    table, width = model.embedding.weight, model.embedding.hidden_size
    if not all(type(n) is LayerNorm and n.size == width and n.weight.data_ptr() % 16 == 0 for n in norms):
        return None
    if width % 4 or width > 4096 or table.data_ptr() % 16 or table.dtype != model.precision.act:
        return None
    # coefficients of every source in every stream, from the tables' numbers in double precision
    each = [[1.0] * streams]
    reads, until, at_streams = [], 0, None
    most = 1 + results_most(streams, table.element_size())      # (the embedding's rows stay in its table; a sublayer adds up to two)

    def take(weights, most):
        nonlocal until, at_streams
        if at_streams is not None:
            return
        if len(each) > most:
            at_streams = [[c[s] for c in each] for s in range(streams)]
            return
        reads.append([sum(w * x for w, x in zip(weights, c)) for c in each])
        until += 1

    # every table's numbers in one copy to the host
    tables = [t for block in blocks for q, _ in block.sublayer_scales() for t in block.tables[q]]
    flat, numbers = torch.cat([t.reshape(-1) for t in tables]).tolist(), {}
    for i, block in enumerate(blocks):
        for q, _ in block.sublayer_scales():
            read, write, mix = flat[:streams], flat[streams:2 * streams], flat[2 * streams:2 * streams + streams * streams]
            numbers[i, q] = read, write, [mix[s * streams:(s + 1) * streams] for s in range(streams)]
            flat = flat[2 * streams + streams * streams:]
    for step in order:
        for q, scales in blocks[step.layer].sublayer_scales():
            read, write, mix = numbers[step.layer, q]
            take(read, most)
            each = [[sum(c[s] * mix[s][t] for s in range(streams)) for t in range(streams)] for c in each]
            each += [[w * scale for w in write] for scale in scales]
            if at_streams is not None:
                break
    take([1.0] * streams, ops.SOURCES_MOST)      # (nothing follows that streams would serve)
    if until == 0 or not all(math.isfinite(x) and abs(x) < 2.0 ** 127 for row in reads + (at_streams or []) for x in row):
        return None
    if at_streams is not None:
        at_streams = torch.tensor(at_streams, dtype=torch.float32, device=model.device)
    return StreamPlan(reads, until, at_streams, blocks)
