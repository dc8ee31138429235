"""A stretch of equal decoder layers as one native call (csrc/layers.hip): what the layers' parts would do operation by
operation, for steps whose time is the host's."""

import ctypes
from typing import NamedTuple

import torch

from . import (_DECLINED, _DT, _check, _matmul, _splits, _stream, few_rows_limit, fused_rows_most, library, matmul_fused_plan, sums_stride,
               FUSED_ROWS_SMALL, OperandError)

_P, _I, _F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float


class _Layer(ctypes.Structure):
    _fields_ = [(n, _P) for n in ("qkv", "out", "gate_up", "down", "q_norm", "k_norm", "middle_norm", "next_norm", "keys", "values")
                ] + [("entry_eps", _F), ("middle_eps", _F)]


class _Step(ctypes.Structure):
    _fields_ = ([(n, _P) for n in ("scaled", "residual", "prepare", "attention", "stream")]
                + [(n, _I) for n in ("rows", "width", "heads", "kv_heads", "dim", "inner", "norm_dtype", "qk_dtype")]
                + [("qk_eps", _F), ("scale", _F), ("window", _I), ("table", _P), ("rotary_dim", _I), ("max_pos", _I)]
                + [(n, _P) for n in ("positions", "seq_index", "block_table", "cu_q", "kv_lens")]
                + [(n, _I) for n in ("table_width", "sequences", "page", "num_pages", "max_q_len", "min_q_len", "max_kv_len", "longest",
                                     "splits", "prompt_splits")]
                + [(n, _P) for n in ("workspace", "prompt_workspace", "residual_rows", "entry_values", "entry_sums")]
                + [(n, _I) for n in ("entry_chunks", "sums_stride", "middle_chunks", "exit_chunks")]
                + [(n, _P) for n in ("qkv_rows", "attended", "hidden", "norm_rows", "middle_sums", "exit_sums")])


_OPERATIONS = ("the product of queries, keys and values", "qk_norm_rope_store", "paged_attention", "the attention's output product",
               "the gated product", "the product back into the stream")
_ATTENTION_OUT, _DOWN = 3, 5        # the two that add into the stream


class Declined(NamedTuple):
    """Where a stretch ended early: `layer` (from the first one run) whose product into the stream was left to the plain product and
    the norm's own kernel, the attention's output product (`of_attention`) or the feed-forward's, and the rows that lack it."""

    layer: int
    of_attention: bool
    rows: torch.Tensor


def _matrix(t, shape):
    return (t is not None and t.is_cuda and t.dtype == torch.bfloat16 and t.shape == shape and t.is_contiguous()
            and fused_rows_most(t) == FUSED_ROWS_SMALL and shape[1] % 64 == 0 and shape[0] % 4 == 0)


def _vector(t, size, dtype):
    return t is not None and t.is_cuda and t.shape == (size,) and t.dtype == dtype and t.is_contiguous()


class DecoderLayers:
    """Layers of one shape: `layers`, per layer a dict of its tensors (`qkv`, `out`, `gate_up` with its rows interleaved, `down`;
    `q_norm`, `k_norm` or None; `middle_norm`, `next_norm`) and `entry_eps`, `middle_eps`; and the sizes they share. The
    tensors are looked at here, once; `None` from `of` if they are not what the native call takes."""

    def __init__(self, layers, heads, kv_heads, dim, width, inner, qk_eps, scale, window):
        self.layers = layers
        self.heads, self.kv_heads, self.dim, self.width, self.inner = heads, kv_heads, dim, width, inner
        self.qk_eps, self.scale, self.window = float(qk_eps), float(scale), int(window)
        self.norm_dtype = layers[0]["middle_norm"].dtype
        self.qk_dtype = layers[0]["q_norm"].dtype if layers[0]["q_norm"] is not None else torch.float32
        self.least_rows = 1 + max(few_rows_limit(l[n]) for l in layers for n in ("qkv", "out", "gate_up", "down"))

    @classmethod
    def of(cls, layers, heads, kv_heads, dim, width, inner, qk_eps, scale, window):
        norm_dtype = getattr(layers[0]["middle_norm"], "dtype", None)
        for l in layers:
            if not (_matrix(l["qkv"], ((heads + 2 * kv_heads) * dim, width)) and _matrix(l["out"], (width, heads * dim))
                    and _matrix(l["gate_up"], (2 * inner, width)) and _matrix(l["down"], (width, inner))
                    and norm_dtype in _DT and _vector(l["middle_norm"], width, norm_dtype) and _vector(l["next_norm"], width, norm_dtype)):
                return None
            if (l["q_norm"] is None) != (l["k_norm"] is None) or (l["q_norm"] is None) != (layers[0]["q_norm"] is None):
                return None
            if l["q_norm"] is not None and not (l["q_norm"].dtype in _DT and _vector(l["q_norm"], dim, layers[0]["q_norm"].dtype)
                                                and _vector(l["k_norm"], dim, layers[0]["q_norm"].dtype)):
                return None
        if not library("attention").q3_paged_attention_fast_path(heads, kv_heads, dim, 16, _DT[torch.bfloat16]):
            return None                               # (a head size whose attention is another kernel's at any page)
        return cls(layers, heads, kv_heads, dim, width, inner, qk_eps, scale, window)

    def rows_fit(self, rows):
        """Whether a step of so many rows is one whose four products all carry their norms by kernels that take row-major weights."""
        if not self.least_rows <= rows <= FUSED_ROWS_SMALL:
            return False
        plans = [matmul_fused_plan("residual", rows, self.width, k) for k in (self.heads * self.dim, self.inner)]
        return all(plan is not None and plan[0] >= 0 for plan in plans)

    def run(self, first, count, stream, values, sums, caches, block_table, positions, seq_index, cu_seqlens_q, kv_lens, max_q_len,
            min_q_len, max_kv_len, max_kv_len_of_many, table):
        """Layers `first` .. `first + count - 1` over the residual `stream` (T, width) float32, in place, from rows
        (`values`, `sums`: see `linear_residual_norm`) that lack the first one's entry norm. `caches`: per layer (keys, values), as
        `paged_attention` takes them, all of one shape. Returns the rows that lack the norm behind the last layer, as (values,
        sums); None, and nothing is done, where the attention is not one for the matrix cores; Declined where a product into the
        stream is not one of those that carry a norm after all (`rows_fit` was asked, and another thread has changed which kernels serve)."""
        if not (0 <= first and 0 < count <= len(self.layers) - first and len(caches) == count and caches[0][0].dim() == 4):
            raise OperandError("a cache for each of the layers, keys (pages, Hkv, page, D)")
        T = values.shape[0]
        H, G, D, page = self.heads, self.kv_heads, self.dim, caches[0][0].shape[2]
        attention = library("attention")
        if not attention.q3_paged_attention_fast_path(H, G, D, page, _DT[torch.bfloat16]):
            return None
        B = kv_lens.shape[0]
        stride = sums_stride(T)
        if not (stream.is_cuda and stream.shape == (T, self.width) and stream.dtype == torch.float32 and stream.is_contiguous()
                and values.shape == (T, self.width) and values.dtype == torch.bfloat16 and values.is_cuda and values.is_contiguous()
                and sums.is_cuda and sums.dim() == 2 and sums.shape[1] == stride and sums.dtype == torch.float32 and sums.is_contiguous()):
            raise OperandError("a float32 stream, bfloat16 rows and float32 sums of squares, contiguous")
        for t, shape in ((positions, (T,)), (seq_index, (T,)), (cu_seqlens_q, (B + 1,)), (kv_lens, (B,))):
            if not (t.is_cuda and t.dtype == torch.int32 and t.shape == shape and t.is_contiguous()):
                raise OperandError("positions and seq_index int32 (T,), cu_seqlens_q int32 (B+1,), kv_lens int32 (B,)")
        if not (block_table.is_cuda and block_table.dim() == 2 and block_table.dtype == torch.int32 and block_table.shape[0] >= B
                and block_table.is_contiguous() and block_table.shape[1] * page >= max_kv_len and 1 <= min_q_len <= max_q_len):
            raise OperandError("block_table must be int32 (B, W) and hold the longest sequence")
        pages = caches[0][0].shape[0]
        for keys, held in caches:
            if not (keys.is_cuda and keys.dtype == torch.bfloat16 and keys.shape == (pages, G, page, D) and keys.is_contiguous()
                    and held.is_cuda and held.dtype == torch.bfloat16 and held.shape == (pages, G, D, page) and held.is_contiguous()
                    and pages > 0):
                raise OperandError("caches must be keys (pages, Hkv, page, D) and values (pages, Hkv, D, page) in bfloat16")
        rotary_dim, max_pos = 0, 0
        if table is not None:
            if not (table.is_cuda and table.dim() == 2 and table.dtype == torch.float32 and table.is_contiguous()
                    and table.shape[1] % 2 == 0 and table.shape[1] <= D and max_kv_len <= table.shape[0]):
                raise OperandError("table must be float32 (P, R) and hold the step's last position")
            max_pos, rotary_dim = table.shape
        matmul, rotary = _matmul(), library("rotary")

        def empty(*shape, dtype=torch.bfloat16):
            return torch.empty(shape, dtype=dtype, device=values.device)

        splits, workspace, prompt_splits, prompt_workspace = 1, None, 1, None
        if min_q_len * (H // G) <= 16:
            splits = _splits(B, G, int(max_kv_len))
            if splits > 1:
                attention.q3_paged_attention_workspace.restype = ctypes.c_long
                workspace = empty(attention.q3_paged_attention_workspace(B, G, D, splits), dtype=torch.float32)
        longest = int(max_kv_len if max_kv_len_of_many is None else max_kv_len_of_many)
        if max_q_len * (H // G) > 16:
            prompt_splits = attention.q3_paged_attention_prompt_splits(
                T, H, G, min(longest, self.window + 128) if self.window else longest)
            if prompt_splits > 1:
                prompt_workspace = empty(T * H * prompt_splits * (D + 2), dtype=torch.float32)
        out = empty(T, self.width)
        middle = empty(matmul.q3_tiles_residual_chunks(T, self.width, H * D), stride, dtype=torch.float32)
        exit_ = empty(matmul.q3_tiles_residual_chunks(T, self.width, self.inner), stride, dtype=torch.float32)
        qkv, attended, hidden = empty(T, (H + 2 * G) * D), empty(T, H * D), empty(T, self.inner)

        def at(t):
            return None if t is None else t.data_ptr()

        step = _Step(
            scaled=ctypes.cast(matmul.q3_tiles_scaled, _P), residual=ctypes.cast(matmul.q3_tiles_residual, _P),
            prepare=ctypes.cast(rotary.q3_qk_norm_rope_store, _P), attention=ctypes.cast(attention.q3_paged_attention, _P),
            stream=_stream(), rows=T, width=self.width, heads=H, kv_heads=G, dim=D, inner=self.inner,
            norm_dtype=_DT[self.norm_dtype], qk_dtype=_DT[self.qk_dtype], qk_eps=self.qk_eps, scale=self.scale, window=self.window,
            table=at(table), rotary_dim=rotary_dim, max_pos=max_pos, positions=at(positions), seq_index=at(seq_index),
            block_table=at(block_table), cu_q=at(cu_seqlens_q), kv_lens=at(kv_lens), table_width=block_table.shape[1], sequences=B,
            page=page, num_pages=pages, max_q_len=int(max_q_len), min_q_len=int(min_q_len), max_kv_len=int(max_kv_len), longest=longest,
            splits=splits, prompt_splits=prompt_splits, workspace=at(workspace), prompt_workspace=at(prompt_workspace),
            residual_rows=at(stream), entry_values=at(values), entry_sums=at(sums), entry_chunks=sums.shape[0], sums_stride=stride,
            middle_chunks=middle.shape[0], exit_chunks=exit_.shape[0], qkv_rows=at(qkv), attended=at(attended), hidden=at(hidden),
            norm_rows=at(out), middle_sums=at(middle), exit_sums=at(exit_))
        layers = (_Layer * count)()
        for native, l, (keys, held) in zip(layers, self.layers[first:first + count], caches):
            native.qkv, native.out, native.gate_up, native.down = at(l["qkv"]), at(l["out"]), at(l["gate_up"]), at(l["down"])
            native.q_norm, native.k_norm = at(l["q_norm"]), at(l["k_norm"])
            native.middle_norm, native.next_norm = at(l["middle_norm"]), at(l["next_norm"])
            native.keys, native.values = keys.data_ptr(), held.data_ptr()
            native.entry_eps, native.middle_eps = l["entry_eps"], l["middle_eps"]
        failed = ctypes.c_int(0)
        status = library("layers").q3_decoder_layers(layers, count, ctypes.byref(step), ctypes.byref(failed))
        layer, operation = divmod(failed.value, len(_OPERATIONS))
        if status == _DECLINED and operation in (_ATTENTION_OUT, _DOWN):
            return Declined(layer, operation == _ATTENTION_OUT, attended if operation == _ATTENTION_OUT else hidden)
        _check(status, _OPERATIONS[operation])
        return out, exit_


DECODE_ROWS_MOST = 32          # rows of a step of single tokens that `DecodeLayers` takes (of some shapes 24 or 16, and of very wide models fewer)


class _DecodeLayer(ctypes.Structure):
    _fields_ = [(n, _P) for n in ("qkv", "out", "gate_up", "down", "q_norm", "k_norm", "entry_norm", "middle_norm", "keys", "values")
                ] + [("entry_eps", _F), ("middle_eps", _F)]


class DecodeLayers:
    """All layers of one shape for steps of single tokens, in one launch (csrc/decode_layers.hip): `layers` as `DecoderLayers` has
    them, and their tile-ordered matrices (`qkv_tiles`, `out_tiles`, `gate_up_tiles`, `down_tiles`) and `entry_norm`. The tensors
    are looked at here, once; `None` from `of` if they are not what the launch takes."""

    def __init__(self, layers, heads, kv_heads, dim, width, inner, qk_eps, scale):
        self.layers = layers
        self.heads, self.kv_heads, self.dim, self.width, self.inner = heads, kv_heads, dim, width, inner
        self.qk_eps, self.scale = float(qk_eps), float(scale)
        self.norm_dtype = layers[0]["middle_norm"].dtype
        self.qk_dtype = layers[0]["q_norm"].dtype if layers[0]["q_norm"] is not None else torch.float32
        lib = library("decode_layers")
        lib.q3_decode_layers_workspace.restype = ctypes.c_long
        self._workspace = lib.q3_decode_layers_workspace

    @classmethod
    def of(cls, layers, heads, kv_heads, dim, width, inner, qk_eps, scale, window):
        norm_dtype = getattr(layers[0]["middle_norm"], "dtype", None)
        if window or norm_dtype not in _DT:
            return None
        for l in layers:
            for name, shape in (("qkv", ((heads + 2 * kv_heads) * dim, width)), ("out", (width, heads * dim)),
                                ("gate_up", (2 * inner, width)), ("down", (width, inner))):
                if not (l[name] is not None and l[name].shape == shape and shape[0] % 16 == 0
                        and _vector(l[name + "_tiles"], shape[0] * shape[1], torch.bfloat16)):
                    return None
            if not (_vector(l["entry_norm"], width, norm_dtype) and _vector(l["middle_norm"], width, norm_dtype)):
                return None
            if (l["q_norm"] is None) != (l["k_norm"] is None) or (l["q_norm"] is None) != (layers[0]["q_norm"] is None):
                return None
            if l["q_norm"] is not None and not (l["q_norm"].dtype in _DT and _vector(l["q_norm"], dim, layers[0]["q_norm"].dtype)
                                                and _vector(l["k_norm"], dim, layers[0]["q_norm"].dtype)):
                return None
            if any(l[n].data_ptr() % 16 for n in ("entry_norm", "middle_norm", "q_norm", "k_norm") if l[n] is not None):
                return None
        found = cls(layers, heads, kv_heads, dim, width, inner, qk_eps, scale)
        return found if found._workspace(1, 1, width, heads, kv_heads, dim, inner, 1) > 0 else None

    def parts(self, max_kv_len):
        """Into how many parts, at most, a sequence's keys are shared out over blocks: as many as leave each wavefront a tile of 32 keys.
        How many it is, the launch finds from the lengths themselves."""
        return max(1, min(-(-int(max_kv_len) // 256), 32))

    def shares(self, kv_lens, max_kv_len):
        """How a step over these lengths (int32, on the GPU) shares out their keys: int32 (rows, 2), a row's first piece and its parts."""
        rows = kv_lens.shape[0]
        if not (kv_lens.is_cuda and kv_lens.dtype == torch.int32 and kv_lens.dim() == 1 and kv_lens.is_contiguous()
                and 1 <= rows <= DECODE_ROWS_MOST):
            raise OperandError("kv_lens int32, of 1 to %d rows" % DECODE_ROWS_MOST)
        out = torch.empty((rows, 2), dtype=torch.int32, device=kv_lens.device)
        _check(library("decode_layers").q3_decode_layers_shares(
            _P(kv_lens.data_ptr()), rows, self.kv_heads, self.parts(max_kv_len), _P(out.data_ptr()), _stream()), "the shares of a step's keys")
        return out

    def run(self, stream, caches, block_table, kv_lens, max_kv_len, table, blocks=0, patience=64, limit=1 << 18):
        """The layers over the residual `stream` (T, width) float32, in place: row b is sequence b's one token, at position
        kv_lens[b] - 1 of its caches (per layer keys and values as `decode_attention` takes them). Whether that was done: not for a step
        or pages that the launch does not take. `blocks`, `patience`: of how many blocks (0: one per compute unit), and how often they
        look for each other before those that are there go on by themselves. `limit`: how often a block looks for another's results before it
        gives up; the stream is then not numbers, all of it, or where that was in the last product, that block's columns of every row (a look takes a
        microsecond: it is there so that every launch ends)."""
        if not (stream.dim() == 2 and caches and caches[0][0].dim() == 4):
            raise OperandError("a stream (T, width), keys (pages, Hkv, page, D)")
        T = stream.shape[0]
        H, G, D, page = self.heads, self.kv_heads, self.dim, caches[0][0].shape[2]
        if not 1 <= T <= DECODE_ROWS_MOST or page < 16 or page & (page - 1) or (table is not None and table.shape[1] != D):
            return False
        if max_kv_len < 1 or not caches[0][0].shape[0]:          # (`decode_attention` has steps over nothing, and caches without a page)
            return False
        count = len(self.layers)
        if len(caches) != count:
            raise OperandError("a cache for each of the layers")
        parts = self.parts(max_kv_len)
        size = self._workspace(count, T, self.width, H, G, D, self.inner, parts)
        if size <= 0:
            return False
        if not (stream.is_cuda and stream.shape == (T, self.width) and stream.dtype == torch.float32 and stream.is_contiguous()):
            raise OperandError("a float32 stream (T, width), contiguous")
        if not (kv_lens.is_cuda and kv_lens.dtype == torch.int32 and kv_lens.shape == (T,) and kv_lens.is_contiguous()):
            raise OperandError("kv_lens int32, one per row")
        if not (block_table.is_cuda and block_table.dim() == 2 and block_table.dtype == torch.int32 and block_table.shape[0] >= T
                and block_table.is_contiguous() and block_table.shape[1] * page >= max_kv_len):
            raise OperandError("block_table must be int32 (B, W) and hold the longest sequence")
        pages = caches[0][0].shape[0]
        for keys, held in caches:
            if not (keys.is_cuda and keys.dtype == torch.bfloat16 and keys.shape == (pages, G, page, D) and keys.is_contiguous()
                    and held.is_cuda and held.dtype == torch.bfloat16 and held.shape == (pages, G, D, page) and held.is_contiguous()
                    and pages > 0):
                raise OperandError("caches must be keys (pages, Hkv, page, D) and values (pages, Hkv, D, page) in bfloat16")
        max_pos = 0
        if table is not None:
            if not (table.is_cuda and table.dim() == 2 and table.dtype == torch.float32 and table.is_contiguous()
                    and max_kv_len <= table.shape[0]):
                raise OperandError("table must be float32 (P, D) and hold the step's last position")
            max_pos = table.shape[0]
        if any(t.data_ptr() % 16 for t in (stream, *(table,) * (table is not None), *(t for pair in caches for t in pair))):
            return False
        workspace = torch.empty(size, dtype=torch.uint8, device=stream.device)
        layers = (_DecodeLayer * count)()

        def at(t):
            return None if t is None else t.data_ptr()

        for native, l, (keys, held) in zip(layers, self.layers, caches):
            for name in ("qkv", "out", "gate_up", "down"):
                setattr(native, name, at(l[name + "_tiles"]))
            for name in ("q_norm", "k_norm", "entry_norm", "middle_norm"):
                setattr(native, name, at(l[name]))
            native.keys, native.values = keys.data_ptr(), held.data_ptr()
            native.entry_eps, native.middle_eps = l["entry_eps"], l["middle_eps"]
        _check(library("decode_layers").q3_decode_layers(
            layers, count, _P(at(stream)), T, self.width, H, G, D, self.inner, _DT[self.norm_dtype], _DT[self.qk_dtype],
            _F(self.qk_eps), _F(self.scale), _P(at(table)), D if table is not None else 0, max_pos, _P(at(block_table)),
            block_table.shape[1], _P(at(kv_lens)), int(max_kv_len), page, pages, parts, _P(at(workspace)), int(blocks), int(patience),
            int(limit), _stream()), "the layers of a step of single tokens")
        return True
