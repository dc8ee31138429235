"""A weight matrix as the parts hold it: row-major, and a second copy for its kernels: of bfloat16 in the
order the few-row product kernel streams it, of float32 in bfloat16 where that loses nothing."""

import torch

from .. import ops
from .base import Part, UnscaledRows

COPIES_MOST = 4                 # float32 matrices' bfloat16 copies take a quarter at most of the memory that is free


def free_memory(device):
    """Bytes of the device that nobody holds, what PyTorch keeps for later among them."""
    return (torch.cuda.mem_get_info(device)[0] + torch.cuda.memory_reserved(device) - torch.cuda.memory_allocated(device))


def _matrices(held, seen):
    """Every LinearWeight that a part, or a list of parts, holds, once each, in their order."""
    if id(held) in seen:
        return
    seen.add(id(held))
    if isinstance(held, LinearWeight):
        yield held
    elif isinstance(held, (Part, list, tuple, dict)):
        inner = vars(held).values() if isinstance(held, Part) else held.values() if isinstance(held, dict) else held
        for value in inner:
            yield from _matrices(value, seen)


def copy_float32_matrices(parts):
    """Give the float32 matrices of `parts`, one after the other, the bfloat16 copies that `LinearWeight` multiplies with, once
    all are loaded: so that whatever fits without them fits with them, and most of what is left stays the cache's."""
    matrices = [m for m in _matrices(list(parts), set()) if m.wants_copy]
    if not matrices:
        return
    room = free_memory(matrices[0].weight.device) // COPIES_MOST
    for m in matrices:
        size = 2 * m.weight.numel()
        if size <= room:
            m.narrow = ops.narrow_weight(m.weight)
            room -= size if m.narrow is not None else 0


def joined_rows(matrices, multiple=16):
    """Matrices of one inner size as one, below each other, filled up with rows of zeros to a multiple
    of `multiple` rows: one product for all of them, in a size that every product kernel takes."""
    rows = sum(m.shape[0] for m in matrices)
    out = torch.zeros((-(-rows // multiple) * multiple, matrices[0].shape[1]), dtype=matrices[0].dtype,
                      device=matrices[0].device)
    at = 0
    for m in matrices:
        out[at:at + m.shape[0]].copy_(m)
        at += m.shape[0]
    return out


class LinearWeight:
    """y = x @ W^T, no bias. W (N, K) is kept row-major for products with many
    rows (the vendor library's) and for float32; when the precision asks for
    it, a tile-ordered bfloat16 copy serves steps with few rows (16, or 32 or 64
    for a small weight), where every weight is read once and the order in memory
    decides the bandwidth. The copy doubles the weight's memory. A float32 weight that
    bfloat16 holds exactly may have a bfloat16 copy instead (`copy_float32_matrices`), half its memory more: the products
    then read half as much and run on the bfloat16 matrix cores, in float32 precision."""

    def __init__(self, weight, precision):
        self.weight = weight
        self.tiled = ops.tile_weight(weight) if precision.tiled else None
        self.narrow = None
        self.wants_copy = precision.tiled and weight.is_cuda and weight.dtype == torch.float32
        if weight.is_cuda and weight.dtype == torch.bfloat16:
            ops.matmul_init()          # the many-row products' buffers: now, not inside a step

    def forward(self, x, out_dtype=None):
        """x @ W^T; x may be UnscaledRows (see `fuses`)."""
        if isinstance(x, UnscaledRows):
            return ops.linear(x.values, self.weight, out_dtype=out_dtype, tiled=self.tiled, unscaled=x.scale_args())
        if self.narrow is not None:
            return ops.linear(x, self.weight, out_dtype=out_dtype, narrow=self.narrow)
        return ops.linear(x, self.weight, out_dtype=out_dtype, tiled=self.tiled)

    def forward_swiglu(self, x, kind="silu"):
        """act(gate) * up of x @ W^T for a W whose rows interleave gate and up; `kind` names the activation."""
        if isinstance(x, UnscaledRows):
            return ops.linear_swiglu(x.values, self.weight, tiled=self.tiled, unscaled=x.scale_args(), kind=kind)
        if self.narrow is not None:
            return ops.linear_swiglu(x, self.weight, kind=kind, narrow=self.narrow)
        return ops.linear_swiglu(x, self.weight, tiled=self.tiled, kind=kind)

    @property
    def fuses(self):
        """Whether steps of few rows go through kernels whose epilogues carry the
        norm fusion, UnscaledRows in, a NormSink out: up to 16 rows (32 or 64 for a
        small weight) the few-row kernel on the tiled copy, up to 128 (or 640) the tiled
        matrix-core kernel. A
        reader of UnscaledRows must have output rows in steps of 4."""
        return self.tiled is not None and self.weight.shape[0] % 4 == 0

    @property
    def fused_rows_most(self):
        """Up to how many rows those kernels take UnscaledRows for this weight."""
        return ops.fused_rows_most(self.weight)

    def forward_into(self, x, sink):
        """x @ W^T added into the sink's residual and prepared for its norm, as
        UnscaledRows; or, where the kernels do not take the case, returned. SplitRows
        (see `ops.decode_attention`) are added in any case."""
        if isinstance(x, ops.SplitRows):
            return UnscaledRows(*ops.linear_residual_norm(x, self.weight, self.tiled, sink.residual, sink.weight),
                                sink.eps, sink.width)
        rows = x.shape[0]
        if self.tiled is None or not (self.weight.shape[0] % 16 == 0 if rows <= ops.few_rows_limit(self.weight)
                                      else ops.fused_rows_take(self.weight, rows)):
            return self.forward(x)
        fused = ops.linear_residual_norm(x, self.weight, self.tiled, sink.residual, sink.weight)
        if fused is None:                       # the kernel leaves this size to the plain product
            return self.forward(x)
        return UnscaledRows(fused[0], fused[1], sink.eps, sink.width)
