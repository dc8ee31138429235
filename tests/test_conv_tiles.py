"""Rows of a tile of the short convolution: what was measured to be the faster, and the same numbers whichever it is."""

import pytest
import torch

from qwen3_from_scratch_amd.ops.build import library


@pytest.mark.parametrize("T,C,taps,act,f32_out,rows", [
    (2048, 4352, 4, 1, False, 4), (8192, 4352, 4, 1, False, 4), (256, 512, 4, 1, True, 4), (2048, 2048, 4, 1, True, 8), (2048, 2048, 4, 0, True, 8),
    (512, 2048, 4, 0, True, 4), (1024, 2048, 4, 0, False, 4), (2048, 2048, 4, 0, False, 8), (2048, 2048, 3, 1, False, 8), (2048, 512, 3, 1, False, 4),
    (2048, 4352, 8, 1, False, 8), (512, 512, 8, 0, True, 4), (512, 2048, 8, 0, True, 8)])
def test_rows_that_are_faster(T, C, taps, act, f32_out, rows):
    from qwen3_from_scratch_amd import ops

    assert library("recurrent").q3_conv_tile(T, C, taps, act, ops._DT[torch.float32 if f32_out else torch.bfloat16]) == rows


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("C,taps,act,out_dtype", [(2048, 4, None, torch.float32), (4096, 3, "silu", None), (1024, 8, None, torch.float32),
                                                  (4096, 4, None, torch.bfloat16), (4096, 4, "silu", torch.float32), (520, 4, "silu", None)])
def test_tiles_of_either_size(dtype, C, taps, act, out_dtype):
    """A prompt, with sequences that begin and end inside a tile, beside the same rows in steps too short for tiles of eight."""
    from test_kernels_gpu import _ops, _rand

    ops = _ops()
    out_dtype = out_dtype or dtype
    lengths = [1021, 3, 1, 0, 9, 1006]
    T, B = sum(lengths), len(lengths)
    x, w, bias = _rand((T, C), dtype, 1), _rand((C, taps), torch.float32, 2), _rand((C,), torch.float32, 3)
    state = _rand((B, (taps - 1) * C), torch.float32, 4)

    def run(first, rows, held):
        """Rows `first` .. of every sequence, as many as `rows` says."""
        ends = torch.tensor([0] + lengths).cumsum(0).tolist()
        at = torch.cat([torch.arange(ends[b] + f, ends[b] + f + n) for b, (f, n) in enumerate(zip(first, rows))])
        cu = torch.tensor([0] + rows).cumsum(0).int().cuda()
        seq = torch.repeat_interleave(torch.arange(B), torch.tensor(rows)).int().cuda()
        slots = torch.arange(B, dtype=torch.int32).cuda()
        out = ops.causal_conv(x[at.cuda()].contiguous(), w, bias, held, slots, cu, seq, activation=act, out_dtype=out_dtype, max_q_len=max(rows))
        return at, out

    whole, parts, want = state.clone(), state.clone(), torch.empty((T, C), dtype=out_dtype, device="cuda")
    at, got = run([0] * B, lengths, whole)
    done = [0] * B
    while done != lengths:
        rows = [min(300, n - d) for n, d in zip(lengths, done)]
        places, out = run(done, rows, parts)
        want[places.cuda()] = out
        done = [d + n for d, n in zip(done, rows)]
    # the same expressions in another kernel, in which the compiler may form a multiply-add where it does not here
    assert torch.allclose(got.float(), want.float(), rtol=2.0 ** -7 if out_dtype == torch.bfloat16 else 2.0 ** -18, atol=1e-5)
    assert torch.equal(whole, parts)
