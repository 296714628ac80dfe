"""The single-token kernels of the block (csrc/mixer_decode.hip) where their dispatch changes: columns and tiles per block of
the products, rows per block of the head kernel, wavefronts of the first product, and a few tokens per sequence.  Against
the same step on the sequence kernels, at the gates of tests/test_gpu_time_mixer_state.py (both sides round to bf16 between
stages; they differ in summation order)."""
from collections import namedtuple

import pytest
import torch

from oracle import seq_ref

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _model(H, seed):
    from wind_rwkv.rwkv7 import TimeMixer
    gen = torch.Generator().manual_seed(seed)
    model = TimeMixer(namedtuple('Config', ['n_layer', 'n_head', 'n_embd'])(4, H, 64 * H), 1)
    with torch.no_grad():
        for p in model.parameters():
            p.copy_(torch.randn(p.shape, generator=gen) * 0.1)
    return model.to(DEV), gen


@pytest.mark.parametrize('B,H', [(2, 1), (17, 12), (47, 12), (80, 12), (200, 12), (3, 20), (300, 3)])
@pytest.mark.parametrize('state_dtype', [torch.float32, torch.bfloat16])
def test_step_over_the_dispatch_of_its_kernels(B, H, state_dtype):
    model, gen = _model(H, seed=B)
    C = 64 * H
    x, prev = torch.randn(2, B, C, generator=gen).bfloat16().to(DEV)
    S = torch.randn(B, H, 64, 64, generator=gen).to(DEV, state_dtype)
    with torch.no_grad():
        want, (_, Sw) = model._step_on_kernels(x, prev, S.clone())
        got, (carry, Sg) = model.step(x, (prev, S.clone()))
    assert torch.equal(carry, x)
    assert seq_ref.rel_err(got.float().cpu(), want.float().cpu()) <= 5e-3
    assert seq_ref.rel_err(Sg.float().cpu(), Sw.float().cpu()) <= (2e-3 if state_dtype == torch.float32 else 8e-3)


# rows no multiple of 16 or 64 and one past a multiple, heads past 256 and 2048 channels; (750, 32) also with the output grouped,
# (978, 10) by rows x channels^2 alone; (33, 35) one round of the linear kernel's widest blocks, (33, 43) more
@pytest.mark.parametrize('B,H', [(161, 13), (33, 35), (257, 12), (400, 29), (33, 43), (750, 32), (978, 10)])
def test_step_with_the_streams_in_memory(B, H):
    test_step_over_the_dispatch_of_its_kernels(B, H, torch.float32)


# the widths of the linear kernels' blocks: up to 256 blocks of 16, 32, 64 columns by a tile, else 64 by two tiles; at each line the
# largest that fits and the smallest that does not, for the products with the interpolation (up to (64, 20)) and for the output
@pytest.mark.parametrize('B,H', [(16, 20), (16, 21), (16, 1), (48, 12), (49, 12), (64, 19), (64, 20), (64, 16), (65, 16), (128, 16), (129, 16),
                                 (256, 16), (257, 16)])
def test_step_at_the_lines_of_its_linear_kernels(B, H):
    test_step_over_the_dispatch_of_its_kernels(B, H, torch.float32)


@pytest.mark.parametrize('B,T,H', [(1, 3, 2), (5, 17, 3), (8, 63, 12)])
def test_a_few_tokens_equal_as_many_steps(B, T, H):
    """Within one rounding of the outputs: the same kernels' arithmetic, the state in registers between the tokens (fp32)."""
    model, gen = _model(H, seed=T)
    x = torch.randn(B, T, 64 * H, generator=gen).bfloat16().to(DEV)
    state = (torch.randn(B, 64 * H, generator=gen).bfloat16().to(DEV), torch.randn(B, H, 64, 64, generator=gen).to(DEV))
    with torch.no_grad():
        y, (last, S) = model(x, state=state, return_state=True)
        st, ys = (state[0], state[1].clone()), []
        for t in range(T):
            yt, st = model.step(x[:, t], st)
            ys.append(yt)
    assert torch.equal(last, x[:, -1])
    assert seq_ref.rel_err(y.float().cpu(), torch.stack(ys, 1).float().cpu()) <= 2e-3
    assert seq_ref.rel_err(S.cpu(), st[1].cpu()) <= 1e-4


@pytest.mark.parametrize('B,T,H', [(1, 1003, 3), (3, 100, 4), (2, 79, 12), (9, 65, 2), (40, 15, 2), (300, 2, 1), (66000, 2, 1)])
@pytest.mark.parametrize('continued', [False, True])
def test_a_ragged_prompt_is_whole_chunks_and_then_steps(B, T, H, continued):
    """The tokens after the last whole chunk keep the state in fp32 from token to token, as steps do: the same sums in
    registers, so the state is theirs to 1e-4 (operands of a chunk's products in bf16 would leave 2^-9 of every token's
    share) and the outputs to a rounding here and there.  More than eight sequences, one token left and no whole chunk
    take other launches."""
    model, gen = _model(H, seed=B + T)
    C, T0 = 64 * H, T - T % 16
    x = torch.randn(B, T, C, generator=gen).bfloat16().to(DEV)
    state = (torch.randn(B, C, generator=gen).bfloat16().to(DEV), torch.randn(B, H, 64, 64, generator=gen).to(DEV))
    given = (state[0], state[1].clone()) if continued else None
    with torch.no_grad():
        y, (last, S) = model(x, state=given, return_state=True)
        st = (state[0], state[1].clone()) if continued else (torch.zeros_like(state[0]), torch.zeros_like(state[1]))
        ys = []
        if T0:
            y0, st = model(x[:, :T0].contiguous(), state=given, return_state=True)
            ys.append(y0)
        for t in range(T0, T):
            yt, st = model.step(x[:, t], st)
            ys.append(yt[:, None])
    assert not continued or torch.equal(given[1], state[1])   # (the caller's is not written)
    assert y.is_contiguous() and torch.equal(last, x[:, -1])
    want = torch.cat(ys, 1)
    start = 0 if continued else 1     # from a zero state the first token's GroupNorm is ill conditioned
    # The sequence kernels mix a continued prompt's first token in fp32 where `step` rounds its weights to bf16.  Where a step
    # is that token's reference (no whole chunk) its operands differ by up to a rounding each, 2^-8 of k, v, a and b and half of
    # that in the mean: 2^-7 of its share of the state, and the block's gate on the outputs.
    y_gate, S_gate = (1.27e-2, 2 ** -7) if continued and T0 == 0 else (2e-3, 1e-4)
    for first in {start, max(start, T0)}:
        assert seq_ref.rel_err(y[:, first:].float().cpu(), want[:, first:].float().cpu()) <= y_gate
    assert seq_ref.rel_err(S.cpu(), st[1].cpu()) <= S_gate


def test_a_ragged_prompt_at_another_head_size_is_whole_chunks_and_then_steps():
    from wind_rwkv.rwkv7 import TimeMixer
    gen = torch.Generator().manual_seed(8)
    model = TimeMixer(namedtuple('Config', ['n_layer', 'n_head', 'n_embd'])(4, 2, 256), 1)
    with torch.no_grad():
        for p in model.parameters():
            p.copy_(torch.randn(p.shape, generator=gen) * 0.1)
    model = model.to(DEV)
    x = torch.randn(2, 37, 256, generator=gen).bfloat16().to(DEV)
    with torch.no_grad():
        y, (_, S) = model(x, return_state=True)
        y0, st = model(x[:, :32].contiguous(), return_state=True)
        ys = [y0]
        for t in range(32, 37):
            yt, st = model.step(x[:, t], st)
            ys.append(yt[:, None])
    assert torch.equal(y, torch.cat(ys, 1)) and torch.equal(S, st[1])


@pytest.mark.parametrize('B,T,T_out,C', [(1, 1, 16, 64), (2, 1003, 1008, 768), (3, 32, 19, 72), (1, 5, 5, 8)])
def test_pad_rows(B, T, T_out, C):
    """Whole numbers through a copy: exact."""
    from wind_rwkv import _native
    x = torch.randn(B, T, C, device='cuda').bfloat16()
    out, last = torch.full((B, T_out, C), 7., device='cuda').bfloat16(), torch.empty(B, C, device='cuda').bfloat16()
    _native.check(_native.lib().wind_rwkv7_pad_rows(B, T, T_out, C, x.data_ptr(), out.data_ptr(), last.data_ptr() if T_out >= T else None,
                                                    torch.cuda.current_stream().cuda_stream))
    n = min(T, T_out)
    assert torch.equal(out[:, :n], x[:, :n]) and not out[:, n:].any()
    assert T_out < T or torch.equal(last, x[:, -1])


# one sequence and more, two chunks and more; from 16 heads on the epilogue goes through the chunks head by head; 140 (batch, head)s: the one-kernel form
@pytest.mark.parametrize('B,T,H,n', [(1, 32, 1, 1), (2, 48, 3, 15), (3, 112, 17, 7), (1, 1024, 12, 9), (140, 32, 1, 3)])
@pytest.mark.parametrize('f32', [True, False])
def test_ragged_prefill_is_prefill_and_tokens(B, T, H, n, f32):
    from wind_rwkv import _native
    lib, stream, gen = _native.lib(), torch.cuda.current_stream().cuda_stream, torch.Generator().manual_seed(T + H)
    rn = lambda *s: torch.randn(*s, generator=gen).to(DEV)
    seqs = [(rn(B, T, H * 64) * 0.3).bfloat16() for _ in range(7)]   # w q k v a b g
    params, s0 = rn(3, H * 64), rn(B, H, 64, 64).to(torch.float32 if f32 else torch.bfloat16)
    kept = torch.empty(3, B, 16, H * 64, device=DEV, dtype=torch.bfloat16)
    _native.check(lib.wind_rwkv7_neutral_rows_keep(B, T, H * 64, T - 16, seqs[0].data_ptr(), seqs[2].data_ptr(), seqs[5].data_ptr(), kept.data_ptr(), stream))
    ptrs, state = [t.data_ptr() for t in (*seqs, params)], _native.F32 if f32 else _native.BF16
    ws = torch.empty(max(16, lib.wind_rwkv7_attn_fwd_workspace_bytes(B, T, H, 64)), device=DEV, dtype=torch.uint8)
    scratch = torch.empty(lib.wind_rwkv7_attn_ln_saved_bytes(B, T, H, 64), device=DEV, dtype=torch.uint8)
    (y1, S1), (y2, S2) = ((torch.full_like(seqs[0], float('nan')), torch.empty_like(s0)) for _ in range(2))
    end = lambda S: (scratch.data_ptr(), S.data_ptr(), ws.data_ptr(), ws.numel(), stream)
    _native.check(lib.wind_rwkv7_attn_ln_prefill(B, T, H, 64, _native.BF16, state, *ptrs, s0.data_ptr(), y1.data_ptr(), *end(S1)))
    _native.check(lib.wind_rwkv7_attn_ln_tokens(B, T, H, 64, T - 16, n, state, kept[0].data_ptr(), ptrs[1], kept[1].data_ptr(), ptrs[3], ptrs[4],
                                                kept[2].data_ptr(), ptrs[6], ptrs[7], 16, 0, S1.data_ptr(), y1.data_ptr(), S1.data_ptr(), stream))
    _native.check(lib.wind_rwkv7_attn_ln_prefill_ragged(B, T, H, 64, n, state, *ptrs, kept.data_ptr(), s0.data_ptr(), y2.data_ptr(), *end(S2)))
    valid = T - 16 + n
    assert torch.equal(S1, S2) and torch.equal(y1[:, :valid], y2[:, :valid])
