"""WKV7 on few heads, the sequence cut into segments of uneven lengths, against the way that a call with the least scratch takes, and
against the fp64 oracle with states that outlive a segment: with the decays of the other tests, 0.75 a token, nothing of one is left behind it,
and what the segments' matrices do to it would not be seen."""
import pytest
import torch

from oracle import inputs, seq_ref

DEV = 'cuda'
C = 64


def _scratch(B, T, H, segments):
    return max(B * H * segments * 3 * C * C * 4, 256)


@pytest.mark.gpu
@pytest.mark.parametrize('B,T,H,segments,least,states,interval', [
    (1, 3200, 40, 5, 4, torch.float32, 32),     # 200 chunks, the shortest segments there are; with less scratch as four
    (1, 3872, 48, 5, 0, torch.bfloat16, 32),    # 242 chunks: no equal segments; with less scratch one block per head
    (3, 4896, 12, 7, 0, torch.float32, 32),     # 36 pairs, 306 chunks
    (3, 4896, 12, 7, 0, torch.float32, 16),     # a state per chunk
    (2, 3328, 16, 5, 4, None, 32),              # 208 chunks, no states in
    (1, 7744, 24, 10, 4, torch.float32, 32),    # 484 chunks; more than eight segments
    (1, 8176, 24, 10, 0, torch.bfloat16, 32),   # 511 chunks: a state per chunk
    (1, 3216, 40, 5, 0, None, 32),              # 201
    (2, 6160, 8, 8, 0, torch.float32, 32),      # 385, two blocks per segment
])
def test_segments_agree_with_the_other_way(B, T, H, segments, least, states, interval):
    """Every token goes through the same products; only the states at the cuts come from elsewhere, in fp32 (2e-3: a bf16 rounding
    of what follows from them, as between one call and two that carry the state)."""
    from wind_rwkv import _native
    from wind_rwkv.rwkv7 import set_checkpoint_interval
    lib = _native.lib()
    d = inputs.wkv7_inputs(B, T, H, C, seed=T + H, dtype=torch.bfloat16, s0_scale=0.3, dsT_scale=0.3)
    x = [d[n].to(DEV).contiguous() for n in ('w', 'q', 'k', 'v', 'a', 'b')]
    dy = d['dy'].to(DEV).contiguous()
    dt = states or torch.float32
    s0, dsT = (d[n].to(dt).to(DEV).contiguous() for n in ('s0', 'dsT'))
    ptr = lambda t: t.data_ptr()
    given = (ptr(s0), ptr(dsT)) if states else (None, None)
    head = (B, T, H, C, _native.BF16, _native.F32 if dt == torch.float32 else _native.BF16)
    stream = torch.cuda.current_stream().cuda_stream
    mem = lambda n: torch.zeros(n, dtype=torch.uint8, device=DEV)
    nan = lambda t: torch.full_like(t, float('nan'))
    kept = B * H * ((T // 32) * 12288 if T % 32 == 0 and interval == 32 else (T // 16) * 10240)
    set_checkpoint_interval(interval)
    try:
        full = _scratch(B, T, H, segments)
        assert lib.wind_rwkv7_attn_fwd_workspace_bytes(B, T, H, C) == full and lib.wind_rwkv7_attn_bwd_workspace_bytes(B, T, H, C) == kept + full
        out = []
        assert lib.wind_rwkv7_attn_fwd_workspace_least_bytes(B, T, H, C) == _scratch(B, T, H, least)
        for f in (full, _scratch(B, T, H, least)):
            b = kept + (f if f > 256 else 0)
            ws, saved = mem(max(f, b)), mem(lib.wind_rwkv7_attn_saved_bytes(*head[:4]))
            y, y0, sT, s1, ds0 = nan(x[0]), nan(x[0]), nan(s0), nan(s0), nan(s0)
            grads = [nan(x[0]) for _ in range(6)]
            _native.check(lib.wind_rwkv7_attn_forward(*head, *map(ptr, x), given[0], ptr(y), ptr(saved), ptr(sT), ptr(ws), f, stream))
            _native.check(lib.wind_rwkv7_attn_backward(*head, *map(ptr, x), ptr(dy), ptr(saved), given[1], *map(ptr, grads), ptr(ds0), ptr(ws), b, stream))
            scratch = torch.empty_like(saved)
            _native.check(lib.wind_rwkv7_attn_prefill(*head, *map(ptr, x), given[0], ptr(y0), ptr(scratch), ptr(s1), ptr(ws), f, stream))
            if f > 256:
                assert lib.wind_rwkv7_attn_forward(*head, *map(ptr, x), given[0], ptr(y), ptr(saved), ptr(sT), ptr(ws), _scratch(B, T, H, least) - 1, stream) == 6
            torch.cuda.synchronize()
            assert torch.equal(y, y0) and torch.equal(sT, s1)
            out.append([y, sT, ds0] + grads)
    finally:
        set_checkpoint_interval(32)
    for i, (t, r) in enumerate(zip(*out)):
        assert torch.isfinite(t.float()).all(), i
        assert (t.float() - r.float()).norm() <= (4e-3 if t.dtype == torch.bfloat16 and i in (1, 2) else 2e-3) * r.float().norm(), i


@pytest.mark.gpu
@pytest.mark.parametrize('B,T,H,segments', [
    (1, 4096, 3, 8),      # eight equal ones and the first
    (1, 5760, 17, 9),     # more than eight
    (1, 7744, 17, 12),    # as many as there are
    (1, 3232, 32, 5),     # 202 chunks, uneven
    (1, 3088, 33, 4),     # 193, a state per chunk
    (1, 6160, 17, 9),     # 385
])
def test_segments_with_long_memory_against_the_oracle(c_oracle, B, T, H, segments):
    """Decays of 0.9985 a token and a tenth of the removal: half of what enters a segment leaves it (without it y, sT and the gradients
    are off by half of themselves).  1e-2: the gate of every bf16 pass."""
    from wind_rwkv import _native
    from wind_rwkv.rwkv7.wkv_attn import WindRWKV7
    assert _native.lib().wind_rwkv7_attn_train_workspace_bytes(B, T, H, C) == _scratch(B, T, H, segments)
    d = inputs.wkv7_inputs(B, T, H, C, seed=T + H, dtype=torch.bfloat16, s0_scale=1.0, dsT_scale=1.0)
    d['w'], d['b'] = (d['w'].float() - 6).bfloat16(), (d['b'].float() * 0.1).bfloat16()
    xs = [d[n].to(DEV).requires_grad_() for n in ('w', 'q', 'k', 'v', 'a', 'b')]
    s0 = d['s0'].to(DEV).requires_grad_()
    y, sT, _ = WindRWKV7.apply(*xs, s0)
    torch.autograd.backward([y, sT], [d['dy'].to(DEV), d['dsT'].to(DEV)])
    args = [d[n] for n in 'qwkvab']
    ref = list(c_oracle.forward(*args, d['s0'])) + list(c_oracle.backward(*args, d['s0'], d['dy'], d['dsT']))
    got = [y, sT] + [xs[i].grad for i in (1, 0, 2, 3, 4, 5)] + [s0.grad]
    errs = {n: seq_ref.rel_err(t.detach().float().cpu(), r) for n, t, r in zip(('y', 'sT', 'dq', 'dw', 'dk', 'dv', 'da', 'db', 'ds0'), got, ref)}
    print({n: f'{e:.1e}' for n, e in errs.items()})
    assert all(e <= 1e-2 for e in errs.values()), errs


@pytest.mark.gpu
@pytest.mark.parametrize('B,T,H,segments', [
    (1, 3872, 48, 5),     # 242 chunks
    (1, 8176, 24, 10),    # 511: a state per chunk
    (1, 4096, 3, 8),      # two blocks per segment
])
def test_attn_ln_in_segments_agrees_with_the_other_way(B, T, H, segments):
    """attn_ln's kept output centred in segments, its parameter gradients beside or behind the segmented scan, and the workspace's order, against
    the call with the least scratch (eight equal segments have no other way: there the plain operator and the epilogue's kernels)."""
    from wind_rwkv import _native
    lib = _native.lib()
    d = inputs.attn_ln_inputs(B, T, H, C, seed=T + H, dtype=torch.bfloat16)
    x = [d[n].to(DEV).contiguous() for n in ('w', 'q', 'k', 'v', 'a', 'b', 'g')]
    gen = torch.Generator().manual_seed(T)
    s0, dsT = ((torch.randn(B, H, C, C, generator=gen)).to(DEV) for _ in range(2))
    dy, params = d['dy'].to(DEV).contiguous(), d['params'].to(DEV)
    ptr = lambda t: t.data_ptr()
    nan = lambda t: torch.full_like(t, float('nan'))
    mem = lambda n: torch.zeros(n, dtype=torch.uint8, device=DEV)
    head = (B, T, H, C, _native.BF16, _native.F32)
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.wind_rwkv7_attn_train_workspace_bytes(B, T, H, C) == _scratch(B, T, H, segments)
    fwd = lib.wind_rwkv7_attn_train_workspace_bytes(B, T, H, C), lib.wind_rwkv7_attn_fwd_workspace_least_bytes(B, T, H, C)
    bwd = lib.wind_rwkv7_attn_ln_bwd_workspace_bytes(B, T, H, C), lib.wind_rwkv7_attn_ln_bwd_workspace_least_bytes(B, T, H, C)
    out = []
    for f, b in zip(fwd, bwd):
        guard = 4096
        ws, saved = mem(max(f, b) + guard), mem(lib.wind_rwkv7_attn_ln_saved_bytes(B, T, H, C))
        y, sT, ds0, dparams, grads = nan(dy), nan(s0), nan(s0), nan(params), [nan(dy) for _ in range(7)]
        ws[f:] = 77
        _native.check(lib.wind_rwkv7_attn_ln_forward(*head, *map(ptr, x), ptr(params), ptr(s0), ptr(y), ptr(saved), ptr(sT), ptr(ws), f, stream))
        assert (ws[f:] == 77).all()
        ws[b:] = 77
        _native.check(lib.wind_rwkv7_attn_ln_backward(*head, *map(ptr, x), ptr(params), ptr(dy), ptr(saved), ptr(dsT), *map(ptr, grads), ptr(dparams),
                                                      ptr(ds0), ptr(ws), b, stream))
        assert (ws[b:] == 77).all()
        out.append(dict(y=y, sT=sT, ds0=ds0, dparams=dparams, **dict(zip(('dw', 'dq', 'dk', 'dv', 'da', 'db', 'dg'), grads))))
    if fwd[0] == fwd[1]:   # one way only: the plain operator, the epilogue on its output and back
        out[1] = {}
        from wind_rwkv.rwkv7.wkv_attn import WindRWKV7
        seqs = [t.clone().requires_grad_() for t in x[:6]]
        h0 = s0.clone().requires_grad_()
        y, sT, _ = WindRWKV7.apply(*seqs, h0)
        leaf = {n: t.detach().double().requires_grad_() for n, t in dict(y=y, q=x[1], k=x[2], v=x[3], g=x[6], p=params).items()}
        z = seq_ref.attn_ln_epilogue(leaf['y'], leaf['q'], leaf['k'], leaf['v'], leaf['g'], leaf['p'])
        z.backward(dy.double())
        torch.autograd.backward([y, sT], [leaf['y'].grad.bfloat16(), dsT])
        out[1] = dict(y=z.detach(), sT=sT, ds0=h0.grad, dparams=leaf['p'].grad, dg=leaf['g'].grad, dw=seqs[0].grad, da=seqs[4].grad, db=seqs[5].grad,
                      **{'d' + n: seqs[i].grad.double() + leaf[n].grad for n, i in (('q', 1), ('k', 2), ('v', 3))})
    for n, t in out[0].items():
        e = seq_ref.rel_err(t.detach().double().cpu(), out[1][n].detach().double().cpu())
        assert e <= (1e-2 if fwd[0] == fwd[1] else 2e-3), (n, e)
