"""WKV7 by records in memory (few (batch, head) pairs) against the one-kernel form and against segments.

The two ways run the same instructions on the same operands, so every output has to be the same bits.  A call takes records when
its workspace holds them and the other way with the least that it accepts, so both are had through the C interface by the size of
the workspace alone.
"""
import pytest
import torch

from oracle import inputs

DEV = 'cuda'
C = 64


def test_workspace_sizes_at_the_lines_of_the_rule():
    """Records from eight chunks (backward, and a forward that keeps something for it: from 96, or 48 and 2048 in all), for up to a quarter
    of the compute units' worth of (batch, head) pairs and 6144 chunks (forward 5120 where a sequence runs as four segments otherwise, 3584 as
    five), and not where a sequence runs as six or more."""
    from wind_rwkv import _native
    lib = _native.lib()
    # prefill, training forward, backward by records; equal segments of the least scratch, and the segments otherwise
    for (B, T, H), (ahead, train, back, least, most) in {
            (1, 112, 4): (False, False, False, 0, 0), (1, 128, 4): (True, False, False, 0, 0), (1, 1520, 4): (True, False, False, 0, 0),
            (1, 1536, 4): (True, True, True, 0, 0), (1, 752, 44): (True, False, False, 0, 0), (1, 768, 43): (True, True, True, 0, 0),
            (1, 768, 42): (True, False, False, 0, 0), (1, 1536, 64): (True, True, True, 0, 0), (1, 1536, 65): (False, False, False, 0, 0),
            (1, 2048, 40): (True, True, True, 4, 4), (1, 2048, 48): (False, False, True, 4, 4), (1, 2064, 48): (False, False, False, 0, 0),
            (1, 3200, 17): (True, True, True, 4, 5), (1, 3200, 18): (False, False, True, 4, 5), (1, 3216, 12): (True, True, True, 0, 5),
            (1, 3840, 12): (False, False, False, 4, 6), (1, 4096, 12): (False, False, False, 8, 8), (1, 4080, 12): (False, False, False, 0, 6),
            (8, 1024, 12): (False, False, False, 0, 0)}.items():
        chunks = B * H * (T // 16)
        kept = B * H * (T // 32 * 12288 if T % 32 == 0 else T // 16 * 10240)
        maps = lambda segments: segments * B * H * 3 * C * C * 4
        assert lib.wind_rwkv7_attn_fwd_workspace_bytes(B, T, H, C) == (chunks * 13568 if ahead else max(maps(most), 256)), (B, T, H)
        assert lib.wind_rwkv7_attn_train_workspace_bytes(B, T, H, C) == (chunks * 13568 if train else max(maps(most), 256)), (B, T, H)
        assert lib.wind_rwkv7_attn_bwd_workspace_bytes(B, T, H, C) == kept + (chunks * 10496 if back else maps(most)), (B, T, H)
        assert lib.wind_rwkv7_attn_fwd_workspace_least_bytes(B, T, H, C) == max(maps(least), 256), (B, T, H)
        assert lib.wind_rwkv7_attn_bwd_workspace_least_bytes(B, T, H, C) == kept + maps(least), (B, T, H)


@pytest.mark.gpu
@pytest.mark.parametrize('ln', [False, True])
@pytest.mark.parametrize('B,T,H,scratch', [(1, 1536, 64, False), (1, 496, 64, False), (1, 256, 4, False), (1, 1536, 4, True)])
def test_a_node_keeps_what_its_backward_reads(B, T, H, scratch, ln):
    """Between forward and backward a node holds the saved tensor beside its outputs, and of the scan's scratch no more than 32 MiB: records
    (6144 chunks, 80 MiB), records that only a forward without gradients would write (64 pairs x 31 chunks), none, few of them."""
    from wind_rwkv import _native
    from wind_rwkv.rwkv7 import attn, attn_ln
    lib = _native.lib()
    d = inputs.wkv7_inputs(B, T, H, C, seed=H, dtype=torch.bfloat16)
    x = [d[n].reshape(B, T, H * C).to(DEV).requires_grad_() for n in ('q', 'w', 'k', 'v', 'a', 'b')]
    g = x[0].detach().clone()
    params = torch.ones(3, H * C, device=DEV)
    go = lambda: attn_ln(*x, g, params, C) if ln else attn(*x, C)
    requested = lambda: torch.cuda.memory_stats()['requested_bytes.all.current']   # (not the pool's blocks, which may be larger)
    before = requested()
    y = go()
    held = requested() - before
    saved = (lib.wind_rwkv7_attn_ln_saved_bytes if ln else lib.wind_rwkv7_attn_saved_bytes)(B, T, H, C)
    wanted = y.numel() * 2 + saved
    if scratch:
        wanted += lib.wind_rwkv7_attn_train_workspace_bytes(B, T, H, C)
        assert B * H * T // 16 * 13568 == lib.wind_rwkv7_attn_train_workspace_bytes(B, T, H, C) <= 32 << 20
    assert wanted <= held <= wanted + 256, (held, wanted)   # the 256 of a call without scratch; (sT goes where nobody asked for it)


@pytest.mark.gpu
@pytest.mark.parametrize('interval', [32, 16])
@pytest.mark.parametrize('B,T,H,state', [(1, 128, 1, True), (3, 144, 3, False), (2, 160, 5, True), (1, 176, 8, True), (1, 1536, 1, False),
                                         (2, 1552, 5, True), (1, 1568, 8, True), (3, 1584, 3, False), (1, 2048, 4, True), (1, 1024, 64, True),
                                         (33, 1536, 1, False)])
def test_records_give_the_bits_of_the_other_way(B, T, H, state, interval):
    """Plain and attn_ln, forward without the kept states and, from 96 chunks, with them and backward; 8 to 11 and 96 to 99 chunks are
    every remainder of the chain's registers, 2048 tokens run as four segments otherwise, 33 sequences reduce the parameter gradients in a launch of their own
    (those sums alone are taken in another order)."""
    from wind_rwkv import _native
    from wind_rwkv.rwkv7 import set_checkpoint_interval
    lib = _native.lib()
    d = inputs.wkv7_inputs(B, T, H, C, seed=B + T + H, dtype=torch.bfloat16, s0_scale=0.3, dsT_scale=0.3)
    x = [d[n].to(DEV).contiguous() for n in ('w', 'q', 'k', 'v', 'a', 'b')]
    dy, s0, dsT = d['dy'].to(DEV).contiguous(), d['s0'].float().to(DEV).contiguous(), d['dsT'].float().to(DEV).contiguous()
    gen = torch.Generator().manual_seed(T)
    g = torch.randn(x[0].shape, generator=gen).bfloat16().to(DEV)
    params = torch.randn(3, H * C, generator=gen).to(DEV)
    stream = torch.cuda.current_stream().cuda_stream
    ptr = lambda t: t.data_ptr()
    ins, states = [ptr(t) for t in x], (ptr(s0), ptr(dsT)) if state else (None, None)
    head = (B, T, H, C, _native.BF16, _native.F32)
    mem = lambda n: torch.zeros(n, dtype=torch.uint8, device=DEV)
    nan = lambda t: torch.full_like(t, float('nan'))
    set_checkpoint_interval(interval)
    try:
        fwd, bwd = lib.wind_rwkv7_attn_fwd_workspace_bytes(B, T, H, C), lib.wind_rwkv7_attn_bwd_workspace_bytes(B, T, H, C)
        ln_bwd = lib.wind_rwkv7_attn_ln_bwd_workspace_bytes(B, T, H, C)
        least_fwd, least_bwd = lib.wind_rwkv7_attn_fwd_workspace_least_bytes(B, T, H, C), lib.wind_rwkv7_attn_bwd_workspace_least_bytes(B, T, H, C)
        least_ln_bwd = lib.wind_rwkv7_attn_ln_bwd_workspace_least_bytes(B, T, H, C)
        assert ln_bwd - least_ln_bwd == bwd - least_bwd
        assert fwd > least_fwd and (bwd > least_bwd) == (T >= 1024)
        out = {}
        for way, (f, b, lb) in {'records': (fwd, bwd, ln_bwd), 'least': (least_fwd, least_bwd, least_ln_bwd)}.items():
            ws, saved, ln_saved = mem(max(f, b, lb)), mem(lib.wind_rwkv7_attn_saved_bytes(*head[:4])), mem(lib.wind_rwkv7_attn_ln_saved_bytes(*head[:4]))
            y, y0, z, z0 = (nan(x[0]) for _ in range(4))
            sT, s1, t0, t1 = (nan(s0) for _ in range(4))
            grads, ln_grads = [nan(x[0]) for _ in range(6)], [nan(x[0]) for _ in range(7)]
            ds0, ln_ds0, dparams = nan(s0), nan(s0), nan(params)
            scratch, ln_scratch = torch.empty_like(saved), torch.empty_like(ln_saved)
            _native.check(lib.wind_rwkv7_attn_prefill(*head, *ins, states[0], ptr(y0), ptr(scratch), ptr(s1), ptr(ws), f, stream))
            _native.check(lib.wind_rwkv7_attn_forward(*head, *ins, states[0], ptr(y), ptr(saved), ptr(sT), ptr(ws), f, stream))
            _native.check(lib.wind_rwkv7_attn_backward(*head, *ins, ptr(dy), ptr(saved), states[1], *map(ptr, grads), ptr(ds0), ptr(ws), b, stream))
            ln = (ptr(g), ptr(params))
            _native.check(lib.wind_rwkv7_attn_ln_prefill(*head, *ins, *ln, states[0], ptr(z0), ptr(ln_scratch), ptr(t0), ptr(ws), f, stream))
            _native.check(lib.wind_rwkv7_attn_ln_forward(*head, *ins, *ln, states[0], ptr(z), ptr(ln_saved), ptr(t1), ptr(ws), f, stream))
            _native.check(lib.wind_rwkv7_attn_ln_backward(*head, *ins, *ln, ptr(dy), ptr(ln_saved), states[1], *map(ptr, ln_grads), ptr(dparams),
                                                          ptr(ln_ds0), ptr(ws), lb, stream))
            assert lib.wind_rwkv7_attn_forward(*head, *ins, states[0], ptr(y), ptr(saved), ptr(sT), ptr(ws), least_fwd - 1, stream) == 6
            assert lib.wind_rwkv7_attn_backward(*head, *ins, ptr(dy), ptr(saved), states[1], *map(ptr, grads), ptr(ds0), ptr(ws), least_bwd - 1, stream) == 6
            assert lib.wind_rwkv7_attn_ln_forward(*head, *ins, *ln, states[0], ptr(z), ptr(ln_saved), ptr(t1), ptr(ws), least_fwd - 1, stream) == 6
            assert lib.wind_rwkv7_attn_ln_backward(*head, *ins, *ln, ptr(dy), ptr(ln_saved), states[1], *map(ptr, ln_grads), ptr(dparams),
                                                   ptr(ln_ds0), ptr(ws), least_ln_bwd - 1, stream) == 6
            torch.cuda.synchronize()
            assert torch.equal(y, y0) and torch.equal(sT, s1) and torch.equal(z, z0) and torch.equal(t0, t1) and torch.equal(sT, t1)
            out[way] = dict(y=y, sT=sT, z=z, ds0=ds0, ln_ds0=ln_ds0, dparams=dparams, **{f'd{i}': t for i, t in enumerate(grads)},
                            **{f'ln_d{i}': t for i, t in enumerate(ln_grads)})
        segmented = least_fwd > 256   # (the states entering the segments are composed there: fp32, but other sums)
        for n, t in out['records'].items():
            r = out['least'][n]
            assert torch.isfinite(t.float()).all(), n
            if segmented:
                assert (t.float() - r.float()).norm() <= 2e-3 * r.float().norm(), n
            elif n == 'dparams':
                assert (t - r).norm() <= 1e-6 * r.norm()   # sums of B T terms in fp32, in another order
            else:
                assert torch.equal(t, r), n
    finally:
        set_checkpoint_interval(32)
