"""GPU parity of the WKV7 kernels against the fp64 oracle, through the C ABI.

Gate (tests/utils.py:18,24 of the reference, restated): for bf16 sequences every output, final state and
input gradient must satisfy ||x - ref||_2 / ||ref||_2 <= 1e-2 against the fp64 sequential recurrence run
on the same (bf16-rounded) inputs.
"""
import pytest
import torch

from oracle import inputs, seq_ref

pytestmark = pytest.mark.gpu
TOL_BF16 = 1e-2
DEV = 'cuda'


def run_device(d, state_dtype, backward=True):
    from wind_rwkv.rwkv7.wkv_attn import WindRWKV7
    xs = [d[n].to(DEV).requires_grad_(backward) for n in ('w', 'q', 'k', 'v', 'a', 'b')]
    s0 = d['s0'].to(state_dtype).to(DEV).requires_grad_(backward)
    y, sT, _ = WindRWKV7.apply(*xs, s0)
    out = {'y': y, 'sT': sT}
    if backward:
        torch.autograd.backward([y, sT], [d['dy'].to(DEV), d['dsT'].to(state_dtype).to(DEV)])
        out.update(dw=xs[0].grad, dq=xs[1].grad, dk=xs[2].grad, dv=xs[3].grad, da=xs[4].grad, db=xs[5].grad,
                   ds0=s0.grad)
    torch.cuda.synchronize()
    return {k: v.detach().float().cpu() for k, v in out.items()}


def run_oracle(c_oracle, d, state_dtype, backward=True):
    s0 = d['s0'].to(state_dtype)
    dsT = d['dsT'].to(state_dtype)
    args = [d[n] for n in 'qwkvab']
    y, sT = c_oracle.forward(*args, s0)
    out = {'y': y, 'sT': sT}
    if backward:
        g = c_oracle.backward(*args, s0, d['dy'], dsT)
        out.update(dq=g[0], dw=g[1], dk=g[2], dv=g[3], da=g[4], db=g[5], ds0=g[6])
    return out


def check(got, ref, tol=TOL_BF16):
    errs = {k: seq_ref.rel_err(got[k], ref[k]) for k in ref}
    bad = {k: e for k, e in errs.items() if not e <= tol}
    assert not bad, f'over tolerance {tol}: {bad} (all: {errs})'
    return errs


@pytest.mark.parametrize('B,T,H,state_dtype,s0s,dsTs', [
    (1, 16, 1, torch.float32, 0.0, 0.0),        # a single chunk
    (1, 32, 1, torch.float32, 0.5, 0.5),
    (2, 64, 3, torch.float32, 0.1, 0.1),
    (2, 64, 3, torch.bfloat16, 0.1, 0.1),       # the reference's state dtype
    (3, 272, 5, torch.float32, 0.1, 0.0),       # chunk count not a multiple of the scan's prefetch depth
    (1, 2048, 2, torch.float32, 0.1, 0.1),      # this one and the next three by records of their chunks
    (1, 2080, 2, torch.float32, 0.1, 0.1),
    (1, 2112, 2, torch.float32, 0.1, 0.1),
    (1, 6160, 3, torch.bfloat16, 0.1, 0.1),     # 385 chunks, a state per chunk
    (25, 32, 12, torch.float32, 0.1, 0.1),      # 300 (batch, head) pairs: more blocks than compute units
    (19, 48, 12, torch.float32, 0.0, 0.1),      # 228 pairs
    (5, 2048, 12, torch.float32, 0.1, 0.1),     # 60 pairs, 7680 chunks: four segments, one block per segment
    (1, 4096, 3, torch.bfloat16, 0.1, 0.1),     # eight segments, two blocks per segment
])
def test_parity_small(c_oracle, B, T, H, state_dtype, s0s, dsTs):
    d = inputs.wkv7_inputs(B, T, H, 64, seed=100 + T + H, dtype=torch.bfloat16, s0_scale=s0s, dsT_scale=dsTs)
    check(run_device(d, state_dtype), run_oracle(c_oracle, d, state_dtype))


@pytest.mark.parametrize('w_max', [-0.5, 0.5, 1.5])
def test_parity_strong_decay(c_oracle, w_max):
    """Decay inputs up to w_max on whole runs of tokens: decay exp(-exp(w)) down to 0.011 per token, 1e-31 over a
    chunk (the reference's time mixer keeps w <= -0.5, decay >= 0.545, rwkv7_expand_loras.py:65).  The chunked form
    divides by cumulative decays inside a chunk; beyond the fp32 range (sum of exp(w) over a chunk above ~87)
    this implementation, like the reference's chunked kernels (rwkv7_attn_triton.py:44-51), is not defined."""
    B, T, H = 2, 128, 3
    d = inputs.wkv7_inputs(B, T, H, 64, seed=77, dtype=torch.bfloat16, s0_scale=0.1, dsT_scale=0.1)
    gen = torch.Generator().manual_seed(78)
    w = torch.rand(B, T, H, 64, generator=gen) * (w_max + 6) - 6
    w[:, 16:48] = w_max          # two whole chunks at the strongest decay
    w[:, 60:70, 1] = w_max       # and a run across a chunk boundary in one head
    d['w'] = w.bfloat16()
    check(run_device(d, torch.float32), run_oracle(c_oracle, d, torch.float32))


@pytest.mark.parametrize('corr,gate', [(0.5, 0.95), (0.2, 1.0)])
def test_parity_strongly_coupled_tokens(c_oracle, corr, gate):
    """Neighbouring tokens with nearly the same removal direction kk, a = -kk, b = gate * kk and slow decay: the
    strictly lower-triangular matrix whose inverse every chunk needs then has ALL its entries near -gate (they are
    near zero for the random directions of the other cases), the regime in which a less accurate inverse (a Neumann
    product, single bf16 operands) loses digits.  Measured: every tensor within 4e-3 except da, db at 6.7e-3 (gate 0.95)
    and 9.8e-3 (gate 1), identical to three digits with the inverse on the fp32 matrix instruction - the bf16
    operands of the chunk algebra set these errors, not the hi/lo inverse."""
    B, T, H = 2, 96, 3
    d = inputs.wkv7_inputs(B, T, H, 64, seed=91, dtype=torch.bfloat16, s0_scale=0.1, dsT_scale=0.1)
    gen = torch.Generator().manual_seed(92)
    u = torch.randn(B, 1, H, 64, generator=gen)
    kk = torch.nn.functional.normalize(u + corr * torch.randn(B, T, H, 64, generator=gen), dim=-1)
    d['a'] = (-kk).bfloat16()
    d['b'] = (gate * kk).bfloat16()
    d['w'] = (-4.0 - 2.0 * torch.rand(B, T, H, 64, generator=gen)).bfloat16()
    errs = check(run_device(d, torch.float32), run_oracle(c_oracle, d, torch.float32))
    print('strongly coupled tokens, errors', {k: f'{v:.2e}' for k, v in errs.items()})


def test_parity_cfg1_full(c_oracle):
    """B=8, T=1024, H=12, N=64, bf16, zero initial state: the shape the headline metric is quoted on."""
    d = inputs.wkv7_inputs(8, 1024, 12, 64, seed=1, dtype=torch.bfloat16)
    errs = check(run_device(d, torch.float32), run_oracle(c_oracle, d, torch.float32))
    print('cfg1 errors', {k: f'{v:.2e}' for k, v in errs.items()})


@pytest.mark.parametrize('B,T,H', [(8, 1024, 13), (17, 1024, 12), (131, 64, 12), (260, 32, 12), (8, 1024, 32)])
def test_parity_runs_of_pairs_that_do_not_divide_evenly(c_oracle, B, T, H):
    """From 3072 pairs of chunks on (6144 on), the gradient kernel's wavefronts take runs of three (six) consecutive
    pairs and carry the dstate along a run themselves; the reverse scan keeps it only where a run starts.  Heads of 32
    pairs: runs straddle the heads' boundaries, the last run is short, and some wavefronts take two runs.  Heads of
    two pairs and of one: a run covers several heads, and with one pair per head nothing is carried at all.  32 heads:
    from 16 heads on the runs are cut per head (32 pairs: ten runs of three and one of two) and handed out head-major."""
    d = inputs.wkv7_inputs(B, T, H, 64, seed=77, dtype=torch.bfloat16, s0_scale=0.1, dsT_scale=0.1)
    errs = check(run_device(d, torch.float32), run_oracle(c_oracle, d, torch.float32))
    print('runs of pairs, errors', {k: f'{v:.2e}' for k, v in errs.items()})


@pytest.mark.parametrize('B,T,H,ln', [(2, 1024, 16, False), (3, 768, 15, False), (33, 32, 16, False), (9, 480, 4, False), (2, 1024, 16, True),
                                      (3, 768, 15, True), (9, 480, 4, True)])
def test_a_chunk_per_wavefront_gives_the_bits_of_a_pair_per_wavefront(B, T, H, ln):
    """Gradients of a batch with more chunks than four per compute unit (2048, 2160, 1056, 1080), a pair of chunks per wavefront, and
    of its sequences one by one (1024, 720, 32, 120), a chunk per wavefront.  (attn_ln up to 128 heads, where its forward has one form.)"""
    from wind_rwkv.rwkv7 import attn, attn_ln
    d = inputs.wkv7_inputs(B, T, H, 64, seed=B + T, dtype=torch.bfloat16, s0_scale=0.3)
    x = [d[n].reshape(B, T, H * 64).to(DEV) for n in ('q', 'w', 'k', 'v', 'a', 'b')]
    s0, dy = d['s0'].float().to(DEV), d['dy'].reshape(B, T, H * 64).to(DEV)
    gen = torch.Generator().manual_seed(T)
    g, params = torch.randn(x[0].shape, generator=gen).bfloat16().to(DEV), torch.randn(3, H * 64, generator=gen).to(DEV)

    def grads(rows):
        leaves = [t[rows].detach().clone().requires_grad_() for t in x + [g]]
        y = attn_ln(*leaves, params, 64, s0=s0[rows]) if ln else attn(*leaves[:6], 64, s0=s0[rows])
        return torch.autograd.grad(y, leaves if ln else leaves[:6], dy[rows])

    whole = grads(slice(None))
    assert all(torch.isfinite(t.float()).all() for t in whole)
    for b in range(0, B, max(1, B - 1)):   # the first and the last sequence
        for n, t in zip('qwkvabg', grads(slice(b, b + 1))):
            assert torch.equal(t[0], whole['qwkvabg'.index(n)][b]), n


@pytest.fixture
def checkpoint_interval(request):
    """Runs the test under the given number of tokens between kept states and restores the default (32)."""
    from wind_rwkv.rwkv7 import set_checkpoint_interval
    set_checkpoint_interval(request.param)
    yield request.param
    set_checkpoint_interval(32)


@pytest.mark.parametrize('checkpoint_interval', [16, 32], indirect=True)
@pytest.mark.parametrize('B,T,H,s0s', [(8, 1024, 12, 0.0), (3, 96, 5, 0.3), (2, 48, 2, 0.1)])
def test_parity_at_either_checkpoint_interval(c_oracle, checkpoint_interval, B, T, H, s0s):
    """A state checkpoint per 16-token chunk (the reference's layout) or per pair of chunks (two-level chunking, the
    default): both against the oracle at the same gate, the headline shape among the cases, and the kept bytes as the
    size query reports them.  (48 tokens = three chunks: a state per chunk whatever the setting.)"""
    from wind_rwkv import _native
    assert _native.lib().wind_rwkv7_checkpoint_interval() == checkpoint_interval
    per_chunk = _native.lib().wind_rwkv7_attn_bwd_workspace_bytes(B, T, H, 64) / (B * H * (T // 16))
    assert per_chunk == (12 * 512 if checkpoint_interval == 32 and (T // 16) % 2 == 0 else 20 * 512)
    d = inputs.wkv7_inputs(B, T, H, 64, seed=1 if T == 1024 else 40 + T, dtype=torch.bfloat16, s0_scale=s0s, dsT_scale=s0s)
    errs = check(run_device(d, torch.float32), run_oracle(c_oracle, d, torch.float32))
    print(f'checkpoint interval {checkpoint_interval}, B{B} T{T} H{H}:', {k: f'{v:.2e}' for k, v in errs.items()})


def test_interval_change_between_forward_and_backward_is_an_error():
    """The saved tensor's layout follows the checkpoint interval of the forward; a backward under another value raises
    instead of misreading it (attn and attn_ln alike)."""
    from wind_rwkv.rwkv7 import set_checkpoint_interval
    from wind_rwkv.rwkv7.wkv_attn import WindRWKV7
    from wind_rwkv.rwkv7.wkv_attn_ln import WindRWKV7LN
    d = inputs.wkv7_inputs(1, 64, 2, 64, seed=77, dtype=torch.bfloat16)
    x = [d[n].to(DEV).requires_grad_() for n in ('w', 'q', 'k', 'v', 'a', 'b')]
    s0 = torch.zeros(1, 2, 64, 64, device=DEV)
    try:
        y = WindRWKV7.apply(*x, s0)[0]
        g = torch.ones_like(x[0])
        params = torch.ones(3, 128, device=DEV)
        y2 = WindRWKV7LN.apply(*x, g, params, s0)[0]
        set_checkpoint_interval(16)
        with pytest.raises(RuntimeError, match='checkpoint interval changed'):
            y.sum().backward()
        with pytest.raises(RuntimeError, match='checkpoint interval changed'):
            y2.sum().backward()
    finally:
        set_checkpoint_interval(32)
    y = WindRWKV7.apply(*x, s0)[0]
    y.sum().backward()    # (and under one value all is well)
    assert all(torch.isfinite(t.grad.float()).all() for t in x)


def test_parity_long_sequences_on_a_quarter_of_the_machine(c_oracle):
    """64 (batch, head) pairs x 2048 tokens: as many pairs as the segmented scans take (a quarter of the compute units), four
    segments each; y, sT, the six gradients and ds0 against the oracle."""
    d = inputs.wkv7_inputs(2, 2048, 32, 64, seed=61, dtype=torch.bfloat16, s0_scale=0.1, dsT_scale=0.1)
    errs = check(run_device(d, torch.float32), run_oracle(c_oracle, d, torch.float32))
    print('B2 T2048 H32:', {k: f'{v:.2e}' for k, v in errs.items()})


def test_parity_cfg3_long_context_slice(c_oracle):
    """T=16384 with a non-zero initial state (4 of the 32 heads, so that the oracle finishes in seconds),
    checking y, sT, the six gradients and ds0."""
    d = inputs.wkv7_inputs(1, 16384, 4, 64, seed=3, dtype=torch.bfloat16, s0_scale=0.1)
    check(run_device(d, torch.float32), run_oracle(c_oracle, d, torch.float32))


def test_cfg3_full_size_properties():
    """B=1, T=16384, H=32 at full size through size-independent properties: splitting the sequence in two
    calls that carry the state reproduces the one-call result, and the map is linear in v."""
    from wind_rwkv.rwkv7.wkv_attn import WindRWKV7
    d = inputs.wkv7_inputs(1, 16384, 32, 64, seed=3, dtype=torch.bfloat16, s0_scale=0.1, with_dy=False)
    xs = [d[n].to(DEV) for n in ('w', 'q', 'k', 'v', 'a', 'b')]
    s0 = d['s0'].to(DEV)
    y, sT, _ = WindRWKV7.apply(*xs, s0)
    half = 8192
    y1, s1, _ = WindRWKV7.apply(*[x[:, :half].contiguous() for x in xs], s0)
    y2, s2, _ = WindRWKV7.apply(*[x[:, half:].contiguous() for x in xs], s1)
    assert seq_ref.rel_err(torch.cat([y1, y2], 1).float().cpu(), y.float().cpu()) < 1e-5
    assert seq_ref.rel_err(s2.cpu(), sT.cpu()) < 1e-5
    xs2 = list(xs)
    xs2[3] = (xs[3].float() * 2).bfloat16()  # exact in bf16
    yv, sTv, _ = WindRWKV7.apply(*xs2, s0 * 2)
    assert seq_ref.rel_err(yv.float().cpu(), 2 * y.float().cpu()) < 1e-5
    assert seq_ref.rel_err(sTv.cpu(), 2 * sT.cpu()) < 1e-5


def test_cfg3_full_size_backward_properties():
    """B=1, T=16384, H=32 at full size, backward included: one call against the same sequence cut in two calls that
    carry the state forward and the state gradient back (dsT of the first piece = ds0 of the second).  Every piece
    runs the same per-chunk arithmetic; only the segment maps and the fp32 states crossing the cut differ."""
    from wind_rwkv.rwkv7.wkv_attn import WindRWKV7
    T, Q = 16384, 8192
    d = inputs.wkv7_inputs(1, T, 32, 64, seed=3, dtype=torch.bfloat16, s0_scale=0.1, dsT_scale=0.1)
    xs = [d[n].to(DEV).requires_grad_() for n in ('w', 'q', 'k', 'v', 'a', 'b')]
    s0 = d['s0'].to(DEV).requires_grad_()
    dy, dsT = d['dy'].to(DEV), d['dsT'].to(DEV)
    y, sT, _ = WindRWKV7.apply(*xs, s0)
    torch.autograd.backward([y, sT], [dy, dsT])
    whole = [y.detach(), sT.detach(), s0.grad.clone()] + [x.grad.clone() for x in xs]
    for x in xs:
        x.grad = None
    s0.grad = None
    y1, s1, _ = WindRWKV7.apply(*[x[:, :Q].contiguous() for x in xs], s0)
    y2, s2, _ = WindRWKV7.apply(*[x[:, Q:].contiguous() for x in xs], s1)
    torch.autograd.backward([torch.cat([y1, y2], 1), s2], [dy, dsT])
    parts = [torch.cat([y1, y2], 1).detach(), s2.detach(), s0.grad] + [x.grad for x in xs]
    for n, a, b in zip(['y', 'sT', 'ds0', 'dw', 'dq', 'dk', 'dv', 'da', 'db'], parts, whole):
        assert torch.isfinite(a).all() and torch.isfinite(b).all(), n
        assert seq_ref.rel_err(a.float().cpu(), b.float().cpu()) < 2e-3, n


def test_very_long_sequence_properties():
    """B=1, T=65536, H=2 (4096 chunks per head, eight scan segments of 512): forward and backward in one call
    against the same sequence cut in four calls that carry the state forward and the state gradient back."""
    from wind_rwkv.rwkv7.wkv_attn import WindRWKV7
    T, Q = 65536, 16384
    d = inputs.wkv7_inputs(1, T, 2, 64, seed=11, dtype=torch.bfloat16, s0_scale=0.1)
    xs = [d[n].to(DEV).requires_grad_() for n in ('w', 'q', 'k', 'v', 'a', 'b')]
    s0 = d['s0'].to(DEV).requires_grad_()
    dy = d['dy'].to(DEV)
    y, sT, _ = WindRWKV7.apply(*xs, s0)
    torch.autograd.backward([y], [dy])
    whole = [y.detach(), sT.detach(), s0.grad.clone()] + [x.grad.clone() for x in xs]
    for x in xs:
        x.grad = None
    s0.grad = None
    state, ys = s0, []
    for i in range(4):
        yi, state, _ = WindRWKV7.apply(*[x[:, i * Q:(i + 1) * Q].contiguous() for x in xs], state)
        ys.append(yi)
    torch.autograd.backward([torch.cat(ys, 1)], [dy])
    parts = [torch.cat(ys, 1).detach(), state.detach(), s0.grad] + [x.grad for x in xs]
    names = ['y', 'sT', 'ds0', 'dw', 'dq', 'dk', 'dv', 'da', 'db']
    for n, a, b in zip(names, parts, whole):
        assert torch.isfinite(a).all() and torch.isfinite(b).all(), n
        # same arithmetic per chunk; the states crossing a cut are fp32 either way, the segment maps differ
        assert seq_ref.rel_err(a.float().cpu(), b.float().cpu()) < 2e-3, n


def test_public_wrapper_matches_function(c_oracle):
    """attn(r,w,k,v,a,b,HEAD_SIZE) takes [B,T,H*C] tensors in the reference's argument order."""
    from wind_rwkv.rwkv7 import attn, load_attn
    load_attn(64)
    d = inputs.wkv7_inputs(2, 48, 2, 64, seed=5, dtype=torch.bfloat16)
    flat = {n: d[n].view(2, 48, 128).to(DEV) for n in 'qwkvab'}
    y = attn(flat['q'], flat['w'], flat['k'], flat['v'], flat['a'], flat['b'], 64)
    yo, _ = c_oracle.forward(*[d[n] for n in 'qwkvab'], d['s0'])
    assert y.shape == (2, 48, 128) and y.dtype == torch.bfloat16
    assert seq_ref.rel_err(y.float().cpu().view(2, 48, 2, 64), yo) < TOL_BF16


def test_missing_upstream_gradients():
    """Only y is used downstream (dsT is None), as in the reference's wrappers (rwkv7_attn.py:38)."""
    from wind_rwkv.rwkv7.wkv_attn import WindRWKV7
    d = inputs.wkv7_inputs(1, 32, 1, 64, seed=6, dtype=torch.bfloat16)
    xs = [d[n].to(DEV).requires_grad_() for n in ('w', 'q', 'k', 'v', 'a', 'b')]
    s0 = torch.zeros(1, 1, 64, 64, device=DEV, dtype=torch.bfloat16)
    y = WindRWKV7.apply(*xs, s0)[0]
    y.float().sum().backward()
    assert all(x.grad is not None and torch.isfinite(x.grad.float()).all() for x in xs)


def test_rejects_bad_shapes():
    from wind_rwkv import _native
    from wind_rwkv.rwkv7.wkv_attn import fw_attn
    x = torch.zeros(1, 24, 1, 64, dtype=torch.bfloat16, device=DEV)
    s0 = torch.zeros(1, 1, 64, 64, device=DEV)
    with pytest.raises(_native.WindRwkv7Error):
        fw_attn(x, x, x, x, x, x, s0)


def test_primitives_selftest():
    """Fragment primitives (matrix products, transposes, row scans, triangular inverse) on one wavefront."""
    import ctypes
    import os
    from wind_rwkv import _native
    st = ctypes.CDLL(os.path.join(os.path.dirname(_native.LIB_PATH), 'libwind_rwkv7_selftest.so'))
    st.wind_rwkv7_selftest_primitives.argtypes = [ctypes.c_void_p] * 4
    gen = torch.Generator().manual_seed(0)
    X = torch.randn(16, 16, generator=gen).bfloat16().float()
    Y = torch.randn(16, 16, generator=gen).bfloat16().float()
    out = torch.zeros(11, 16, 16, device=DEV)
    Xd, Yd = X.to(DEV), Y.to(DEV)
    assert st.wind_rwkv7_selftest_primitives(Xd.data_ptr(), Yd.data_ptr(), out.data_ptr(), None) == 0
    torch.cuda.synchronize()
    o = out.cpu()
    Xl = torch.tril(X, -1)
    inv = torch.linalg.inv(torch.eye(16, dtype=torch.float64) - Xl.double()).float()
    expect = [X @ Y.T, X @ Y.T, X.T, torch.cumsum(X, 0), torch.flip(torch.cumsum(torch.flip(X, [0]), 0), [0]),
              X[15:16].expand(16, 16), X.sum(0, keepdim=True).expand(16, 16), inv, inv.T,
              X.view(16, 4, 4).sum(1).repeat(1, 4), X.sum(1, keepdim=True).expand(16, 16)]
    for i, e in enumerate(expect):
        assert seq_ref.rel_err(o[i], e) < 1e-5, i


@pytest.mark.parametrize('B,T,H', [(2, 64, 3), (25, 32, 12)])   # two blocks per head / one block per head
def test_absent_states_equal_zero_states(B, T, H):
    """An empty s0 (the C ABI's NULL: zero initial state), no gradient for sT (NULL dsT) and no request for ds0
    (NULL ds0) give bit for bit what explicit tensors of zeros give."""
    from wind_rwkv.rwkv7.wkv_attn import WindRWKV7, no_state
    d = inputs.wkv7_inputs(B, T, H, 64, seed=77, dtype=torch.bfloat16)
    dy = d['dy'].to(DEV)

    def run(s0, dsT):
        xs = [d[n].to(DEV).requires_grad_() for n in ('w', 'q', 'k', 'v', 'a', 'b')]
        y, sT, _ = WindRWKV7.apply(*xs, s0)
        torch.autograd.backward([y] if dsT is None else [y, sT], [dy] if dsT is None else [dy, dsT])
        return [y.detach(), sT.detach()] + [x.grad for x in xs]

    zeros = torch.zeros(B, H, 64, 64, dtype=torch.bfloat16, device=DEV)
    ref = run(zeros.clone().requires_grad_(), torch.zeros_like(zeros))
    got = run(no_state(torch.bfloat16, DEV), None)
    for r, g in zip(ref, got):
        assert torch.equal(r, g)


# (rows of 16 tokens and 2^26 channels on reach past 2 GiB of a tile's first byte)
@pytest.mark.parametrize('at', [0, (1 << 31) - 1024, (1 << 31) - 512, 1 << 31, (1 << 32) - 2048])
def test_stores_through_the_l2_reach_four_gib(at):
    import ctypes
    import os
    from wind_rwkv import _native
    st = ctypes.CDLL(os.path.join(os.path.dirname(_native.LIB_PATH), 'libwind_rwkv7_selftest.so'))
    st.wind_rwkv7_selftest_store_through.argtypes = [ctypes.c_void_p, ctypes.c_longlong, ctypes.c_longlong, ctypes.c_void_p]
    out = torch.empty(1 << 30, dtype=torch.int32, device=DEV)
    here = out[at // 4:at // 4 + 256].fill_(-1)
    assert st.wind_rwkv7_selftest_store_through(out.data_ptr(), at, 1 << 32, None) == 0
    torch.cuda.synchronize()
    want = torch.arange(64, dtype=torch.int32)[:, None] + torch.arange(4, dtype=torch.int32)
    assert bool((here.view(64, 4).cpu() == want).all())


def test_global_to_lds_load_lane_mapping():
    """The hardware fact the gradient kernel's state prefetch is built on: a global -> LDS load of 16 bytes per lane
    (global_load_lds_dwordx4) takes one memory address per lane but writes lane l's piece at the wave-uniform LDS
    base + 16 l; the immediate offset moves both the memory address and the LDS address, a buffer load's scalar
    offset the memory address only."""
    import ctypes
    import os
    from wind_rwkv import _native
    st = ctypes.CDLL(os.path.join(os.path.dirname(_native.LIB_PATH), 'libwind_rwkv7_selftest.so'))
    st.wind_rwkv7_selftest_lds_dma.argtypes = [ctypes.c_void_p] * 3
    src = torch.arange(1536, dtype=torch.int32, device=DEV)
    out = torch.full((2048,), -1, dtype=torch.int32, device=DEV)
    assert st.wind_rwkv7_selftest_lds_dma(src.data_ptr(), out.data_ptr(), None) == 0
    torch.cuda.synchronize()
    got = out.cpu().view(2048)
    for t in range(256):
        wave, lane = divmod(t, 64)
        piece = (37 * t + 11) & 255
        first = got[wave * 256 + 4 * lane:][:4].tolist()
        second = got[wave * 256 + 512 + 512 + 4 * lane:][:4].tolist()      # base + 2 KiB + immediate 2 KiB
        assert first == [4 * (piece + 128) + i for i in range(4)], (t, first)   # buffer form: the scalar offset moves the memory address only
        assert second == [4 * (255 - piece + 128) + i for i in range(4)], (t, second)
