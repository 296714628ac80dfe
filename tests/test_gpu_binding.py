"""The native eager path (csrc/torch_binding.cpp) against the Python autograd Functions, which call the same kernels: same
bits in outputs and gradients, whichever inputs ask for a gradient, and the same errors for what the kernels do not take."""
import pytest
import torch

from oracle import inputs, seq_ref

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _flat(d, n, dtype=torch.bfloat16):
    B, T, H, C = d[n].shape
    return d[n].reshape(B, T, H * C).to(DEV, dtype)


def _run(fn, leaves, wanted, grads):
    xs = [t.detach().clone().requires_grad_(i in wanted) for i, t in enumerate(leaves)]
    outs = fn(*xs)
    gs = torch.autograd.grad(outs, [x for i, x in enumerate(xs) if i in wanted], grads)
    return [o.detach() for o in outs] + list(gs)


def _same(native, function, leaves, grads, wanted_sets):
    for wanted in wanted_sets:
        for x, y in zip(_run(native, leaves, wanted, grads), _run(function, leaves, wanted, grads)):
            assert x.dtype == y.dtype and torch.equal(x.reshape(-1), y.reshape(-1))


@pytest.mark.parametrize('state_dtype', [torch.float32, torch.bfloat16, None])
@pytest.mark.parametrize('B,T,H,C', [(1, 16, 1, 64), (2, 48, 3, 64), (2, 32, 3, 128), (1, 2048, 2, 64)])
def test_attn_and_attn_ln_equal_the_python_functions(B, T, H, C, state_dtype):
    from wind_rwkv.rwkv7 import attn, attn_ln
    from wind_rwkv.rwkv7.wkv_attn import WindRWKV7, no_state
    from wind_rwkv.rwkv7.wkv_attn_ln import WindRWKV7LN
    d = inputs.attn_ln_inputs(B, T, H, C, 3, dtype=torch.bfloat16)
    gen = torch.Generator().manual_seed(4)
    seqs = [_flat(d, n) for n in 'qwkvab']
    heads = lambda t: t.view(B, T, H, C)
    state = [] if state_dtype is None else [torch.randn(B, H, C, C, generator=gen).to(DEV, state_dtype)]
    s0_of = lambda st: st[0] if st else no_state(torch.bfloat16, DEV)
    dy = _flat(d, 'dy')
    dsT = torch.randn(B, H, C, C, generator=gen).to(DEV, state_dtype or torch.bfloat16)
    every = set(range(6 + len(state)))
    def function(r, w, k, v, a, b, *st):
        y, sT, _ = WindRWKV7.apply(*map(heads, (w, r, k, v, a, b)), s0_of(st))
        return y.view(B, T, H * C), sT
    native = lambda *x: attn(*x[:6], C, s0=x[6] if x[6:] else None, return_state=True)
    _same(native, function, seqs + state, [dy, dsT], [every, {1, 3}, {max(every)}])
    def function_ln(r, w, k, v, a, b, g, p, *st):
        y, sT, _ = WindRWKV7LN.apply(*map(heads, (w, r, k, v, a, b, g)), p, s0_of(st))
        return y.view(B, T, H * C), sT
    native_ln = lambda *x: attn_ln(*x[:8], C, s0=x[8] if x[8:] else None, return_state=True)
    every = set(range(8 + len(state)))
    _same(native_ln, function_ln, seqs + [_flat(d, 'g'), d['params'].to(DEV)] + state, [dy, dsT], [every, {6, 7}, {max(every)}])


@pytest.mark.parametrize('param_dtype', [torch.float32, torch.bfloat16])
def test_ddlerp_and_expand_loras_equal_the_python_functions(param_dtype):
    from wind_rwkv.rwkv7 import ddlerp, expand_loras
    from wind_rwkv.rwkv7.loras import ExpandLoras
    from wind_rwkv.rwkv7.token_shift import DDLerp
    B, T, C = 2, 48, 128
    d = inputs.ddlerp_inputs(B, T, C, 32, 5, dtype=torch.bfloat16)
    leaves = [d['x'].to(DEV)] + [d[n].to(DEV, param_dtype) for n in ('alpha', 'L', 'R', 'beta')]
    _same(ddlerp, DDLerp.apply, leaves, [g.to(DEV) for g in d['dy']], [set(range(5)), {0}, {2}])
    d = inputs.expand_loras_inputs(B, T, C, 16, 6, dtype=torch.bfloat16)
    acts = [d[n].to(DEV) for n in ('w_in', 'k_in', 'z_in', 'a_in', 'ma_in', 'mk_in')]
    params = [d[n].to(DEV, param_dtype) for n in ('Wz', 'Wa', 'Wma', 'Wmk', 'w_bias', 'a_bias', 'ma_bias', 'mk_bias')]
    _same(lambda *x: expand_loras(*x, 64), lambda *x: ExpandLoras.apply(*x, 64), acts + params, [g.to(DEV) for g in d['dy']],
          [set(range(14)), {2, 5}, {9, 13}])


def test_what_the_native_path_leaves_to_python():
    """Strided inputs and wrong types raise as before; a changed checkpoint interval is an error in backward."""
    from wind_rwkv.rwkv7 import attn, checkpoint_interval, set_checkpoint_interval
    d = inputs.wkv7_inputs(1, 32, 2, 64, 7, dtype=torch.bfloat16)
    seqs = [_flat(d, n).requires_grad_() for n in 'qwkvab']
    with pytest.raises(AssertionError):
        attn(*[t.mT.contiguous().mT for t in seqs], 64)
    with pytest.raises(AssertionError):
        attn(seqs[0].half(), *seqs[1:], 64)
    before = checkpoint_interval()
    y = attn(*seqs, 64)
    set_checkpoint_interval(48 - before)
    try:
        with pytest.raises(RuntimeError, match='checkpoint interval'):
            y.sum().backward()
    finally:
        set_checkpoint_interval(before)


class _Absent:
    """A binding that takes no case: every call falls to the Python path."""
    def __getattr__(self, name):
        return lambda *args: None


@pytest.mark.parametrize('C,H,x_dtype,param_dtype,frozen', [
    (128, 2, torch.bfloat16, torch.float32, ()), (192, 6, torch.float32, torch.float32, ('Wr', 'gate_w2', 'ln_x.weight')),
    (256, 2, torch.bfloat16, torch.bfloat16, ('Wo', 'time_maa_w1'))])
def test_block_equals_the_python_path(monkeypatch, C, H, x_dtype, param_dtype, frozen):
    """Forward, backward and the forward without autograd of the whole block, with some parameters frozen, against the
    Python path, whose products are the BLAS library's: other summation orders inside them, so bf16 values differ by a
    rounding here and there, and what follows from those: a gate of 5e-3 on the output and 1e-2 on gradients (what the block
    is held to against its oracle is 1e-2 to 1.6e-2)."""
    from collections import namedtuple
    from oracle import seq_ref
    from wind_rwkv import _native
    from wind_rwkv.rwkv7 import TimeMixer
    gen = torch.Generator().manual_seed(C)
    model = TimeMixer(namedtuple('Config', ['n_layer', 'n_head', 'n_embd'])(4, H, C), 1)
    with torch.no_grad():
        for n, p in model.named_parameters():
            p.copy_(torch.randn(p.shape, generator=gen) * 0.1)
            p.requires_grad_(n not in frozen)
    model = model.to(DEV, param_dtype)
    x = torch.randn(2, 48, C, generator=gen).to(DEV, x_dtype)
    dy = torch.randn(2, 48, C, generator=gen).to(DEV, torch.bfloat16)
    results = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(_native, 'binding', lambda: _Absent())
        leaves = [x.clone().requires_grad_()] + [p for p in model.parameters() if p.requires_grad]
        y = model(leaves[0])
        with torch.no_grad():
            z = model(x)
        results.append([y.detach(), z] + list(torch.autograd.grad(y, leaves, dy)))
    for i, (a, b) in enumerate(zip(*results)):
        assert a.dtype == b.dtype and a.shape == b.shape
        assert seq_ref.rel_err(a.float().cpu(), b.float().cpu()) <= (5e-3 if i < 2 else 1e-2), i


@pytest.mark.parametrize('C,H,B', [(2048, 32, 6), (768, 12, 42)])
def test_a_block_of_large_products_equals_the_python_path(monkeypatch, C, H, B):
    """Products of 2.5e10 and more, which go to the BLAS library: all of them at 2048 channels, those of one segment at 768.  At
    the gates of the test above, the output's first token apart (its GroupNorm after a zero state is ill conditioned)."""
    from wind_rwkv import _native
    assert B * 1024 * C * C >= 2.5e10
    model, gen = _small_model(C, H, torch.float32)
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() == 2:
                p.mul_(10 * C ** -0.5)   # (unit gain: 0.1 N(0,1) as above is for small blocks)
    x, dy = (torch.randn(B, 1024, C, generator=gen).bfloat16().to(DEV) for _ in range(2))
    dy[:, 0] = 0
    results = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(_native, 'binding', lambda: _Absent())
        leaves = [x.clone().requires_grad_()] + list(model.parameters())
        y = model(leaves[0])
        results.append([y.detach()[:, 1:]] + list(torch.autograd.grad(y, leaves, dy)))
    for i, (a, b) in enumerate(zip(*results)):
        assert seq_ref.rel_err(a.float(), b.float()) <= (5e-3 if i < 1 else 1e-2), i


@pytest.mark.parametrize('T', [2, 15, 17, 100])
@pytest.mark.parametrize('continued', [False, True])
def test_prompt_of_any_length_equals_the_python_path(monkeypatch, T, continued):
    """The native prompt against the Python path of whole chunks and single-token steps: other summation orders, so at the
    block's gate (1.27e-2 where `step` computed the tokens, see tests/test_gpu_time_mixer_state.py), state at 1e-2."""
    from collections import namedtuple
    from oracle import seq_ref
    from wind_rwkv import _native
    from wind_rwkv.rwkv7 import TimeMixer
    gen = torch.Generator().manual_seed(T)
    C, H, B = 256, 4, 3
    model = TimeMixer(namedtuple('Config', ['n_layer', 'n_head', 'n_embd'])(4, H, C), 1)
    with torch.no_grad():
        for p in model.parameters():
            p.copy_(torch.randn(p.shape, generator=gen) * 0.1)
    model = model.to(DEV)
    x = torch.randn(B, T, C, generator=gen).bfloat16().to(DEV)
    state = (torch.randn(B, C, generator=gen).bfloat16().to(DEV), torch.randn(B, H, 64, 64, generator=gen).to(DEV)) if continued else None
    with torch.no_grad():
        y, (last, S) = model(x, state=state, return_state=True)
        monkeypatch.setattr(_native, 'binding', lambda: _Absent())
        y0, (last0, S0) = model(x, state=state, return_state=True)
    assert y.shape == y0.shape and y.is_contiguous() and torch.equal(last, last0) and torch.equal(last, x[:, -1])
    assert S.dtype == S0.dtype == torch.float32
    first = 0 if continued else 1     # from a zero state the first token's GroupNorm is ill conditioned
    assert seq_ref.rel_err(y[:, first:].float().cpu(), y0[:, first:].float().cpu()) <= 1.27e-2
    assert seq_ref.rel_err(S.cpu(), S0.cpu()) <= 1e-2


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_parameters_and_gradients_that_start_anywhere(dtype):
    """Parameters as views into one flat buffer (flat optimizers), the input and its gradient one element off a 16-byte
    boundary: the bits of the same values in tensors of their own, for the block, prompts, steps and the two stages."""
    from collections import namedtuple
    from wind_rwkv.rwkv7 import TimeMixer, ddlerp, expand_loras
    C, H, B, T = 128, 2, 2, 48
    gen = torch.Generator().manual_seed(5)
    model = TimeMixer(namedtuple('Config', ['n_layer', 'n_head', 'n_embd'])(4, H, C), 1)
    with torch.no_grad():
        for p in model.parameters():
            p.copy_(torch.randn(p.shape, generator=gen) * 0.1)
    model = model.to(DEV, dtype)
    off = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)
    x, dy = (torch.randn(B, T, C, generator=gen).bfloat16().to(DEV) for _ in range(2))
    state = (torch.randn(B, C, generator=gen).bfloat16().to(DEV), torch.randn(B, H, 64, 64, generator=gen).to(DEV))
    def passes(move):
        leaf = move(x).requires_grad_()
        y = model(leaf)
        out = [y] + list(torch.autograd.grad(y, [leaf] + list(model.parameters()), move(dy)))
        with torch.no_grad():
            for n in (T, 7, 35):
                y, st = model(move(x[:, :n].contiguous()), state=(move(state[0]), state[1].clone()), return_state=True)
                y2, st = model.step(move(x[:, n - 1].contiguous()), (move(st[0]), st[1]))
                out += [y, y2, *st]
            compiled = torch.compile(model, fullgraph=True)
            out.append(compiled(move(x)))
        m = model
        out += ddlerp(x, m.time_maa_x, m.time_maa_w1, m.time_maa_w2, m.time_maa)
        a16 = x[..., :16].contiguous()
        out += expand_loras(x, dy, a16, a16, a16, a16, m.time_kkk_w2, m.time_aaa_w2, m.ma_w2, m.mk_w2, m.time_decay, m.time_aaaaa, m.time_misc_a, m.time_misc_k, 64)
        return [t.detach().clone() for t in out]
    want = passes(lambda t: t.clone())
    flat = torch.cat([torch.zeros(1, dtype=dtype, device=DEV)] + [p.detach().reshape(-1) for p in model.parameters()])
    at = 1
    for p in model.parameters():
        p.data = flat[at:at + p.numel()].view(p.shape)
        at += p.numel()
    assert all(p.data_ptr() % 16 for p in model.parameters())
    model.invalidate_decode_cache()
    for i, (a, b) in enumerate(zip(passes(off), want)):
        assert torch.equal(a, b), i


def _small_model(C, H, dtype, seed=5):
    from collections import namedtuple
    from wind_rwkv.rwkv7 import TimeMixer
    gen = torch.Generator().manual_seed(seed)
    model = TimeMixer(namedtuple('Config', ['n_layer', 'n_head', 'n_embd'])(4, H, C), 1)
    with torch.no_grad():
        for p in model.parameters():
            p.copy_(torch.randn(p.shape, generator=gen) * 0.1)
    return model.to(DEV, dtype), gen


EXPANSION = ('time_kkk_w2', 'time_aaa_w2', 'ma_w2', 'mk_w2', 'time_decay', 'time_aaaaa', 'time_misc_a', 'time_misc_k')


@pytest.mark.parametrize('compiled', [False, True])
@pytest.mark.parametrize('wanted', [('Wo',), ('ln_x.weight',), ('Wo', 'Wv'), ('gate_w1',), ('gate_w2', 'Wr'), ('mk_w1',), ('time_aaa_w1',),
                                    ('time_decay_w2', 'Wk'), EXPANSION[1:2], EXPANSION, ('time_maa_w2',), ('x',), ('x', 'Wo', 'ma_w1')])
def test_a_backward_pass_stops_behind_what_is_wanted(wanted, compiled):
    """Any choice of wanted gradients: the values are those of the whole backward (the same products; a weight gradient alone or in
    a smaller group is cut into other token ranges, fp32 sums: 1e-5).  With the output projection alone nothing of the
    recurrence runs or is kept, and the buffer handed out holds the wanted gradients only."""
    from wind_rwkv import _native
    B, T, C, H = 2, 64, 128, 2
    model, gen = _small_model(C, H, torch.float32)
    x, dy = (torch.randn(B, T, C, generator=gen).bfloat16().to(DEV) for _ in range(2))
    params = dict(model.named_parameters())
    leaf = x.clone().requires_grad_()
    every = dict(zip(['x'] + list(params), torch.autograd.grad(model(leaf), [leaf] + list(params.values()), dy)))
    for n, p in params.items():
        p.requires_grad_(n in wanted)
    leaf = x.clone().requires_grad_('x' in wanted)
    torch._dynamo.reset()   # (every case is another graph of the same code)
    fn = torch.compile(model, fullgraph=True) if compiled else model
    fn(leaf)   # (compiled, warmed up)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    y = fn(leaf)
    kept = torch.cuda.memory_allocated() - before
    _native.lib().wind_rwkv7_profile_enable(1)
    try:
        got = dict(zip(wanted, torch.autograd.grad(y, [leaf if n == 'x' else params[n] for n in wanted], dy)))
        import ctypes
        ran = _native.lib().wind_rwkv7_profile_read(1, (ctypes.c_float * 16)(), 16)
    finally:
        _native.lib().wind_rwkv7_profile_enable(0)
    assert (ran > 0) == (wanted != ('Wo',))   # kernels of the recurrence's backward
    for n in wanted:
        assert seq_ref.rel_err(got[n].float().cpu(), every[n].float().cpu()) <= 1e-5, n
    if wanted == ('Wo',):
        assert kept <= 2 * x.numel() * 2 + 4096         # the output and what the projection multiplied
        if not compiled:
            assert got['Wo'].untyped_storage().nbytes() == 4 * C * C


@pytest.mark.parametrize('mixed', [False, True])
def test_gradients_of_bf16_parameters_are_converted_once(mixed):
    model, gen = _small_model(128, 2, torch.bfloat16)
    if mixed:
        model.ln_x.float()
    x, dy = (torch.randn(2, 32, 128, generator=gen).bfloat16().to(DEV) for _ in range(2))
    params = list(model.parameters())
    grads = torch.autograd.grad(model(x), params, dy)
    assert all(g.dtype == p.dtype and g.shape == p.shape and g.is_contiguous() for g, p in zip(grads, params))
    assert len({g.untyped_storage().data_ptr() for g in grads}) == (2 if mixed else 1)
    for p in params:
        p.data = p.data.float()
    for a, b in zip(grads, torch.autograd.grad(model(x), params, dy)):
        assert torch.equal(a, b.to(a.dtype))


@pytest.mark.parametrize('T', [1024, 1003])
def test_memory_of_a_pass_without_gradients(T):
    """Nine planes of activations, what the output projection multiplies, the output, the LoRA activations, the recurrence's
    scratch and the weights' copies; a ragged prompt also its padded input and the sequences it does not cut in place.  (All
    planes held to the end: 3.5 planes more.)"""
    from wind_rwkv import _native
    B, C, H = 2, 768, 12
    model, gen = _small_model(C, H, torch.float32)
    x = torch.randn(B, T, C, generator=gen).bfloat16().to(DEV)
    Tp = -(-T // 16) * 16
    plane = 2 * B * Tp * C
    saved = _native.lib().wind_rwkv7_attn_ln_saved_bytes(B, Tp, H, 64) + _native.lib().wind_rwkv7_attn_ln_fwd_workspace_bytes(B, Tp, H, 64)
    weights = 2 * sum(p.numel() for p in model.parameters()) + 12 * C
    loras = 2 * B * Tp * (8 * 32 + 128 + 64 + 64)
    with torch.no_grad():
        model(x, return_state=True)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        model(x, return_state=True)
        peak = torch.cuda.max_memory_allocated() - base
    assert peak <= (11 + (T != Tp)) * plane + saved + weights + loras + 4 * B * H * 4096 + 3 * 32 * B * C + (2 << 20)


@pytest.mark.parametrize('stage', ['ddlerp', 'expand_loras', 'block'])
def test_float32_parameters_may_be_written_to_before_the_backward_pass(stage):
    """What a backward pass multiplies with is the bf16 copies that the forward made, as in the Python Functions: an optimizer
    step or a swap of weights in between changes nothing and is no error."""
    from wind_rwkv.rwkv7 import ddlerp, expand_loras
    model, gen = _small_model(128, 2, torch.float32)
    x = torch.randn(2, 32, 128, generator=gen).bfloat16().to(DEV)
    a16 = torch.randn(2, 32, 16, generator=gen).bfloat16().to(DEV)
    names = {'ddlerp': ('time_maa_x', 'time_maa_w1', 'time_maa_w2', 'time_maa'), 'expand_loras': EXPANSION,
             'block': [n for n, _ in model.named_parameters()]}[stage]
    params = [dict(model.named_parameters())[n] for n in names]
    leaf = x.clone().requires_grad_()
    grads = []
    for write in (False, True):
        y = {'ddlerp': lambda: ddlerp(leaf, *params), 'expand_loras': lambda: expand_loras(leaf, x, a16, a16, a16, a16, *params, 64),
             'block': lambda: (model(leaf),)}[stage]()
        if write:
            with torch.no_grad():
                for p in params:
                    p.mul_(2)
        grads.append(torch.autograd.grad(y, [leaf] + params, [x] * len(y)))
    for a, b in zip(*grads):
        assert torch.equal(a, b)


def test_errors_of_the_library_keep_their_class_and_code(tmp_path):
    """With a library in the kernels' place that does nothing but return codes: the forward's error out of the call, the
    backward's out of autograd."""
    import ctypes
    import subprocess
    from wind_rwkv import _native
    from wind_rwkv.rwkv7 import attn
    codes = {'wind_rwkv7_attn_prefill': 5, 'wind_rwkv7_attn_backward': 7}
    source = ['#include <stddef.h>']
    for name, (res, _) in _native.SIGNATURES.items():
        kind, value = {ctypes.c_char_p: ('const char*', '"nothing here"'), ctypes.c_size_t: ('size_t', 256)}.get(res, ('int', codes.get(name, 0)))
        source.append(f'{kind} {name}() {{ return {value}; }}')
    (tmp_path / 'stub.c').write_text('\n'.join(source))
    subprocess.run(['cc', '-shared', '-fPIC', '-w', '-o', str(tmp_path / 'stub.so'), str(tmp_path / 'stub.c')], check=True)
    x = torch.zeros(1, 16, 64, dtype=torch.bfloat16, device=DEV)
    _native.binding().load(str(tmp_path / 'stub.so'), _native.WindRwkv7Error)
    try:
        for _ in range(2):   # (nothing is left over from an error)
            with torch.no_grad(), pytest.raises(_native.WindRwkv7Error, match='nothing here') as info:
                attn(x, x, x, x, x, x, 64)
            assert info.value.code == 5
            y = attn(x.clone().requires_grad_(), x, x, x, x, x, 64)
            with pytest.raises(_native.WindRwkv7Error, match='nothing here') as info:
                y.sum().backward()
            assert info.value.code == 7
    finally:
        _native.binding().load(_native.LIB_PATH, _native.WindRwkv7Error)
