"""Grouped products (wind_rwkv7_linear_group) and packed weights (wind_rwkv7_pack_weights) through the C ABI.

Inputs are bf16, sums are fp32, results are rounded to bf16 once: within 2^-9 of each value plus the fp32 sums' error, so
4e-3 in norm; tanh and its derivative are applied to the rounded value and rounded again."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _problem(segments, pieces):
    from wind_rwkv import _native
    p = _native.Linear()
    for g, (A, W) in enumerate(segments):
        p.A[g], p.W[g], p.lda[g], p.ldw[g], p.K[g] = A.data_ptr(), W.data_ptr(), A.stride(0), W.stride(0), A.shape[1]
        p.N = W.shape[0]
    p.npieces = len(pieces)
    for t, (out, op, aux) in enumerate(pieces):
        p.out[t], p.ld_out[t], p.width[t], p.op[t] = out.data_ptr(), out.stride(0), out.shape[1], op
        p.aux[t] = None if aux is None else aux.data_ptr()
    return p


def _pad_and_pack(x, T_out):
    from wind_rwkv import _native
    B, T, C = x.shape
    a = torch.randn(80, 192, device=DEV)
    dst, out, last = torch.zeros(80, 192, device=DEV, dtype=torch.bfloat16), torch.full((B, T_out, C), 7., device=DEV, dtype=torch.bfloat16), torch.empty_like(x[:, 0])
    arr = (_native.Pack * 1)()
    p = arr[0]
    p.src, p.dst, p.rows, p.cols, p.src_dtype, p.dst_dtype, p.dstT, p.ldT = a.data_ptr(), dst.data_ptr(), 80, 192, _native.F32, _native.BF16, None, 0
    _native.check(_native.lib().wind_rwkv7_pack_weights_pad_rows(1, arr, B, T, T_out, C, x.data_ptr(), out.data_ptr(), last.data_ptr(),
                                                                 torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return torch.equal(dst, a.bfloat16()), out, last


@pytest.mark.parametrize('B,T,T_out,C', [(1, 1, 16, 8), (3, 33, 48, 72), (2, 1003, 1008, 768)])
def test_rows_padded_beside_packed_weights(B, T, T_out, C):
    x = torch.randn(B, T, C, device=DEV).bfloat16()
    packed, out, last = _pad_and_pack(x, T_out)
    assert packed and torch.equal(out[:, :T], x) and not out[:, T:].any() and torch.equal(last, x[:, -1])


def _run(problems, M):
    from wind_rwkv import _native
    arr = (_native.Linear * len(problems))(*problems)
    _native.check(_native.lib().wind_rwkv7_linear_group(len(problems), M, arr, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30))


# one tile and less, tile edges in every direction, K tails (16, 48, 96), each tile shape: 64 x 64 .. 64 x 192 on four stages, 64 and
# 128 tokens on two
@pytest.mark.parametrize('M,N,K', [(1, 16, 16), (16, 16, 16), (33, 48, 80), (64, 192, 64), (65, 208, 96), (129, 64, 768),
                                   (515, 768, 768), (2006, 768, 128), (2006, 2304, 96), (8200, 400, 80), (16, 2048, 2048)])
def test_one_product(M, N, K):
    gen = torch.Generator().manual_seed(M + N + K)
    A, W = (torch.randn(*s, generator=gen).bfloat16().to(DEV) for s in ((M, K), (N, K)))
    out = torch.full((M, N), float('nan'), device=DEV, dtype=torch.bfloat16)
    _run([_problem([(A, W)], [(out, 0, None)])], M)
    assert _rel(out, A.float() @ W.float().T) <= 4e-3
    # a one-hot row picks a row of W exactly: which column of A meets which column of W, and where the result goes
    A.zero_()
    A[M // 2, K - 1] = 1
    _run([_problem([(A, W)], [(out, 0, None)])], M)
    want = torch.zeros_like(out)
    want[M // 2] = W[:, K - 1]
    assert torch.equal(out, want)


@pytest.mark.parametrize('M', [7, 300, 5000])
def test_group_with_two_segments_and_cut_columns(M):
    gen = torch.Generator().manual_seed(M)
    rn = lambda *s: torch.randn(*s, generator=gen).bfloat16().to(DEV)
    wide = rn(M, 256)
    A, A2, W, W2 = wide[:, 64:160], rn(M, 128), rn(96, 96), rn(96, 128)      # a strided input
    target = torch.full((M, 160), 7.0, device=DEV, dtype=torch.bfloat16)      # columns of a wider output
    outs = [target[:, 16:80], torch.empty(M, 16, device=DEV, dtype=torch.bfloat16), target[:, 96:112]]
    aux, B, V, plain = rn(M, 16), rn(M, 32), rn(768, 32), torch.empty(M, 768, device=DEV, dtype=torch.bfloat16)
    _run([_problem([(A, W), (A2, W2)], [(outs[0], 1, None), (outs[1], 0, None), (outs[2], 2, aux)]),
          _problem([(B, V)], [(plain, 0, None)])], M)
    ref = A.float() @ W.float().T + A2.float() @ W2.float().T
    assert _rel(outs[0], torch.tanh(ref[:, :64])) <= 6e-3 and _rel(outs[1], ref[:, 64:80]) <= 4e-3
    assert _rel(outs[2], ref[:, 80:] * (1 - aux.float() ** 2)) <= 6e-3 and _rel(plain, B.float() @ V.float().T) <= 4e-3
    assert bool((target[:, :16] == 7).all() and (target[:, 80:96] == 7).all() and (target[:, 112:] == 7).all())


def _steps(x):
    """The distance of neighbouring bf16 values at x (float64)."""
    return torch.exp2(torch.floor(torch.log2(x.abs().clamp_min(2.0 ** -126))) - 7)


# the two sides of the series' line among them, in every column of a tile; 64 tokens and 128 of it
@pytest.mark.parametrize('tokens', [510, 20400])
def test_tanh_of_every_finite_bf16_value(tokens):
    """W = 1, so the sums are the inputs: tanh is the bf16 value nearest to its own in 64 bits.  (That is never closer to the middle between
    two of them than 8e-6 of itself, so the step through 32 bits that torch's conversion takes does not matter.)"""
    values = torch.arange(0, 65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    values = values[values.isfinite()]
    A = values.repeat(-(-tokens * 128 // values.numel()))[:tokens * 128].view(tokens, 128).contiguous().to(DEV)
    assert tokens * 128 >= values.numel()
    eye = torch.eye(128, device=DEV, dtype=torch.bfloat16)
    out, plain = torch.empty_like(A), torch.empty(tokens, 64, device=DEV, dtype=torch.bfloat16)
    _run([_problem([(A, eye)], [(out[:, :64], 1, None), (out[:, 64:], 1, None)]), _problem([(A[:, :64], eye[:64, :64])], [(plain, 0, None)])], tokens)
    assert torch.equal(plain, A[:, :64])
    assert torch.equal(out, torch.tanh(A.double()).bfloat16())


# columns to one, two and four tensors: the derivative's operands are read four columns a lane
@pytest.mark.parametrize('M', [1, 33, 129, 2500])
@pytest.mark.parametrize('widths', [(16,), (16, 32), (64, 48, 16, 80)])
def test_derivative_in_every_column(M, widths):
    gen = torch.Generator().manual_seed(M + sum(widths))
    N = sum(widths)
    A = torch.randn(M, N, generator=gen).bfloat16().to(DEV)
    aux = [torch.rand(M, w, generator=gen).bfloat16().to(DEV) for w in widths]
    outs = [torch.full((M, w), float('nan'), device=DEV, dtype=torch.bfloat16) for w in widths]
    _run([_problem([(A, torch.eye(N, device=DEV, dtype=torch.bfloat16))], [(o, 2, y) for o, y in zip(outs, aux)])], M)
    want = A.double() * (1 - torch.cat(aux, 1).double() ** 2)
    assert bool(((torch.cat(outs, 1).double() - want).abs() <= 0.501 * _steps(want) + 2.0 ** -22 * A.double().abs()).all())


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('off', [0, 1])
def test_packed_weights(dtype, off):
    """`off`: elements that the sources start off a 16-byte boundary."""
    from wind_rwkv import _native
    gen = torch.Generator().manual_seed(3)
    a, b, v = (torch.cat([torch.zeros(off), torch.randn(s[0] * s[1], generator=gen)]).to(DEV, dtype)[off:].view(s) for s in ((16, 192), (80, 192), (1, 208)))
    assert all((t.data_ptr() % 16 == 0) == (off == 0) for t in (a, b, v))
    dst = [torch.zeros(t.shape, device=DEV, dtype=torch.bfloat16) for t in (a, b)] + [torch.zeros(v.shape, device=DEV)]
    both = torch.zeros(192, 96, device=DEV, dtype=torch.bfloat16)             # the transposed concatenation [a; b]
    arr = (_native.Pack * 3)()
    for p, s, d in zip(arr, (a, b, v), dst):
        p.src, p.dst, p.rows, p.cols = s.data_ptr(), d.data_ptr(), *s.shape
        p.src_dtype, p.dst_dtype = (_native.F32 if t.dtype == torch.float32 else _native.BF16 for t in (s, d))
    arr[0].dstT, arr[0].ldT, arr[1].dstT, arr[1].ldT = both.data_ptr(), 96, both[:, 16:].data_ptr(), 96
    _native.check(_native.lib().wind_rwkv7_pack_weights(3, arr, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(dst[0], a.bfloat16()) and torch.equal(dst[1], b.bfloat16()) and torch.equal(dst[2], v.float())
    assert torch.equal(both, torch.cat([a, b]).bfloat16().T)


def test_arguments_are_checked_on_the_host():
    from wind_rwkv import _native
    lib, x = _native.lib(), torch.zeros(64, 64, device=DEV, dtype=torch.bfloat16)
    call = lambda p, n=1, M=64: lib.wind_rwkv7_linear_group(n, M, (_native.Linear * 1)(p), None)
    good = lambda: _problem([(x, x)], [(x, 0, None)])
    for change, code in ((dict(N=48), 2), (dict(N=0), 2), (dict(npieces=0), 2), (dict(npieces=5), 2)):
        p = good()
        for k, val in change.items():
            setattr(p, k, val)
        assert call(p) == code, change
    assert call(good(), n=0) == 2 and call(good(), M=0) == 2
    for field, val, code in (('K', 24, 9), ('lda', 60, 2), ('ldw', 68, 2), ('A', None, 1), ('A', x.data_ptr() + 8, 2), ('width', 24, 9),
                             ('out', None, 1), ('op', 3, 2), ('op', 2, 1), ('ld_out', 56, 2)):
        p = good()
        getattr(p, field)[0] = val
        assert call(p) == code, field
