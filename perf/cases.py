"""Timed passes of the RWKV-7 time mixer, each through the package's public entry points.

A case is a plain dict; its "kind" says which entry points one pass calls:

  step      TimeMixer.step: one token for each of B sequences (token-by-token generation)
  prompt    TimeMixer(x, return_state=True) under no_grad: a prompt of any length, or its next piece (`continued`)
  block     TimeMixer forward + backward, the training step of one block
  attn      WKV7 forward + backward on bf16 sequences, head size 64; `state`: from a carried state, whose gradient and
            that of the final state belong to the pass
  attn_ln   WKV7 with the GroupNorm + bonus + gate epilogue, forward + backward; `state`: from a carried state
  attn_f32  WKV7 forward + backward on float32 sequences (the accuracy mode)
  bighead   attn_triton_bighead(dot_prec='bf16') forward + backward: head sizes other than 64
  stages    ddlerp and expand_loras, forward + backward: the block's two elementwise stages as operators

Sizes follow the benchmark configurations (768 channels as 12 heads of 64 at B = 8 or 64, T = 1024; 32 heads at
T = 16384; B = 1, T = 256, 4 heads) and the ranges of the tests.
"""
import os
import sys
from collections import namedtuple

import torch

PACKAGE = os.path.join(os.getcwd(), 'wind-rwkv7_amd')
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

from wind_rwkv.rwkv7 import TimeMixer, attn, attn_ln, attn_triton_bighead, ddlerp, expand_loras  # noqa: E402

DEV = 'cuda'
Config = namedtuple('Config', ['n_layer', 'n_head', 'n_embd'])
F = torch.nn.functional


def listed():
    return [
        # generation for one user: nothing but launches and latency
        {'name': 'step_one', 'kind': 'step', 'B': 1, 'H': 12, 'N': 64},
        # generation for a full serving batch: the states and the products both count
        {'name': 'step_batch', 'kind': 'step', 'B': 256, 'H': 12, 'N': 64},
        # two prompts of a length that is no multiple of anything, ahead of generation
        {'name': 'prompt_ragged', 'kind': 'prompt', 'B': 2, 'T': 1003, 'H': 12, 'N': 64, 'continued': False},
        # one block of a 124M-parameter model in training, the benchmark's batch
        {'name': 'block_train', 'kind': 'block', 'B': 8, 'T': 1024, 'H': 12, 'N': 64},
        # the smallest training call of the configurations: latency and host work
        {'name': 'attn_small', 'kind': 'attn', 'B': 1, 'T': 256, 'H': 4, 'state': False},
        # the headline configuration
        {'name': 'attn_train', 'kind': 'attn', 'B': 8, 'T': 1024, 'H': 12, 'state': False},
        # the same at the batch that fills the card
        {'name': 'attn_train_large', 'kind': 'attn', 'B': 64, 'T': 1024, 'H': 12, 'state': False},
        # long context: one sequence, few heads, from a carried state
        {'name': 'attn_long', 'kind': 'attn', 'B': 1, 'T': 16384, 'H': 32, 'state': True},
        # the fused operator that the block calls, at the benchmark's batch
        {'name': 'attn_ln_train', 'kind': 'attn_ln', 'B': 8, 'T': 1024, 'H': 12, 'state': False},
        # the accuracy mode at the headline shape
        {'name': 'attn_float32', 'kind': 'attn_f32', 'B': 8, 'T': 1024, 'H': 12, 'N': 64},
        # the same 768 channels as 6 large heads
        {'name': 'bighead_train', 'kind': 'bighead', 'B': 8, 'T': 1024, 'H': 6, 'N': 128},
        # token shift and LoRA expansion at the block's shape, an odd batch and length
        {'name': 'stages_ragged', 'kind': 'stages', 'B': 7, 'T': 1008, 'H': 12, 'N': 64, 'mix_rank': 32, 'rank': 16},
    ]


def _log_int(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm."""
    return max(lo, min(hi, int(lo * ((hi + 1) / lo) ** rng.random())))


def _batch_and_length(rng, tokens, longest, most, shortest=16):
    """B and T (a multiple of 16) with about `tokens` in all."""
    T = 16 * _log_int(rng, shortest // 16, max(shortest, min(longest, tokens)) // 16)
    return max(1, min(most, tokens // T)), T


def draw(rng):
    kind = rng.choice(['step', 'prompt', 'block', 'attn', 'attn_ln', 'attn_f32', 'bighead', 'stages'])
    if kind == 'step':
        return {'kind': kind, 'B': _log_int(rng, 1, 512), 'H': rng.randint(3, 32), 'N': 64}
    if kind == 'prompt':
        T = _log_int(rng, 1, 4096)
        return {'kind': kind, 'B': _log_int(rng, 1, max(1, min(8, 8192 // T))), 'T': T, 'H': rng.randint(3, 24), 'N': 64,
                'continued': rng.random() < 0.5}
    if kind == 'block':
        H = rng.randint(3, 24)
        B, T = _batch_and_length(rng, _log_int(rng, 256, min(32768, 8192 * 144 // (H * H))), 4096, 64, 128)
        return {'kind': kind, 'B': B, 'T': T, 'H': H, 'N': 64}
    if kind in ('attn', 'attn_ln'):
        H = rng.randint(1, 32)
        B, T = _batch_and_length(rng, max(16, _log_int(rng, 1024, 786432 if kind == 'attn' else 524288) // H), 16384, 64,
                                 16 if kind == 'attn' else 128)
        # (attn_ln over very many sequences from a zero state: some of their first tokens are always ill conditioned)
        return {'kind': kind, 'B': B, 'T': T, 'H': H, 'state': rng.random() < (0.3 if kind == 'attn' else 0.6) or (kind == 'attn_ln' and B * H > 128)}
    if kind == 'attn_f32':
        N = rng.choice([64, 64, 64, 32, 96, 128])
        H = rng.randint(1, 16)
        B, T = _batch_and_length(rng, max(16, _log_int(rng, 256, 98304) * 64 // (H * N)), 65536 // max(N, 64), 32)
        return {'kind': kind, 'B': B, 'T': T, 'H': H, 'N': N}
    if kind == 'bighead':
        N = rng.choice([16, 32, 48, 80, 96, 112, 128, 128, 128])
        H = rng.randint(1, 16)
        B, T = _batch_and_length(rng, max(16, _log_int(rng, 512, 98304) * 64 // (H * N)), 2048, 32)
        return {'kind': kind, 'B': B, 'T': T, 'H': H, 'N': N}
    H = rng.randint(1, 32)
    B, T = _batch_and_length(rng, max(16, _log_int(rng, 512, 98304) // H), 4096, 64)
    return {'kind': kind, 'B': B, 'T': T, 'H': H, 'N': 64, 'mix_rank': rng.choice([32, 32, 64]), 'rank': rng.choice([16, 16, 32, 64])}


class _Normal:
    """Seeded values on the device."""

    def __init__(self, seed):
        self.gen = torch.Generator(DEV).manual_seed(seed)

    def __call__(self, *shape):
        return torch.randn(*shape, generator=self.gen, device=DEV)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.gen, device=DEV)


def _wkv7_inputs(rn, B, T, H, N, dtype):
    """r, w, k, v, a, b [B,T,H*N] as the time mixer makes them: w = -softplus(.) - 0.5, a = -kk, b = kk * sigmoid(.)
    with kk of unit length per head."""
    q, k, v = rn(B, T, H, N), rn(B, T, H, N), rn(B, T, H, N)
    w = -F.softplus(-rn(B, T, H, N)) - 0.5
    kk = F.normalize(rn(B, T, H, N), dim=-1)
    seqs = (q, w, k, v, -kk, kk * torch.sigmoid(rn(B, T, H, N)))
    return [t.reshape(B, T, H * N).to(dtype).contiguous() for t in seqs]


def _model(rn, H, N):
    """A TimeMixer with mix parameters ~ U(0,1), LoRA weights ~ 0.02 N(0,1), projections ~ N(0, 1/C); the remaining
    vectors keep their deterministic initialisation.  float32 master weights."""
    C = H * N
    model = TimeMixer(Config(12, H, C), 6).to(DEV)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name in ('time_maa_x', 'time_maa'):
                p.copy_(rn.uniform(*p.shape))
            elif name in ('Wr', 'Wk', 'Wv', 'Wo'):
                p.copy_(rn(*p.shape) * C ** -0.5)
            elif name.endswith('_w1') or name.endswith('_w2'):
                p.copy_(rn(*p.shape) * 0.02)
    return model


def _leaves(tensors):
    return [t.detach().requires_grad_() for t in tensors]


def prepare(case, seed):
    rn = _Normal(seed)
    kind, B, H = case['kind'], case['B'], case['H']
    N = case.get('N', 64)
    C, T = H * N, case.get('T')
    if kind in ('step', 'prompt'):
        s = {'model': _model(rn, H, N)}
        # a state that a sequence leaves behind: the last token, and sums of decayed outer products
        state = (rn(B, C).bfloat16(), rn(B, H, N, N) * 0.5)
        if kind == 'step':
            s.update(x=rn(B, C).bfloat16(), state=state)
        else:
            s.update(x=rn(B, T, C).bfloat16(), state=state if case['continued'] else None)
    elif kind == 'block':
        model = _model(rn, H, N)
        s = {'model': model, 'x': rn(B, T, C).bfloat16().requires_grad_(), 'dy': rn(B, T, C).bfloat16()}
        s['dy'][:, 0] = 0   # no loss on the opening token: its GroupNorm, after a zero state, is ill conditioned
        s['leaves'] = [s['x']] + list(model.parameters())
    elif kind in ('attn', 'attn_ln', 'attn_f32', 'bighead'):
        dtype = torch.float32 if kind == 'attn_f32' else torch.bfloat16
        seqs = _wkv7_inputs(rn, B, T, H, N, dtype)
        if kind == 'attn_ln' and not case['state']:
            # after a zero state the first output is (k.r) v: where k.r is near zero its GroupNorm is ill conditioned and
            # no two bf16 results agree, so the first token's k and r point the same way
            seqs[2][:, 0] = seqs[0][:, 0]
        s = {'seqs': _leaves(seqs), 'dy': rn(B, T, C).to(dtype)}
        if kind == 'attn_ln':
            s['g'] = rn(B, T, C).bfloat16().requires_grad_()
            s['params'] = torch.stack([1 + 0.1 * rn(C), 0.1 * rn(C), 0.1 * rn(C)]).requires_grad_()
            s['s0'] = rn(B, H, N, N) * 0.5 if case['state'] else None
        elif case.get('state'):
            s['s0'] = (rn(B, H, N, N) * 0.1).requires_grad_()
            s['dsT'] = rn(B, H, N, N) * 0.1
    else:
        D, M = case['rank'], case['mix_rank']
        s = {'mix': _leaves([rn(B, T, C).bfloat16(), rn.uniform(C), rn(4 * M, C) * 0.02, rn(4, C, M) * 0.02, rn.uniform(4, 1, 1, C)]),
             'expand': _leaves([rn(B, T, C).bfloat16() for _ in range(2)] + [rn(B, T, D).bfloat16() for _ in range(4)]
                               + [rn(C, D) * 0.1 for _ in range(4)] + [rn(C) for _ in range(4)]),
             'dmix': [rn(B, T, C).bfloat16() for _ in range(4)], 'dexpand': [rn(B, T, C).bfloat16() for _ in range(4)]}
    s['case'] = case
    return s


def run(s):
    case = s['case']
    kind, N = case['kind'], case.get('N', 64)
    if kind == 'step':
        y, s['state'] = s['model'].step(s['x'], s['state'])
        return y, s['state']
    if kind == 'prompt':
        with torch.no_grad():
            return s['model'](s['x'], state=s['state'], return_state=True)
    if kind == 'block':
        y = s['model'](s['x'])
        return (y,) + torch.autograd.grad(y, s['leaves'], s['dy'])
    if kind == 'stages':
        ys = ddlerp(*s['mix'])
        zs = expand_loras(*s['expand'], N)
        return (ys, zs, torch.autograd.grad(ys, s['mix'], s['dmix']), torch.autograd.grad(zs, s['expand'], s['dexpand']))
    if kind == 'attn_ln':
        y = attn_ln(*s['seqs'], s['g'], s['params'], N, s0=s['s0'])
        return (y,) + torch.autograd.grad(y, s['seqs'] + [s['g'], s['params']], s['dy'])
    if kind == 'bighead':
        y = attn_triton_bighead(*s['seqs'], N, dot_prec='bf16')
    elif 's0' in s:
        y, sT = attn(*s['seqs'], N, s0=s['s0'], return_state=True)
        return (y, sT) + torch.autograd.grad([y, sT], s['seqs'] + [s['s0']], [s['dy'], s['dsT']])
    else:
        y = attn(*s['seqs'], N)
    return (y,) + torch.autograd.grad(y, s['seqs'], s['dy'])


def _block_parameters(C):
    """(weights of the matrix products, vector parameters) of one TimeMixer: the four projections, the mix LoRA (4 x 32),
    gate 128, decay 64 and four of rank 16, each with two factors; mix (5), decay, bonus, three biases, GroupNorm (2)."""
    return 4 * C * C + 2 * C * (4 * 32 + 128 + 64 + 4 * 16), 12 * C


def work(case):
    """Bytes: the forward and the backward are two calls, so each reads its inputs and writes its outputs once (a
    backward also reads the forward's inputs).  Flops: the matrix products, and per token and head of the recurrence
    8 N^2 forward (state times a, two outer products, state times r) and twice that backward."""
    kind, B, H = case['kind'], case['B'], case['H']
    N, T = case.get('N', 64), case.get('T', 1)
    C = H * N
    rows = B * T
    scan = 8 * N * N * H * rows
    state = 4 * B * H * N * N
    weights, vectors = _block_parameters(C)
    if kind == 'step':        # the kept weights are bf16; the state is updated in place
        return {'bytes': 2 * weights + 4 * vectors + 2 * state + 3 * 2 * B * C, 'flops': 2 * weights * B + scan}
    if kind == 'prompt':
        return {'bytes': 4 * (weights + vectors) + state * (2 if case['continued'] else 1) + 2 * 2 * rows * C,
                'flops': 2 * weights * rows + scan}
    if kind == 'block':       # forward: x, parameters, y; backward: x, dy, parameters, dx, their gradients
        return {'bytes': 3 * 4 * (weights + vectors) + 5 * 2 * rows * C, 'flops': 6 * weights * rows + 3 * scan}
    if kind == 'stages':
        D, M = case['rank'], case['mix_rank']
        wide = 5 + 6 + 6 + 8   # ddlerp: x, 4 y | x, 4 dy, dx;  expand_loras: 2 in, 4 out | 2 in, 4 dy, 2 gradients
        return {'bytes': 2 * rows * (wide * C + 3 * 4 * D) + 3 * 4 * (8 * M * C + 5 * C + 4 * D * C + 4 * C),
                'flops': 6 * rows * C * (8 * M + 4 * D)}
    width = 4 if kind == 'attn_f32' else 2
    passes = 23 if kind == 'attn_ln' else 20
    return {'bytes': passes * width * rows * C + ((state if kind == 'attn_ln' else 4 * state) if case.get('state') else 0), 'flops': 3 * scan}


def tolerance(case):
    """bf16 sequences and bf16 matrix operands with fp32 sums: half a unit in the last place is 2e-3 of a value, and a
    gradient passes several roundings in a row, each implementation with its own (float32 kernels on the same values
    differ from bf16 ones by 5e-3).  A GroupNorm divides by the spread of a token's outputs, which for a few tokens near
    the start of a sequence is small: single values there, and through them a whole gradient, move further."""
    kind = case['kind']
    if kind == 'attn_f32':
        return {'rel': 1e-5}
    if kind in ('attn_ln', 'block'):
        return {'rel': 2e-2, 'max': 0.99}
    return {'rel': 1e-2}
