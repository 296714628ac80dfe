"""The entry point that allocates nothing: wind_rwkv7_attn_prefill_static keeps its scratch in a device array that is
part of the library, so a caller passes inputs and outputs only.  Checked through the C ABI against
wind_rwkv7_attn_prefill (caller-provided scratch) bit for bit, on calls in a row, each with a smaller input than the one before (the array keeps
the earlier call's contents).  A few heads run by records of their chunks in the array, long sequences on them as segments, whose
affine maps and entering states lie there; what needs no scratch are sequences of fewer than eight chunks and many heads."""
import pytest
import torch

from oracle import inputs

DEV = 'cuda'


def _run_pair(lib, _native, B, T, H, seed, slower=0.):
    C = 64
    d = inputs.wkv7_inputs(B, T, H, C, seed, dtype=torch.bfloat16)
    d['w'] = d['w'] - slower
    x = [d[n].to(DEV).contiguous() for n in ('w', 'q', 'k', 'v', 'a', 'b')]
    s0 = (torch.randn(B, H, C, C, generator=torch.Generator().manual_seed(seed)) * 0.3).to(DEV)
    stream = torch.cuda.current_stream().cuda_stream
    ptrs = [t.data_ptr() for t in x]
    # reference: the existing entry point with caller-provided scratch and workspace
    scratch = torch.empty(lib.wind_rwkv7_attn_saved_bytes(B, T, H, C), dtype=torch.uint8, device=DEV)
    ws = torch.empty(max(lib.wind_rwkv7_attn_fwd_workspace_bytes(B, T, H, C), 256), dtype=torch.uint8, device=DEV)
    y0, sT0 = torch.empty_like(x[3]), torch.empty_like(s0)
    _native.check(lib.wind_rwkv7_attn_prefill(B, T, H, C, _native.BF16, _native.F32, *ptrs, s0.data_ptr(), y0.data_ptr(),
                                              scratch.data_ptr(), sT0.data_ptr(), ws.data_ptr(), ws.numel(), stream))
    # under test: outputs allocated beforehand, nothing else passed
    y1, sT1 = torch.full_like(x[3], float('nan')), torch.full_like(s0, float('nan'))
    torch.cuda.synchronize()
    # neither the framework's allocator nor the device itself (an allocation made inside the library would only show
    # in the device's free bytes) may have handed out memory
    before, free_before = torch.cuda.memory_allocated(), torch.cuda.mem_get_info()[0]
    _native.check(lib.wind_rwkv7_attn_prefill_static(B, T, H, C, _native.BF16, _native.F32, *ptrs, s0.data_ptr(),
                                                     y1.data_ptr(), sT1.data_ptr(), stream))
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == before
    assert torch.cuda.mem_get_info()[0] >= free_before
    assert torch.equal(y0, y1) and torch.equal(sT0, sT1)
    assert torch.isfinite(y1.float()).all() and torch.isfinite(sT1).all()


@pytest.mark.gpu
def test_prefill_static_matches_prefill_on_two_calls_in_a_row():
    from wind_rwkv import _native
    lib = _native.lib()
    assert lib.wind_rwkv7_attn_prefill_static_bytes(1, 4096, 2, 64) > 0   # (also the array's address lookup)
    _run_pair(lib, _native, B=1, T=4096, H=2, seed=33)    # a long sequence on few heads as eight segments
    _run_pair(lib, _native, B=1, T=2048, H=1, seed=34)    # records; the array is dirty with the call before
    _run_pair(lib, _native, B=2, T=256, H=3, seed=31)     # records of 96 chunks
    _run_pair(lib, _native, B=1, T=64, H=2, seed=32)      # 8 chunks, one-kernel forward: no scratch touched


@pytest.mark.gpu
@pytest.mark.parametrize('B,T,H', [(1, 2048, 12), (1, 3200, 14), (1, 2576, 19)])
def test_prefill_static_takes_the_same_way_up_to_its_limit(B, T, H):
    """1536, 2800 and 3059 chunks: records of 20, 36 and 40 MiB; without them all three run in segments, whose states
    are composed in another order.  (Decays near one, exp(-exp(-7)) a token: else nothing is left of a state behind a segment.)"""
    from wind_rwkv import _native
    lib = _native.lib()
    assert lib.wind_rwkv7_attn_prefill_static_bytes(B, T, H, 64) <= 32 << 20
    assert lib.wind_rwkv7_attn_fwd_workspace_bytes(B, T, H, 64) == B * H * (T // 16) * 13568
    _run_pair(lib, _native, B, T, H, seed=T, slower=6.)


def test_the_array_holds_every_problem_within_the_limit():
    from wind_rwkv import _native
    lib = _native.lib()
    array, limit, seen = 44 << 20, 32 << 20, 0
    for heads in range(1, 3277):
        most = 3276 // heads
        for chunks in set(range(1, min(most, 40) + 1)) | set(range(most, 0, -max(1, most // 64))):
            if lib.wind_rwkv7_attn_prefill_static_bytes(1, 16 * chunks, heads, 64) <= limit:
                seen += 1
                assert lib.wind_rwkv7_attn_fwd_workspace_bytes(1, 16 * chunks, heads, 64) <= array, (chunks, heads)
    assert seen > 1000


def test_prefill_static_rejects_what_does_not_fit():
    """Host-side validation only: the limit is checked before anything touches a device."""
    from wind_rwkv import _native
    lib = _native.lib()
    limit = 32 << 20
    assert lib.wind_rwkv7_attn_prefill_static_bytes(2, 256, 3, 64) <= limit
    B, T, H = 8, 1024, 12
    assert lib.wind_rwkv7_attn_prefill_static_bytes(B, T, H, 64) > limit
    one = 1   # never dereferenced: validation fails first
    rc = lib.wind_rwkv7_attn_prefill_static(B, T, H, 64, _native.BF16, _native.F32, *([one] * 7), one, one, None)
    assert rc == 10 and b'scratch' in lib.wind_rwkv7_strerror(rc)
    assert lib.wind_rwkv7_attn_prefill_static(2, 250, 3, 64, _native.BF16, _native.F32, *([one] * 7), one, one, None) == 4
    assert lib.wind_rwkv7_attn_prefill_static(2, 256, 3, 64, _native.BF16, _native.F32, *([0] * 7), one, one, None) == 1
