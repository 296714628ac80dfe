"""A guard on the compiled kernels (no GPU needed: hipcc cross-compiles to assembly here).

This compiler release places no wait states between two matrix instructions of DIFFERENT shapes when the second takes
the first one's result as its accumulator (seen with v_mfma_f32_16x16x32_bf16 followed by v_mfma_f32_16x16x16_bf16:
emitted back to back, and the triangular inverse built that way came out wrong by 1e-3 on the GPU).  The sources
therefore never chain shapes through the accumulator; this test scans the assembly of every kernel file that uses
matrix instructions for such a pair, so that a later edit cannot reintroduce one unnoticed.
"""
import os
import re
import shutil
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, 'wind-rwkv7_amd', 'csrc')
HIPCC = shutil.which('hipcc') or '/opt/rocm/bin/hipcc'
MAKEFILE = os.path.join(ROOT, 'wind-rwkv7_amd', 'Makefile')


def makefile_flags():
    """(common flags, {file name: extra flags}) as the package's Makefile sets them, so that the assembly scanned here
    is that of the shipped objects: HIPFLAGS for every file, and the per-target `EXTRA := $(VAR)` lines."""
    text = open(MAKEFILE).read()
    var = dict(re.findall(r'^(\w+)\s*[:?]?=\s*(.*)$', text, flags=re.M))
    expand = lambda v: re.sub(r'\$\((\w+)\)', lambda m: expand(var.get(m.group(1), '')), v)
    common = [f for f in expand(var['HIPFLAGS']).split() if f != '-fPIC']
    extra = {}
    for targets, value in re.findall(r'^((?:build/\w+\.o\s*)+):\s*EXTRA\s*:=\s*(.*)$', text, flags=re.M):
        for t in targets.split():
            extra[os.path.basename(t)[:-2] + '.hip'] = expand(value).split()
    return common, extra


FLAGS, EXTRA = makefile_flags()
FLAGS = FLAGS + ['-S', '--cuda-device-only']
FILES = ['wkv7_fused.hip', 'wkv7_bwd.hip', 'wkv7_fwd.hip', 'wkv7_wide.hip', 'ddlerp.hip', 'expand_loras.hip', 'expand_loras16.hip', 'mixer_decode.hip',
         'linear_wgrad.hip', 'selftest.hip', 'wkv7_f32.hip', 'linear_group.hip', 'cast_bf16.hip', 'cols.hip']
WINDOW = 16   # instructions; a matrix instruction has long finished after that many

MFMA = re.compile(r'(v_mfma_\w+)\s+([av]\[\d+:\d+\]),\s*(?:[av]\[\d+:\d+\]|v\d+),\s*(?:[av]\[\d+:\d+\]|v\d+),\s*([av]\[\d+:\d+\]|0)')


DEST = re.compile(r'v_\w+\s+(v\d+|v\[\d+:\d+\])')


def _regs(operand):
    m = re.match(r'[av]\[(\d+):(\d+)\]', operand)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    return {int(operand[1:])}


def mixed_pairs(asm):
    ins = [t.strip() for t in asm.split('\n')]
    ins = [t for t in ins if t and not t.startswith((';', '.')) and not t.endswith(':')]
    found = []
    for i, t in enumerate(ins):
        m = MFMA.match(t)
        if not m or m.group(3) == '0':
            continue
        pending = _regs(m.group(3)) if m.group(3)[0] == 'v' else None   # accumulator registers not yet seen rewritten
        for j in range(i - 1, max(i - 1 - WINDOW, -1), -1):
            p = MFMA.match(ins[j])
            if p and p.group(2) == m.group(3):      # the producer of this instruction's accumulator
                if p.group(1) != m.group(1):
                    found.append((ins[j], t))
                break
            # a vector instruction in between that rewrites the whole accumulator range: the matrix instruction before
            # it is not what this one accumulates onto (the registers were merely reused)
            d = DEST.match(ins[j])
            if d and pending is not None and not p:
                pending -= _regs(d.group(1))
                if not pending:
                    break
    return found


class Flow:
    """Instructions and labels of an assembly listing in their order, and which may have run right before each."""

    def __init__(self, asm):
        self.ins, self.written_as_such = [], set()   # (the second: indices of what the sources write as assembly)
        inside = False
        for line in asm.split('\n'):
            if '#ASMSTART' in line or '#ASMEND' in line:
                inside = '#ASMSTART' in line
                continue
            t = line.split(';')[0].strip()
            if not t or (t.startswith('.') and not t.endswith(':')):   # (directives; labels stay)
                continue
            if inside:
                self.written_as_such.add(len(self.ins))
            self.ins.append(t)
        self.jumps = {}
        for i, t in enumerate(self.ins):
            m = re.match(r's_c?branch\S*\s+(\S+)', t)
            if m:
                self.jumps.setdefault(m.group(1) + ':', []).append(i)

    def before(self, i):
        """Indices of the instructions (no labels) that may have run right before instruction i."""
        found, seen, todo = set(), set(), [i]
        while todo:
            j = todo.pop()
            from_jumps = self.jumps.get(self.ins[j], []) if j != i else []
            above = [j - 1] if j > 0 and not re.match(r's_branch\b|s_endpgm|s_setpc', self.ins[j - 1]) else []
            for k in from_jumps + above:
                if k in seen:
                    continue
                seen.add(k)
                (todo.append if self.ins[k].endswith(':') else found.add)(k)
        return found

    def writers(self, i, regs, reach=None):
        """The vector instructions that may have written the vector registers `regs` last before instruction i, with the wait states
        between (those of another path from the same one: the fewest); `reach`: only those with fewer."""
        found, best, todo = {}, {}, [(i, 0, frozenset(regs))]
        while todo:
            j, waits, left = todo.pop()
            for k in self.before(j):
                t = self.ins[k]
                hit = left & written(t)
                if hit:
                    found[k] = min(waits, found.get(k, waits))
                rest = left - hit
                then = waits + 1 + (int(t.split()[1], 0) if t.startswith('s_nop') else 0)
                rest = frozenset(r for r in rest if best.get((k, r), then + 1) > then)
                best.update({(k, r): then for r in rest})
                if rest and (reach is None or then < reach):
                    todo.append((k, then, rest))
        return found


def written(t):
    """Vector registers that an instruction writes."""
    m = re.match(r'(v_\w+|ds_\w+|(?:global|buffer|flat|scratch)_load\w*)\s+(v\d+|v\[\d+:\d+\])(?:,\s*(v\d+))?', t)
    if not m or (m.group(1).startswith('ds_') and not re.match(r'ds_(read|bpermute|permute|swizzle)', t)) or re.search(r'\slds\b', t):
        return set()
    return _regs(m.group(2)) | (_regs(m.group(3)) if 'swap' in m.group(1) and m.group(3) else set())


def stores_of_matrix_results(asm):
    """Stores that the sources write as assembly, of registers that a matrix instruction wrote last (or at an address in such): the compiler
    keeps the distance which these need only for the stores that it makes itself."""
    f, found = Flow(asm), []
    for i in sorted(f.written_as_such):
        if re.match(r'(global|buffer|flat)_store', f.ins[i]):
            regs = set().union(*map(_regs, re.findall(r'\bv\d+\b|\bv\[\d+:\d+\]', f.ins[i])))
            found += [(f.ins[k], f.ins[i]) for k in f.writers(i, regs) if 'mfma' in f.ins[k]]
    return found


def test_scanner_sees_a_store_of_matrix_results():
    asm = '''
        v_mfma_f32_32x32x16_bf16 v[16:31], v[0:3], v[4:7], v[16:31]
        s_cbranch_scc1 .LBB0_2
        v_mov_b32_e32 v20, 0
    .LBB0_2:                                ; %some block
        v_lshl_add_u64 v[8:9], s[0:1], 0, v[10:11]
        ;;#ASMSTART
        global_store_dwordx4 v[8:9], v[20:23], off sc1
        s_nop 1
        ;;#ASMEND
        global_store_dwordx4 v[8:9], v[24:27], off
        s_endpgm
    '''
    assert len(stores_of_matrix_results(asm)) == 1
    assert not stores_of_matrix_results(asm.replace('v[20:23], off', 'v[32:35], off'))
    assert not stores_of_matrix_results(asm.replace('v_lshl_add', 'ds_read_b128 v[20:23], v4\nv_lshl_add'))
    assert stores_of_matrix_results(asm.replace('v_mov_b32_e32 v20, 0', 's_branch .LBB0_3'))   # (through the jump alone)


def early_lane_reads(asm):
    """v_fmac_f32_dpp instructions (written as such in the sources, so that the compiler does not place the two wait states a
    lane-crossing operand needs behind a vector instruction that writes it) with a writer of that operand less than two before them."""
    f, found = Flow(asm), []
    for i, t in enumerate(f.ins):
        m = re.match(r'v_fmac_f32_dpp v\d+, v(\d+),', t)
        if m:
            found += [(f.ins[k], t) for k, waits in f.writers(i, {int(m.group(1))}, reach=2).items() if waits < 2 and f.ins[k].startswith('v_')]
    return found


def test_scanner_sees_an_early_lane_read():
    asm = '''
        v_mul_f32_e32 v7, v1, v2
        v_add_f32_e32 v9, v1, v2
        v_fmac_f32_dpp v3, v7, v4 row_ror:8 row_mask:0xf bank_mask:0xf
    '''
    assert len(early_lane_reads(asm)) == 1 and not early_lane_reads(asm.replace('v_add', 's_nop 0\nv_add'))
    # the writer at the end of a loop, the reader right behind its label: the branch is one wait state, the label none
    loop = '''
        v_mov_b32_e32 v7, 0
        s_nop 1
    .LBB0_2:                                ; =>This Inner Loop Header: Depth=1
        v_fmac_f32_dpp v3, v7, v4 row_ror:8 row_mask:0xf bank_mask:0xf
        v_mul_f32_e32 v7, v1, v2
        s_cbranch_scc1 .LBB0_2
        s_endpgm
    '''
    assert [w for w, _ in early_lane_reads(loop)] == ['v_mul_f32_e32 v7, v1, v2']
    assert not early_lane_reads(loop.replace('s_cbranch', 's_add_u32 s0, s0, 1\ns_cbranch'))
    # and one that the code falls through to
    assert len(early_lane_reads(asm.replace('v_add_f32_e32 v9, v1, v2', '.LBB0_4:   ; %x'))) == 1


def test_flags_are_the_makefiles():
    assert '--offload-arch=gfx950' in FLAGS and '-O3' in FLAGS
    assert EXTRA['wkv7_fused.hip'] == ['-mllvm', '-amdgpu-mfma-vgpr-form'] and 'expand_loras.hip' not in EXTRA


def test_scanner_sees_a_mixed_pair():
    asm = '''
        v_mfma_f32_16x16x32_bf16 v[68:71], v[76:79], v[68:71], v[2:5]
        v_mfma_f32_16x16x16_bf16 v[66:69], v[66:67], v[72:73], v[68:71]
        v_mfma_f32_16x16x16_bf16 v[66:69], v[66:67], v[72:73], v[66:69]
    '''
    assert len(mixed_pairs(asm)) == 1
    reused = '''
        v_mfma_f32_16x16x16_bf16 v[56:59], v[24:25], v[252:253], 0
        v_cvt_pk_bf16_f32 v62, v56, v57
        v_and_b32_e32 v59, 0xffff0000, v43
        v_lshlrev_b32_e32 v58, 16, v43
        v_and_b32_e32 v57, 0xffff0000, v42
        v_lshlrev_b32_e32 v56, 16, v42
        v_mfma_f32_16x16x32_bf16 v[56:59], v[60:63], v[12:15], v[56:59]
    '''
    assert mixed_pairs(reused) == []       # the accumulator registers were rewritten in between
    partly = reused.replace('v_and_b32_e32 v59, 0xffff0000, v43', '')
    assert len(mixed_pairs(partly)) == 1   # one register still holds the first instruction's result


@pytest.fixture(scope='module')
def assembly():
    """[(file name, its assembly)]."""
    if not os.path.exists(HIPCC):
        pytest.skip('hipcc not found')
    with tempfile.TemporaryDirectory() as tmp:
        def compile_one(name):
            out = os.path.join(tmp, name + '.s')
            extra = EXTRA.get(name, [])
            subprocess.run([HIPCC, *FLAGS, *extra, '-o', out, os.path.join(CSRC, name)], check=True,
                           stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
            with open(out) as f:
                return name, f.read()
        with ThreadPoolExecutor(max_workers=4) as pool:
            return list(pool.map(compile_one, FILES))


def test_a_steps_linear_kernels_take_no_more_arguments_than_they_read(assembly):
    """The host writes a kernel's arguments for every launch, which bounds a step of few sequences: nine pairs of 32 bytes, the plan and
    the token shift's operands; one pair, the plan and a pointer for the output projection."""
    sizes = {}
    for size, name in re.findall(r'\.kernarg_segment_size:\s+(\d+)\n(?:.*\n)*?\s+\.name:\s+(\S+)', dict(assembly)['mixer_decode.hip']):
        m = re.search(r'decode_linear_kernelILb([01])E', name)
        if m:
            sizes.setdefault(m.group(1), set()).add(int(size))
    assert sizes == {'1': {64 + 9 * 32 + 48}, '0': {64 + 32 + 8}}


def test_no_matrix_instructions_of_different_shapes_chained_through_the_accumulator(assembly):
    results = assembly
    bad = {name: pairs[:3] for name, asm in results if (pairs := mixed_pairs(asm))}
    assert not bad, bad
    stored = {name: pairs[:3] for name, asm in results if (pairs := stores_of_matrix_results(asm))}
    assert not stored, stored
    assert sum(len(Flow(asm).written_as_such) for name, asm in results if name == 'linear_group.hip')   # (what the scan is for)
    early = {name: pairs[:3] for name, asm in results if (pairs := early_lane_reads(asm))}
    assert not early, early
    assert any('v_fmac_f32_dpp' in asm for _, asm in results)   # (what the scan is for)
    # The WKV7 kernels must not spill to scratch memory.  In the lock-step kernels a spilling wavefront holds up all
    # the others at every barrier; in the gradient kernel every reload of a spilled register makes the compiler wait
    # for ALL outstanding memory operations (scratch accesses count as loads of unknown order), which ends the overlap
    # of the next chunk's prefetch with this chunk's arithmetic.
    spilling = {}
    for name, asm in results:
        # (the fp32 kernels: their backward sits at the register limit of a wavefront, so a change that tips it over shows here)
        if name in ('wkv7_fused.hip', 'wkv7_bwd.hip', 'wkv7_fwd.hip', 'wkv7_f32.hip'):
            for kernel, size in re.findall(r'\.name:\s+(\S+)\n(?:.*\n)*?\s+\.private_segment_fixed_size:\s+(\d+)', asm):
                if int(size):
                    spilling[kernel] = int(size)
    assert not spilling, spilling
