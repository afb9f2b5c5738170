"""Hazards around the kernels' written-out instructions, read off the built library's own code.

The compiler keeps the wait states that its own instructions need and looks at no written-out ones
(csrc/mfma.h, mlp16.h, mlp_impl.h).  Checked, over every way that leads to an instruction (branches included):

* a copy global -> LDS reads its scalar address five wait states after a vector instruction wrote it, at least;
* no matrix instruction of the 16-bit MLP chains writes accumulation registers, which to_agpr writes without
  the compiler knowing what may still be in flight to them;
* a written-out vector instruction writes no register that a matrix instruction still in flight writes, and no
  matrix instruction reads its result within two wait states.
"""
import re
import shutil
import struct
import subprocess
from pathlib import Path

import pytest

from srf_hip import build

WRITTEN_OUT = ('v_accvgpr_write_b32', 'v_pk_min_u16', 'v_lshl_or_b32', 'v_mbcnt_lo_u32_b32', 'v_mbcnt_hi_u32_b32',
               'v_cndmask_b32')
# wait states from a matrix instruction to a vector instruction that writes the same register
IN_FLIGHT = {'16x16x32': 8, '32x32x16': 12, '16x16x4': 10}


def code_objects(data):
    """The GPU code objects of a host library (one bundle a source)."""
    at = data.find(b'__CLANG_OFFLOAD_BUNDLE__')
    while at >= 0:
        n, = struct.unpack_from('<Q', data, at + 24)
        o = at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from('<QQQ', data, o)
            if b'gfx' in data[o + 24:o + 24 + length] and size:
                yield data[at + off:at + off + size]
            o += 24 + length
        at = data.find(b'__CLANG_OFFLOAD_BUNDLE__', at + 24)


def regs(text):
    """Registers named by an operand: {('v', 3), ...}."""
    m = re.match(r'([sva])(\d+)$', text)
    if m:
        return {(m.group(1), int(m.group(2)))}
    m = re.match(r'([sva])\[(\d+):(\d+)\]$', text)
    return {(m.group(1), k) for k in range(int(m.group(2)), int(m.group(3)) + 1)} if m else set()


@pytest.fixture(scope='module')
def kernels(tmp_path_factory):
    """Kernel name -> (instructions, {index of an instruction: indexes of the branches to it})."""
    objdump = shutil.which('llvm-objdump') or '/opt/rocm/llvm/bin/llvm-objdump'
    if not (build.LIB_PATH.exists() and Path(objdump).exists()):
        pytest.skip('no built library or no llvm-objdump')
    out, name = {}, None
    for i, obj in enumerate(code_objects(build.LIB_PATH.read_bytes())):
        path = tmp_path_factory.mktemp('code') / f'{i}.co'
        path.write_bytes(obj)
        text = subprocess.run([objdump, '-d', f'--mcpu={build.ARCH}', str(path)], check=True, capture_output=True,
                              text=True).stdout
        for line in text.splitlines():
            head = re.match(r'[0-9a-f]+ <(.+)>:', line)
            ins = re.match(r'\s+(\S.*?)\s*// ([0-9A-F]+):', line)
            if head:
                name = head.group(1)
                out[name] = ([], [])
            elif name and ins:
                out[name][0].append(re.split(r'[\s,]+', ins.group(1)))
                out[name][1].append(int(ins.group(2), 16))
    assert len(out) > 100
    for name, (code, address) in out.items():
        at = {a: i for i, a in enumerate(address)}
        branches = {}
        for i, ins in enumerate(code):
            if re.match(r's_c?branch', ins[0]):
                words = int(ins[1])
                target = address[i] + 4 + 4 * (words - 65536 if words >= 32768 else words)
                branches.setdefault(at[target], []).append(i)
        out[name] = (code, branches)
    return out


def back(kernel, at, states):
    """(instruction, wait states between it and instruction `at`) of those up to `states` before it, on every way;
    send(True) ends the way that the last one lies on."""
    code, branches = kernel
    ways, seen = [(at, 0)], set()
    while ways:
        i, passed = ways.pop()
        for before in ([i - 1] if i and code[i - 1][0] not in ('s_branch', 's_endpgm') else []) + branches.get(i, []):
            if (before, passed) in seen:
                continue
            seen.add((before, passed))
            ins = code[before]
            if (yield ins, passed):
                continue
            more = passed + 1 + (int(ins[1], 0) if ins[0] == 's_nop' else 0)
            if more < states:
                ways.append((before, more))


def all_back(kernel, at, states, ends=lambda ins: False):
    walk, stop = back(kernel, at, states), None
    while True:
        try:
            ins, passed = walk.send(stop)
        except StopIteration:
            return
        stop = ends(ins)
        yield ins, passed


def test_copies(kernels):
    found = 0
    for name, kernel in kernels.items():
        for at, ins in enumerate(kernel[0]):
            if ins[0].startswith('global_load_lds') and regs(ins[2]):
                found += 1
                # a scalar copy of the address is kept in order with both sides
                copied = lambda before: before[0].startswith('s_mov') and regs(before[1]) == regs(ins[2])
                for before, _ in all_back(kernel, at, 5, copied):
                    assert not (before[0].startswith('v_') and regs(before[1]) & regs(ins[2])), (name, before, ins)
    assert found > 1000


def test_accumulation_registers_are_not_written_by_matrix_instructions(kernels):
    chains = {k: v for k, v in kernels.items() if 'mlp16_fwd' in k or 'mlp16_bwd' in k}
    assert len(chains) >= 12
    for name, (code, _) in chains.items():
        for ins in code:
            if ins[0].startswith('v_mfma'):
                assert ins[1].startswith('v'), (name, ins)


def test_vector_instructions(kernels):
    found = 0
    for name, kernel in kernels.items():
        if not any(ins[0].startswith('v_mfma') for ins in kernel[0]):
            continue
        for at, ins in enumerate(kernel[0]):
            if ins[0].startswith('v_mfma'):
                reads = set().union(*(regs(r) for r in ins[2:5]))
                for before, _ in all_back(kernel, at, 2):
                    assert not (before[0].startswith(WRITTEN_OUT) and regs(before[1]) & reads), (name, before, ins)
            elif ins[0].startswith(WRITTEN_OUT):
                found += 1
                for before, passed in all_back(kernel, at, 12):
                    if before[0].startswith('v_mfma') and regs(before[1]) & regs(ins[1]):
                        shape = re.search(r'(16x16x32|32x32x16|16x16x4)', before[0]).group(1)
                        assert passed >= IN_FLIGHT[shape], (name, before, ins, passed)
    assert found > 1000
