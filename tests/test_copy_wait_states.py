"""Wait states of the written-out global -> LDS copies (csrc/mfma.h), read off the assembly of a small kernel.

A vector-memory instruction may read a scalar register five wait states after a vector instruction wrote it
at the earliest.  The compiler sees to that for its own instructions, not for written-out ones.
"""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from srf_hip import build

SOURCE = r"""
#include "mfma.h"
namespace srf {
// the address of a copy comes from a vector register directly before it
__global__ void copies(const uint8_t* base, const int* off, float* out) {
  __shared__ uint8_t buf[4096];
  const int lane = threadIdx.x & 63;
  lds_dma_1k(base + off[lane], buf);
  lds_dma_1k(base + off[lane + 64], buf + 1024);
  wait_vmem();
  out[lane] = buf[lane] + buf[1024 + lane];
}
}  // namespace srf
"""


def regs(text):
    """Scalar registers named in an operand."""
    m = re.match(r's\[(\d+):(\d+)\]$', text)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.match(r's(\d+)$', text)
    return {int(m.group(1))} if m else set()


def test_copies_wait_for_their_scalar_address(tmp_path):
    if not (shutil.which('hipcc') or Path('/opt/rocm/bin/hipcc').exists()):
        pytest.skip('no hipcc')
    src, asm = tmp_path / 'copies.hip', tmp_path / 'copies.s'
    src.write_text(SOURCE)
    subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, f'-I{build.CSRC_DIR}', '-w', '--cuda-device-only', '-S',
                    str(src), '-o', str(asm)], check=True, capture_output=True, text=True)
    code = [re.split(r'[\s,]+', line.split(';')[0].strip()) for line in asm.read_text().splitlines()
            if re.match(r'\t[sv]_|\tglobal_|\tds_', line)]
    found = 0
    for at, ins in enumerate(code):
        if not ins[0].startswith('global_load_lds'):
            continue
        found += 1
        address, states = regs(ins[2]), 0
        assert address
        for before in reversed(code[:at]):
            if before[0].startswith('s_mov') and regs(before[1]) == address:
                break  # scalar instructions are kept in order with both sides
            if before[0].startswith('v_') and regs(before[1]) & address:
                assert states >= 5, (before, ins, states)
                break
            states += 1 + (int(before[1]) if before[0] == 's_nop' else 0)
    assert found == 2
