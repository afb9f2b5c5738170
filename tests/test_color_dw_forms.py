"""The tiles that the waves of the colour network's weight-gradient kernel multiply, and their cost
(csrc/color_dw.h), for every number of row and column tiles: all tiles of the product are covered, no wave
multiplies a column more than the widest share, and the cost that cuts the ranges is that of these tiles."""
import shutil
import subprocess
from pathlib import Path

import pytest

from srf_hip import build

SOURCE = r"""
#include <cstdio>
#include "color_dw.h"
using namespace srf::color;
template <bool SPLIT>
void table() {
  for (int a = 1; a <= kCdwMaxA; ++a)
    for (int b = 1; b <= kCdwMaxB; ++b) {
      const CdwForm f = cdw_form<SPLIT>(a, b);
      std::printf("%d %d %d %d %d %d\n", SPLIT, a, b, f.rows, f.cols, cdw_cost<SPLIT>(a, b));
    }
}
int main() { table<false>(); table<true>(); }
"""


def test_forms_and_costs(tmp_path):
    if not (shutil.which('hipcc') or Path('/opt/rocm/bin/hipcc').exists()):
        pytest.skip('no hipcc')
    src, exe = tmp_path / 'forms.hip', tmp_path / 'forms'
    src.write_text(SOURCE)
    subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, f'-I{build.CSRC_DIR}', '-w', str(src), '-o', str(exe)],
                   check=True, capture_output=True, text=True)
    lines = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split('\n')[:-1]
    assert len(lines) == 2 * 8 * 16
    for line in lines:
        split, a, b, rows, cols, cost = map(int, line.split())
        tile = 2 if split else 1                       # 16-row tiles of a wave's tile
        need_cols = -(-b // tile)
        if a <= 2:                                     # eight waves across the columns
            assert rows * tile >= a and cols == -(-need_cols // 8), line
        else:                                          # four across the rows, two across the columns
            assert rows * tile * 4 >= a and cols == -(-need_cols // 2), line
        # MFMAs of 16 points: FP32 four of 32 cycles a tile, split three of 16 passes (64 cycles) and the
        # planes' work, 256 cycles in all; two waves share a SIMD
        mfma = 2 * (256 if split else 128) * rows * cols
        reads = (90 if split else 60) * (a + b)
        assert cost == max(mfma, reads) + 200, line
