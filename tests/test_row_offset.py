"""Offsets of rows that go to LDS directly (csrc/row_offset.h), on the CPU: rows beyond the last stay outside of the window at the largest pitches
that mpa_linear_run accepts, where a tile's rows times the pitch are more than 32 bits."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mamba.py_amd", "csrc")
PROGRAM = r"""
#include <stdio.h>
#include "row_offset.h"
int main() {
    unsigned long long row, rows, pitch, k, element;
    while (scanf("%llu %llu %llu %llu %llu", &row, &rows, &pitch, &k, &element) == 5)
        for (int tile = 32; tile <= 128; tile *= 2) {  // (the largest tile's are the last)
            const uint32_t at = (uint32_t)((row * pitch + k) * element);
            if (row / tile * tile < rows) printf("%u ", mpa::rows_wrap(rows, tile, pitch, element) ? mpa::row_offset((int)row, (int)rows, at) : at);
            else printf("%u ", mpa::kNoRow);  // (no workgroup)
        }
}
"""


def test_rows_beyond_the_last_are_outside_of_the_window(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "offsets.cpp", tmp_path / "offsets"
    src.write_text(PROGRAM)
    subprocess.run([gxx, "-O1", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    cases = []
    # (rows, K, pitch): rows * pitch below 2^29 elements
    for rows, K, pitch in [(1, 8, (1 << 29) - 8), (2, 8, 1 << 27), (2, 64, (1 << 28) - 8), (4, (1 << 24) - 8, (1 << 24) - 8), (31, 1 << 24, (1 << 24) + 8),
                           (3, 264, 89478480), (100, 768, 768), (129, 8, 4161792)]:
        for element in (2, 4):
            for t0 in sorted({0, (rows - 1) // 64 * 64}):
                for row in range(t0, t0 + 128):
                    for k in {0, K - 16 // element}:
                        cases.append((row, rows, pitch, k, element, K))
    out = subprocess.run([str(exe)], input="".join("%d %d %d %d %d\n" % c[:5] for c in cases), capture_output=True, text=True, check=True).stdout.split()
    assert len(out) == 3 * len(cases)
    wrapped = 0
    for (row, rows, pitch, k, element, K), got in zip((c for c in cases for _ in range(3)), map(int, out)):
        window = ((rows - 1) * pitch + K) * element
        assert window < 1 << 31
        if row < rows:
            assert got == (row * pitch + k) * element and got + 16 <= window
        else:
            assert got >= window
            wrapped += (row * pitch + k) * element % (1 << 32) < window
    assert wrapped > 0  # (offsets that grow by the pitch are within the window there)
