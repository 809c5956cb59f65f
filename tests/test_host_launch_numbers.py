"""Launch numbers (csrc/launch_number.h) against what a recycled workspace may hold: no word of ordinary data carries one,
two processes do not share them, and none comes twice."""
import os
import subprocess

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include "launch_number.h"
int main() { for (int i = 0; i < 20000; ++i) std::printf("%llu\n", (unsigned long long)msgl::next_launch_number()); }
"""


def test_numbers_are_unlike_data(tmp_path):
    src, exe = tmp_path / "numbers.cpp", tmp_path / "numbers"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "mini-sglang-mlx_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    first, second = (np.array(subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split(), dtype=np.uint64)
                     for _ in range(2))
    assert np.unique(first).size == first.size and first.max() < 2 ** 48  # a count of 16 bits goes below
    # a process that starts where another did would meet its numbers in the same order: two seeds of 36 bits
    assert first[0] != second[0]
    for count in (0, 1, 0xffff):
        words = (first << np.uint64(16)) | np.uint64(count)
        assert (words > 2 ** 62).all() and (words < 2 ** 63).all()            # token ids, positions, offsets, masks; -1
        assert not np.isfinite(words.view(np.float64)).any()
        high = (words >> np.uint64(32)).astype(np.uint32)
        assert np.isnan(high.view(np.float32)).all()                           # pairs of fp32
        top = (words >> np.uint64(48)).astype(np.uint16)
        assert np.isnan(top.view(np.float16)).all()                            # half
        assert np.isnan((top.astype(np.uint32) << np.uint32(16)).view(np.float32)).all()  # bf16
