"""Grids of the fills (csrc/launch.h), compiled for the host: every word of the
largest buffers is reached and the work-items of a launch fit in 32 bits."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "entropicthreadsafe_amd", "csrc")
PROGRAM = """
#include <cstdio>
#include <cstdlib>
namespace {
#include "launch.h"
}
int main(int n, char **a) {
  for (int i = 1; i < n; i++) printf("%u\\n", fill_blocks(atoll(a[i])));
}
"""
NODES = 2**31 - 1
# a word; around a block; a state buffer of 390 million nodes and the largest one in FP32 (with padding), normals
WORDS = [0, 1, 255, 256, 257, 2**32 - 256, 2**32 - 255, 2**32, 2**32 + 1, 11 * 390_500_000, 4 * NODES, 11 * NODES,
         16 * NODES]


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_fill_grids(tmp_path):
    src, exe = tmp_path / "p.cpp", tmp_path / "p"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I" + CSRC, "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)] + [str(w) for w in WORDS], check=True, capture_output=True, text=True).stdout
    for words, blocks in zip(WORDS, map(int, out.split())):
        assert 1 <= blocks and blocks * 256 < 2**32
        assert blocks * 256 >= words or blocks >= 1 << 16  # one word a thread, or enough threads to stride
