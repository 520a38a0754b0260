"""The blocks of a nibble column that the digit kernel loads stay inside the
column: its workspace is sized exactly, and every step loads one step ahead."""
from __future__ import annotations

import subprocess

from conftest import PACKAGE_DIR

SOURCE = r"""
#include "onehot_blocks.hpp"
#include <cstdio>
int main() {
  for (unsigned blocks = 1; blocks <= 70; ++blocks) {
    const unsigned steps = (blocks + 1) / 2;
    for (unsigned s = 0; s <= steps; ++s)       // step `steps` is loaded ahead of the end
      for (unsigned h = 0; h < 2; ++h) {
        const unsigned at = ackvq::digit_block(s, h, blocks);
        if (at >= blocks || (2 * s + h < blocks && at != 2 * s + h)) {
          std::printf("blocks %u step %u half %u reads block %u\n", blocks, s, h, at);
          return 1;
        }
      }
  }
  return 0;
}
"""


def test_every_load_lies_in_its_column(tmp_path):
    source, program = tmp_path / "blocks.cpp", tmp_path / "blocks"
    source.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-Wall", f"-I{PACKAGE_DIR / 'csrc'}", str(source), "-o",
                    str(program)], check=True)
    done = subprocess.run([str(program)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
