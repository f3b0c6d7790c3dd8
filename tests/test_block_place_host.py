"""The block matrix's ScaleAddI carries each thread's place in its block along
the grid's stride (block_place.h).  On the CPU, for block sizes up to the last
whose m*m fits 32 bits and the strides the kernel uses: the carried place is
the 64-bit remainder at every step, also where the sum of place and step would
leave 32 bits (m = 65280 .. 65535 at a stride of 2^25)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include "block_place.h"
template <typename U>
int walk(unsigned long m, unsigned long stride)
{
  const unsigned long mm = m * m;
  const unsigned long firsts[] = {0, 2, 510, m, mm - 1, mm / 2, stride - 2};
  for (unsigned long first : firsts)
  {
    U at = (U)(first % mm);
    for (unsigned long k = 0; k < 600; k++)
    {
      if (at != (first + k * stride) % mm)
      {
        std::printf("m %lu stride %lu first %lu step %lu\n", m, stride, first, k);
        return 1;
      }
      at = block_place_after<U>(at, (U)(stride % mm), (U)mm);
    }
  }
  return 0;
}
int main()
{
  const unsigned long ms[] = {1,     2,     3,     21,    32,    64,    32767, 32768,
                              46340, 46341, 65279, 65280, 65281, 65500, 65534, 65535};
  const unsigned long strides[] = {512, 3 * 512, 2UL * 65536 * 256};
  int bad = 0;
  for (unsigned long m : ms)
  {
    for (unsigned long s : strides) { bad += walk<unsigned>(m, s) + walk<unsigned long>(m, s); }
  }
  return bad != 0;
}
"""


def test_carried_place_is_the_remainder(tmp_path):
    cc = shutil.which("g++") or shutil.which("c++")
    if cc is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "place.cpp", tmp_path / "place"
    src.write_text(SRC)
    subprocess.run([cc, "-std=c++17", "-I" + os.path.join(ROOT, "sundials_amd", "csrc", "sunmatrix"),
                    str(src), "-o", str(exe)], check=True, capture_output=True, text=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
