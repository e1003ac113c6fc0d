"""Bit positions of the many-lanes lossless-JPEG decode (lj92_pos.h) on the
CPU: a scan that runs on past its data, as a truncated one does, never comes
back into it, over more bits than 32-bit positions count."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "lj92_pos.h"
#include <stdio.h>
int main(void)
{
  const uint32_t bits[] = { 0, 8, 1000, (1u << 31) - 8 };
  for(int k = 0; k < 4; k++)
  {
    uint32_t pos = bits[k] > 100 ? bits[k] - 100 : 0;
    uint64_t exact = pos;
    for(long s = 0; s < 150000000L; s++)      // 31 bits a sample: past 2^32
    {
      const uint32_t n = 1 + (uint32_t)(s % 31 ? 30 : s & 15);
      pos = lj92_next(pos, n, bits[k]);
      exact += n;
      if(exact <= bits[k] + 64ull ? pos != exact : pos < bits[k] + 32) { printf("%u: sample %ld at %u\n", bits[k], s, pos); return 1; }
    }
  }
  return 0;
}
"""


def test_positions_past_the_data(tmp_path):
    (tmp_path / "pos.c").write_text(SRC)
    exe = str(tmp_path / "pos")
    try:
        subprocess.run(["gcc", "-O2", "-I" + os.path.join(ROOT, "vkdt_amd", "csrc"), "-o", exe, str(tmp_path / "pos.c")], check=True,
                       capture_output=True)
    except (OSError, subprocess.CalledProcessError) as e:
        pytest.skip(f"no C compiler: {e}")
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
