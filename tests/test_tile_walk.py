"""The deal of a product's tiles to the XCDs (csrc/kernels.h: xcd_walk), compiled for the host: every tile has a slot, and
an uneven deal never takes a round of workgroups more than the even one."""

import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "distributed-xfold_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include <cstdio>
#include "kernels.h"
int main() {
  long bad = 0, uneven = 0;
  for (int bm : {32, 64, 128, 192, 256})
    for (int bn : {64, 128, 192, 256})
      for (int per_round : {32, 64, 96, 128})
        for (long tm = 1; tm <= 130; ++tm)
          for (long tn = 1; tn <= 80; ++tn) {
            const XcdWalk w = xcd_walk(tm, tn, 1, bm, bn, per_round);
            const long even = (tm * tn + 7) / 8;
            long most = even;
            if (w.rows) {
              most = 0;
              long all = 0;
              for (int xcd = 0; xcd < 8; ++xcd) {
                const long r = w.rows, c = 8 / r, i = xcd & (r - 1), j = xcd / r;
                const long tiles = (tm * (i + 1) / r - tm * i / r) * (tn * (j + 1) / c - tn * j / c);
                all += tiles;
                if (tiles > most) most = tiles;
              }
              if (all != tm * tn) ++bad;
              uneven += most > even;
            }
            if (most > w.slots || (most + per_round - 1) / per_round > (even + per_round - 1) / per_round) ++bad;
          }
  std::printf("bad %ld uneven %ld\n", bad, uneven);
}
"""


def test_no_deal_takes_a_round_more_than_the_even_one(tmp_path):
    if not shutil.which(HIPCC):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "walk.hip", tmp_path / "walk"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "-std=c++17", "-O1", "--offload-arch=gfx950", "-Wno-everything", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    assert int(out[1]) == 0 and int(out[3]) > 0, out
