"""The coefficient rows of the many-density synthesis (napmo_amd/csrc/synth_rows.hpp), walked on the
CPU for every lmax as the kernel walks them: two or four loads ahead of the first step, then whole
groups of two or four steps, each with one load. The steps read the rows of their harmonics, and no
load, those past the last step included, goes beyond the last row."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

WALK = r'''
#include <cstdio>
#include "synth_rows.hpp"
int main() {
  for (int lmax = 0; lmax <= 24; ++lmax)
    for (int depth = 2; depth <= 4; depth += 2)
      for (int ndp = 16; ndp <= 48; ndp += 16)
        for (int qbytes = 8 * ndp; qbytes <= 32 * ndp; qbytes += 24 * ndp) {
          const int L = (lmax + 1) * (lmax + 1), steps = (lmax + 1) * (lmax + 2) / 2, last = (L - 1) * qbytes;
          const int loads = depth + (steps + depth - 1) / depth * depth;
          napmo::SynthRows s;
          for (int k = 0; k < loads; ++k) {
            std::printf("%d %d %d %d %d %d %d %d\n", lmax, qbytes, k, steps, s.cos_row(last), s.sin_row(qbytes, last), s.l, s.m);
            s.next(lmax, qbytes);
          }
        }
}
'''


@pytest.mark.skipif(shutil.which('g++') is None, reason='g++ is absent')
def test_no_load_leaves_the_table(tmp_path):
    src, exe = tmp_path / 'walk.cpp', str(tmp_path / 'walk')
    src.write_text(WALK)
    subprocess.run(['g++', '-std=c++17', '-I' + os.path.join(ROOT, 'napmo_amd', 'csrc'), str(src), '-o', exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    count = 0
    for line in out.splitlines():
        lmax, qbytes, k, steps, cos, sin, l, m = map(int, line.split())
        last = (lmax + 1) ** 2 - 1
        assert 0 <= cos <= last * qbytes and 0 <= sin <= last * qbytes, line
        if k >= steps:
            continue
        # harmonics of m = 0 first, then (cos, sin) pairs of each m; l runs inside m
        lm = [(a, b) for b in range(lmax + 1) for a in range(b, lmax + 1)]
        q = k if m == 0 else lmax + 1 + 2 * (k - lmax - 1)
        assert (l, m) == lm[k] and cos == q * qbytes, line
        assert m == 0 or sin == (q + 1) * qbytes, line
        count += 1
    assert count > 0
