"""Index rules of the CSF kernels (csrc/csf_index.hpp), compiled for the host.

The up kernel takes whole tiles of x1 rows, past the last virtual of a vector
too: no position it reads may lie behind the vector's end, at every occupied
count it takes (2..32) and virtual counts through several tiles; the rows that
exist are read from their own position."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "adc_ottawa_amd", "csrc")

SOURCE = r"""
#include <cstdio>
#include "csf_index.hpp"
using namespace adc2g;
int main() {
  for (int o = 2; o <= 32; ++o)
    for (int v = 2; v <= 40; ++v) {
      const long n1 = (long)o * v, po = o * (o - 1) / 2, pv = v * (v - 1) / 2;
      const long ndim = 2 * n1 + pv * o + po * v + 2 * po * pv;
      for (int c0 = 0; c0 < v; c0 += CSF_UP_ROWS)
        for (int g = 0; g < 4; ++g)
          for (int s = 0; s < 2; ++s)
            for (int k = 0; k < o; ++k) {
              const int c = c0 + 4 * s + g;
              const long at = (long)(c0 + csf_up_first(g, v) + s * csf_up_half(v)) * o + k;
              if (at < 0 || at >= ndim || (c < v && at != (long)c * o + k)) {
                std::printf("o=%d v=%d c=%d k=%d reads %ld of %ld\n", o, v, c, k, at, ndim);
                return 1;
              }
            }
    }
  return 0;
}
"""


def test_up_rows_within_the_vector(tmp_path):
    src, exe = tmp_path / "rows.cpp", tmp_path / "rows"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
