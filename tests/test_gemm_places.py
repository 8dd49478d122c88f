"""Where the dequantising tiles load (csrc/kernels/gemm_dq_places.h), on the host: every step that they ask for, those past a slice's
last one too, lies inside the operand, and the steps of the slice cover the row's stream in order."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "gemm_dq_places.h"
#include <cstdio>
#include <initializer_list>
using namespace omx;
#define CHECK(c) do { if (!(c)) { std::printf("%s: SB %d rows %d slice %d step %d\n", #c, SB, rows, z, s); return 1; } } while (0)
int main() {
  const int AHEAD = 8;  // steps past the end; the tiles ask for four
  for (int SB = 1; SB <= 9; ++SB)
    for (int rows : {1, 2, 128})
      for (int sk = 1; sk <= 3 && sk <= SB; ++sk)
        for (int z = 0; z < sk; ++z) {
          const int ks0 = 4 * (z * SB / sk), ks1 = 4 * ((z + 1) * SB / sk), kl = ks1 - 1, r = rows - 1;
          const unsigned Kp = 256u * SB;
          for (int s = ks0; s < ks1 + AHEAD; ++s) {
            for (unsigned xc = 0; xc < 8; ++xc) {
              const unsigned at = ds_x_at(r, Kp, xc) + ds_x_step(s, kl);
              CHECK(at + 16 <= 2u * rows * Kp);
              if (s < ks1) CHECK(at == 2u * (r * Kp + 64u * s + 8u * xc));
            }
            for (unsigned fq = 0; fq < 2; ++fq) {
              for (unsigned block : {32u, 64u, 128u, 256u}) {  // high bits (Q5_K, Q6_K), 4-bit codes, Q8_0 codes
                const unsigned at = ds_w_at(r * SB, block, fq) + ds_w_step(s, kl, block);
                CHECK(at + block / 8 <= (unsigned)rows * SB * block);
                if (s < ks1) CHECK(at == r * SB * block + (2u * s + fq) * (block / 8));
              }
              const unsigned pc = 2u * s + fq, lt = pc / SB, sb = pc - lt * SB;
              const unsigned at = ds_scale_at(r * SB + sb, lt);
              CHECK(at + 2 <= 16u * rows * SB);
              if (s < ks1) CHECK(at == 16u * (r * SB + sb) + 2u * lt);
            }
          }
        }
  return 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="needs g++")
def test_loads_stay_inside_their_operands(tmp_path):
    src, exe = tmp_path / "places.cpp", tmp_path / "places"
    src.write_text(PROGRAM)
    kernels = os.path.join(ROOT, "csrc", "kernels")
    subprocess.run(["g++", "-std=c++17", "-I", kernels, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
